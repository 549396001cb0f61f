"""bench.py pieces that need no GPU: the refusal of more than one GPU, the workload table (FLOP
counts of the five configurations against figures worked out by hand from their layer shapes), and
the CPU-baseline leg on a tiny sample."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT


def test_more_than_one_gpu_is_refused_with_a_message():
    res = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                         text=True, timeout=120)
    assert res.returncode != 0 and "ONE GPU" in res.stderr and res.stdout.strip() == ""


def test_workload_flops_match_the_configurations():
    sys.path.insert(0, ROOT)
    import bench
    want = {"vgg16": 982.18e9, "resnet50": 523.15e9, "unet": 1745.1e9, "block": 14.797e9, "conv": 14155776.0}
    for name, (kwargs, seed, dist, desc) in bench.WORKLOADS.items():
        m = bench.builder_of(name)(**kwargs)
        flops = 0
        for l in m.layers:
            if l.kind == "conv2d":
                cd = l.attrs["cd"]
                N, Kf, P, Q = cd.out_shape
                flops += 2 * N * Kf * cd.kz * cd.kr * cd.kc * P * Q
        assert abs(flops - want[name]) / want[name] < 2e-3, (name, flops)


def test_every_plan_number_has_a_form_and_the_split_form_a_peak_of_its_own(tmp_path):
    """The benchmark names every plan that the library's loader accepts and no other, and prices the split form by the bf16 instruction."""
    sys.path.insert(0, ROOT)
    import bench
    from eddl_amd import _lib
    lib = _lib.load()
    path = tmp_path / "plans.txt"
    for tile in range(-2, 30):
        path.write_text("4 128 64 1 1 1 1 28 28 1 | %d 1\n" % tile)
        if lib.eddlhip_conv2d_tuned_load(0, str(path).encode()) == 0:
            assert (bench.form_of_plan(tile) == "split") == (tile >= 16)
            assert (bench.form_of_plan(tile) == "upsampled_2x2") == (tile in (8, 9))
        else:
            with pytest.raises(ValueError):
                bench.form_of_plan(tile)
    lib.eddlhip_conv2d_autotune(-1)
    assert bench.peak_of_form("direct") == bench.peak_of_form("winograd") == 157.3
    assert bench.peak_of_form("split") == pytest.approx(16 * 157.3 / 6)


def test_cpu_baseline_leg_runs_on_a_small_sample(monkeypatch):
    sys.path.insert(0, ROOT)
    import bench
    monkeypatch.setitem(bench.WORKLOADS, "block", ({"batch": 2, "channels": 4, "size": 8, "filters": 4}, 2, "normal", "tiny block"))
    out = bench.cpu_baseline("block", want_seconds=0.2)
    assert out["kind"] == "port" and out["unit"] == "images/sec" and out["cores"] >= 1
    assert out["value"] > 0 and out["value_strict"] > 0 and "sample" in out
    json.dumps(out)


def test_cpu_baseline_leg_checks_a_device_output_against_the_oracle(monkeypatch):
    """The parity gate of the benchmark: an output equal to the oracle's passes, one that is off by 1e-3 of the
    output scale does not; a larger batch than the sample is compared on its first images."""
    sys.path.insert(0, ROOT)
    import bench
    from eddl_amd import models
    from oracle import net_oracle
    from oracle.oracle import Oracle
    kwargs = {"batch": 2, "channels": 4, "size": 8, "filters": 4}
    monkeypatch.setitem(bench.WORKLOADS, "block", (kwargs, 2, "normal", "tiny block"))
    monkeypatch.setattr(os, "cpu_count", lambda: 1)   # a sample of one image out of the batch of two
    monkeypatch.setattr(os, "sched_getaffinity", lambda pid: {0}, raising=False)
    model = models.conv_bn_relu_pool_block(**kwargs)
    models.init_he_normal(model, 2)
    x = models.synthetic_input(model.lin[0].out_shape, 1002, "normal")   # the benchmark's own input: seed + 1000
    full = net_oracle.forward(Oracle(hpc=False), model, [x])[0]
    good = bench.cpu_baseline("block", want_seconds=0.1, device_output=full)["parity"]
    assert good["ok"] and good["images"] == 1 and good["max_abs_err"] == 0.0
    bad = bench.cpu_baseline("block", want_seconds=0.1, device_output=full + 1e-3 * np.abs(full).max())["parity"]
    assert not bad["ok"] and bad["err_over_max_ref"] > bench.PARITY_BOUND


def test_matrix_counter_table_counts_the_split_kernel_in_bf16_products(tmp_path):
    """The counter summary has a row for every kind of matrix kernel, the split one from the bf16 counter and at that peak."""
    from eddl_amd import profsum
    names = ["void (anonymous namespace)::%s(ConvParams)" % k for k in ("conv_split_kernel<4, 1, 1, 2, 3>", "conv_tap_kernel<2, 2, 1, 1, 1, 1, 16, true>")]
    with open(tmp_path / "m_counter_collection.csv", "w") as fh:
        fh.write("Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value\n")
        for i, k in enumerate(names):
            for counter, value in (("SQ_INSTS_VALU_MFMA_MOPS_F32", 2e6 * i), ("SQ_INSTS_VALU_MFMA_MOPS_BF16", 2e7 * (1 - i)),
                                   ("SQ_VALU_MFMA_BUSY_CYCLES", 1024e4), ("GRBM_GUI_ACTIVE", 16e4)):
                fh.write('%d,"%s",%s,%f\n' % (i, k, counter, value))
    with open(tmp_path / "m_kernel_trace.csv", "w") as fh:
        fh.write("Kernel_Name,Start_Timestamp,End_Timestamp\n")
        for k in names:
            fh.write('"%s",1000,11000\n' % k)
    profsum.mfma("resnet50", str(tmp_path), str(tmp_path / "out.txt"))
    rows = {l.split("<")[0]: l.split("(ConvParams)")[1].split() for l in open(tmp_path / "out.txt") if "(ConvParams)" in l}
    assert set(rows) == {"conv_split_kernel", "conv_tap_kernel"}
    for name, ops, peak in (("conv_split_kernel", 2e7, 16 * 157.3), ("conv_tap_kernel", 2e6, 157.3)):
        rate = ops * 512 / 10e-6 / 1e12        # TFLOP/s of a 10 us dispatch
        assert float(rows[name][3]) == round(rate, 1) and float(rows[name][4]) == round(100 * rate / peak, 1)


def test_stall_table_and_trace_find_the_split_kernels_under_the_traces_names(tmp_path):
    """Every convolution kernel has its row of stall counters, and the benchmark's dominant kernel is found in a trace that writes enumerators as numbers."""
    import json
    import os
    import re
    from eddl_amd import profsum
    split = "conv_split_kernel<4, 1, 1, 2, 3, ((anonymous namespace)::SplitTaps)2>"
    names = ["void (anonymous namespace)::%s((anonymous namespace)::ConvParams)" % k for k in
             (split, "wino_split_kernel<true>", "wino_fused_kernel<2, 1, 4, 3, true>", "conv_up2x2_split_kernel<4, 1>", "softmax_kernel")]
    for d, counters in (("sq", profsum.STALL_SQ), ("tcp", profsum.STALL_TCP)):
        os.makedirs(str(tmp_path / d))
        with open(tmp_path / d / "m_counter_collection.csv", "w") as fh:
            fh.write("Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value\n")
            for i, k in enumerate(names):
                for c in counters.split():
                    fh.write('%d,"%s",%s,1000\n' % (i, k, c))
        with open(tmp_path / d / "m_kernel_trace.csv", "w") as fh:
            fh.write("Kernel_Name,Start_Timestamp,End_Timestamp\n")
            for k in names:
                fh.write('"%s",1000,11000\n' % k)
    profsum.stalls("vgg16", str(tmp_path / "sq"), str(tmp_path / "tcp"), str(tmp_path / "stalls.txt"))
    text = open(tmp_path / "stalls.txt").read()
    assert all(re.search("^%s<" % k, text, re.M) for k in ("conv_split_kernel", "wino_split_kernel", "wino_fused_kernel", "conv_up2x2_split_kernel"))
    assert not re.search("^softmax", text, re.M)

    with open(tmp_path / "t_kernel_stats.csv", "w") as fh:
        fh.write("Name,Calls,TotalDurationNs,AverageNs,Percentage\n")
        for i, k in enumerate(names):
            fh.write('"%s",%d,1000,%d000,10\n' % (k, i + 1, i + 1))
    for kernel, found in (("conv_split_kernel<4,1,1,2,3,ONE_TAP>", "average 0.0010 ms over 1 calls"), ("wino_split_kernel<true>", "average 0.0020 ms over 2 calls"),
                          ("wino_fused_kernel<2,1,4,3,true>", "average 0.0030 ms over 3 calls"), ("conv_split_kernel<4,1,1,2,3,STORED>", "NOT FOUND")):
        (tmp_path / "bench.log").write_text(json.dumps({"metric": "x", "value": 1.0, "unit": "u", "ms_per_step": 1.0,
                                                        "roofline": {"kernel": kernel, "achieved": 1.0, "unit": "TFLOP/s", "frac": 0.1, "peak": 10.0}}) + "\n")
        profsum.trace("vgg16", str(tmp_path), str(tmp_path / "bench.log"), str(tmp_path / "trace.txt"))
        assert "same kernel in the trace above: %s" % found in open(tmp_path / "trace.txt").read()


def test_traffic_table_has_a_row_for_each_build_of_the_split_kernel(tmp_path):
    import json
    import os
    from eddl_amd import profsum
    names = ["void (anonymous namespace)::conv_split_kernel<4, 1, 1, 2, 3, ((anonymous namespace)::SplitTaps)%d>((anonymous namespace)::ConvParams)" % i for i in range(3)]
    probe = "void (anonymous namespace)::unary_kernel<0>(float const*, float*, unsigned long)"
    for d, c in (("f", "FETCH_SIZE"), ("w", "WRITE_SIZE")):
        os.makedirs(str(tmp_path / d))
        with open(tmp_path / d / "m_counter_collection.csv", "w") as fh:
            fh.write("Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value\n")
            for i, k in enumerate(names + [probe]):
                fh.write('%d,"%s",%s,%f\n' % (i, k, c, 262144.0 if k == probe else 1000.0 * (i + 1)))
    with open(tmp_path / "t_kernel_stats.csv", "w") as fh:
        fh.write("Name,Calls,TotalDurationNs,AverageNs,Percentage\n")
        for k in names + [probe]:
            fh.write('"%s",1,1000,1000,10\n' % k)
    (tmp_path / "bench.log").write_text(json.dumps({"metric": "x", "value": 1.0, "unit": "u", "ms_per_step": 1.0, "roofline": {
        "kernel": "conv_split_kernel<4,1,1,2,3,ONE_TAP>", "launches_per_step": 1, "achieved": 1.0, "unit": "TFLOP/s", "frac": 0.1, "peak": 10.0}}) + "\n")
    profsum.traffic("resnet50", str(tmp_path), str(tmp_path / "f"), str(tmp_path / "w"), str(tmp_path / "bench.log"), str(tmp_path / "o.txt"), str(tmp_path / "o.json"))
    table = json.load(open(tmp_path / "o.json"))
    assert [table["kernels"]["conv_split_kernel<4,1,1,2,3,%s>" % t]["fetch_bytes_per_launch"] for t in ("UPSAMPLED", "STORED", "ONE_TAP")] == [1024e3, 2048e3, 3072e3]
    assert table["steps_in_counter_run"] == 1.0


def test_a_form_has_one_name_and_its_peak():
    import bench
    for tile in (16, 19, 32, 33, 34):
        assert bench.peak_of_form(bench.form_of_plan(tile)) == pytest.approx(16 * 157.3 / 6)
    for tile in (-1, 0, 3, 4, 5, 6, 7, 8, 9):
        assert bench.peak_of_form(bench.form_of_plan(tile)) == 157.3
    assert bench.peak_of_form(None) == 157.3
