"""eddlhip_conv2d_fwd_noalloc, the convolution entry point that allocates nothing, against
eddlhip_conv2d_fwd on the same inputs: same kernels, same launch plan, so the outputs are compared
bit for bit.  Every case makes two calls in a row, the second on a smaller input, because every call on
a device shares that device's one scratch array, which keeps the previous call's contents.

Called through the C ABI (ctypes), device memory from eddlhip_malloc.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCRATCH_BYTES = 64 << 20  # EDDLHIP_CONV_NOALLOC_SCRATCH_BYTES of include/eddlhip.h


def _out_dim(size, k, stride, pad_lo, pad_hi):
    return (size + pad_lo + pad_hi - k) // stride + 1


def _both(hip, rng, N, C, H, W, Kf, R, S, stride, pad, epilogue):
    """Runs eddlhip_conv2d_fwd and eddlhip_conv2d_fwd_noalloc on one seeded case; returns both outputs and
    the kernel each call reported."""
    x = rng.standard_normal((N, C, H, W), dtype=np.float32)
    w = (rng.standard_normal((Kf, C, R, S)) * np.sqrt(2.0 / (C * R * S))).astype(np.float32)
    P, Q = _out_dim(H, R, stride, pad, pad), _out_dim(W, S, stride, pad, pad)
    dx, dw = hip.array(x), hip.array(w)
    bias = g = b = mean = var = res = None
    if epilogue:
        bias = hip.array(rng.standard_normal(Kf).astype(np.float32))
        g = hip.array(rng.uniform(0.8, 1.2, Kf).astype(np.float32))
        b = hip.array((rng.standard_normal(Kf) * 0.1).astype(np.float32))
        mean = hip.array((rng.standard_normal(Kf) * 0.1).astype(np.float32))
        var = hip.array(rng.uniform(0.5, 1.5, Kf).astype(np.float32))
        res = hip.array(rng.standard_normal((N, Kf, P, Q), dtype=np.float32))
    ptr = lambda t: None if t is None else t.ptr
    outs, kernels = [], []
    for fn in (hip.lib.eddlhip_conv2d_fwd, hip.lib.eddlhip_conv2d_fwd_noalloc):
        O = hip.full((N, Kf, P, Q), float("nan"))
        hip._check(fn(hip.dev, dx.ptr, dw.ptr, ptr(bias), O.ptr, N, C, H, W, Kf, R, S, stride, stride, pad, pad, P, Q,
                      ptr(g), ptr(b), ptr(mean), ptr(var), 1e-5, ptr(res), int(epilogue)))
        kernels.append(hip.last_conv_kernel())
        outs.append(O.numpy())
    return outs, kernels


# (first call, second smaller call): N, C, H, W, Kf, R, S, stride, pad
CASES = {
    # 3x3, 128x128 tiles; 28x28x512 at batch 32 leaves tiles over that are divided along K: repacked filters + partial tiles
    "3x3_ksplit": ((32, 256, 28, 28, 512, 3, 3, 1, 1), (3, 64, 14, 14, 96, 3, 3, 1, 1)),
    # 7x7 stride 2 (the 16-tap kernel): repacked filters + tap table; then a 5x5
    "7x7_taptable": ((8, 3, 112, 112, 64, 7, 7, 2, 3), (2, 5, 30, 30, 40, 5, 5, 1, 2)),
    # 1x1 short K with the whole fused tail, then a 2x2
    "1x1_epilogue": ((16, 64, 56, 56, 256, 1, 1, 1, 0), (4, 32, 17, 17, 48, 2, 2, 1, 0)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_noalloc_equals_conv2d_fwd_two_calls_in_a_row(hip, name):
    rng = np.random.default_rng(71)
    saw_split = False
    for shape in CASES[name]:
        N, C, H, W, Kf, R, S, stride, pad = shape
        (ref, got), (k_ref, k_got) = _both(hip, rng, N, C, H, W, Kf, R, S, stride, pad, epilogue=(name == "1x1_epilogue"))
        assert k_ref == k_got, "the two entry points planned different launches: %s vs %s" % (k_ref, k_got)
        assert np.all(np.isfinite(got)), "%s %s: the output holds values that were never written" % (name, shape)
        assert np.array_equal(ref, got), "%s %s (%s): %d values differ" % (name, shape, k_got, int((ref != got).sum()))
        saw_split = saw_split or "+ksplit" in k_got
    if name == "3x3_ksplit":
        assert saw_split, "this case is meant to cover the partial tiles of a K-split launch"


def test_noalloc_leaves_the_workspace_alone(hip):
    """The property the entry point exists for: with the library's workspace released beforehand, a call larger than any
    before it (repacked filters and the partial tiles of a K-split launch come from the fixed array) leaves the workspace
    at zero bytes - nothing was allocated - and the allocating entry point, called afterwards, gives the same bits."""
    rng = np.random.default_rng(73)
    N, C, H, W, Kf = 32, 320, 28, 28, 512
    x = rng.standard_normal((N, C, H, W), dtype=np.float32)
    w = (rng.standard_normal((Kf, C, 3, 3)) * 0.03).astype(np.float32)
    dx, dw = hip.array(x), hip.array(w)
    O1, O2 = hip.full((N, Kf, H, W), float("nan")), hip.full((N, Kf, H, W), float("nan"))
    hip.synchronize()
    hip.workspace_trim()
    assert hip.workspace_bytes() == 0
    args = lambda O: (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 3, 3, 1, 1, 1, 1, H, W, None, None, None, None, 0.0, None, 0)
    hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))
    kernel = hip.last_conv_kernel()
    assert hip.workspace_bytes() == 0, "eddlhip_conv2d_fwd_noalloc took a workspace"
    assert "+ksplit" in kernel, kernel
    hip._check(hip.lib.eddlhip_conv2d_fwd(*args(O2)))
    assert hip.last_conv_kernel() == kernel and hip.workspace_bytes() > 0
    assert np.array_equal(O1.numpy(), O2.numpy())


def test_noalloc_uses_registered_filters(hip):
    """With the filters registered the call needs no room for a repacked copy; the result is unchanged."""
    rng = np.random.default_rng(72)
    N, C, H, W, Kf = 4, 64, 28, 28, 128
    x = rng.standard_normal((N, C, H, W), dtype=np.float32)
    w = (rng.standard_normal((Kf, C, 3, 3)) * 0.05).astype(np.float32)
    dx, dw = hip.array(x), hip.array(w)
    outs = []
    for cached in (False, True):
        if cached:
            hip.cache_conv_filters(dw)
        O = hip.full((N, Kf, H, W), float("nan"))
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 3, 3, 1, 1, 1, 1, H, W,
                                                      None, None, None, None, 0.0, None, 0))
        outs.append(O.numpy())
    hip.uncache_conv_filters(dw)
    assert np.array_equal(outs[0], outs[1])


def test_noalloc_refuses_what_does_not_fit(hip):
    """A filter tensor whose repacked copy is larger than the scratch array: EDDLHIP_EINVAL with the figures, nothing
    launched, nothing written; the allocating entry point takes the same call."""
    Kf, C = 2048, 1024  # 3x3: 9216 taps x 2048 channels x 4 bytes = 75 MB
    assert 9 * C * Kf * 4 > SCRATCH_BYTES
    N, H, W = 1, 8, 8
    dx, dw = hip.full((N, C, H, W), 1.0), hip.full((Kf, C, 3, 3), 0.5)
    O = hip.full((N, Kf, H, W), -7.0)
    args = (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 3, 3, 1, 1, 1, 1, H, W, None, None, None, None, 0.0, None, 0)
    rc = hip.lib.eddlhip_conv2d_fwd_noalloc(*args)
    assert rc == -1
    text = hip.lib.eddlhip_last_error().decode()
    assert "scratch" in text and str(SCRATCH_BYTES) in text, text
    hip.synchronize()
    assert np.all(O.numpy() == -7.0)
    hip._check(hip.lib.eddlhip_conv2d_fwd(*args))
    out = O.numpy()
    assert out[0, 0, 4, 4] == np.float32(9 * C * 0.5) and out[0, 0, 0, 0] == np.float32(4 * C * 0.5)


def test_noalloc_refused_while_profiling(hip):
    dx, dw, O = hip.full((1, 8, 8, 8), 1.0), hip.full((8, 8, 3, 3), 1.0), hip.empty((1, 8, 8, 8))
    hip.conv_profile(True)
    try:
        rc = hip.lib.eddlhip_conv2d_fwd_noalloc(hip.dev, dx.ptr, dw.ptr, None, O.ptr, 1, 8, 8, 8, 8, 3, 3, 1, 1, 1, 1, 8, 8,
                                                None, None, None, None, 0.0, None, 0)
    finally:
        hip.conv_profile(False)
    assert rc == -1 and "profile" in hip.lib.eddlhip_last_error().decode()


# (N, C, H, W, Kf, R, stride, pad), plan tile and K slices: the split form kept for a geometry
SPLIT_PLANS = {"1x1": ((4, 96, 15, 17, 200, 1, 1, 0), 17, 4), "3x3 stride 2": ((3, 64, 28, 28, 128, 3, 2, 1), 19, 1), "3x3": ((2, 128, 13, 11, 72, 3, 1, 1), 18, 6)}


@pytest.mark.parametrize("registered", [False, True])
@pytest.mark.parametrize("name", sorted(SPLIT_PLANS))
def test_noalloc_runs_the_split_plan_that_was_found(hip, tmp_path, name, registered):
    """A plan of the split form is used like any found plan: same kernel and bits as conv2d_fwd, nothing allocated."""
    (N, C, H, W, Kf, R, stride, pad), tile, slices = SPLIT_PLANS[name]
    P, Q = _out_dim(H, R, stride, pad, pad), _out_dim(W, R, stride, pad, pad)
    path = tmp_path / "plans.txt"
    path.write_text("%d %d %d %d %d %d %d %d %d 1 | %d %d\n" % (N, C, Kf, R, R, stride, stride, P, Q, tile, slices))
    rng = np.random.default_rng(74)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.array((rng.standard_normal((Kf, C, R, R)) * 0.05).astype(np.float32))
    O1, O2 = hip.full((N, Kf, P, Q), float("nan")), hip.full((N, Kf, P, Q), float("nan"))
    args = lambda O: (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, R, R, stride, stride, pad, pad, P, Q, None, None, None, None, 0.0, None, 0)
    hip.conv_autotune(-1)
    try:
        hip.conv_tuned_load(str(path))
        hip.conv_autotune(True)
        if registered:
            hip.cache_conv_filters(dw)
        hip.synchronize()
        hip.workspace_trim()
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))
        kernel = hip.last_conv_kernel()
        assert kernel.startswith("conv_split") and ("+ksplit" in kernel) == (slices > 1), kernel
        assert hip.workspace_bytes() == 0
        hip._check(hip.lib.eddlhip_conv2d_fwd(*args(O2)))
        assert hip.last_conv_kernel() == kernel
        assert np.array_equal(O1.numpy(), O2.numpy())
        hip.fill_(O1, float("nan"))
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))   # (registered: with the split copy that conv2d_fwd has made)
        assert np.array_equal(O1.numpy(), O2.numpy())
    finally:
        hip.conv_autotune(-1)
        hip.uncache_conv_filters(dw)


def test_noalloc_takes_the_planners_plan_where_the_split_filters_do_not_fit(hip, tmp_path):
    """6 bytes a weight are beyond the array, the repacked 4 are not: the call is accepted as without a found plan."""
    N, C, H, W, Kf = 1, 3840, 8, 8, 3072
    assert 4 * C * Kf < SCRATCH_BYTES < 6 * C * Kf
    path = tmp_path / "plans.txt"
    path.write_text("%d %d %d 1 1 1 1 %d %d 1 | 17 1\n" % (N, C, Kf, H, W))
    rng = np.random.default_rng(75)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.full((Kf, C, 1, 1), 0.25)
    O1, O2 = hip.empty((N, Kf, H, W)), hip.empty((N, Kf, H, W))
    args = lambda O: (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 1, 1, 1, 1, 0, 0, H, W, None, None, None, None, 0.0, None, 0)
    hip.conv_autotune(-1)
    try:
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))
        kernel = hip.last_conv_kernel()
        hip.conv_tuned_load(str(path))
        hip.conv_autotune(True)
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O2)))
        assert hip.last_conv_kernel() == kernel
        assert np.array_equal(O1.numpy(), O2.numpy())
    finally:
        hip.conv_autotune(-1)


@pytest.mark.parametrize("registered", [False, True])
@pytest.mark.parametrize("W,slices", [(14, 1), (16, 4)])
def test_noalloc_runs_the_split_winograd_plan_that_was_found(hip, tmp_path, W, slices, registered):
    """The one-launch Winograd form in the split arithmetic is used like any found plan: same kernel and bits as conv2d_fwd, nothing allocated."""
    N, C, H, Kf = 3, 128, 18, 72
    path = tmp_path / "plans.txt"
    path.write_text("%d %d %d 3 3 1 1 %d %d 1 | 32 %d\n" % (N, C, Kf, H, W, slices))
    rng = np.random.default_rng(76)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.array((rng.standard_normal((Kf, C, 3, 3)) * 0.05).astype(np.float32))
    O1, O2 = hip.full((N, Kf, H, W), float("nan")), hip.full((N, Kf, H, W), float("nan"))
    args = lambda O: (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 3, 3, 1, 1, 1, 1, H, W, None, None, None, None, 0.0, None, 0)
    hip.conv_autotune(-1)
    try:
        hip.conv_tuned_load(str(path))
        hip.conv_autotune(True)
        if registered:
            hip.cache_conv_filters(dw)
        hip.synchronize()
        hip.workspace_trim()
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))
        kernel = hip.last_conv_kernel()
        assert "wino_split_kernel" in kernel and ("+ksplit" in kernel) == (slices > 1), kernel
        assert hip.workspace_bytes() == 0
        hip._check(hip.lib.eddlhip_conv2d_fwd(*args(O2)))
        assert hip.last_conv_kernel() == kernel
        assert np.array_equal(O1.numpy(), O2.numpy())
        hip.fill_(O1, float("nan"))
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))   # (registered: with the copy that conv2d_fwd has made)
        assert np.array_equal(O1.numpy(), O2.numpy())
    finally:
        hip.conv_autotune(-1)
        hip.uncache_conv_filters(dw)


def test_noalloc_takes_the_planners_plan_where_the_split_winograd_filters_do_not_fit(hip, tmp_path):
    N, C, H, W, Kf = 1, 1024, 8, 8, 1024
    assert 4 * 9 * C * Kf < SCRATCH_BYTES < 96 * C * Kf
    path = tmp_path / "plans.txt"
    path.write_text("%d %d %d 3 3 1 1 %d %d 1 | 32 1\n" % (N, C, Kf, H, W))
    rng = np.random.default_rng(77)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.full((Kf, C, 3, 3), 0.25)
    O1, O2 = hip.empty((N, Kf, H, W)), hip.empty((N, Kf, H, W))
    args = lambda O: (hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, 3, 3, 1, 1, 1, 1, H, W, None, None, None, None, 0.0, None, 0)
    hip.conv_autotune(-1)
    try:
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O1)))
        kernel = hip.last_conv_kernel()
        hip.conv_tuned_load(str(path))
        hip.conv_autotune(True)
        hip._check(hip.lib.eddlhip_conv2d_fwd_noalloc(*args(O2)))
        assert hip.last_conv_kernel() == kernel
        assert np.array_equal(O1.numpy(), O2.numpy())
    finally:
        hip.conv_autotune(-1)


# the planner takes a tile of the split form for these (the last in slices, where the direct kernels divide nothing)
CHOSEN = [(2, 128, 28, 30, 128, 3, 3, 1, 1), (8, 256, 28, 28, 256, 1, 1, 1, 0), (1, 48, 8, 18, 256, 3, 3, 1, 1)]


@pytest.mark.parametrize("N,C,H,W,Kf,R,S,stride,pad", CHOSEN)
def test_noalloc_first_call_on_registered_filters_reads_their_copy(hip, N, C, H, W, Kf, R, S, stride, pad):
    """No call of the other entry point came before: the filters are not split (or repacked) once more.  Seen from a filter tensor that
    a kernel has written behind the library's back, which is registered again only after that."""
    rng = np.random.default_rng(74)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.array((rng.standard_normal((Kf, C, R, S)) * 0.05).astype(np.float32))
    O = hip.full((N, Kf, H, W), float("nan"))

    def run(fn):
        hip.fill_(O, float("nan"))
        hip._check(fn(hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, R, S, stride, stride, pad, pad, H, W, None, None, None, None, 0.0, None, 0))
        assert "split_kernel" in hip.last_conv_kernel()
        return O.numpy()
    before = run(hip.lib.eddlhip_conv2d_fwd)
    hip.cache_conv_filters(dw)
    try:
        hip.relu(dw, dw)
        assert np.array_equal(run(hip.lib.eddlhip_conv2d_fwd_noalloc), before)
        hip.cache_conv_filters(dw)
        after = run(hip.lib.eddlhip_conv2d_fwd_noalloc)
        assert not np.array_equal(after, before) and np.array_equal(run(hip.lib.eddlhip_conv2d_fwd), after)
        dw.copy_from(dw.numpy() * 0.5)  # through the library: followed without another registration
        assert np.array_equal(run(hip.lib.eddlhip_conv2d_fwd_noalloc), after * np.float32(0.5))
    finally:
        hip.uncache_conv_filters(dw)
    assert np.array_equal(run(hip.lib.eddlhip_conv2d_fwd_noalloc), after * np.float32(0.5))


@pytest.mark.parametrize("N,C,H,W,Kf,R,S,stride,pad", CHOSEN)
def test_first_call_recorded_with_registered_filters_and_no_workspace(hip, N, C, H, W, Kf, R, S, stride, pad):
    """An undivided launch on registered filters takes no workspace in any form, so it is recorded without an eager call before it; where the
    chosen form is divided and the direct kernels are not, those run."""
    rng = np.random.default_rng(75)
    X, K, O = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.array((rng.standard_normal((Kf, C, R, S)) * 0.05).astype(np.float32)), hip.empty((N, Kf, H, W))
    hip.workspace_trim()
    hip.cache_conv_filters(K)
    try:
        graph = hip.record(lambda: hip.conv2D(X, K, None, O, stride, stride, pad, pad))
        recorded = hip.last_conv_kernel()
        got = []
        for _ in range(3):
            hip.fill_(O, float("nan"))
            graph.launch()
            got.append(O.numpy())
        divided = "slices" in recorded or "ksplit" in recorded
        assert not divided and hip.workspace_bytes() == 0
        hip.conv2D(X, K, None, O, stride, stride, pad, pad)
        eager = hip.last_conv_kernel()
        assert "split_kernel" in eager
        if eager != recorded:
            assert "split_kernel" not in recorded and "slices" in eager
            hip.set_conv_algo("winograd_never")
            hip.conv2D(X, K, None, O, stride, stride, pad, pad)
            hip.set_conv_algo("winograd_off")
        assert all(np.array_equal(g, O.numpy()) for g in got)
    finally:
        hip.uncache_conv_filters(K)


def test_dense_recorded_with_the_workspace_of_the_fp32_product(hip):
    """Many rows recorded with a workspace that holds what the fp32 product takes and not the rows in three parts: that product is recorded."""
    rng = np.random.default_rng(76)
    m, k, n = 64, 16384, 16
    A, W, C = hip.array(rng.standard_normal((m, k), dtype=np.float32)), hip.array(rng.standard_normal((k, n), dtype=np.float32)), hip.empty((m, n))
    hip.workspace_trim()
    hip.set_conv_algo("winograd_never")
    try:
        hip.mult2D(A, W, C)
    finally:
        hip.set_conv_algo("winograd_off")
    want = C.numpy()
    graph = hip.record(lambda: hip.mult2D(A, W, C))
    for _ in range(3):
        hip.fill_(C, float("nan"))
        graph.launch()
        assert np.array_equal(C.numpy(), want)


def test_registered_under_the_search_and_called_without_allocating_first(hip):
    """A tensor that was registered while the plan search was on has no split copy until a call makes it: a call that cannot runs the direct
    kernels on the copy that there is, and the planner's choice from then on."""
    N, C, H, W, Kf, R, S, stride, pad = CHOSEN[1]
    rng = np.random.default_rng(77)
    dx, dw = hip.array(rng.standard_normal((N, C, H, W), dtype=np.float32)), hip.array((rng.standard_normal((Kf, C, R, S)) * 0.05).astype(np.float32))
    O = hip.full((N, Kf, H, W), float("nan"))

    def run(fn):
        hip.fill_(O, float("nan"))
        hip._check(fn(hip.dev, dx.ptr, dw.ptr, None, O.ptr, N, C, H, W, Kf, R, S, stride, stride, pad, pad, H, W, None, None, None, None, 0.0, None, 0))
        return "split_kernel" in hip.last_conv_kernel(), O.numpy()
    split, want = run(hip.lib.eddlhip_conv2d_fwd)
    hip.set_conv_algo("winograd_never")
    direct = run(hip.lib.eddlhip_conv2d_fwd)[1]
    hip.set_conv_algo("winograd_off")
    hip.conv_autotune(True)
    hip.cache_conv_filters(dw)
    hip.conv_autotune(False)
    try:
        first, got = run(hip.lib.eddlhip_conv2d_fwd_noalloc)
        assert split and not first and np.array_equal(got, direct)
        for fn in (hip.lib.eddlhip_conv2d_fwd, hip.lib.eddlhip_conv2d_fwd_noalloc):
            chosen, got = run(fn)
            assert chosen and np.array_equal(got, want)
    finally:
        hip.conv_autotune(-1)
        hip.uncache_conv_filters(dw)
