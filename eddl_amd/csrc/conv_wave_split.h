// The split form (conv_split.h) for launches of few tiles (included by conv.hip only): one image of a network, the deep layers of a few.
//
// Such a launch is bound by latencies, not by a pipe: conv_split_kernel has a barrier per 32 channels, between them a trip to L2 or the
// last-level cache, and the K slices that fill the device need a second launch to be added.  Here the K range of a tile is divided
// over the eight wavefronts of a workgroup and then over workgroups.  A wavefront multiplies its own part of the K range alone: it
// loads pixels and filters straight into registers, DEPTH units of 16 channels under one tap ahead, and splits the pixels there;
// nothing is shared, so nothing is waited for until the sums of the eight meet in LDS, once.  Divided tiles are finished by the
// wavefronts that come last: each writes its sums past the caches of its XCD (agent-scope stores), counts itself in, and the one that
// completes the count reads them back and adds them in the order of the slices.  Nobody waits for another; no fence, whose
// write-back of a whole L2 is what made such a finish too dear behind a large launch.
// Bound: a chain of latencies.  256 -> 1024 on 14x14, one image, lasts 4.0 us on the device: 0.6 until the last workgroup runs, 1.1 until the first
// loads are on their way (address arithmetic and cold instructions; 2.1 with divisions), 0.9 in the loop (two units), 1.5 from there to the last
// acknowledged store; K slices add 2 (store, count, read back).  Three units in flight instead of two, or the constants asked for later,
// gain nothing; the counts of a tile's wavefronts side by side in one cache line cost 0.4 - 1.2 us.
// Sums: a wavefront's as in conv_split.h (hi hi in one accumulator, the five small products in another), then eight wavefronts
// in increasing K order, then the slices: a fixed order, shorter chains than one workgroup's.

// Pixels of 16 channels from c0 on for lane half `half`, channels past C zero, two tensors with any division between them.
// (Channels past the last must not be read: they belong to the next image, and what they hold times a filter's zero need not be zero.)
__device__ __forceinline__ void wave_split_load_any(const ConvParams &p, __amdgpu_buffer_rsrc_t in1, __amdgpu_buffer_rsrc_t in2, int voff, int c0, int half, int HW4, float (&raw)[8]) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int c = c0 + 8 * half + j;
        const bool second = c >= p.Csplit, ok = voff != OOB && c < p.C;
        const int off = voff + (second ? c - p.Csplit : c) * HW4;
        const float f1 = buf_load(in1, ok && !second ? off : OOB, 0), f2 = buf_load(in2, ok && second ? off : OOB, 0);
        raw[j] = second ? f2 : f1;
    }
}

// What a launch of this form needs besides: the host's reciprocals of the divisions at a workgroup's start (split_divide), which would
// be several hundred instructions of it, and the units of the K range of a wavefront (one more for the first `more` of them).
struct WaveSplitParams : ConvParams {
    unsigned magic_gn, magic_gm, magic_pq, magic_q, magic_rs, magic_s;
    int units_each, more;
};

template <int TM, int TN, SplitTaps TAPS>
__global__ __launch_bounds__(512, TM *TN == 1 ? 4 : 2) void conv_wave_split_kernel(const WaveSplitParams p) {
    constexpr int W = WAVE_SPLIT_WAVES, DEPTH = 2;
    __shared__ float red[W][TN][16][64];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    trace_mark(p, 0);
    // workgroup -> (pixel tile fastest, filter tile, K slice); ids that share an XCD get consecutive ones, so that the workgroups which read
    // the same filters share an L2
    const unsigned total = gridDim.x, per = total / EDDLHIP_NUM_XCD, rest = total % EDDLHIP_NUM_XCD;
    const unsigned xcd = blockIdx.x % EDDLHIP_NUM_XCD, slot = blockIdx.x / EDDLHIP_NUM_XCD;
    const unsigned vid = (xcd < rest ? xcd * (per + 1) : rest * (per + 1) + (xcd - rest) * per) + slot;
    const unsigned row = split_divide(vid, (unsigned)p.gn, p.magic_gn);  // (slice, filter tile)
    const int n_tile = (int)(vid - row * (unsigned)p.gn), slice = (int)split_divide(row, (unsigned)p.gm, p.magic_gm), m_tile = (int)row - slice * p.gm;
    const int tile = m_tile * p.gn + n_tile, m0 = m_tile * TM * 32, n0 = n_tile * TN * 32;

    // ---- this wavefront's units of the K range: 16 channels under one tap, taps fastest
    const int RS = p.R * p.S, part = slice * W + wave;
    const int lo = part * p.units_each + min(part, p.more), hi = lo + p.units_each + (part < p.more ? 1 : 0);
    const int first_c16 = (int)split_divide((unsigned)lo, (unsigned)RS, p.magic_rs), first_tap = lo - first_c16 * RS;

    // ---- what the epilogue needs of this lane's rows 2 wave and 2 wave + 1 of each 32 filters, asked for first
    float c_bias[TM][2], c_mean[TM][2], c_var[TM][2], c_g[TM][2], c_b[TM][2];
    int mrow[TM][2];
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int v = 2 * wave + k;
            mrow[tm][k] = m0 + tm * 32 + 8 * (v / 4) + 4 * half + v % 4;
            const int m = mrow[tm][k] < p.Kf ? mrow[tm][k] : p.Kf - 1;
            c_bias[tm][k] = p.bias ? p.bias[m] : 0.0f;
            c_mean[tm][k] = p.bn_mean ? p.bn_mean[m] : 0.0f;
            c_var[tm][k] = p.bn_mean ? p.bn_var[m] : 0.0f;
            c_g[tm][k] = p.bn_g ? p.bn_g[m] : 1.0f;
            c_b[tm][k] = p.bn_g ? p.bn_b[m] : 0.0f;
        }

    // ---- filters (past the wavefront's last unit the descriptors cover nothing: the loads bring zeros without touching memory)
    const int mblocks = p.Mp / 32, a_voff = lane * 16 + (m0 / 32) * SPLIT_UNIT;
    uintx4 a[DEPTH][TM][3];
    int wt_c16 = first_c16, wt_tap = first_tap;  // the unit that is loaded next
    auto load_filters = [&](int s, bool exists) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)p.Wp, 0, exists ? p.wp_bytes : 0u, RSRC_WORD3);
        const int soff = (2 * ((wt_c16 >> 1) * RS + wt_tap) + (wt_c16 & 1)) * mblocks * SPLIT_UNIT;
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                a[s][tm][k] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, a_voff + tm * SPLIT_UNIT + k * 1024, soff, 0));
        const int wrap = TAPS == ONE_TAP || wt_tap + 1 == RS ? 1 : 0;
        wt_tap = wrap ? 0 : wt_tap + 1;
        wt_c16 += wrap;
    };
#pragma unroll
    for (int s = 0; s < DEPTH; s++) load_filters(s, lo + s < hi);

    // ---- pixels
    const __amdgpu_buffer_rsrc_t in1 = __builtin_amdgcn_make_buffer_rsrc((void *)p.I, 0, p.in_bytes, RSRC_WORD3);
    const __amdgpu_buffer_rsrc_t in2 = __builtin_amdgcn_make_buffer_rsrc((void *)p.I2, 0, p.in_bytes, RSRC_WORD3);
    const int HW4 = p.H * p.W * 4, half_off = half * 8 * HW4;
    const unsigned magic_h = TAPS == UPSAMPLED ? split_magic(p.uh) : 0u, magic_w = TAPS == UPSAMPLED ? split_magic(p.uw) : 0u;
    int base[TN], ih0[TN], iw0[TN], only[TN];
    unsigned img[TN], pq[TN];
    bool pvalid[TN];
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        const int n = n0 + tn * 32 + l32;
        pvalid[tn] = n < (int)p.npix;
        const unsigned nc = pvalid[tn] ? (unsigned)n : 0u;
        img[tn] = split_divide(nc, (unsigned)p.PQ, p.magic_pq);
        pq[tn] = nc - img[tn] * (unsigned)p.PQ;
        const int op = (int)split_divide(pq[tn], (unsigned)p.Q, p.magic_q), oq = (int)pq[tn] - op * p.Q;
        base[tn] = (int)img[tn] * (p.Cimg * p.H * p.W);
        ih0[tn] = op * p.sr - p.pt;
        iw0[tn] = oq * p.sc - p.pl;
        only[tn] = pvalid[tn] && (unsigned)ih0[tn] < (unsigned)p.H && (unsigned)iw0[tn] < (unsigned)p.W ? (base[tn] + ih0[tn] * p.W + iw0[tn]) * 4 : OOB;  // (ONE_TAP)
    }
    int px_c16 = first_c16, px_ky = (int)split_divide((unsigned)first_tap, (unsigned)p.S, p.magic_s), px_kx = first_tap - px_ky * p.S;
    float raw[DEPTH][TN][8];
    auto load_pixels = [&](int s, bool exists) __attribute__((always_inline)) {
        const int c0 = px_c16 * 16;
        const bool second = c0 >= p.Csplit;
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            int voff = only[tn];
            if constexpr (TAPS == UPSAMPLED) voff = split_pixel(p, magic_h, magic_w, pvalid[tn], base[tn], ih0[tn], iw0[tn], px_ky, px_kx);
            if constexpr (TAPS == STORED) {
                const int y = ih0[tn] + px_ky, x = iw0[tn] + px_kx;
                const bool ok = pvalid[tn] && (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W;
                voff = ok ? (base[tn] + y * p.W + x) * 4 : OOB;
            }
            if (TAPS == UPSAMPLED && (c0 + 16 > p.C || (!second && c0 + 16 > p.Csplit))) {
                wave_split_load_any(p, in1, in2, exists ? voff : OOB, c0, half, HW4, raw[s][tn]);
            } else {
                const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(second ? p.I2 : p.I), 0, exists ? p.in_bytes : 0u, RSRC_WORD3);
                const int at = voff == OOB ? OOB : voff + half_off;
                int soff = (second ? c0 - p.Csplit : c0) * HW4;
#pragma unroll
                for (int j = 0; j < 8; j++, soff += HW4) raw[s][tn][j] = buf_load(rsrc, at, soff);
            }
        }
        if constexpr (TAPS == ONE_TAP) {
            px_c16++;
        } else {
            const int kx = px_kx + 1, wrap_x = kx == p.S ? 1 : 0, ky = px_ky + wrap_x, wrap_y = ky == p.R ? 1 : 0;
            px_kx = wrap_x ? 0 : kx;
            px_ky = wrap_y ? 0 : ky;
            px_c16 += wrap_y;
        }
    };
#pragma unroll
    for (int s = 0; s < DEPTH; s++) load_pixels(s, lo + s < hi);

    floatx16 acc[TM][TN], small[TM][TN];
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[tm][tn][v] = small[tm][tn][v] = 0.0f;
    trace_mark(p, 1);
    auto multiply_unit = [&](int s, bool more, bool exists) __attribute__((always_inline)) {
        uintx4 b[TN][3];
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                unsigned h, m, l;
                split_pair(SPLIT_UP * raw[s][tn][2 * q], SPLIT_UP * raw[s][tn][2 * q + 1], h, m, l);
                b[tn][0][q] = h;
                b[tn][1][q] = m;
                b[tn][2][q] = l;
            }
        if (more) load_pixels(s, exists);
        constexpr int kA[6] = {0, 1, 2, 0, 1, 0}, kB[6] = {0, 0, 0, 1, 1, 2};
#pragma unroll
        for (int k = 0; k < 6; k++)
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int tn = 0; tn < TN; tn++) {
                    floatx16 &d = k == 0 ? acc[tm][tn] : small[tm][tn];
                    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[s][tm][kA[k]]), __builtin_bit_cast(bf16x8, b[tn][kB[k]]), d, 0, 0, 0);
                }
        if (more) load_filters(s, exists);
    };
    // (no branch between the units of the loop: behind one the compiler can only wait for every load in flight)
    int u = lo;
    for (; u + DEPTH <= hi; u += DEPTH) {
#pragma unroll
        for (int s = 0; s < DEPTH; s++) multiply_unit(s, true, u + s + DEPTH < hi);
    }
#pragma unroll
    for (int s = 0; s < DEPTH - 1; s++)
        if (u + s < hi) multiply_unit(s, false, false);
    trace_mark(p, 2);

    float finite = 0.0f;
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                acc[tm][tn][v] = SPLIT_DOWN * __fadd_rn(acc[tm][tn][v], small[tm][tn][v]);
                finite = __builtin_fmaf(acc[tm][tn][v], 0.0f, finite);
            }
    if (__any(finite != 0.0f)) {
        split_tile_again<TM, TN, 16>(p, small, in1, in2, m0, n0, lo, hi, lane);
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int tn = 0; tn < TN; tn++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[tm][tn][v] = acc[tm][tn][v] * 0.0f == 0.0f ? acc[tm][tn][v] : small[tm][tn][v];
    }

    size_t oidx[TM][TN][2];
    bool ok[TM][TN][2];
    float res[TM][TN][2];
#pragma unroll
    for (int tn = 0; tn < TN; tn++)
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                ok[tm][tn][k] = pvalid[tn] && mrow[tm][k] < p.Kf;
                oidx[tm][tn][k] = ok[tm][tn][k] ? ((size_t)img[tn] * p.Kf + mrow[tm][k]) * p.PQ + pq[tn] : 0;
                res[tm][tn][k] = p.residual ? p.residual[oidx[tm][tn][k]] : 0.0f;
            }

    // ---- the eight wavefronts' sums meet: each adds two rows of accumulators of every 32 x 32 block
    float sum[TM][TN][2];
#pragma unroll
    for (int tm = 0; tm < TM; tm++) {
        if (tm > 0) __syncthreads();
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) red[wave][tn][v][lane] = acc[tm][tn][v];
        __syncthreads();
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                float s = red[0][tn][2 * wave + k][lane];
#pragma unroll
                for (int w = 1; w < W; w++) s = __fadd_rn(s, red[w][tn][2 * wave + k][lane]);
                sum[tm][tn][k] = s;
            }
    }

    if (p.nslices > 1) {
        const size_t tiles = (size_t)p.gm * p.gn, stride = tiles * (TM * TN * 1024);
        float *mine = p.partial + (size_t)tile * (TM * TN * 1024) + 2 * wave * 64 + lane;
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int tn = 0; tn < TN; tn++)
#pragma unroll
                for (int k = 0; k < 2; k++)
                    __hip_atomic_store(mine + (size_t)slice * stride + (tm * TN + tn) * 1024 + k * 64, sum[tm][tn][k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // A wavefront's rows are its own in every slice: it counts itself in as soon as its stores have reached the memory that all XCDs see,
        // and the last of the slices' wavefronts goes on.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        unsigned *count = p.count + (tile * W + wave) * WAVE_SPLIT_COUNT_WORDS;
        unsigned before = 0;
        if (lane == 0) before = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__builtin_amdgcn_readfirstlane((int)before) != p.nslices - 1) return;
        if (lane == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // as the next launch expects it
        constexpr int AHEAD = 16 / (TM * TN);
#pragma unroll 1
        for (int s0 = 0; s0 < p.nslices; s0 += AHEAD) {
            float x[AHEAD][TM][TN][2];
#pragma unroll
            for (int s = 0; s < AHEAD; s++)
                if (s0 + s < p.nslices) {
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
#pragma unroll
                        for (int tn = 0; tn < TN; tn++)
#pragma unroll
                            for (int k = 0; k < 2; k++)
                                x[s][tm][tn][k] =
                                    __hip_atomic_load(mine + (size_t)(s0 + s) * stride + (tm * TN + tn) * 1024 + k * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
            for (int s = 0; s < AHEAD; s++)
                if (s0 + s < p.nslices) {
#pragma unroll
                    for (int tm = 0; tm < TM; tm++)
#pragma unroll
                        for (int tn = 0; tn < TN; tn++)
#pragma unroll
                            for (int k = 0; k < 2; k++) sum[tm][tn][k] = s0 + s == 0 ? x[s][tm][tn][k] : __fadd_rn(sum[tm][tn][k], x[s][tm][tn][k]);
                }
        }
    }
    ChannelEpilogue chan[TM][2];
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            // (not before the loop, where it would wait for the loads)
            asm volatile("" : "+v"(c_var[tm][k]));
            chan[tm][k] = {c_bias[tm][k], c_mean[tm][k], p.bn_mean ? sqrtf(__fadd_rn(c_var[tm][k], p.bn_eps)) : 1.0f, c_g[tm][k], c_b[tm][k]};
        }
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float x = finish_value(p, chan[tm][k], sum[tm][tn][k], res[tm][tn][k]);
                if (ok[tm][tn][k]) p.O[oidx[tm][tn][k]] = x;
            }
    if (p.trace != nullptr) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        trace_mark(p, 3);
    }
}
