// The 2x2 convolution of an image upsampled twice (conv_up2x2_kernel) in the split arithmetic of conv_split.h (included by conv.hip
// only): the nine weight sums per filter and channel, added up in 64 bits, and the stored pixels are split into three
// bf16 numbers, the six largest products of two such sums summed in fp32, the smallest first.  The instruction rounds what it
// shifts out on the way to an accumulator downwards and several times a step, so that products added straight to the long sums are up to
// 14 % further from 64 bits than the fp32 kernel's behind a ReLU: as in wino_split.h the products of 16 channels (of one to three
// weight sums of a parity) are summed from zero and added to the long sum by vector instructions, rounded once and to nearest.
// What remains of the bias has opposite signs for the outputs (0,1) and (1,0) of a block and for every other block of a plane.
// Error against 64 bits behind a ReLU relative to the outputs' root mean square, of the fp32 kernel -> of this one (in brackets with the products
// added straight to the long sums): 16 channels 9.0e-8 -> 4.4e-8 (7.2e-8), 128 2.2e-7 -> 1.0e-7 (2.4e-7), 512 4.2e-7 -> 1.7e-7 (4.7e-7), 1024
// 6.1e-7 -> 2.5e-7 (7.0e-7); of the mean of a plane at 512 channels 1.9e-8 -> 5.0e-9 (3.2e-8).

constexpr int UPSPLIT_UNIT = 9 * SPLIT_UNIT;  // bytes of 32 filters x 16 channels, all nine weight sums

// Weight sum `row` (up2x2_filter_kernel's numbering) of the 2x2 filter at k.
template <typename T>
__device__ __forceinline__ T up2x2_sum(const float *k, int row) {
    const T w00 = k[0], w01 = k[1], w10 = k[2], w11 = k[3];
    return row == 0 ? (w00 + w01) + (w10 + w11) : row == 1 ? w00 + w10 : row == 2 ? w01 + w11 : row == 3 ? w00 + w01 : row == 4 ? w10 + w11 : (T)k[row - 5];
}

// K[Kf][C][2][2] -> Ws[c / 16][Mp / 32][weight sum][part][lane][8], operands of the matrix instruction as in split_filter_kernel;
// channels past C and filters past Kf are zeros; the sums of the outputs (0,1) and (1,0) negated.  Bound by the write (54 bytes per filter and channel).
__global__ __launch_bounds__(256) void up2x2_split_filter_kernel(const float *__restrict__ K, uintx4 *__restrict__ Ws, int Kf, int C, int mblocks, int k16s) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)k16s * mblocks * 64) return;
    const int lane = (int)(idx & 63);
    const int unit = (int)(idx >> 6), mb = unit % mblocks, k16 = unit / mblocks;
    const int c0 = k16 * 16 + (lane >> 5) * 8, m = mb * 32 + (lane & 31);
    uintx4 *dst = Ws + (size_t)unit * (9 * 192) + lane;
#pragma unroll
    for (int row = 0; row < 9; row++) {
        const double up = row >= 1 && row <= 4 ? -SPLIT_UP : SPLIT_UP;
        uintx4 hi, mid, lo;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int c = c0 + 2 * q;
            const float *k = K + ((size_t)(m < Kf ? m : 0) * C + (c < C ? c : 0)) * 4;  // (channels come in pairs: C is a multiple of 16)
            const bool ok = m < Kf && c < C;
            unsigned h, md, l;
            split_pair(ok ? up * up2x2_sum<double>(k, row) : 0.0, ok ? up * up2x2_sum<double>(k + 4, row) : 0.0, h, md, l);
            hi[q] = h;
            mid[q] = md;
            lo[q] = l;
        }
        dst[row * 192] = hi;
        dst[row * 192 + 64] = mid;
        dst[row * 192 + 128] = lo;
    }
}

template <typename F, int... I>
__device__ __forceinline__ void for_each_index(std::integer_sequence<int, I...>, F f) {
    (f(std::integral_constant<int, I>()), ...);
}

// One 32x32 block of one parity's sums once more with the fp32 instruction (see split_tile_again), channels [c_lo, c_hi): this
// lane's filter m, the byte offsets of its block's four stored pixels.
__device__ __forceinline__ void up2x2_block_again(const ConvParams &p, floatx16 &sum, __amdgpu_buffer_rsrc_t in, int m, const int (&voff)[4], int parity, int c_lo,
                                                  int c_hi, int half) {
    const int HW4 = p.H * p.W * 4;
#pragma unroll
    for (int v = 0; v < 16; v++) sum[v] = 0.0f;
#pragma unroll 1
    for (int c0 = c_lo; c0 < c_hi && c0 < p.C; c0 += 2) {
        const int c = c0 + half;
        const float *k = p.K + ((size_t)(m < p.Kf ? m : 0) * p.C + c) * 4;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if ((t & parity) != t) continue;  // (uniform: tap (t / 2, t % 2) is seen by the parities that have its bits)
            const int row = parity == 0 ? 0 : (parity == 1 ? 1 + t : (parity == 2 ? 3 + t / 2 : 5 + t));
            const float a = up2x2_sum<float>(k, row), b = buf_load(in, voff[t] == OOB ? OOB : voff[t] + c * HW4, 0);
            sum = __builtin_amdgcn_mfma_f32_32x32x2f32(m < p.Kf ? a : 0.0f, b, sum, 0, 0, 0);
        }
    }
}

// A workgroup takes 32 WM filters x 64 WN blocks (stored pixels), a wavefront 32 x 64 of them with the four parities' accumulators
// (128 registers).  A K-step is 32 channels: their four stored pixels per block come one tap after the other as in
// conv_split_kernel (loaded a tap ahead, split between the matrix instructions on their way into LDS), and tap t is multiplied by the
// weight sums that see it - 4, 2, 2 and 1 of the nine - straight from L2, the next sum's requested while the current one
// multiplies.  216 matrix instructions of a wavefront share four reads of the pixels; their splitting and the additions to the long
// sums are three to five vector instructions per matrix instruction.  Measured (4 images, us, with the products added straight to the
// long sums -> this): 1024 -> 512 on 32x32 193 -> 195, 512 -> 256 on 64x64 171 -> 182, 256 -> 128 on 128x128 175 -> 186, 128 -> 64 on
// 256x256 (64 x 128 tile) 218 -> 232; the fp32 kernel 314, 280, 288, 314.  Bound: in U-Net's launches the matrix pipe is busy 49 % of the cycles
// at 2.26 GHz (46 % of the bf16 instruction's rate; 64 x 128 tile 41 %), the vector L1 holds requests back half of them (every filter
// comes from L2 for 64 or 128 blocks only) and a wavefront waits 37 %.
// All 256 registers are taken; three values of either build lie in scratch.
template <int WM, int WN>
__global__ __launch_bounds__(256, 2) void conv_up2x2_split_kernel(const ConvParams p) {
    static_assert(WM * WN == 4, "four wavefronts per workgroup");
    constexpr int BM = 32 * WM, BN = 64 * WN, TN = 2;
    constexpr int CHUNKS = SPLIT_K / (256 / BN) / 8;
    static_assert(CHUNKS == 1 || CHUNKS == 2, "BN is 64 or 128");
    __shared__ uintx4 Bs[2][3][SPLIT_K / 8][BN];
    __shared__ __attribute__((aligned(16))) float epi[EPI_ROWS * BM];

    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int m_tile, n_tile, local_tile, slice;
    bool split;
    trace_mark(p, 0);
    tile_of_block(p, m_tile, n_tile, local_tile, slice, split);
    const int step_lo = split ? slice * p.slice_steps : 0;
    const int step_hi = split ? min(step_lo + p.slice_steps, p.nsteps) : p.nsteps;
    const int m0 = m_tile * BM, n0 = n_tile * BN;
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)p.Wp, 0, p.wp_bytes, RSRC_WORD3);
    const int per_img = p.wth * p.wtw, HW4 = p.H * p.W * 4;

    // the byte offsets of block n's four stored pixels (channel 0)
    auto pixels_of = [&](int n, int (&voff)[4]) {
        const int nc = n < p.wT ? n : 0, img = nc / per_img, r = nc - img * per_img, ty = r / p.wtw, tx = r - ty * p.wtw;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int y = ty + (t >> 1), x = tx + (t & 1);
            voff[t] = n < p.wT && y < p.H && x < p.W ? (img * (p.C * p.H * p.W) + y * p.W + x) * 4 : OOB;
        }
    };
    const int pix = tid % BN;
    const int kgroup = __builtin_amdgcn_readfirstlane(tid / BN) * CHUNKS;
    int voff[4];
    pixels_of(n0 + pix, voff);
    float raw[CHUNKS][8];
    auto load_pixels = [&](int step, int tap, int chunk) __attribute__((always_inline)) {
        const int c0 = step * SPLIT_K + (kgroup + chunk) * 8;
        const bool there = c0 < p.C;  // (past the last channel, and behind the last step: zeros, without touching memory)
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.I, 0, there ? p.in_bytes : 0u, RSRC_WORD3);
        int soff = there ? c0 * HW4 : 0;
#pragma unroll
        for (int j = 0; j < 8; j++, soff += HW4) raw[chunk][j] = buf_load(rsrc, voff[tap], soff);
    };
    // every other block of a plane is accumulated with the opposite sign
    auto odd_block = [&](int n) { return ((n / p.wtw + n % p.wtw - n / per_img * p.wth) & 1) != 0; };
    const float up = odd_block(n0 + pix) ? -SPLIT_UP : SPLIT_UP;
    auto put_pixels = [&](int buf, int chunk) __attribute__((always_inline)) {
        uintx4 hi, mid, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            unsigned h, m, l;
            split_pair(up * raw[chunk][2 * j], up * raw[chunk][2 * j + 1], h, m, l);
            hi[j] = h;
            mid[j] = m;
            lo[j] = l;
        }
        Bs[buf][0][kgroup + chunk][pix] = hi;
        Bs[buf][1][kgroup + chunk][pix] = mid;
        Bs[buf][2][kgroup + chunk][pix] = lo;
    };

    const int a_voff = lane * 16, a_base = (m0 / 32 + wm) * UPSPLIT_UNIT, a_k16 = p.Mp / 32 * UPSPLIT_UNIT;
    uintx4 a[2][3];
    auto load_a = [&](int set, int k16, int row) __attribute__((always_inline)) {
#pragma unroll
        for (int part = 0; part < 3; part++)
            a[set][part] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, a_voff, a_base + k16 * a_k16 + row * SPLIT_UNIT + part * 1024, 0));
    };
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; chunk++) load_pixels(step_lo, 0, chunk);
    load_a(0, 2 * step_lo, 0);
    TileChannel chan = NO_CHANNEL;
    if (!split) chan = fetch_channel_constants<BM>(p, m0, tid);
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; chunk++) put_pixels(0, chunk), load_pixels(step_lo, 1, chunk);
    if (!split) put_channel_constants<BM>(epi, chan, tid);

    floatx16 acc[4][TN];  // [parity 2 i + j][block group]
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[e][tn][v] = 0.0f;
    __syncthreads();
    trace_mark(p, 1);

    // The step's 18 groups of products: tap, 16 channels and the parity that they belong to, two or three in a row of one parity where
    // that can be, as their products are added up before they go to the long sum
    constexpr int GROUPS = 18;
    constexpr int kTap[GROUPS] = {0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 2, 2, 2, 2, 3, 3}, kHalf[GROUPS] = {0, 0, 0, 0, 1, 1, 1, 1, 0, 0, 1, 1, 0, 0, 1, 1, 0, 1};
    constexpr int kParity[GROUPS] = {0, 1, 2, 3, 3, 2, 0, 1, 1, 3, 1, 3, 3, 2, 2, 3, 3, 3}, kRow[4][4] = {{0, 1, 3, 5}, {0, 2, 0, 6}, {0, 0, 4, 7}, {0, 0, 0, 8}};  // [tap][parity]
    constexpr int kA[6] = {2, 1, 1, 0, 0, 0}, kB[6] = {0, 1, 0, 2, 1, 0};  // the smallest products first
    uintx4 b[TN][3];
    floatx16 own[TN];  // the products of a run of groups of one parity
#pragma unroll
    for (int v = 0; v < 16; v++) own[1][v] = 0.0f;
    auto add_own = [&](int parity, int tn) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < 16; v++) acc[parity][tn][v] = __fadd_rn(acc[parity][tn][v], own[tn][v]);
    };
    // Group I of a step; the filters of the group after it are requested first.  Products of 32 blocks are added to their long sum
    // while those of the next 32 multiply: the second 32 blocks' in the next group.
    auto group = [&](int step, int next, auto i_c) __attribute__((always_inline)) {
        constexpr int I = decltype(i_c)::value, N = (I + 1) % GROUPS, B = (I + GROUPS - 1) % GROUPS;
        constexpr int tap = kTap[I], g = kHalf[I], parity = kParity[I], set = I & 1;
        constexpr bool fresh = tap != kTap[B] || g != kHalf[B];
        // (the build with twice the pixels in flight has the registers for runs of one group only: with longer ones it spills in the loop, 350 us instead of 232)
        constexpr bool run_starts = CHUNKS == 2 || parity != kParity[B], run_ends = CHUNKS == 2 || parity != kParity[N];
        constexpr bool put = fresh && g < CHUNKS;  // the next tap's pixels into the other buffer, those of the tap after it in their place
        const floatx16 zero = {0.0f};
        load_a(set ^ 1, 2 * (N == 0 ? next : step) + kHalf[N], kRow[kTap[N]][kParity[N]]);
#pragma unroll
        for (int tn = 0; tn < TN; tn++) {
            if (fresh) {
#pragma unroll
                for (int part = 0; part < 3; part++) b[tn][part] = Bs[tap & 1][part][2 * g + half][wn * 64 + tn * 32 + (lane & 31)];
            }
            if (tn == 0 ? run_starts : run_ends) add_own(tn == 0 ? kParity[B] : parity, tn ^ 1);
#pragma unroll
            for (int k = 0; k < 6; k++)
                own[tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[set][kA[k]]), __builtin_bit_cast(bf16x8, b[tn][kB[k]]), k == 0 && run_starts ? zero : own[tn],
                                                                  0, 0, 0);
            if (put && tn == 0) put_pixels((tap & 1) ^ 1, g);
            if (put && tn == 1) load_pixels(tap < 2 ? step : step + 1, (tap + 2) & 3, g);
#pragma unroll
            for (int i = 0; i < 6; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (put && tn == 0 && i > 0) __builtin_amdgcn_sched_group_barrier(0x002, 13, 0);
                else if (i > 0 && i < 5) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (tap != kTap[N]) __syncthreads();
    };
    for (int step = step_lo; step < step_hi; step++) {
        const int next = step + 1 < step_hi ? step + 1 : step;
        for_each_index(std::make_integer_sequence<int, GROUPS>(), [&](auto i_c) __attribute__((always_inline)) { group(step, next, i_c); });
    }
    add_own(3, 1);
    trace_mark(p, 2);

    // (the lane's number once more, so that nothing that follows from it lives through the loop: registers)
    const int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), half_e = lane_e >> 5;
    const int m_first = m0 + wm * 32 + (lane_e & 31);
    auto finish = [&](auto tn_c) __attribute__((always_inline)) {
        constexpr int tn = decltype(tn_c)::value;
        const int n_first = n0 + wn * 64 + tn * 32;
        const float down = odd_block(n_first + (lane_e & 31)) ? -SPLIT_DOWN : SPLIT_DOWN;
        floatx16 y[2][2];
        float finite = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                y[e >> 1][e & 1][v] = __builtin_fmaf(e == 1 || e == 2 ? -down : down, acc[e][tn][v], 0.0f);  // (a sum of zeros is +0 under either sign)
                finite = __builtin_fmaf(y[e >> 1][e & 1][v], 0.0f, finite);
            }
        if (__any(finite != 0.0f)) {
            const __amdgpu_buffer_rsrc_t in = __builtin_amdgcn_make_buffer_rsrc((void *)p.I, 0, p.in_bytes, RSRC_WORD3);
            int at[4];
            pixels_of(n_first + (lane_e & 31), at);
#pragma unroll 1
            for (int e = 0; e < 4; e++) {
                floatx16 sum;
                up2x2_block_again(p, sum, in, m_first, at, e, step_lo * SPLIT_K, step_hi * SPLIT_K, half_e);
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float x = y[s >> 1][s & 1][v];
                        y[s >> 1][s & 1][v] = s != e || x * 0.0f == 0.0f ? x : sum[v];
                    }
            }
        }
        if (split) {
            // this slice's share, raw: wino_fused_reduce_kernel's layout
            const size_t tiles = (gridDim.x - (unsigned)p.main_tiles) / p.nslices;
            floatx4 *dst = reinterpret_cast<floatx4 *>(p.partial) + (((size_t)slice * tiles + local_tile) * (WM * 2 * WN) + wm * (2 * WN) + wn * 2 + tn) * 16 * 64 + lane_e;
#pragma unroll
            for (int v = 0; v < 16; v++) dst[v * 64] = (floatx4){y[0][0][v], y[0][1][v], y[1][0][v], y[1][1][v]};
        } else {
            wino_store_tile<BM>(p, y, epi, m0, wm * 32, n_first, lane_e);
        }
    };
    finish(std::integral_constant<int, 0>());
    finish(std::integral_constant<int, 1>());
    if (p.trace != nullptr) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        trace_mark(p, 3);
    }
}
