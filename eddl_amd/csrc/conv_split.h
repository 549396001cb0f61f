// Convolution in fp32 accuracy on the bf16 matrix instructions (included by conv.hip only).
//
// Every fp32 number x, enlarged 2^24 times, is the sum of three bf16 numbers (Henry, Tang and Heinecke, "Leveraging the bfloat16
// artificial intelligence datatype for higher-precision computations", 2019): hi = bf16(y), mid = bf16(y - hi),
// lo = y - hi - mid with y = 2^24 x.  A bf16 holds 8 significant bits with the exponent range of an fp32, both differences are
// exact, and 3 x 8 bits hold the 24 of the fp32.  The factor keeps the last bit of the smallest number in range: y is a
// multiple of 2^-125, so every part is zero or a normal bf16 and nothing of x is lost, subnormal numbers included (without it
// numbers below 2^-110 lost bits of lo, below 2^-118 of mid).  The finished sums, 2^48 times too large, are scaled back.
// Of the nine products of two such sums the six largest are multiplied -
//   hi hi + (hi mid + mid hi) + (hi lo + mid mid + lo hi)
// - and the three left out are together below 2^-24 of the product (each of mid lo and lo mid can reach 2^-25), the rounding of
// one fp32 product.  The products are exact in the instruction and the sums stay in fp32 accumulators.
// v_mfma_f32_32x32x16_bf16 does 16 times the work of v_mfma_f32_32x32x2_f32 in the same cycles per flop of K, so six of them
// per 16 taps cost 6/16 of the fp32 instruction's.
//
// Not for infinities: inf - inf is NaN, and inf times the zero mid of a short factor is too; numbers from 2^104 and sums from
// 2^80 on are infinite here as well.  A wavefront whose finished accumulators are not all finite computes its tile with the
// fp32 instruction too, from the original filters (split_tile_again), and every sum that is not finite takes that value: the
// others keep theirs, whatever stands beside them in the tile.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int SPLIT_K = 32;                   // channels of a K-step (of one filter tap): two matrix instructions deep
constexpr int SPLIT_UNIT = 3 * 64 * 16;       // bytes of 32 filters x 16 channels: [part][lane][8 bf16]

__device__ __forceinline__ unsigned split_round(float a, float b) {  // two bf16, rounded to nearest even
    return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2){a, b}, bf16x2));
}
__device__ __forceinline__ void split_pair(float a, float b, unsigned &hi, unsigned &mid, unsigned &lo) {
    hi = split_round(a, b);
    const float ra = a - __builtin_bit_cast(float, hi << 16), rb = b - __builtin_bit_cast(float, hi & 0xffff0000u);
    mid = split_round(ra, rb);
    lo = split_round(ra - __builtin_bit_cast(float, mid << 16), rb - __builtin_bit_cast(float, mid & 0xffff0000u));
}

// The same of numbers that are known in 64 bits (transformed filters): the three parts, each rounded to nearest, hold 26 bits of them.
__device__ __forceinline__ void split_pair(double a, double b, unsigned &hi, unsigned &mid, unsigned &lo) {
    hi = split_round((float)a, (float)b);
    const double ra = a - (double)__builtin_bit_cast(float, hi << 16), rb = b - (double)__builtin_bit_cast(float, hi & 0xffff0000u);
    mid = split_round((float)ra, (float)rb);
    lo = split_round((float)(ra - (double)__builtin_bit_cast(float, mid << 16)), (float)(rb - (double)__builtin_bit_cast(float, mid & 0xffff0000u)));
}

constexpr float SPLIT_UP = 16777216.0f;                    // 2^24, of pixels and filters
constexpr float SPLIT_DOWN = 1.0f / SPLIT_UP / SPLIT_UP;   // of their products

// K[Kf][C][RS] -> Ws[k16][Mp / 32][part][lane][8]: the operand of lane l of the matrix instruction is filter l % 32 of the
// block, channels 8 (l / 32) .. + 7 of the 16.  k16 = 2 (cb RS + tap) + g covers channels 32 cb + 16 g .. + 15 under one tap;
// channels past C and filters past Kf are zeros.  Bound by the write (6 bytes a weight); once per registered filter tensor.
__global__ __launch_bounds__(256) void split_filter_kernel(const float *__restrict__ K, uintx4 *__restrict__ Ws, int Kf, int C, int RS, int mblocks, int k16s) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)k16s * mblocks * 64) return;
    const int lane = (int)(i & 63);
    const int unit = (int)(i >> 6), mb = unit % mblocks, k16 = unit / mblocks;
    const int step = k16 >> 1, cb = step / RS, tap = step - cb * RS;
    const int c0 = cb * SPLIT_K + (k16 & 1) * 16 + (lane >> 5) * 8, m = mb * 32 + (lane & 31);
    uintx4 hi, mid, lo;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = c0 + 2 * j;
        const float a = m < Kf && c < C ? SPLIT_UP * K[((size_t)m * C + c) * RS + tap] : 0.0f;
        const float b = m < Kf && c + 1 < C ? SPLIT_UP * K[((size_t)m * C + c + 1) * RS + tap] : 0.0f;
        unsigned h, md, l;
        split_pair(a, b, h, md, l);
        hi[j] = h;
        mid[j] = md;
        lo[j] = l;
    }
    uintx4 *dst = Ws + (size_t)unit * 192 + lane;
    dst[0] = hi;
    dst[64] = mid;
    dst[128] = lo;
}

// The same for filters of 2 ... 9 taps: a workgroup takes 32 filters and 16 channels, whose weights lie in 32 runs of memory, through LDS, so that
// reads are whole lines (one weight at a time they are 4 bytes at the stride of the taps).  us with the launch,
// one weight at a time -> this: 512 -> 512 16.6 -> 11.6, 1024 -> 1024 37 -> 15.9, 128 -> 128 3.2 -> 4.9, 256 -> 512 9.1 -> 11.2; so from 2 million weights on.
constexpr int SPLIT_FILTER_TAPS = 9;
constexpr long long SPLIT_FILTER_MANY = 2000000;
__global__ __launch_bounds__(256) void split_filter_taps_kernel(const float *__restrict__ K, uintx4 *__restrict__ Ws, int Kf, int C, int RS, int mblocks) {
    constexpr int PITCH = 16 * SPLIT_FILTER_TAPS + 1;  // odd: the 32 filters of a read lie in 32 banks
    __shared__ float rows[32 * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mb = blockIdx.x % mblocks, c16 = blockIdx.x / mblocks, run = 16 * RS, there = min(run, C * RS - c16 * run);  // (fewer, or none, past C)
    constexpr int PASSES = (16 * SPLIT_FILTER_TAPS + 63) / 64;
    float w[8][PASSES];  // (all of a wavefront's eight runs are asked for before the first is stored)
#pragma unroll
    for (int f8 = 0; f8 < 8; f8++)
#pragma unroll
        for (int i = 0; i < PASSES; i++) {
            const int m = mb * 32 + 8 * wave + f8, r = lane + 64 * i;
            w[f8][i] = m < Kf && r < there ? K[((size_t)m * C + c16 * 16) * RS + r] : 0.0f;
        }
#pragma unroll
    for (int f8 = 0; f8 < 8; f8++)
#pragma unroll
        for (int i = 0; i < PASSES; i++)
            if (lane + 64 * i < run) rows[(8 * wave + f8) * PITCH + lane + 64 * i] = SPLIT_UP * w[f8][i];
    __syncthreads();
    for (int t = wave; t < RS; t += 4) {
        const float *src = rows + (lane & 31) * PITCH + (lane >> 5) * 8 * RS + t;
        uintx4 hi, mid, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            unsigned h, md, l;
            split_pair(src[2 * j * RS], src[(2 * j + 1) * RS], h, md, l);
            hi[j] = h;
            mid[j] = md;
            lo[j] = l;
        }
        uintx4 *dst = Ws + ((size_t)(2 * ((c16 >> 1) * RS + t) + (c16 & 1)) * mblocks + mb) * 192 + lane;
        dst[0] = hi;
        dst[64] = mid;
        dst[128] = lo;
    }
}

// Division by an upsampling factor as one multiplication, with no branch (a branch would end the block that the matrix
// instructions are scheduled in): magic = ceil(2^32 / factor), 0 for factor 1.  The sides of the enlarged image are at most
// 2^20, so the product overestimates the quotient by less than 2^-12 and by one whole at most.
__device__ __forceinline__ unsigned split_magic(int factor) { return factor == 1 ? 0u : 0xffffffffu / (unsigned)factor + 1u; }
__device__ __forceinline__ unsigned split_divide(unsigned y, unsigned factor, unsigned magic) {
    unsigned q = __umulhi(y, magic);
    q -= q * factor > y ? 1u : 0u;
    return magic == 0u ? y : q;
}

// Byte offset of the stored pixel that tap (ky, kx) of a window at (ih0, iw0) reads (channel 0), OOB outside the image.
__device__ __forceinline__ int split_pixel(const ConvParams &p, unsigned magic_h, unsigned magic_w, bool valid, int base, int ih0, int iw0, int ky, int kx) {
    const unsigned y = (unsigned)(ih0 + ky), x = (unsigned)(iw0 + kx);
    const bool ok = valid && y < (unsigned)(p.H * p.uh) && x < (unsigned)(p.W * p.uw);
    const int at = (base + (int)split_divide(y, (unsigned)p.uh, magic_h) * p.W + (int)split_divide(x, (unsigned)p.uw, magic_w)) * 4;
    return ok ? at : OOB;
}

// The K-steps [step_lo, step_hi) (of GROUP channels each) of a wavefront's blocks once more with the fp32 instruction, two channels at
// a time in the order of the split sums; reads the image and the original filters where they are.  Only infinities, NaN and numbers near
// the end of the fp32 range come here.  (The fp32 kernels take the channels slowest: a sum that overflows in one of the two
// orders and not in the other can differ.)
template <int TM, int TN, int GROUP>
__device__ __forceinline__ void split_tile_again(const ConvParams &p, floatx16 (&acc)[TM][TN], __amdgpu_buffer_rsrc_t in1, __amdgpu_buffer_rsrc_t in2, int m_first,
                                                 int n_first, int step_lo, int step_hi, int lane) {
    const int RS = p.R * p.S, half = lane >> 5, HW4 = p.H * p.W * 4;
    const unsigned magic_h = split_magic(p.uh), magic_w = split_magic(p.uw);
    int base[TN], ih0[TN], iw0[TN];
    bool valid[TN];
#pragma unroll
    for (int tn = 0; tn < TN; tn++) {
        const int n = n_first + tn * 32 + (lane & 31);
        valid[tn] = n < (int)p.npix;
        const unsigned nc = valid[tn] ? (unsigned)n : 0u, img = nc / (unsigned)p.PQ, pq = nc - img * (unsigned)p.PQ;
        const int op = (int)(pq / (unsigned)p.Q), oq = (int)pq - op * p.Q;
        base[tn] = (int)img * (p.Cimg * p.H * p.W);
        ih0[tn] = op * p.sr - p.pt;
        iw0[tn] = oq * p.sc - p.pl;
    }
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[tm][tn][v] = 0.0f;
#pragma unroll 1
    for (int step = step_lo; step < step_hi; step++) {
        const int cb = step / RS, tap = step - cb * RS, ky = tap / p.S, kx = tap - ky * p.S;
#pragma unroll 1
        for (int c0 = cb * GROUP; c0 < cb * GROUP + GROUP && c0 < p.C; c0 += 2) {
            const int c = c0 + half;
            float a[TM], b[TN];
#pragma unroll
            for (int tm = 0; tm < TM; tm++) {
                const int m = m_first + tm * 32 + (lane & 31);
                a[tm] = m < p.Kf && c < p.C ? p.K[((size_t)m * p.C + c) * RS + tap] : 0.0f;
            }
#pragma unroll
            for (int tn = 0; tn < TN; tn++) {
                const bool second = c >= p.Csplit;
                int off = split_pixel(p, magic_h, magic_w, valid[tn] && c < p.C, base[tn], ih0[tn], iw0[tn], ky, kx);
                if (off != OOB) off += (second ? c - p.Csplit : c) * HW4;
                const float from1 = buf_load(in1, second ? OOB : off, 0), from2 = buf_load(in2, second ? off : OOB, 0);
                b[tn] = second ? from2 : from1;
            }
#pragma unroll
            for (int tm = 0; tm < TM; tm++)
#pragma unroll
                for (int tn = 0; tn < TN; tn++) acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[tm], b[tn], acc[tm][tn], 0, 0, 0);
        }
    }
}

// Issue order of a stretch of code: its VALU vector instructions behind its MFMA matrix instructions, evenly.
template <int MFMA, int VALU>
__device__ __forceinline__ void split_issue_order() {
#pragma unroll
    for (int i = 0; i < MFMA; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (VALU + MFMA - 1) / MFMA, 0);
    }
}

// Implicit GEMM, any filter shape and stride: a K-step is 32 channels of one filter tap.  A thread loads the tap's pixel of
// one output position for 8 or 16 channels (coalesced along the image row), splits them and puts them into LDS in the
// operand layout, [buffer][part][8 channels][pixel][8 bf16]: every LDS access is 16 bytes per lane of consecutive lanes.
// Split filters go from L2 straight to registers (two wavefronts read the same 1 KB; the second meets the first's in L1).
// How a step finds its pixel.  UPSAMPLED: any convolution; STORED: of the image as it is stored; ONE_TAP: the filter has one tap, so
// that the offset is the same in every step.  A general offset takes two divisions (25 vector instructions a step and thread, beside
// the 52 that split its eight pixels), which slow a kernel that multiplies little per pixel (batch 64, best plans, us, all on one card;
// UPSAMPLED -> ONE_TAP: 256 -> 64 on 56x56 55.8 -> 52.4, 512 -> 256 on 28x28 78.4 -> 76.5, 128 -> 512 53.1 -> 51.2, 256 -> 1024 on
// 14x14 46.6 -> 45.2, 1024 -> 256 45.2 -> 43.2, 2048 -> 512 on 7x7 51.8 -> 49.5; UPSAMPLED -> STORED: 128 3x3 stride 2 on 56x56
// 91.2 -> 89.9, tile 128x128 95.8 -> 94.4).  ROW_BIAS: ONE_TAP with a residual of one row for all filters, a dense layer's bias.
enum SplitTaps { UPSAMPLED, STORED, ONE_TAP, ROW_BIAS };
template <int WM, int WN, int TM, int TN, int WGS, SplitTaps TAPS>
__global__ __launch_bounds__(256, WGS) void conv_split_kernel(const ConvParams p) {
    static_assert(WM * WN == 4, "four wavefronts per workgroup");
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    constexpr int CHUNKS = SPLIT_K / (256 / BN) / 8;  // groups of 8 channels a thread loads per step
    static_assert(CHUNKS == 1 || CHUNKS == 2, "BN is 64 or 128");
    constexpr int RD = CHUNKS == 1 ? 2 : 1;  // steps whose pixels are in registers or on their way there
    __shared__ uintx4 Bs[2][3][SPLIT_K / 8][BN];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int m_tile, n_tile, local_tile, slice;
    bool split;
    trace_mark(p, 0);
    tile_of_block(p, m_tile, n_tile, local_tile, slice, split);
    const int step_lo = split ? slice * p.slice_steps : 0;
    const int step_hi = split ? min(step_lo + p.slice_steps, p.nsteps) : p.nsteps;
    const int m0 = m_tile * BM;
    const int n0 = n_tile * BN;
    TileChannel chan = NO_CHANNEL;
    if (!split) chan = fetch_channel_constants<BM>(p, m0, tid);

    const __amdgpu_buffer_rsrc_t rsrc_in = __builtin_amdgcn_make_buffer_rsrc((void *)p.I, 0, p.in_bytes, RSRC_WORD3);
    const __amdgpu_buffer_rsrc_t rsrc_in2 = __builtin_amdgcn_make_buffer_rsrc((void *)p.I2, 0, p.in_bytes, RSRC_WORD3);
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)p.Wp, 0, p.wp_bytes, RSRC_WORD3);

    // ---- this thread's pixel and its channels of a step: kgroup * 8 .. + 8 CHUNKS - 1
    const int pix = tid % BN;
    const int kgroup = __builtin_amdgcn_readfirstlane(tid / BN) * CHUNKS;
    int base, ih0, iw0;
    bool pvalid;
    {
        const int n = n0 + pix;
        pvalid = n < (int)p.npix;
        const unsigned nc = pvalid ? (unsigned)n : 0u, img = nc / (unsigned)p.PQ, pq = nc - img * (unsigned)p.PQ;
        const int op = (int)(pq / (unsigned)p.Q), oq = (int)pq - op * p.Q;
        base = (int)img * (p.Cimg * p.H * p.W);
        ih0 = op * p.sr - p.pt;
        iw0 = oq * p.sc - p.pl;
    }
    const int HW4 = p.H * p.W * 4, RS = p.R * p.S;
    const unsigned magic_h = split_magic(p.uh), magic_w = split_magic(p.uw);
    // the step whose pixels are loaded next
    int ld_c = step_lo / RS * SPLIT_K, ld_ky, ld_kx;
    {
        const int tap = step_lo - step_lo / RS * RS;
        ld_ky = tap / p.S;
        ld_kx = tap - ld_ky * p.S;
    }
    float raw[RD][CHUNKS][8];
    const int origin = (base + ih0 * p.W + iw0) * 4;  // (the window's first pixel, which may lie outside)
    const int only = split_pixel(p, magic_h, magic_w, pvalid, base, ih0, iw0, 0, 0);
    // (the channel counts of this form are multiples of 16, of each tensor's of 8: eight channels are one tensor's or nobody's)
    auto load_pixels = [&](int at, int chunk) __attribute__((always_inline)) {
        int voff = only;
        if constexpr (TAPS == UPSAMPLED) voff = split_pixel(p, magic_h, magic_w, pvalid, base, ih0, iw0, ld_ky, ld_kx);
        if constexpr (TAPS == STORED) {
            const bool ok = pvalid && (unsigned)(ih0 + ld_ky) < (unsigned)p.H && (unsigned)(iw0 + ld_kx) < (unsigned)p.W;
            voff = ok ? origin + (ld_ky * p.W + ld_kx) * 4 : OOB;
        }
        const int c0 = ld_c + (kgroup + chunk) * 8;
        const bool second = c0 >= p.Csplit;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(second ? p.I2 : p.I), 0, c0 < p.C ? p.in_bytes : 0u, RSRC_WORD3);
        int soff = (second ? c0 - p.Csplit : c0) * HW4;
#pragma unroll
        for (int j = 0; j < 8; j++, soff += HW4) raw[at][chunk][j] = buf_load(rsrc, voff, soff);
    };
    auto next_load_step = [&]() {
        // (selects: a branch would end the block that the matrix instructions are scheduled in; behind the last step the
        // channels run past the last and the loads bring zeros without touching memory)
        if constexpr (TAPS == ONE_TAP || TAPS == ROW_BIAS) {
            ld_c += SPLIT_K;
            return;
        }
        const int kx = ld_kx + 1, wrap_x = kx == p.S ? 1 : 0, ky = ld_ky + wrap_x, wrap_y = ky == p.R ? 1 : 0;
        ld_kx = wrap_x ? 0 : kx;
        ld_ky = wrap_y ? 0 : ky;
        ld_c += wrap_y ? SPLIT_K : 0;
    };
    uintx4 parts[CHUNKS][3];
    auto split_pixels = [&](int at, int chunk, int q) __attribute__((always_inline)) {  // pair q of the four
        unsigned h, m, l;
        split_pair(SPLIT_UP * raw[at][chunk][2 * q], SPLIT_UP * raw[at][chunk][2 * q + 1], h, m, l);
        parts[chunk][0][q] = h;
        parts[chunk][1][q] = m;
        parts[chunk][2][q] = l;
    };
    auto put_pixels = [&](int chunk, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int part = 0; part < 3; part++) Bs[buf][part][kgroup + chunk][pix] = parts[chunk][part];
    };

    // ---- filters: 3 x 16 bytes per lane, block and 16 channels
    const int mblocks = p.Mp / 32;
    const int a_voff = lane * 16 + (m0 / 32 + wm * TM) * SPLIT_UNIT;
    uintx4 a[2][TM][3];
    auto load_a = [&](int g, int step) __attribute__((always_inline)) {
        const int soff = (min(step, step_hi - 1) * 2 + g) * mblocks * SPLIT_UNIT;
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int part = 0; part < 3; part++)
                a[g][tm][part] = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, a_voff + tm * SPLIT_UNIT + part * 1024, soff, 0));
    };

    // hi hi is summed on its own (one rounding per 16 taps), the five small products in a second accumulator whose roundings are
    // 2^-8 of the first's; the two meet after the last step
    floatx16 acc[TM][TN], small[TM][TN];
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[tm][tn][v] = small[tm][tn][v] = 0.0f;

    uintx4 b[TN][3];
    auto read_b = [&](int part, int g, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int tn = 0; tn < TN; tn++) b[tn][part] = Bs[buf][part][2 * g + (lane >> 5)][wn * TN * 32 + tn * 32 + (lane & 31)];
    };
    constexpr int kA[6] = {0, 1, 2, 0, 1, 0}, kB[6] = {0, 0, 0, 1, 1, 2};
    auto multiply = [&](int g, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int tn = 0; tn < TN; tn++) {
                floatx16 &d = k == 0 ? acc[tm][tn] : small[tm][tn];
                d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[g][tm][kA[k]]), __builtin_bit_cast(bf16x8, b[tn][kB[k]]), d, 0, 0, 0);
            }
    };

#pragma unroll
    for (int i = 0; i < RD; i++) {
#pragma unroll
        for (int chunk = 0; chunk < CHUNKS; chunk++) load_pixels(i, chunk);
        next_load_step();
    }
    load_a(0, step_lo);
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; chunk++) {
#pragma unroll
        for (int q = 0; q < 4; q++) split_pixels(0, chunk, q);
        put_pixels(chunk, 0);
        load_pixels(0, chunk);
    }
    next_load_step();
    __syncthreads();
    trace_mark(p, 1);
    constexpr int T = TM * TN;
    if constexpr (CHUNKS == 1) {
        // Step t multiplies buffer t % 2, splits the pixels of step t + 1 into the other buffer and loads those of step t + 3.  (What the last steps
        // load - nothing behind the last channel, the next slice's first steps otherwise - is not used; without those loads slices took the
        // same time.)  Two things keep the matrix
        // pipe from waiting where a CU has one or two workgroups:
        //   * the six products take the parts of the pixels in turn, so the registers of a part take the next 16 channels' as soon as its
        //     last product has started, and the one barrier of a step stands where the first part of the next step is read, half
        //     a step behind the last write;
        //   * loads arrive in the order in which they were asked for, so a wait for filters waits for the pixels asked for before
        //     them: pixels are asked for right behind the filters of the next half step, which makes theirs a whole step.
        // 12 images, the loop below -> this: 256 3x3 on 14x14 58.7 -> 53.6 us (64x64 tile 49.9 -> 41.0), 128 3x3 stride 2 on 56x56 34.6 -> 31.0,
        // 1024 -> 256 on 14x14 26.9 -> 25.3; 64 images 256 3x3 on 14x14 94.8 -> 91.1, 1x1 layers within 1 %.  Slices of 5 ... 18 steps with more than one
        // workgroup on a CU are 1 - 4 % slower (512 3x3 on 28x28 of one image, 8 slices, 33.3 -> 34.0), from 32 steps on all are faster.
#pragma unroll
        for (int part = 0; part < 3; part++) read_b(part, 0, 0);
        auto whole_step = [&](int step, int s) __attribute__((always_inline)) {  // s: the step's place in the unrolled loop
            const int buf = (step - step_lo) & 1;
#pragma unroll
            for (int g = 0; g < 2; g++) {
                const int next_buf = g == 0 ? buf : buf ^ 1;
                load_a(g ^ 1, step + g);
                if (g == 0) {
#pragma unroll
                    for (int q = 0; q < 3; q++) split_pixels((s + 1) % RD, 0, q);
                    __builtin_amdgcn_sched_group_barrier(0x020, 3 * TM, 0);
                } else {
                    load_pixels((s + 1) % RD, 0);
                    next_load_step();
                    __builtin_amdgcn_sched_group_barrier(0x020, 3 * TM + 8, 0);
                }
#pragma unroll
                for (int k = 0; k < 3; k++) multiply(g, k);
                if (g == 0) split_issue_order<3 * T, 39>();
                __builtin_amdgcn_sched_barrier(0);
                if (g == 1) {
                    __syncthreads();
                    __builtin_amdgcn_sched_barrier(0);
                }
                read_b(0, g ^ 1, next_buf);
                __builtin_amdgcn_sched_barrier(0);
                if (g == 0) split_pixels((s + 1) % RD, 0, 3);
                multiply(g, 3);
                multiply(g, 4);
                if (g == 0) split_issue_order<2 * T, 13>();
                __builtin_amdgcn_sched_barrier(0);
                read_b(1, g ^ 1, next_buf);
                if (g == 0) put_pixels(0, buf ^ 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(g, 5);
                __builtin_amdgcn_sched_barrier(0);
                read_b(2, g ^ 1, next_buf);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int step = step_lo;
        for (; step + 2 <= step_hi; step += 2) {
            whole_step(step, 0);
            whole_step(step + 1, 1);
        }
        if (step < step_hi) whole_step(step, 0);
        __syncthreads();  // (the last reads, before the epilogue writes there)
    } else {
        // The same with a barrier at the end of a step and a chunk split in each half: more registers are not to be had, and the order
        // above without them is 2-6 % slower here.
        for (int step = step_lo; step < step_hi; step++) {
            const int buf = (step - step_lo) & 1;
#pragma unroll
            for (int g = 0; g < 2; g++) {
#pragma unroll
                for (int part = 0; part < 3; part++) read_b(part, g, buf);
                load_a(g ^ 1, step + g);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 6; k++) multiply(g, k);
#pragma unroll
                for (int q = 0; q < 4; q++) split_pixels(0, g, q);
                put_pixels(g, buf ^ 1);
                load_pixels(0, g);
                if (g == 1) next_load_step();
                // issue order: the splitting between the matrix instructions, then what it is for
                split_issue_order<6 * T, 72>();
                __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 8, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        }
    }
    trace_mark(p, 2);
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[tm][tn][v] = SPLIT_DOWN * __fadd_rn(acc[tm][tn][v], small[tm][tn][v]);

    float finite = 0.0f;
#pragma unroll
    for (int tm = 0; tm < TM; tm++)
#pragma unroll
        for (int tn = 0; tn < TN; tn++)
#pragma unroll
            for (int v = 0; v < 16; v++) finite = __builtin_fmaf(acc[tm][tn][v], 0.0f, finite);
    const int m_first = m0 + wm * TM * 32, n_first = n0 + wn * TN * 32;
    if (__any(finite != 0.0f)) {
        split_tile_again<TM, TN, SPLIT_K>(p, small, rsrc_in, rsrc_in2, m_first, n_first, step_lo, step_hi, lane);
#pragma unroll
        for (int tm = 0; tm < TM; tm++)
#pragma unroll
            for (int tn = 0; tn < TN; tn++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[tm][tn][v] = acc[tm][tn][v] * 0.0f == 0.0f ? acc[tm][tn][v] : small[tm][tn][v];
    }

    if (split) {
        store_partial<TM, TN>(p, acc, local_tile, slice, wave, lane);
    } else {
        float *epi = (float *)&Bs[0][0][0][0];  // the K loop ended with a barrier
        put_channel_constants<BM>(epi, chan, tid);
        __syncthreads();
        store_tile<TM, TN, BM, TAPS == ROW_BIAS, true>(p, acc, epi, m0, wm * TM * 32, n_first, lane);
    }
    if (p.trace != nullptr) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        trace_mark(p, 3);
    }
}
