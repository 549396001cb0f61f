// The one-launch Winograd form F(2x2, 3x3) on the bf16 matrix instructions (included by conv.hip only).  Loop order, tiles and
// output transform are wino_fused_kernel's, the arithmetic of the products is conv_split.h's: the transformed pixels V = B^T d B
// are computed in fp32 by the same operations, enlarged 2^24 times and split exactly into three bf16 numbers by the lane that
// multiplies them; the filters are transformed in 64 bits and split once per registered filter tensor (an error in U is the same in
// every pixel of a plane: rounded to fp32 as in the other Winograd forms it is what remains of theirs in a plane's mean).  The six largest of the nine products
// of two such sums are added to fp32 accumulators, the smallest first: six roundings per 16 channels where the fp32 instruction
// (two channels each) makes eight.  That instruction rounds what it shifts out on the way to an accumulator downwards, not to
// nearest, and several times on the way (a product at a time or a few): in an accumulator of a long sum that costs more than the
// eight roundings of the fp32 instruction.  Two things keep the form more accurate than the fp32 one-launch kernel all the same:
//   * The positions (i, 1) of a patch, where pixels of one sign add up and whose sums are the largest by far behind a ReLU, have their
//     six products of a step summed from zero and added to the long sum by vector instructions: one rounding to nearest per 16 channels.
//   * The error that remains has one sign.  Position (i, 2) is accumulated with the opposite sign, so are the position rows 1 and 3,
//     and so is every other block (2x2 outputs) of a plane: what is left in an output is a small fraction of its rounding, and
//     the means of planes, which no pool and no later layer would average away, hold none of it.
// Error against 64 bits on the inputs that the layers of the networks have, relative to the outputs' root mean square, of the fp32 one-launch kernel -> of
// this one (in brackets with all products in one accumulator): 64 channels 1.5e-7 -> 1.1e-7 (1.4e-7), 128 2.0e-7 -> 1.1e-7 (1.9e-7), 256
// 2.5e-7 -> 1.4e-7 (2.7e-7), 512 3.4e-7 -> 1.6e-7 (3.6e-7), 1024 4.8e-7 -> 2.3e-7 (5.2e-7); of the mean of a plane: 64 channels on 56x56
// 4.6e-8 -> 4e-9, 256 on 14x14 6.0e-8 -> 1.6e-8, 512 on 7x7 9.5e-8 -> 4.4e-8.  On normally distributed pixels 2.6e-7 -> 1.8e-7 (64 channels).
// Sums that are not finite - infinities and NaN, and with the
// enlargement numbers from 2^104 and sums from 2^80 on - are computed with the fp32 instruction too and take that value.

// K[Kf][C][3][3] -> Ws[c / 16][Mp / 32][position][part][lane][8]: the transformed filters U = G g G^T, in 64 bits, as
// operands of the matrix instruction: lane l holds filter l % 32 of the block, channels 8 (l / 32) .. + 7 of the 16.
// C is a multiple of 16; filters past Kf are zeros.  Bound by the write (96 bytes per filter and channel).
__global__ __launch_bounds__(256) void wino_split_filter_kernel(const float *__restrict__ K, uintx4 *__restrict__ Ws, int Kf, int C, int mblocks, int k16s) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)k16s * mblocks * 64) return;
    const int lane = (int)(idx & 63);
    const int unit = (int)(idx >> 6), mb = unit % mblocks, k16 = unit / mblocks;
    const int c0 = k16 * 16 + (lane >> 5) * 8, m = mb * 32 + (lane & 31);
    uintx4 *dst = Ws + (size_t)unit * (16 * 192) + lane;
#pragma unroll 1
    for (int i = 0; i < 4; i++) {  // a position row at a time: 4 x 8 values
        double u[8][4];
#pragma unroll
        for (int ch = 0; ch < 8; ch++) {
            double g[9], t[3];
#pragma unroll
            for (int e = 0; e < 9; e++) g[e] = m < Kf ? (double)SPLIT_UP * (double)K[((size_t)m * C + c0 + ch) * 9 + e] : 0.0;
#pragma unroll
            for (int j = 0; j < 3; j++) t[j] = i == 0 ? g[j] : (i == 3 ? g[6 + j] : 0.5 * ((i == 1 ? g[j] + g[3 + j] : g[j] - g[3 + j]) + g[6 + j]));
            u[ch][0] = t[0];
            u[ch][1] = 0.5 * (t[0] + t[1] + t[2]);
            u[ch][2] = 0.5 * (t[0] - t[1] + t[2]);
            u[ch][3] = t[2];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uintx4 hi, mid, lo;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                unsigned h, md, l;
                split_pair(u[2 * q][j], u[2 * q + 1][j], h, md, l);
                hi[q] = h;
                mid[q] = md;
                lo[q] = l;
            }
            dst[(4 * i + j) * 192] = hi;
            dst[(4 * i + j) * 192 + 64] = mid;
            dst[(4 * i + j) * 192 + 128] = lo;
        }
    }
}

constexpr int WSPLIT_UNIT = 16 * SPLIT_UNIT;  // bytes of 32 filters x 16 channels, all positions

// One 32x32 block of one position's sums once more with the fp32 instruction (see split_tile_again), channels [c_lo, c_hi), from
// the image and the original filters: this lane's filter m and block n, patch position (i, j).
__device__ __forceinline__ void wino_block_again(const ConvParams &p, floatx16 &sum, __amdgpu_buffer_rsrc_t in1, __amdgpu_buffer_rsrc_t in2, int m, int n, int i, int j,
                                                 int c_lo, int c_hi, int half) {
    const int per_img = p.wth * p.wtw, HW4 = p.H * p.W * 4;
    const bool nok = n < p.wT;
    const int nc = nok ? n : 0, img = nc / per_img, r = nc - img * per_img, ty = r / p.wtw, tx = r - ty * p.wtw;
    const int base = img * (p.Cimg * p.H * p.W), y0 = 2 * ty - p.pt, x0 = 2 * tx - p.pl;
    const unsigned magic_h = split_magic(p.uh), magic_w = split_magic(p.uw);
    const int ra = i == 0 ? 0 : (i == 2 ? 2 : 1), rb = i == 0 ? 2 : (i == 1 ? 2 : (i == 2 ? 1 : 3));
    const int ca = j == 0 ? 0 : (j == 2 ? 2 : 1), cb = j == 0 ? 2 : (j == 1 ? 2 : (j == 2 ? 1 : 3));
    const float si = i == 1 ? 1.0f : -1.0f, sj = j == 1 ? 1.0f : -1.0f;
    int off[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) off[a][b] = split_pixel(p, magic_h, magic_w, nok, base, y0, x0, a ? rb : ra, b ? cb : ca);
#pragma unroll
    for (int v = 0; v < 16; v++) sum[v] = 0.0f;
#pragma unroll 1
    for (int c0 = c_lo; c0 < c_hi; c0 += 2) {
        const int c = c0 + half;
        const bool second = c >= p.Csplit;
        const int coff = (second ? c - p.Csplit : c) * HW4;
        float d[2][2], t[3];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const int o = off[a][b] == OOB ? OOB : off[a][b] + coff;
                const float f1 = buf_load(in1, second ? OOB : o, 0), f2 = buf_load(in2, second ? o : OOB, 0);
                d[a][b] = second ? f2 : f1;
            }
        const float vv = __builtin_fmaf(__builtin_fmaf(d[1][1], si, d[0][1]), sj, __builtin_fmaf(d[1][0], si, d[0][0]));
        const float *g = p.K + ((size_t)(m < p.Kf ? m : 0) * p.C + c) * 9;
#pragma unroll
        for (int x = 0; x < 3; x++) {
            const float a0 = g[x], a1 = g[3 + x], a2 = g[6 + x];
            t[x] = i == 0 ? a0 : (i == 3 ? a2 : __fmul_rn(0.5f, __fadd_rn(i == 1 ? __fadd_rn(a0, a1) : __fsub_rn(a0, a1), a2)));
        }
        const float uu = j == 0 ? t[0] : (j == 3 ? t[2] : __fmul_rn(0.5f, __fadd_rn(j == 1 ? __fadd_rn(t[0], t[1]) : __fsub_rn(t[0], t[1]), t[2])));
        sum = __builtin_amdgcn_mfma_f32_32x32x2f32(m < p.Kf ? uu : 0.0f, vv, sum, 0, 0, 0);
    }
}

// A workgroup owns 64 filters x 32 blocks (2x2 outputs) and keeps the accumulators of all 16 positions, wavefront i those of
// position row i (8 blocks of 32x32: 128 registers).  A K-step is 16 channels, one matrix instruction deep:
//   * the load unit writes the step's raw pixels into LDS, every pixel once, in the segments of wino_fused_kernel (there for the
//     layout), two steps ahead;
//   * a lane reads the two patch rows of its block and position row for its eight channels, forms the four operands and
//     splits them (64 vector instructions per pair of channels).  Positions 0 and 1 of step t + 1 are made during the matrix
//     instructions of positions 2 and 3 of step t, positions 2 and 3 are split during those of 0 and 1: that keeps 48 operand
//     and 16 intermediate registers alive instead of 96;
//   * a step is eight groups of six products (a position and 32 filters).  Position 1's alternate with position 0's: the sum of
//     a group is added to the long one while the next group multiplies, so that 16 registers hold it and nothing waits for it;
//   * filters go from L2 straight to registers (a fragment is one wavefront's alone), two groups ahead, each part into
//     the place of the one that has been multiplied last.
// Why this tile: filters are used for 32 blocks only (192 KB per step and two workgroups, 64 bytes a cycle and CU if the matrix
// pipe never waited, which is what L2 delivers: 138 GB/s per CU measured, 100 where 25 MB of filters come from the last-level
// cache), but two independent workgroups share a CU and cover each other's latencies, prologue and epilogue.  Tried: 64 filters x 64
// blocks on eight wavefronts (half the filter traffic, one workgroup per CU): level on 512 channels, 17-25 % slower on 64 and 128;
// the same on sixteen wavefronts with one position each: 1.5 times the time.
// Bound: neither pipe is full. VGG-16's nine launches of the wide build at batch 32 keep the matrix pipe busy 36 % of the cycles, at 2.2 GHz (power:
// 2.4 with operands of zeros); a wavefront issues 38 % of its cycles, 13 vector instructions per memory instruction, and waits for memory or LDS 28 %; the
// vector L1 holds requests back 35 % of a CU's cycles.  Without filter loads a quarter of the time goes, without pixel loads a tenth.  Narrow build (planes 14
// wide): 26 %, 34 % and 31 %; each step's pixels are four times as many load instructions, and its 62 scalar values beyond the register file lie in
// vector registers (no scratch).  Batch 32, us, wino_fused_kernel -> this one: conv 64->64 on 224x224 541
// -> 495, 128->128 on 112x112 492 -> 410, 256->256 on 56x56 462 -> 368, 512->512 on 28x28 462 -> 363, on 14x14 151 -> 129; 64->64 on
// 512x512, batch 4, 359 -> 328; ResNet-50's at batch 64: 77 -> 65, 73 -> 61, 84 -> 70.
template <bool WIDE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void wino_split_kernel(const ConvParams p) {
    constexpr int FM = 2, MF = 32 * FM, NB = 32, CK = 16, SLOTS = 16 * NB;
    constexpr int R_FLOATS = CK * SLOTS;
    __shared__ __attribute__((aligned(16))) float lds[2 * R_FLOATS];
    __shared__ __attribute__((aligned(16))) float epi[EPI_ROWS * MF];
    static_assert(2 * R_FLOATS >= FM * 4 * 2 * 16 * 64, "the exchange of the filter groups");

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int m_tile, n_tile, local_tile, slice;
    bool split;
    trace_mark(p, 0);
    tile_of_block(p, m_tile, n_tile, local_tile, slice, split);
    const int m0 = m_tile * MF, n0 = n_tile * NB;
    const int step_lo = split ? slice * p.slice_steps : 0;
    const int step_hi = split ? min(step_lo + p.slice_steps, p.nsteps) : p.nsteps;

    // ---- filters: 16 bytes per lane, part and 32 filters
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc((void *)p.Wp, 0, p.wp_bytes, RSRC_WORD3);
    const int a_voff = lane * 16;
    const int a_base = (m0 / 32) * WSPLIT_UNIT + 4 * wave * SPLIT_UNIT, a_step = p.Mp / 32 * WSPLIT_UNIT;
    constexpr int GROUPS = 4 * FM, kPos[GROUPS] = {1, 0, 1, 0, 2, 2, 3, 3}, kFm[GROUPS] = {0, 0, 1, 1, 0, 1, 0, 1};  // a step's groups of products
    uintx4 a[2][3];  // of this group and the next
    auto load_a = [&](int part, int step, int i) __attribute__((always_inline)) {
        a[i & 1][part] = __builtin_bit_cast(
            uintx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, a_voff + part * 1024, a_base + step * a_step + kFm[i] * WSPLIT_UNIT + kPos[i] * SPLIT_UNIT, 0));
    };

    // ---- where the tile's pixels go in LDS and this lane's patch lies there (wino_fused_kernel; a wavefront loads one or two groups of 64 slots)
    constexpr int KG = WIDE ? SLOTS / 256 : 4;     // WIDE: slot group wave % KG of channels CPW (wave / KG) ..; else groups wave, wave + 4 of all
    constexpr int WLC = WIDE ? 1 : SLOTS / 64 / 4;
    constexpr int CPW = WIDE ? CK * KG / 4 : CK;
    const int my_k = wave % KG, my_c = wave / KG * CPW;
    const int per_img = p.wth * p.wtw;
    int voff[WLC], my_base = WIDE ? 1 : 0, my_stride = 0, my_odd = 0;  // (my_odd: the parity of this lane's block in its plane)
#pragma unroll
    for (int k = 0; k < WLC; k++) voff[k] = OOB;
    {
        const int n_end = min(n0 + NB, p.wT);
        const unsigned Hu = (unsigned)(p.H * p.uh), Wu = (unsigned)(p.W * p.uw);
        const int img_elems = p.Cimg * p.H * p.W;
        const bool whole = p.uh == 1 && p.uw == 1;
        int base = 0;
        for (int seg_n = n0; seg_n < n_end;) {
            const int row = seg_n / p.wtw, tx0 = seg_n - row * p.wtw;
            const int cnt = min(p.wtw - tx0, n_end - seg_n), width = 2 * cnt + 2;
            const int img = row / p.wth, ty = row - img * p.wth;
            const int y0 = 2 * ty - p.pt, x0 = 2 * tx0 - p.pl, gbase = img * img_elems;
            const int xs = WIDE ? ((x0 + 4) & ~3) - 4 : x0, shift = x0 - xs;
            const int gpr = WIDE ? (shift + width + 3) >> 2 : width, gb = WIDE ? base >> 2 : base;  // groups (slots) per pixel row
#pragma unroll
            for (int k = 0; k < WLC; k++) {
                const int local = (my_k + k * KG) * 64 + lane - gb;
                const int r = (local >= gpr ? 1 : 0) + (local >= 2 * gpr ? 1 : 0) + (local >= 3 * gpr ? 1 : 0);
                const unsigned y = (unsigned)(y0 + r), x = (unsigned)(xs + (WIDE ? 4 : 1) * (local - r * gpr));
                const bool ok = (unsigned)local < (unsigned)(4 * gpr) && y < Hu && x < Wu;
                int off;
                if (WIDE || whole) off = (gbase + (int)y * p.W + (int)x) * 4;
                else off = (gbase + (int)(y / (unsigned)p.uh) * p.W + (int)(x / (unsigned)p.uw)) * 4;
                voff[k] = ok ? off : voff[k];
            }
            {
                const int n = n0 + l32;
                if (n >= seg_n && n < seg_n + cnt) my_base = base + shift + 2 * (n - seg_n), my_stride = WIDE ? 4 * gpr : width, my_odd = (ty + tx0 + n - seg_n) & 1;
            }
            base += WIDE ? 16 * gpr : 4 * width;
            seg_n += cnt;
        }
    }
    const int HW4 = p.H * p.W * 4;
    const int32x4 dma_in = make_rsrc_words(p.I, p.in_bytes), dma_in2 = make_rsrc_words(p.I2, p.in_bytes);
    auto rs_of = [&](int buf) { return (lds_float *)&lds[buf * R_FLOATS]; };
    // (no branch: it would end the block that the matrix instructions are scheduled in; past the last step zeros arrive)
    auto load_step = [&](int want, lds_float *rs) __attribute__((always_inline)) {
        const int step = min(want, step_hi - 1);
        // (a folded Concat's tensors have multiples of eight channels: eight of a step are one tensor's, not always all sixteen)
#pragma unroll
        for (int c8 = 0; c8 < CPW; c8 += 8) {
            const int first = step * CK + my_c + c8;
            const bool second = first >= p.Csplit;
            const int32x4 dma = second ? dma_in2 : dma_in;
            const int c0 = first - (second ? p.Csplit : 0);
#pragma unroll
            for (int k = 0; k < WLC; k++) {
                const int at = want < step_hi ? voff[k] : OOB;
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    if constexpr (WIDE) lds_dma_b128(dma, rs + (my_c + c8 + c) * SLOTS + my_k * 256, at, (c0 + c) * HW4);
                    else lds_dma_b32(dma, rs + (my_c + c8 + c) * SLOTS + (my_k + KG * k) * 64, at, (c0 + c) * HW4);
                }
            }
        }
    };
    load_step(step_lo, rs_of(0));
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int part = 2; part >= 0; part--) load_a(part, step_lo, i);
    if (!split) stage_channel_constants<MF>(p, epi, m0, tid);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    load_step(step_lo + 1, rs_of(1));
    trace_mark(p, 1);

    floatx16 acc[4][FM];  // (position 1's are sum1)
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int fm = 0; fm < FM; fm++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[j][fm][v] = 0.0f;
    float sum1[FM][16];
#pragma unroll
    for (int fm = 0; fm < FM; fm++)
#pragma unroll
        for (int v = 0; v < 16; v++) sum1[fm][v] = 0.0f;

    const int ra = wave == 0 ? 0 : (wave == 2 ? 2 : 1), rb = wave == 0 ? 2 : (wave == 1 ? 2 : (wave == 2 ? 1 : 3));
    const float sgn = wave == 1 ? 1.0f : -1.0f;
    const int ra_off = half * 8 * SLOTS + my_base + ra * my_stride, rb_off = half * 8 * SLOTS + my_base + rb * my_stride;
    typedef const __attribute__((address_space(3))) floatx2 *lds_f2;
    uintx4 b[4][3];
    const float up = ((wave ^ my_odd) & 1) != 0 ? -SPLIT_UP : SPLIT_UP;  // (position 2 has the other sign)
    float v2[8], v3[8];  // positions 2 and 3, from the turn of 0 and 1 to their own
    float d[2][2][4];           // [channel of a pair][patch row][column]
    auto read_pair = [&](const lds_float *rs, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const lds_float *pp[2] = {rs + ra_off + (2 * q + e) * SLOTS, rs + rb_off + (2 * q + e) * SLOTS};
#pragma unroll
            for (int r = 0; r < 2; r++) {
                if constexpr (WIDE) {  // a patch starts at an odd slot
                    const floatx2 mid = *(lds_f2)(pp[r] + 1);
                    d[e][r][0] = pp[r][0], d[e][r][1] = mid.x, d[e][r][2] = mid.y, d[e][r][3] = pp[r][3];
                } else {
                    const floatx2 lo = *(lds_f2)pp[r], hi = *(lds_f2)(pp[r] + 2);
                    d[e][r][0] = lo.x, d[e][r][1] = lo.y, d[e][r][2] = hi.x, d[e][r][3] = hi.y;
                }
            }
        }
    };
    auto put = [&](int j, int q, float v0, float v1) __attribute__((always_inline)) {
        unsigned h, m, l;
        split_pair(v0, v1, h, m, l);
        b[j][0][q] = h;
        b[j][1][q] = m;
        b[j][2][q] = l;
    };
    // positions 0 and 1 of a pair of channels: u0 - u2, u1 + u2 (and 2 and 3: -(u2 - u1), u1 - u3)
    auto first = [&](int q) __attribute__((always_inline)) {
        float v[2][2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            float u[4];
#pragma unroll
            for (int c = 0; c < 4; c++) u[c] = __builtin_fmaf(d[e][1][c], sgn, d[e][0][c]);
            const float s1 = up * u[1], s2 = up * u[2];
            v[0][e] = __builtin_fmaf(up, u[0], -s2);
            v[1][e] = __fadd_rn(s1, s2);
            v2[2 * q + e] = __fsub_rn(s1, s2);
            v3[2 * q + e] = __builtin_fmaf(-up, u[3], s1);
        }
        put(0, q, v[0][0], v[0][1]);
        put(1, q, v[1][0], v[1][1]);
    };
    auto second = [&](int q) __attribute__((always_inline)) {
        put(2, q, v2[2 * q], v2[2 * q + 1]);
        put(3, q, v3[2 * q], v3[2 * q + 1]);
    };
    constexpr int kA[6] = {2, 1, 1, 0, 0, 0}, kB[6] = {0, 1, 0, 2, 1, 0};
    floatx16 own;  // position 1's products of one step and 32 filters
    auto multiply = [&](int i, int k) __attribute__((always_inline)) {  // product k of group i, the filters' smallest parts first
        const floatx16 zero = {0.0f};
        floatx16 &sum = kPos[i] == 1 ? own : acc[kPos[i]][kFm[i]];
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i & 1][kA[k]]), __builtin_bit_cast(bf16x8, b[kPos[i]][kB[k]]), kPos[i] == 1 && k == 0 ? zero : sum,
                                                      0, 0, 0);
    };
    read_pair(rs_of(0), 0);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        first(q);
        if (q < 3) read_pair(rs_of(0), q + 1);
    }
    for (int step = step_lo; step < step_hi; step++) {
        const int cur = (step - step_lo) & 1;
        const int next = step + 1 < step_hi ? step + 1 : step;
        const lds_float *rs = rs_of(cur ^ 1);
#pragma unroll
        for (int i = 0; i < GROUPS; i++) {
            if (i == GROUPS / 2) {
                // The next step's pixels were requested a step ago; of what was requested since then only the filters of
                // this group and the next may still be on their way.  Behind the barrier nobody reads this step's pixels any more.
                __builtin_amdgcn_s_waitcnt(0x0F70 | 6);
                __syncthreads();
                load_step(step + 2, rs_of(cur));
                __builtin_amdgcn_sched_barrier(0);
                read_pair(rs, 0);
            }
            const int q = i & 3;
#pragma unroll
            for (int k = 0; k < 6; k++) multiply(i, k);
            if (i < GROUPS / 2) {
                second(q);
                if (i & 1) {
#pragma unroll
                    for (int v = 0; v < 16; v++) sum1[kFm[i]][v] = __fadd_rn(sum1[kFm[i]][v], own[v]);
                }
            } else {
                first(q);
                if (q < 3) read_pair(rs, q + 1);
            }
            const int in = (i + 2) % GROUPS, js = i + 2 < GROUPS ? step : next;
            load_a(2, js, in), load_a(1, js, in), load_a(0, js, in);
#pragma unroll
            for (int t = 0; t < 6; t++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i >= GROUPS / 2) __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                else if (i & 1) __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
                else __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                if (i >= GROUPS / 2 && q < 3 && (t == 1 || t == 2)) __builtin_amdgcn_sched_group_barrier(0x100, WIDE ? 6 : 4, 0);
                if (t == 1 || t == 3) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    const float down = up * (SPLIT_DOWN / SPLIT_UP);
    trace_mark(p, 2);

    // ---- output transform: along the position row in registers, across the rows through LDS
    const size_t plane = (size_t)p.wP * p.wQ;
    // (the lane's number once more, so that nothing that follows from it lives through the loop: registers)
    const unsigned lane_again = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int lane_e = (int)lane_again, l32_e = lane_e & 31, half_e = lane_e >> 5;
    const bool pair = (p.wQ % 2 == 0) && (((size_t)p.O | (size_t)(p.residual ? p.residual : p.O)) % 8 == 0);
    floatx4 *xch = reinterpret_cast<floatx4 *>(&lds[0]);  // [filter group][position row][b][v / 4][lane_e] of v % 4
    __builtin_amdgcn_s_waitcnt(0x0F70);                    // (the zeros behind the last step)
    __syncthreads();
    float finite = 0.0f;
#pragma unroll
    for (int fm = 0; fm < FM; fm++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            floatx4 t[2];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float m[4];
#pragma unroll
                for (int j = 0; j < 4; j++) m[j] = (j == 2 ? -down : down) * (j == 1 ? sum1[fm][4 * q + k] : acc[j][fm][4 * q + k]);  // (the sums are 2^48 times too large)
                t[0][k] = __fadd_rn(__fadd_rn(m[0], m[1]), m[2]);
                t[1][k] = __fsub_rn(__fsub_rn(m[1], m[2]), m[3]);
                finite = __builtin_fmaf(t[0][k], 0.0f, finite);
                finite = __builtin_fmaf(t[1][k], 0.0f, finite);
            }
#pragma unroll
            for (int b2 = 0; b2 < 2; b2++) xch[(((fm * 4 + wave) * 2 + b2) * 4 + q) * 64 + lane_e] = t[b2];
        }
    if (__any(finite != 0.0f)) {
        const __amdgpu_buffer_rsrc_t in1 = __builtin_amdgcn_make_buffer_rsrc((void *)p.I, 0, p.in_bytes, RSRC_WORD3);
        const __amdgpu_buffer_rsrc_t in2 = __builtin_amdgcn_make_buffer_rsrc((void *)p.I2, 0, p.in_bytes, RSRC_WORD3);
#pragma unroll 1
        for (int fm = 0; fm < FM; fm++) {
            floatx16 t0 = {0.0f}, t1 = {0.0f};
#pragma unroll 1
            for (int j = 0; j < 4; j++) {
                floatx16 sum;
                wino_block_again(p, sum, in1, in2, m0 + fm * 32 + l32_e, n0 + l32_e, wave, j, step_lo * CK, step_hi * CK, half_e);
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float x0 = j == 0 ? acc[0][0][v] : (j == 1 ? sum1[0][v] : (j == 2 ? acc[2][0][v] : acc[3][0][v]));
                    const float x1 = j == 0 ? acc[0][1][v] : (j == 1 ? sum1[1][v] : (j == 2 ? acc[2][1][v] : acc[3][1][v]));
                    const float x = (j == 2 ? -down : down) * (fm == 0 ? x0 : x1), m = x * 0.0f == 0.0f ? x : sum[v];
                    t0[v] = j == 0 ? m : (j == 3 ? t0[v] : __fadd_rn(t0[v], m));
                    t1[v] = j == 1 ? m : __fsub_rn(t1[v], m);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                xch[(((fm * 4 + wave) * 2 + 0) * 4 + q) * 64 + lane_e] = (floatx4){t0[4 * q], t0[4 * q + 1], t0[4 * q + 2], t0[4 * q + 3]};
                xch[(((fm * 4 + wave) * 2 + 1) * 4 + q) * 64 + lane_e] = (floatx4){t1[4 * q], t1[4 * q + 1], t1[4 * q + 2], t1[4 * q + 3]};
            }
        }
    }
    __syncthreads();
    const int n = n0 + l32_e;
    const int nc = n < p.wT ? n : 0;
    const int img = nc / per_img, r = nc - img * per_img, ty = r / p.wtw, tx = r - ty * p.wtw;
#pragma unroll
    for (int fm = 0; fm < FM; fm++) {
        float yk[4][2][2];  // [k][a][b]: output (2 ty + a, 2 tx + b) of filter row 8 wave + 4 half_e + k of the block
#pragma unroll
        for (int b2 = 0; b2 < 2; b2++) {
            floatx4 t[4];
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = xch[(((fm * 4 + i) * 2 + b2) * 4 + wave) * 64 + lane_e];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                yk[k][0][b2] = __fadd_rn(__fadd_rn(t[0][k], t[1][k]), t[2][k]);
                yk[k][1][b2] = __fsub_rn(__fsub_rn(t[1][k], t[2][k]), t[3][k]);
            }
        }
        const int ml0 = fm * 32 + 8 * wave + 4 * half_e;
        if (split) {
            const size_t tiles = (gridDim.x - (unsigned)p.main_tiles) / p.nslices;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                floatx4 *dst = reinterpret_cast<floatx4 *>(p.partial) + (((((size_t)slice * tiles + local_tile) * FM + fm) * 4 + wave) * 4 + k) * 64 + lane_e;
                floatx4 yv;
                yv.x = yk[k][0][0], yv.y = yk[k][0][1], yv.z = yk[k][1][0], yv.w = yk[k][1][1];
                *dst = yv;
            }
        } else if (n < p.wT) {
            if (pair && 2 * ty + 1 < p.wP && 2 * tx + 1 < p.wQ && m0 + ml0 + 3 < p.Kf) {
                wino_store_rows<MF, 4>(p, epi, ml0, m0 + ml0, img, ty, tx, plane, yk);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    wino_store_row(p, channel_from_lds<MF>(epi, ml0 + k), m0 + ml0 + k, img, ty, tx, plane, pair, yk[k][0][0], yk[k][0][1], yk[k][1][0], yk[k][1][1]);
            }
        }
    }
    if (p.trace != nullptr) {
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        trace_mark(p, 3);
    }
}
