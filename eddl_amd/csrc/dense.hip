// Dense forward: C[m,n] (+)= A[m,k] * B[k,n], row-major fp32, B = W[in, out]
// (what LDense::forward asks of mult2D: src/layers/core/layer_dense.cpp:65-73).
//
// At the batch sizes of CNN heads (m = 32..64 rows against a 25088 x 4096 weight matrix) the
// product is bound by streaming B from HBM once.  One wavefront owns a 32-row x 128-column
// output block over a slice of k: per pair of k it loads ONE float4 of B per lane (lane l of a
// half wavefront covers columns 4l..4l+3: 512 contiguous bytes per k row) and one dword of the
// activations, and issues four v_mfma_f32_32x32x2_f32, one per column phase
// (accumulator j holds columns 4l + j).  Except for one row, or few with not too many weights (reads_rows), the
// activations are transposed first (At[k][32], a few MB, L2-resident) so that their loads are coalesced too.  k is split over wavefronts so the
// whole device streams B; the per-slice partial blocks go to the private workspace and a second
// kernel adds them in slice order (fixed summation order, no atomics).  More rows than 48 take the split form (split_rows).
#include <algorithm>

#include "common.h"

using namespace eddlhip;

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// A[m][k] -> At[mt][k][32] (mt = 32-row block), zero-padded rows
__global__ __launch_bounds__(256) void dense_transpose_kernel(const float *__restrict__ A, float *__restrict__ At, int m, int k) {
    __shared__ float tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int k0 = blockIdx.x * 32, mt = blockIdx.y;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = mt * 32 + ty + 8 * j, kk = k0 + tx;
        tile[ty + 8 * j][tx] = (r < m && kk < k) ? A[(size_t)r * k + kk] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int kk = k0 + ty + 8 * j;
        if (kk < k) At[((size_t)mt * k + kk) * 32 + tx] = tile[tx][ty + 8 * j];
    }
}

// grid: (column tiles of 128, k slices, groups of MT row tiles of 32); block: one wavefront, which multiplies every
// float4 of weights it loads into MT accumulator sets: one pass over B serves MT x 32 rows (a batch of up to 128 rows
// reads the weights once; the activations, transposed, are small and come from L2).
// VEC: n is a multiple of 4 and B is 16-byte aligned, so a lane's four columns are one float4.
// STREAM (with VEC): the weights are read with the streaming (non-temporal) hint - for matrices larger than
// the device's caches, which no later kernel finds there anyway (25088 x 4096: 96 -> 88 us).
// DIRECT (one row tile): At is A[m][k] itself and a lane reads its row where it stands, so there is no transposed copy to make;
// lanes of rows past m read the last row again (their results are not stored).  The same products and sums, bit for bit.
template <bool VEC, bool STREAM, int MT, bool DIRECT = false>
__global__ __launch_bounds__(64) void dense_partial_kernel(const float *__restrict__ At, const float *__restrict__ B,
                                                           float *__restrict__ part, int m, int k, int n, int kslice) {
    const int lane = threadIdx.x, half = lane >> 5, l = lane & 31;
    const int n0 = blockIdx.x * 128, ks = blockIdx.y, mt0 = blockIdx.z * MT;
    const int kbeg = ks * kslice;
    int kend = kbeg + kslice;
    if (kend > k) kend = k;
    const int col0 = n0 + 4 * l;
    const int mtiles = (m + 31) / 32;
    // row tile mt0 + t of this group, or the last existing one again (its results are not stored)
    const float *ap[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) ap[t] = DIRECT ? At + (size_t)(l < m ? l : m - 1) * k : At + (size_t)(mt0 + t < mtiles ? mt0 + t : mtiles - 1) * k * 32 + l;
    constexpr size_t A_STEP = DIRECT ? 1 : 32;  // floats from one tap of a row to the next
    floatx16 acc[MT][4];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[t][j][v] = 0.0f;
    auto load_b = [&](int ki) -> floatx4 {
        floatx4 b = {0.0f, 0.0f, 0.0f, 0.0f};
        if (ki < kend) {
            const float *row = B + (size_t)ki * n;
            if (VEC) {
                if (col0 < n) b = *reinterpret_cast<const floatx4 *>(row + col0);
            } else {
                if (col0 + 0 < n) b.x = row[col0 + 0];
                if (col0 + 1 < n) b.y = row[col0 + 1];
                if (col0 + 2 < n) b.z = row[col0 + 2];
                if (col0 + 3 < n) b.w = row[col0 + 3];
            }
        }
        return b;
    };
    auto multiply = [&](const float (&a)[MT], const floatx4 &b) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < MT; t++) {
            acc[t][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b.x, acc[t][0], 0, 0, 0);
            acc[t][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b.y, acc[t][1], 0, 0, 0);
            acc[t][2] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b.z, acc[t][2], 0, 0, 0);
            acc[t][3] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b.w, acc[t][3], 0, 0, 0);
        }
    };
    constexpr int U = MT == 1 ? 8 : 4;  // k pairs (float4 of weights per lane) in flight
    int kk = kbeg;
    for (; kk + 2 * U <= kend; kk += 2 * U) {
        float a[U][MT];
        floatx4 b[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int ki = kk + 2 * u + half;
#pragma unroll
            for (int t = 0; t < MT; t++) a[u][t] = ap[t][(size_t)ki * A_STEP];
            const float *row = B + (size_t)ki * n;
            if (VEC) {
                const floatx4 *src = reinterpret_cast<const floatx4 *>(row + col0);
                b[u] = col0 < n ? (STREAM ? __builtin_nontemporal_load(src) : *src) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            } else {
                b[u] = load_b(ki);
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) multiply(a[u], b[u]);
    }
    for (; kk < kend; kk += 2) {
        const int ki = kk + half;
        float a[MT];
#pragma unroll
        for (int t = 0; t < MT; t++) a[t] = ki < kend ? ap[t][(size_t)ki * A_STEP] : 0.0f;
        multiply(a, load_b(ki));
    }
    // part[ks][row][col]: accumulator j, lane column l -> column col0 + j; rows 8*(v/4) + 4*half + v%4
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int r = (mt0 + t) * 32 + 8 * (v / 4) + 4 * half + (v % 4);
            if (r < m) {
                float *dst = part + ((size_t)ks * m + r) * n + col0;
                if (VEC) {
                    if (col0 < n) *reinterpret_cast<floatx4 *>(dst) = floatx4{acc[t][0][v], acc[t][1][v], acc[t][2][v], acc[t][3][v]};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (col0 + j < n) dst[j] = acc[t][j][v];
                }
            }
        }
}

// Adds the K slices in slice order; then, in the reference's order, C += (incC), + bias[column]
// (sum2D_rowwise) and ReLU - each an fp32 operation of its own, so the fused tail equals the
// separate launches bit for bit.
__global__ __launch_bounds__(256) void dense_reduce_kernel(const float *__restrict__ part, float *C, size_t mn, int nslices,
                                                           int incC, const float *__restrict__ bias, int n, int relu) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256;
    for (size_t t = i; t < mn; t += stride) {
        // eight slices' loads in flight at a time; the additions keep the slice order
        float s = part[t];
        int ks = 1;
        for (; ks + 8 <= nslices; ks += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = part[(size_t)(ks + u) * mn + t];
#pragma unroll
            for (int u = 0; u < 8; u++) s = __fadd_rn(s, v[u]);
        }
        for (; ks < nslices; ks++) s = __fadd_rn(s, part[(size_t)ks * mn + t]);
        if (incC) s = __fadd_rn(C[t], s);
        if (bias) s = __fadd_rn(s, bias[t % (size_t)n]);
        if (relu) s = s > 0.0f ? s : 0.0f;
        C[t] = s;
    }
}

}  // namespace

namespace {

// Whether a product reads the activations where they are instead of from a transposed copy.  The copy is a launch of its own,
// 2 to 6 us.  In place a lane reads its own row, a cache line a row and not one for 32, and the wavefronts beside it read those
// lines again while they stream the weights: the more rows and the more weights, the less of that the caches hold.  Measured over
// 29 matrices of 512 .. 25088 x 128 .. 25088, the weights from memory (us, in place against the copy): one row is faster in place
// everywhere (4096 x 1000 14.8 against 17.5, 25088 x 4096 81.8 against 83.2).  More rows are up to 17 M weights, whatever the
// shape (32 rows: 4096 x 4096 26.4 against 28.9, 16384 x 1000 30.0 against 35.3; 6144 x 2048 alone 27.2 against 26.7).  At 25 M
// up to 16 rows are (eight: 4096 x 6144 31.1 against 33.5, 25088 x 1000 40.0 against 43.0; sixteen 33.5 against 34.8, 45.2 against
// 44.2) and 32 are not (43.7 against 38.2); from 34 M on only one row is (8192 x 4096: two rows 38.8 against 39.8, eight 42.9
// against 41.4, 32 58.9 against 47.5).
bool reads_rows(int m, int k, int n) { return m == 1 || (m <= 32 && (size_t)k * n <= (size_t)(m <= 16 ? 28 : 20) << 20); }

// Many rows are bound by the fp32 matrix instruction as much as by the weights, and take the split form of a convolution (dense_split) where that
// can run it: whole groups of 16 inputs.  us, before -> after: 64 rows 25088 x 4096 159 -> 116, 4096 x 4096 39.3 -> 28.8, 4096 x 1000 26.4
// -> 18.2, 512 x 10 22.3 -> 11.3; 128 rows 297 -> 171, 63.6 -> 37.2, 37.1 -> 21.6, 33.6 -> 12.4; error against 64 bits 3.7e-7 -> 2.4e-7 ... 3.3e-7,
// 1.8e-7 -> 1.0e-7, 1.6e-7 -> 9.7e-8.
// The line at 48 rows is not where the times cross: 33 to 48 rows would gain as much (48 rows 37.7 -> 28.7; up to 32 the weights are streamed no
// faster, 25088 x 4096 110 against 112).  It is a choice for calls of varying row counts: up to 48 rows (and, in the fp32 product, up to 128) a row has the
// same bits in every batch, which the split form's tiles and K slices end.
// Few columns under a long sum have few tiles, which the K slices do not make enough of, and the rows cost more to split than to multiply: the fp32
// product from 4 M row elements or 16 K inputs on, up to 256 columns (us, fp32 against split: 256 rows 25088 x 10 60.7 against 66.1, 256 rows 50176 x 64 76
// against 119, 768 rows 12544 x 100 55 against 68, 1024 rows 16384 x 128 80 against 84; below it 512 rows 8192 x 10 1.26 times as fast in the split form,
// 256 rows 12544 x 64 1.08, beyond it 384 columns 0.93 ... 1.6, 1000 columns 1.2 ... 1.9).
bool split_rows(int m, int k, int n) { return m > 48 && (n > 256 || (k <= 16384 && (long long)m * k <= 1LL << 22)); }

int dense_impl(int dev, const float *A, const float *B, float *C, int m, int k, int n, int incC, const float *bias, int relu,
               const char *what) {
    EH_REQUIRE(m >= 0 && k > 0 && n > 0, "%s: bad shape %dx%d * %dx%d", what, m, k, k, n);
    if (m == 0) return 0;
    EH_REQUIRE(A && B && C, "%s: NULL tensor", what);
    EH_TRY(use_device(dev));
    hipStream_t st = state(dev).stream;
    if (split_rows(m, k, n)) {
        bool taken = false;
        EH_TRY(dense_split(dev, A, B, C, m, k, n, incC, bias, relu, &taken));
        if (taken) return 0;
    }
    const int nt = (n + 127) / 128, mt = (m + 31) / 32;
    // Wavefronts to cover the device eight times over, in slices of at least 128 taps (shorter
    // slices cost more in partial blocks written and read back than they gain) - unless that
    // leaves fewer than four wavefronts per CU, when slices go down to 64 taps.
    const int MT = mt >= 3 ? 4 : mt;  // row tiles one wavefront serves with each float4 of weights it loads
    const int mgroups = (mt + MT - 1) / MT;
    const long long blocks = (long long)nt * mgroups;
    const long long num_cu = state(dev).num_cu;
    long long nsl = (8 * num_cu + blocks - 1) / blocks;
    const long long max128 = (k + 127) / 128, max64 = (k + 63) / 64;
    if (nsl > max128) nsl = std::max(max128, std::min((4 * num_cu + blocks - 1) / blocks, max64));
    int nslices = (int)std::max(1LL, nsl);
    int kslice = ((k + nslices - 1) / nslices + 1) & ~1;  // even, so MFMA tap pairs do not straddle slices
    nslices = (k + kslice - 1) / kslice;
    EH_REQUIRE(nslices <= 65535 && mgroups <= 65535, "%s: shape out of range", what);
    const bool direct = reads_rows(m, k, n);
    const size_t at_bytes = direct ? 0 : ((size_t)mt * k * 32 * sizeof(float) + 255) & ~(size_t)255;
    void *ws = nullptr;
    EH_TRY(get_workspace(dev, at_bytes + (size_t)nslices * m * n * sizeof(float), &ws));
    float *At = (float *)ws, *part = (float *)((char *)ws + at_bytes);
    if (!direct) {
        hipLaunchKernelGGL(dense_transpose_kernel, dim3((k + 31) / 32, mt), dim3(256), 0, st, A, At, m, k);
        EH_CHECK_LAUNCH();
    }
    const bool vec = (n % 4 == 0) && (((uintptr_t)B & 15u) == 0);
    const bool stream = vec && (size_t)k * n * sizeof(float) > ((size_t)256 << 20);  // beyond the 256 MB last-level cache
    typedef void (*partial_fn)(const float *, const float *, float *, int, int, int, int);
    static const partial_fn kernels[4][3] = {
        {dense_partial_kernel<false, false, 1>, dense_partial_kernel<true, false, 1>, dense_partial_kernel<true, true, 1>},
        {dense_partial_kernel<false, false, 2>, dense_partial_kernel<true, false, 2>, dense_partial_kernel<true, true, 2>},
        {dense_partial_kernel<false, false, 4>, dense_partial_kernel<true, false, 4>, dense_partial_kernel<true, true, 4>},
        {dense_partial_kernel<false, false, 1, true>, dense_partial_kernel<true, false, 1, true>, dense_partial_kernel<true, true, 1, true>}};
    const partial_fn kern = kernels[direct ? 3 : MT == 1 ? 0 : MT == 2 ? 1 : 2][!vec ? 0 : (stream ? 2 : 1)];
    hipLaunchKernelGGL(kern, dim3(nt, nslices, mgroups), dim3(64), 0, st, direct ? A : (const float *)At, B, part, m, k, n, kslice);
    EH_CHECK_LAUNCH();
    size_t mn = (size_t)m * n;
    hipLaunchKernelGGL(dense_reduce_kernel, dim3(eh_blocks(mn, 256, 65536)), dim3(256), 0, st, (const float *)part, C, mn, nslices, incC,
                       bias, n, relu);
    EH_CHECK_LAUNCH();
    return 0;
}

}  // namespace

extern "C" int eddlhip_mult2d(int dev, const float *A, const float *B, float *C, int m, int k, int n, int incC) {
    return dense_impl(dev, A, B, C, m, k, n, incC, nullptr, 0, "mult2d");
}

extern "C" int eddlhip_dense_fwd(int dev, const float *A, const float *W, const float *bias, float *C, int m, int k, int n, int relu) {
    return dense_impl(dev, A, W, C, m, k, n, 0, bias, relu, "dense_fwd");
}
