// float32 GEMM for the projection operators' float32 compute dtype: the reference runs its
// projections through torch.mm / addmm in whatever compute dtype the model uses
// (kernels/linear.py:16-44, with TF32 off in train.py:80-82), so a float32 model needs
// every product of forward_linear, input_gradient and parameter_gradients in full fp32.
//
//   C[m, n] = op(A)[m, k] op(B)[k, n] (+ C when beta) (+ bias[n])
//
// op(A) is A stored [m, k] (trans_a = 0) or [k, m] (trans_a = 1); op(B) is B stored [k, n]
// (trans_b = 0) or [n, k] (trans_b = 1); leading dimensions are the stored row pitches.
// With beta = 0 the destination is never read (garbage or NaN there is ignored).
//
// Design: v_mfma_f32_16x16x4_f32 (full fp32 products and sums; no TF32 or reduced-
// precision step), bound by the matrix cores' fp32 rate (157 TFLOP/s at 2.4 GHz; rocBLAS's
// 8192^3 product reaches 154 on this card). Each operand keeps its stored order in LDS, so no
// register transposes are needed: [row][32 k] with the bf16 kernels' conflict-free 16-byte
// swizzle (slot()) when it is contiguous along k, [k][rows] with a column XOR when it is
// contiguous along its rows. Either way MFMA t of a 16-k slice takes k 4t .. 4t+3 in index
// order, through conflict-free ds_read_b32 (wider along B's rows). Three tiles by the size of
// the output (choose()):
//   128 x 128 and 64 x 64, 4 waves, two stages of 32 k, sums in one chain in index order;
//   32 x 32, 8 waves that split each 128-k stage between them and add their sums in LDS in a
//   fixed order: an adapter's products (1000 x 64 over 2048) give few tiles, and the split
//   reduction inside the workgroup keeps the chip busy without a workspace.
// Every output element is a fixed-order reduction, so results repeat bit for bit.

#include <type_traits>

#include "gemm_common.hpp"

namespace ct {
namespace {

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct F32Args {
    const float *a, *b, *bias;
    float *c;
    int64_t lda, ldb, ldc, m, n, k;
    int tiles_m, tiles_n, beta, vec_a, vec_b, vec_c;
};

// One operand's tile of a stage of KD * 32 reduction indices, ROWS rows, moved in 16-byte
// chunks that keep the stored order: KFAST, stored [rows, k], goes to [KD][ROWS][32 k] with
// tile row n at LDS row frag_row<FRAG>(n); otherwise stored [k, rows], it goes to
// [k][ROWS], columns XORed with shift(k). VEC: every chunk is one 16-byte load or none of it
// (aligned base, pitch and contiguous extent in multiples of 4). Otherwise `vec` says whether
// whole chunks may be loaded so; the rest go element by element.
template <int ROWS, int KD, int THREADS, bool KFAST, bool VEC, int FRAG>
struct Tile {
    static constexpr int kPer = ROWS * 8 * KD / THREADS;
    static_assert(kPer >= 1 && kPer * THREADS == ROWS * 8 * KD, "whole chunks per thread");
    f32x4 v[kPer];

    // Rows 4t .. 4t+3 of a [k][ROWS] tile start on distinct 16-bank groups under this XOR
    // (a row of 32 floats spans half the banks, so every second row moves).
    __device__ __forceinline__ static int shift(int k) { return ROWS >= 64 ? (k & 3) << 4 : (k & 2) << 3; }

    __device__ __forceinline__ static void place(int tid, int i, int &row, int &kk) {
        const int id = tid + i * THREADS;
        if constexpr (KFAST) {
            row = id / (8 * KD);
            kk = (id % (8 * KD)) * 4;
        } else {
            row = (id % (ROWS / 4)) * 4;
            kk = id / (ROWS / 4);
        }
    }
    __device__ __forceinline__ void load(const float *p, int64_t ld, int64_t r0, int64_t rows, int64_t k0,
                                         int64_t kdim, bool vec, int tid) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            int row, kk;
            place(tid, i, row, kk);
            const int64_t rg = r0 + row, kg = k0 + kk;
            const int64_t left = KFAST ? (rg < rows ? kdim - kg : 0) : (kg < kdim ? rows - rg : 0);
            const float *src = KFAST ? p + rg * ld + kg : p + kg * ld + rg;
            if constexpr (VEC) {
                v[i] = left > 0 ? *reinterpret_cast<const f32x4 *>(src) : f32x4{0.f, 0.f, 0.f, 0.f};
            } else if (vec && left >= 4) {
                v[i] = *reinterpret_cast<const f32x4 *>(src);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[i][j] = j < left ? src[j] : 0.f;
            }
        }
    }
    __device__ __forceinline__ void store(f32x4 *stage, int tid) const {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            int row, kk;
            place(tid, i, row, kk);
            if constexpr (KFAST) stage[(kk >> 5) * ROWS * 8 + slot(frag_row<FRAG>(row), (kk & 31) >> 2)] = v[i];
            else stage[(kk * ROWS + (row ^ shift(kk))) / 4] = v[i];
        }
    }
    // Fragment f (of FRAGS) of the 16 * FRAGS rows from w0, for MFMA t of slice `slice` (k 16
    // slice + 4t + lane / 16): rows w0 + 16 f + lane % 16 with FRAG = 1, else rows
    // w0 + FRAG (lane % 16) + f.
    template <int FRAGS>
    __device__ __forceinline__ static void fragments(const f32x4 *stage, int w0, int slice, int t, int lane,
                                                     float (&out)[FRAGS]) {
        const float *base = reinterpret_cast<const float *>(stage);
        const int g = lane >> 4, c = lane & 15;
        if constexpr (KFAST) {
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                out[f] = base[((slice >> 1) * ROWS * 8 + slot(w0 + f * 16 + c, (slice & 1) * 4 + t)) * 4 + g];
        } else if constexpr (FRAG == 1) {
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                out[f] = base[(16 * slice + 4 * t + g) * ROWS + ((w0 + f * 16 + c) ^ shift(g))];
        } else {
            typedef float vec __attribute__((ext_vector_type(FRAG)));
            const vec q = *reinterpret_cast<const vec *>(base + (16 * slice + 4 * t + g) * ROWS +
                                                         ((w0 + FRAG * c) ^ shift(g)));
#pragma unroll
            for (int f = 0; f < FRAGS; ++f) out[f] = q[f];
        }
    }
};

// Output columns col .. col + N - 1 of one row: + bias, + C when beta.
template <int N>
__device__ __forceinline__ void write_row(const F32Args &g, int64_t row, int64_t col, const float (&acc)[N]) {
    if (row >= g.m || col >= g.n) return;
    float *c = g.c + row * g.ldc + col;
    if (N > 1 && g.vec_c && col + N <= g.n) {
        typedef float vec __attribute__((ext_vector_type(N > 1 ? N : 2)));
        vec w;
#pragma unroll
        for (int j = 0; j < N; ++j) w[j] = acc[j] + (g.bias ? g.bias[col + j] : 0.f);
        if (g.beta) w = *reinterpret_cast<const vec *>(c) + w;
        *reinterpret_cast<vec *>(c) = w;
        return;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
        if (col + j >= g.n) break;
        const float v = acc[j] + (g.bias ? g.bias[col + j] : 0.f);
        c[j] = g.beta ? c[j] + v : v;
    }
}

// BM x BN tile; WAVES_M x WAVES_N waves over it, KW of them along the reduction: a stage
// holds KD * 32 reduction indices in 2 KD slices of 16, of which wave group w multiplies
// slices w * 2 KD / KW and on.
template <int BM, int BN, int WAVES_M, int WAVES_N, int KW, int KD, bool AK, bool BKF, bool VEC>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N * KW) __attribute__((amdgpu_waves_per_eu(2))) void gemm_f32(
    const F32Args g) {
    constexpr int THREADS = 64 * WAVES_M * WAVES_N * KW;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, FM = WM / 16, FN = WN / 16;
    constexpr int kSlices = 2 * KD / KW, kDepth = 32 * KD;
    constexpr int kStage = (BM + BN) * 8 * KD;  // 16-byte units
    static_assert(kSlices >= 1, "every wave group has a slice");
    static_assert(KW == 1 || (WAVES_M == 1 && WAVES_N == 1 && KW * BM * BN * 4 <= 2 * kStage * 16 &&
                              BM * BN % THREADS == 0),
                  "the groups' sums fit the stages");
    __shared__ f32x4 lds[2 * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int group = KW > 1 ? wave : 0;
    const int wm = KW > 1 ? 0 : (wave % WAVES_M) * WM, wn = KW > 1 ? 0 : (wave / WAVES_M) * WN;

    // Tile order: contiguous ranges per XCD, in groups of 8 row tiles that share B panels.
    constexpr int kXcds = 8, kGroupM = 8;
    const int tiles = g.tiles_m * g.tiles_n, xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
    const int per = (tiles + kXcds - 1) / kXcds, tall = tiles % kXcds == 0 ? kXcds : tiles % kXcds;
    const int rid = xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
    const int gm = g.tiles_m < kGroupM ? g.tiles_m : kGroupM;
    const int span = gm * g.tiles_n, first_m = rid / span * gm;
    const int gsize = g.tiles_m - first_m < gm ? g.tiles_m - first_m : gm;
    const int64_t m0 = (int64_t)(first_m + rid % span % gsize) * BM, n0 = (int64_t)(rid % span / gsize) * BN;

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // SETS register sets per operand: step s stores tile s + 1 to the other stage before its
    // products and loads tile s + 1 + SETS into the set that freed, so a load has SETS steps
    // to arrive. Two where registers allow it: the 128 x 128 tile would spill.
    constexpr int SETS = BM >= 128 ? 1 : 2;
    using TileA = Tile<BM, KD, THREADS, AK, VEC, 1>;
    using TileB = Tile<BN, KD, THREADS, BKF, VEC, FN>;
    TileA la[SETS];
    TileB lb[SETS];
    const int64_t steps = (g.k + kDepth - 1) / kDepth;
    const auto load = [&](auto set, int64_t s) {
        la[set].load(g.a, g.lda, m0, g.m, s * kDepth, g.k, g.vec_a, tid);
        lb[set].load(g.b, g.ldb, n0, g.n, s * kDepth, g.k, g.vec_b, tid);
    };
    const auto store = [&](auto set, int stage) {
        la[set].store(lds + stage * kStage, tid);
        lb[set].store(lds + stage * kStage + BM * 8 * KD, tid);
    };
    const auto step = [&](auto cur, int64_t s) {
        constexpr int nxt = decltype(cur)::value ^ 1;
        const std::integral_constant<int, nxt % SETS> set{};
        if (s + 1 < steps) store(set, nxt);
        if (s + 1 + SETS < steps) load(set, s + 1 + SETS);
        const f32x4 *sa = lds + decltype(cur)::value * kStage, *sb = sa + BM * 8 * KD;
#pragma unroll
        for (int q = 0; q < kSlices; ++q) {
            const int slice = group * kSlices + q;
            float af[4][FM], bf[4][FN];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                TileA::template fragments<FM>(sa, wm, slice, t, lane, af[t]);
                TileB::template fragments<FN>(sb, wn, slice, t, lane, bf[t]);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) acc[i][j] = mfma_f32(af[t][i], bf[t][j], acc[i][j]);
        }
        __syncthreads();
    };
    const std::integral_constant<int, 0> even{};
    const std::integral_constant<int, 1> odd{};
    if (steps > 0) {
        load(even, 0);
        if (SETS > 1 && steps > 1) load(std::integral_constant<int, SETS - 1>{}, 1);
        store(even, 0);
        if (steps > SETS) load(even, SETS);
        __syncthreads();
        int64_t s = 0;
        for (; s + 1 < steps; s += 2) {
            step(even, s);
            step(odd, s + 1);
        }
        if (s < steps) step(even, s);
    }

    // Lane l holds rows 4 (l / 16) + e of each 16-row block and, of the wave's columns,
    // FN (l % 16) + j.
    if constexpr (KW > 1) {
        float *sums = reinterpret_cast<float *>(lds);  // free: every wave has left the loop
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    sums[group * BM * BN + (i * 16 + (lane >> 4) * 4 + e) * BN + (lane & 15) * FN + j] = acc[i][j][e];
        __syncthreads();
#pragma unroll
        for (int o = 0; o < BM * BN / THREADS; ++o) {
            const int at = o * THREADS + tid;
            float v[1] = {sums[at]};
#pragma unroll
            for (int w = 1; w < KW; ++w) v[0] += sums[w * BM * BN + at];
            write_row<1>(g, m0 + at / BN, n0 + at % BN, v);
        }
    } else {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v[FN];
#pragma unroll
                for (int j = 0; j < FN; ++j) v[j] = acc[i][j][e];
                write_row<FN>(g, m0 + wm + i * 16 + (lane >> 4) * 4 + e, n0 + wn + (lane & 15) * FN, v);
            }
    }
}

enum Shape { LARGE, MEDIUM, SMALL };
constexpr int kEdge[3] = {128, 64, 32};

// 128 x 128 tiles once they give every CU a workgroup, 64 x 64 ones likewise, and the split
// 32 x 32 tile for everything smaller, unless the reduction fits one of its stages (nothing to
// split: 64 x 64 tiles, which also keep such sums in one chain). MI355X, one launch
// (trans_b = 1): 4096 x 4096 x 4096 1077 us, 1198 on 64 x 64 tiles (1243 with the previous
// 128 x 128 kernel of b32-staged 16-k slices); 1000 x 2048 x 2048 98, 109 on 32 x 32 (219);
// 1000 x 64 x 2048 17 us, 57 on 64 x 64 (215); 64 x 2048 x 1000 10 us, 29 (109).
Shape choose(int64_t m, int64_t n, int64_t k) {
    if (cdiv(m, 128) * cdiv(n, 128) >= 256) return LARGE;
    return cdiv(m, 64) * cdiv(n, 64) >= 256 || k <= 128 ? MEDIUM : SMALL;
}

template <bool AK, bool BKF, bool VEC>
void launch_shape(Shape shape, const F32Args &g, hipStream_t s) {
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n));
    if (shape == LARGE) gemm_f32<128, 128, 2, 2, 1, 1, AK, BKF, VEC><<<grid, dim3(256), 0, s>>>(g);
    else if (shape == MEDIUM) gemm_f32<64, 64, 2, 2, 1, 1, AK, BKF, VEC><<<grid, dim3(256), 0, s>>>(g);
    else gemm_f32<32, 32, 1, 1, 8, 4, AK, BKF, VEC><<<grid, dim3(512), 0, s>>>(g);
}

template <bool AK, bool BKF>
void launch_vec(Shape shape, bool vec, const F32Args &g, hipStream_t s) {
    if (vec) launch_shape<AK, BKF, true>(shape, g, s);
    else launch_shape<AK, BKF, false>(shape, g, s);
}

// 16-byte loads of an operand's whole chunks: aligned base and pitch in multiples of 4.
bool operand_vec(const float *p, int64_t ld) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % 4 == 0; }

}  // namespace
}  // namespace ct

extern "C" int ct_gemm_f32(const float *a, int64_t lda, int32_t trans_a, const float *b, int64_t ldb, int32_t trans_b,
                           float *c, int64_t ldc, int32_t beta, const float *bias, int64_t m, int64_t n, int64_t k,
                           hipStream_t stream) {
    using namespace ct;
    if (m < 0 || n < 0 || k < 0) return -CT_EINVAL_SHAPE;
    if (m == 0 || n == 0) return 0;
    if (!c || (k > 0 && (!a || !b))) return -CT_EINVAL_POINTER;
    const int64_t acols = trans_a ? m : k, bcols = trans_b ? k : n;
    if (ldc < n || (k > 0 && (lda < acols || ldb < bcols))) return -CT_EINVAL_SHAPE;
    F32Args g{};
    g.a = a, g.b = b, g.bias = bias, g.c = c;
    g.lda = lda, g.ldb = ldb, g.ldc = ldc, g.m = m, g.n = n, g.k = k;
    g.beta = beta != 0;
    g.vec_c = reinterpret_cast<uintptr_t>(c) % 16 == 0 && ldc % 4 == 0;
    const Shape shape = choose(m, n, k);
    const int64_t tm = cdiv(m, kEdge[shape]), tn = cdiv(n, kEdge[shape]);
    if (tm * tn > 0x7fffffff) return -CT_EINVAL_SHAPE;
    g.tiles_m = (int)tm;
    g.tiles_n = (int)tn;
    g.vec_a = operand_vec(a, lda);
    g.vec_b = operand_vec(b, ldb);
    // Both operands in whole chunks: the kernels without the per-chunk choice.
    const bool vec = g.vec_a && g.vec_b && acols % 4 == 0 && bcols % 4 == 0;
    if (trans_a && trans_b) launch_vec<false, true>(shape, vec, g, stream);
    else if (trans_a) launch_vec<false, false>(shape, vec, g, stream);
    else if (trans_b) launch_vec<true, true>(shape, vec, g, stream);
    else launch_vec<true, false>(shape, vec, g, stream);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;  // a positive HIP error code
}
