// backward.hip — backward pass of the MoE layer and its load-balancing loss.
//
// The reference has neither: its block backward (src/transformer.c:975-1013)
// skips the FFN/MoE half, and the auxiliary loss exists only as the comment
// aux = n_experts * sum_e f_e * P_e (src/transformer.c:280-282).  Here, for
// the layer of src/transformer.c:287-366 with the routing held as the
// forward decided it, the gradients of L = sum(dout * out) + aux_coef * aux
// (f_e = assignments to e / (T k), a count; P_e = mean_t probs[t][e]):
//
//   recompute  G, U = x W_g, x W_u (rows in dispatch order), H = silu(G) U,
//              Y = H W_d
//   slots      dgw = <Y, dout[t]>, dY = gw dout[t]
//   experts    dH = dY W_d^T, dG = dH U silu'(G), dU = dH silu(G),
//              dXr = dG W_g^T + dU W_u^T; dW_d = H^T dY, dW_g = X^T dG,
//              dW_u = X^T dU over each expert's rows
//   router     gw = p_sel / S: dp_sel = (dgw - <dgw, gw>) / S; dp += aux_coef
//              E f / T; dlogits = p (dp - <dp, p>); dW_r = X^T dlogits
//   dx         = sum over the token's slots of dXr + dlogits W_r^T
//
// The row products run on the forward's grouped GEMMs (gemm_split.hip), the
// weight gradients on reduce_split_kernel (the reduction over an expert's
// rows); shapes they do not tile on the fp32 rows_mfma, rows_gemm and
// reduce_gemm kernels.  Every sum runs in a fixed order (deterministic).
#include "gemm_split.h"
#include "moe_internal.h"
#include "moe_math.h"

namespace moe {
namespace {

constexpr int kRM = 128, kRN = 64, kRK = 16;   // rows_gemm tile
constexpr int kQM = 64, kQN = 64, kQR = 16;    // reduce_gemm tile

// C[pos][n] (+)= sum_kk A(pos, kk) B_e(kk, n) for the rows pos of each
// 128-row tile (expert e).  A(pos, kk) = a[arow * lda + kk] with arow =
// perm[pos] / topk (GATHER) or pos; B_e(kk, n) = b[e * b_e + kk * ldb + n]
// or, BT, b[e * b_e + n * ldb + kk].  Thread (tr, tc) = (tid / 16, tid % 16)
// owns rows 8tr .. 8tr + 7 and columns 4tc .. 4tc + 3; K slices of 16 in LDS.
struct RowsGemm {
    const float *a;
    int lda;
    const int *perm;
    int topk;
    const float *b;
    size_t b_e;
    int ldb;
    float *c;
    int ldc;
    const int *offsets, *tile_off, *tile_expert;
    int E, K, N, max_mtiles, accumulate;
};

template <bool GATHER, bool BT>
__global__ __launch_bounds__(256) void rows_gemm_kernel(RowsGemm g) {
    __shared__ __align__(16) float As[kRK][kRM + 4];
    __shared__ __align__(16) float Bs[kRK][kRN + 4];
    const int ntn = (g.N + kRN - 1) / kRN;
    const int nt = blockIdx.x % ntn, mtg = blockIdx.x / ntn;
    if (mtg >= g.tile_off[g.E]) return;
    const int e = g.tile_expert[mtg];
    const int row0 = g.offsets[e] + (mtg - g.tile_off[e]) * kRM;
    const int rows = min(kRM, g.offsets[e + 1] - row0);
    const int n0 = nt * kRN;
    const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15;

    const float *arow[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = min((tid >> 2) + 64 * i, rows - 1);
        const size_t src = GATHER ? (size_t)(g.perm[row0 + r] / g.topk) : (size_t)(row0 + r);
        arow[i] = g.a + src * g.lda + 4 * (tid & 3);
    }
    const float *bb = g.b + (size_t)e * g.b_e;
    float acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < g.K; k0 += kRK) {
        float4 av[2], bv;
#pragma unroll
        for (int i = 0; i < 2; ++i) av[i] = *reinterpret_cast<const float4 *>(arow[i] + k0);
        int bk, bn;
        if (!BT) {   // 16 k rows x 16 column quads
            bk = tid >> 4;
            bn = 4 * (tid & 15);
            const bool in = n0 + bn < g.N;
            bv = masked4(in, *reinterpret_cast<const float4 *>(bb + (size_t)(k0 + bk) * g.ldb +
                                                              (in ? n0 + bn : 0)));
        } else {     // 64 columns x 4 k quads
            bn = tid >> 2;
            bk = 4 * (tid & 3);
            const bool in = n0 + bn < g.N;
            bv = masked4(in, *reinterpret_cast<const float4 *>(bb + (size_t)(in ? n0 + bn : 0) * g.ldb +
                                                              k0 + bk));
        }
        __syncthreads();   // the previous slice is consumed
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = (tid >> 2) + 64 * i, kq = 4 * (tid & 3);
            As[kq][r] = av[i].x;
            As[kq + 1][r] = av[i].y;
            As[kq + 2][r] = av[i].z;
            As[kq + 3][r] = av[i].w;
        }
        if (!BT) {
            *reinterpret_cast<float4 *>(&Bs[bk][bn]) = bv;
        } else {
            Bs[bk][bn] = bv.x;
            Bs[bk + 1][bn] = bv.y;
            Bs[bk + 2][bn] = bv.z;
            Bs[bk + 3][bn] = bv.w;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kRK; ++kk) {
            const float4 a0 = *reinterpret_cast<const float4 *>(&As[kk][8 * tr]);
            const float4 a1 = *reinterpret_cast<const float4 *>(&As[kk][8 * tr + 4]);
            const float4 b4 = *reinterpret_cast<const float4 *>(&Bs[kk][4 * tc]);
            const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            const float b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
    }
    const int n = n0 + 4 * tc;
    if (n >= g.N) return;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = 8 * tr + i;
        if (r >= rows) break;
        float4 *cp = reinterpret_cast<float4 *>(g.c + (size_t)(row0 + r) * g.ldc + n);
        float4 v = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
        if (g.accumulate) {
            const float4 o = *cp;
            v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
        }
        *cp = v;
    }
}

// The same product on the matrix cores (v_mfma_f32_32x32x2f32): a 128 x 64
// tile per workgroup of two waves, wave w rows 64w .. 64w + 63 and all 64
// columns (2 x 2 blocks of 32 x 32).  K slices of 32 sit in LDS with K
// contiguous per row (As) and per column (Bs); lane (li, lh) = (l % 32,
// l / 32) feeds k = 16 lh + 4q + s of MFMA (q, s), as in the forward's
// grouped GEMM.  The next slice is loaded into registers while the MFMAs
// of this one run.
typedef float fx4 __attribute__((ext_vector_type(4)));
typedef float fx16 __attribute__((ext_vector_type(16)));
constexpr int kMK = 32, kMLd = kMK + 4;

template <bool GATHER, bool BT>
__global__ __launch_bounds__(128) void rows_mfma_kernel(RowsGemm g) {
    __shared__ __align__(16) float As[kRM][kMLd];
    __shared__ __align__(16) float Bs[kRN][kMLd];
    const int ntn = (g.N + kRN - 1) / kRN;
    const int nt = blockIdx.x % ntn, mtg = blockIdx.x / ntn;
    if (mtg >= g.tile_off[g.E]) return;
    const int e = g.tile_expert[mtg];
    const int row0 = g.offsets[e] + (mtg - g.tile_off[e]) * kRM;
    const int rows = min(kRM, g.offsets[e + 1] - row0);
    const int n0 = nt * kRN;
    const int tid = threadIdx.x, lane = tid & 63, wm = tid >> 6;
    const int li = lane & 31, lh = lane >> 5;
    const fx4 zero = {0.f, 0.f, 0.f, 0.f};

    // A: 128 rows x 8 k-quads = 1024 float4s, 8 per thread.
    const float *asrc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = tid + 128 * i, r = min(q >> 3, rows - 1);
        const size_t src = GATHER ? (size_t)(g.perm[row0 + r] / g.topk) : (size_t)(row0 + r);
        asrc[i] = g.a + src * g.lda + 4 * (q & 7);
    }
    const float *bb = g.b + (size_t)e * g.b_e;
    fx4 ra[8], rb[4];
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ra[i] = *reinterpret_cast<const fx4 *>(asrc[i] + k0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = tid + 128 * i;
            if (BT) {   // 64 columns x 8 k-quads
                const int n = n0 + (q >> 3);
                rb[i] = n < g.N ? *reinterpret_cast<const fx4 *>(bb + (size_t)n * g.ldb + k0 +
                                                                   4 * (q & 7))
                                : zero;
            } else {    // 32 k rows x 16 column quads
                const int n = n0 + 4 * (q & 15);
                rb[i] = n < g.N ? *reinterpret_cast<const fx4 *>(bb + (size_t)(k0 + (q >> 4)) *
                                                                           g.ldb + n)
                                : zero;
            }
        }
    };
    auto sstore = [&]() {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int q = tid + 128 * i;
            *reinterpret_cast<fx4 *>(&As[q >> 3][4 * (q & 7)]) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = tid + 128 * i;
            if (BT) {
                *reinterpret_cast<fx4 *>(&Bs[q >> 3][4 * (q & 7)]) = rb[i];
            } else {
                const int k = q >> 4, n = 4 * (q & 15);
                Bs[n][k] = rb[i][0];
                Bs[n + 1][k] = rb[i][1];
                Bs[n + 2][k] = rb[i][2];
                Bs[n + 3][k] = rb[i][3];
            }
        }
    };
    fx16 acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
    const int nk = g.K / kMK;
    gload(0);
    for (int kt = 0; kt < nk; ++kt) {
        if (kt > 0) __syncthreads();   // this slice's LDS is free
        sstore();
        __syncthreads();
        if (kt + 1 < nk) gload((kt + 1) * kMK);
        const float *as = &As[wm * 64 + li][16 * lh];
        const float *bs = &Bs[li][16 * lh];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const fx4 a0 = *reinterpret_cast<const fx4 *>(as + 4 * q);
            const fx4 a1 = *reinterpret_cast<const fx4 *>(as + 32 * kMLd + 4 * q);
            const fx4 b0 = *reinterpret_cast<const fx4 *>(bs + 4 * q);
            const fx4 b1 = *reinterpret_cast<const fx4 *>(bs + 32 * kMLd + 4 * q);
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s2], b0[s2], acc[0][0], 0, 0, 0);
                acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s2], b1[s2], acc[0][1], 0, 0, 0);
                acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s2], b0[s2], acc[1][0], 0, 0, 0);
                acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s2], b1[s2], acc[1][1], 0, 0, 0);
            }
        }
    }
    // Block (m, n), register r: row 8 (r / 4) + 4 lh + r % 4, column li.
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = wm * 64 + m * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
            if (row >= rows) continue;
            float *cr = g.c + (size_t)(row0 + row) * g.ldc;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int col = n0 + n * 32 + li;
                if (col < g.N) cr[col] = g.accumulate ? cr[col] + acc[m][n][r] : acc[m][n][r];
            }
        }
}

// C_e[m][n] (+)= sum over the rows pos of group e (offsets[e] ..
// offsets[e + 1], or 0 .. nrows without offsets) of A(pos, m) B(pos, n),
// A(pos, m) = a[arow * lda + m] (arow = perm[pos] / topk with GATHER),
// B(pos, n) = b[pos * ldb + n].  Thread (tm, tn) = (tid / 16, tid % 16)
// owns rows 4tm .. and columns 4tn .. of the 64 x 64 tile (blockIdx.y,
// blockIdx.x) of group blockIdx.z; rows in slices of 16 through LDS.
struct ReduceGemm {
    const float *a;
    int lda;
    const int *perm;
    int topk;
    const float *b;
    int ldb;
    float *c;
    size_t c_e;
    int ldc;
    const int *offsets;
    int nrows, chunk, M, N, accumulate, vec_a, vec_b;
    // reduce_split_kernel only: N runs over [G | U]'s 2F packed columns and
    // column n's product goes to c (gate, n % 64 < 32) or c_up (up) at
    // feature 32 (n / 64) + n % 32.
    float *c_up = nullptr;
};

template <bool GATHER>
__global__ __launch_bounds__(256) void reduce_gemm_kernel(ReduceGemm g) {
    __shared__ __align__(16) float As[kQR][kQM + 4];
    __shared__ __align__(16) float Bs[kQR][kQN + 4];
    // Groups: the experts' row ranges, or (no offsets) chunks of nrows rows
    // of `chunk` each, whose partials go to C + z * c_e.
    const int e = blockIdx.z, m0 = blockIdx.y * kQM, n0 = blockIdx.x * kQN;
    const int r0 = g.offsets ? g.offsets[e] : e * g.chunk;
    const int r1 = g.offsets ? g.offsets[e + 1] : min(g.nrows, (e + 1) * g.chunk);
    const int tid = threadIdx.x, tm = tid >> 4, tn = tid & 15;
    const int lr = tid >> 4, lq = 4 * (tid & 15);   // load row and column quad
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int r = r0; r < r1; r += kQR) {
        const int row = r + lr;
        const bool in = row < r1;
        float av[4], bv[4];
        const size_t arow = in ? (GATHER ? (size_t)(g.perm[row] / g.topk) : (size_t)row) : 0;
        if (g.vec_a && in && m0 + lq < g.M) {   // (M, lda multiples of 4)
            const float4 v = *reinterpret_cast<const float4 *>(g.a + arow * g.lda + m0 + lq);
            av[0] = v.x; av[1] = v.y; av[2] = v.z; av[3] = v.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                av[j] = in && m0 + lq + j < g.M ? g.a[arow * g.lda + m0 + lq + j] : 0.f;
        }
        if (g.vec_b && in && n0 + lq < g.N) {   // (N, ldb multiples of 4)
            const float4 v = *reinterpret_cast<const float4 *>(g.b + (size_t)row * g.ldb + n0 + lq);
            bv[0] = v.x; bv[1] = v.y; bv[2] = v.z; bv[3] = v.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                bv[j] = in && n0 + lq + j < g.N ? g.b[(size_t)row * g.ldb + n0 + lq + j] : 0.f;
        }
        __syncthreads();
        *reinterpret_cast<float4 *>(&As[lr][lq]) = make_float4(av[0], av[1], av[2], av[3]);
        *reinterpret_cast<float4 *>(&Bs[lr][lq]) = make_float4(bv[0], bv[1], bv[2], bv[3]);
        __syncthreads();
#pragma unroll
        for (int rr = 0; rr < kQR; ++rr) {
            const float4 a4 = *reinterpret_cast<const float4 *>(&As[rr][4 * tm]);
            const float4 b4 = *reinterpret_cast<const float4 *>(&Bs[rr][4 * tn]);
            const float a[4] = {a4.x, a4.y, a4.z, a4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
    }
    float *ce = g.c + (size_t)e * g.c_e;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + 4 * tm + i;
        if (m >= g.M) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + 4 * tn + j;
            if (n >= g.N) break;
            float *cp = ce + (size_t)m * g.ldc + n;
            *cp = g.accumulate ? *cp + acc[i][j] : acc[i][j];
        }
    }
}

// The same product on the bf16 matrix cores with split operands
// (gemm_split.h), for M, N multiples of 64 WM and 64 WN over the experts' row
// ranges: a 64 WM x 64 WN tile per workgroup, 2 x 2 waves of (32 WM) x
// (32 WN).  The reduction runs over rows, so an operand piece is eight rows
// of one column: per step of 16 rows a wave loads eight rows of 64 columns of
// A and of B (one column per lane), splits them and stores them as three
// planes in MFMA operand order (two LDS stages, one barrier per step).  Rows
// are loaded kRedAhead steps ahead: a step is 0.3-0.4 us of MFMAs, a load
// from memory 1-2 us (one step ahead the 128 x 128 tiles of T = 4096, d = 256,
// F = 1024 took 118 us instead of 85).  The gathered rows' perm entries come a
// step earlier still, one per lane.
// KG = 2: two such groups of four waves take the steps in turn and the second
// group's sums are added to the first's at the end: for grids of one tile per
// CU, where four waves leave the splitting, the LDS traffic and the MFMAs of a
// step one after another (dW_g, dW_u 76 -> 71 us, dW_d 59 -> 46 there; with
// four tiles per CU, d = 512, F = 2048, it costs 5 %).
// Bound by the MFMAs, the splitting and the LDS traffic about equally: d =
// 512, F = 2048, 1024 rows per expert: dW_g, dW_u 235 us (146 TFLOP/s), dW_d
// 113; on the fp32 MFMAs 348 and 169.
constexpr int kRedAhead = 4;

// SHORT: loads wholly past the expert's range are left out.  With few rows
// most of the first five are, and a load costs the same there (the gathered
// ones wait for perm one after another).  Up to kRedShortRows rows per expert
// on average; where most loads are in range the branches cost more.  Whole
// backward, us without and with: 6 rows (T = 71, d = 192, F = 128, E = 12,
// top-3) 96.5, 93.0; 12 (T = 200, d = 1024, F = 512, E = 64, top-4) 593, 587;
// 14 (T = 210, d = 320, F = 256, E = 15) 126.9, 119.0; 31 665.7, 664.1; 62 775.8,
// 783.9.
constexpr int kRedShortRows = 32;

template <bool GATHER, int WM, int WN, int KG, bool SHORT>
__global__ __launch_bounds__(256 * KG, 2) void reduce_split_kernel(ReduceGemm g, unsigned topk_magic,
                                                                unsigned topk_one) {
    using namespace split;
    constexpr int PLANE_A = 64 * WM * 32, PLANE_B = 64 * WN * 32;   // bytes of a plane (16 rows)
    constexpr int STAGE = 3 * (PLANE_A + PLANE_B), D = kRedAhead;
    constexpr int SR = 16 * KG;   // rows from one step of a group to its next
    static_assert(KG == 1 || 4 * STAGE >= WM * WN * 16384, "LDS for the second group's sums");
    __shared__ __align__(16) char smem_all[2 * STAGE * KG];
    const int e = blockIdx.z, m0 = blockIdx.y * 64 * WM, n0 = blockIdx.x * 64 * WN;
    const int r0 = g.offsets[e], r1 = g.offsets[e + 1];
    const int lane = threadIdx.x & 63, wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = wave8 & 3, kg = wave8 >> 2;
    char *smem = smem_all + 2 * STAGE * kg;
    const int wm = wave >> 1, wn = wave & 1, li = lane & 31, lh = lane >> 5;
    // What the wave stages: rows 8 half .. of each step, one 64-column group
    // of A and of B (with 64 columns in all, two waves hold the same group
    // and one of them stores it).
    const int half = wave & 1, grp = wave >> 1;
    const bool own_a = WM == 2 || grp == 0, own_b = WN == 2 || grp == (WM == 2 ? 0 : 1);
    const float *pa = g.a + m0 + (WM == 2 ? 64 * grp : 0);   // (uniform)
    const float *pb = g.b + n0 + (WN == 2 ? 64 * grp : 0);

    float ra[D][8], rb[D][8];
    int pix = 0;                         // lane i: perm entry of row i of the next load
    auto token = [&](int p) -> size_t {  // perm / topk
        return __umulhi((unsigned)p, topk_magic) + ((unsigned)p & topk_one);
    };
    auto load_pix = [&](int r) {
        if (GATHER) pix = g.perm[min(r + 8 * half + (lane & 7), r1 - 1)];
    };
    // Rows past the range read its last row.
    auto load = [&](auto set, int r) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = min(r + 8 * half + i, r1 - 1);
            const size_t ar = GATHER ? token(__builtin_amdgcn_readlane(pix, i)) : (size_t)row;
            const float *qa = pa + ar * g.lda, *qb = pb + (size_t)row * g.ldb;
            ra[S][i] = qa[(unsigned)lane];
            rb[S][i] = qb[(unsigned)lane];
        }
        load_pix(r + SR);
    };
    auto load_in = [&](auto set, int r) {
        constexpr int S = decltype(set)::value;
        if (!SHORT || r < r1) load(set, r);
        else
#pragma unroll
            for (int i = 0; i < 8; ++i) ra[S][i] = rb[S][i] = 0.f;
    };
    // Mask: rows past the range count as zeros.
    auto store = [&](auto set, auto mask, int buf, int r) {
        constexpr int S = decltype(set)::value;
        if constexpr (decltype(mask)::value)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool in = r + 8 * half + i < r1;
                ra[S][i] = in ? ra[S][i] : 0.f;
                rb[S][i] = in ? rb[S][i] : 0.f;
            }
        // Column c of a group: its 32-column block's KB, 16 bytes at c % 32
        // of the half.
        char *w = smem + buf * STAGE + (lane >> 5) * 1024 + 512 * half + 16 * li;
        auto put = [&](const float (&v)[8], char *q, int plane) {
            const Frag f = split8(fx4{v[0], v[1], v[2], v[3]}, fx4{v[4], v[5], v[6], v[7]});
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<ux4 *>(q + p * plane) = f.t[p];
        };
        if (own_a) put(ra[S], w + (WM == 2 ? 2048 * grp : 0), PLANE_A);
        if (own_b) put(rb[S], w + 3 * PLANE_A + (WN == 2 ? 2048 * grp : 0), PLANE_B);
    };
    fx16 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    const int aoff = wm * WM * 1024 + 16 * lane, boff = 3 * PLANE_A + wn * WN * 1024 + 16 * lane;
    // Step c of a round: multiply LDS stage c % 2, store the next step's rows
    // (register set (c + 1) % D) and refill that set D steps on.
    auto step = [&](auto cc, auto mask, int r) {
        constexpr int c = decltype(cc)::value, buf = c & 1;
        using Next = std::integral_constant<int, (c + 1) % D>;
        ux4 fa[WM][3], fb[WN][3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < WM; ++i)
                fa[i][p] = *reinterpret_cast<const ux4 *>(smem + buf * STAGE + aoff + p * PLANE_A + i * 1024);
#pragma unroll
            for (int j = 0; j < WN; ++j)
                fb[j][p] = *reinterpret_cast<const ux4 *>(smem + buf * STAGE + boff + p * PLANE_B + j * 1024);
        }
#pragma unroll
        for (int q = 0; q < kPairs; ++q)
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j)
                    acc[i][j] = mma(fa[i][kPairA[q]], fb[j][kPairB[q]], acc[i][j]);
        store(Next{}, mask, buf ^ 1, r + SR);
        load_in(Next{}, r + SR * (D + 1));
        __syncthreads();
    };
    if (r0 < r1) {
        using S0 = std::integral_constant<int, 0>;
        using S1 = std::integral_constant<int, 1>;
        using S2 = std::integral_constant<int, 2>;
        using S3 = std::integral_constant<int, 3>;
        static_assert(D == 4, "register sets");
        using Mask = std::true_type;
        using Whole = std::false_type;
        // (the group's own rows: step i at r + 16 kg)
        const int o = 16 * kg;
        load_pix(r0 + o);
        load_in(S0{}, r0 + o);
        load_in(S1{}, r0 + o + SR);
        load_in(S2{}, r0 + o + 2 * SR);
        load_in(S3{}, r0 + o + 3 * SR);
        store(S0{}, Mask{}, 0, r0 + o);
        load_in(S0{}, r0 + o + 4 * SR);
        __syncthreads();
        int r = r0;
        for (; r + 5 * SR <= r1; r += 4 * SR) {   // (the rows stored are all there)
            step(S0{}, Whole{}, r + o);
            step(S1{}, Whole{}, r + o + SR);
            step(S2{}, Whole{}, r + o + 2 * SR);
            step(S3{}, Whole{}, r + o + 3 * SR);
        }
        for (; r < r1; r += 4 * SR) {
            step(S0{}, Mask{}, r + o);
            if (r + SR < r1) step(S1{}, Mask{}, r + o + SR);
            if (r + 2 * SR < r1) step(S2{}, Mask{}, r + o + 2 * SR);
            if (r + 3 * SR < r1) step(S3{}, Mask{}, r + o + 3 * SR);
        }
    }
    if (KG == 2) {
        // (every wave is past its last fragment reads: a step ends in a barrier)
        float *x = reinterpret_cast<float *>(smem_all) + wave * (WM * WN * 1024) + lane;
        if (kg == 1)
#pragma unroll
            for (int i = 0; i < WM * WN * 16; ++i) x[64 * i] = acc[i / (16 * WN)][i / 16 % WN][i % 16];
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int i = 0; i < WM * WN * 16; ++i) acc[i / (16 * WN)][i / 16 % WN][i % 16] += x[64 * i];
    }
    // Sums that are not finite, or too small for the split: again as float
    // products (gemm_split.h), rows r + lh at a time.
    SumCheck check;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) check.add(acc[i][j]);
    if (!check.fits()) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const float *ca = g.a + m0 + (wm * WM + i) * 32 + li;
                const float *cb = g.b + n0 + (wn * WN + j) * 32 + li;
                fx16 f;
#pragma unroll
                for (int q = 0; q < 16; ++q) f[q] = 0.f;
#pragma unroll 1
                for (int r = r0; r < r1; r += 2) {
                    const int row = min(r + lh, r1 - 1);
                    float x = ca[(GATHER ? token(g.perm[row]) : (size_t)row) * g.lda];
                    float y = cb[(size_t)row * g.ldb];
                    if (r + lh >= r1) x = y = 0.f;
                    f = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, f, 0, 0, 0);
                }
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    acc[i][j][q] = float_sum_needed(acc[i][j][q]) ? f[q] : acc[i][j][q];
            }
    }
    // Lane l, register q of a block: row 8 (q / 4) + 4 (l / 32) + q % 4,
    // column l % 32.
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const int n = n0 + (wn * WN + j) * 32 + li;
        float *ce = (g.c_up && (n & 32) ? g.c_up : g.c) + (size_t)e * g.c_e;
        const int col = g.c_up ? 32 * (n >> 6) + (n & 31) : n;
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = m0 + (wm * WM + i) * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
                float *cp = ce + (size_t)m * g.ldc + col;
                *cp = g.accumulate ? *cp + acc[i][j][q] : acc[i][j][q];
            }
    }
}

// dW_r = X^T dlogits over all T rows, and (CS set) the column sums of
// probs for the aux loss.  Workgroup (column block cb of 64 x columns, row
// chunk z of R rows); thread (c, p) = (t % 64, t / 64) runs the FMA chains of
// kRgEB experts at a time over rows zR + p, zR + p + 4, ..., and the 4 row
// phases are added in phase order through LDS into P[z][d][E].  Every load
// is unconditional (indices clamped, masked terms multiplied by zero).  The
// workgroups of column block 0 also sum probs over their rows into CS[z][E].
// router_grad_final_kernel adds the chunks in order.
constexpr int kRgEB = 8;

__global__ __launch_bounds__(256) void router_grad_kernel(const float *x, const float *dl,
                                                          const float *probs, int T, int d,
                                                          int E, int R, float *P, float *CS) {
    __shared__ float red[4][64][kRgEB + 1];
    const int cb = blockIdx.x, z = blockIdx.y;
    const int t = threadIdx.x, c = t & 63, p = t >> 6;
    const int col = min(cb * 64 + c, d - 1);
    const int r0 = z * R, r1 = min(T, r0 + R);
    for (int e0 = 0; e0 < E; e0 += kRgEB) {
        float acc[kRgEB];
#pragma unroll
        for (int j = 0; j < kRgEB; ++j) acc[j] = 0.f;
        // Rows in batches of 8 (every load of a batch in flight together).
        for (int rb = r0 + p; rb < r1; rb += 32) {
            float xv[8], w[8][kRgEB];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int r = min(rb + 4 * u, r1 - 1);
                xv[u] = x[(size_t)r * d + col];
#pragma unroll
                for (int j = 0; j < kRgEB; ++j) w[u][j] = dl[(size_t)r * E + min(e0 + j, E - 1)];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int j = 0; j < kRgEB; ++j)
                    acc[j] = fmaf(rb + 4 * u < r1 ? xv[u] : 0.f, e0 + j < E ? w[u][j] : 0.f,
                                  acc[j]);
        }
#pragma unroll
        for (int j = 0; j < kRgEB; ++j) red[p][c][j] = acc[j];
        __syncthreads();
        for (int i = t; i < 64 * kRgEB; i += 256) {
            const int cc = i / kRgEB, j = i % kRgEB, oc = cb * 64 + cc;
            if (oc < d && e0 + j < E)
                P[((size_t)z * d + oc) * E + e0 + j] =
                    ((red[0][cc][j] + red[1][cc][j]) + red[2][cc][j]) + red[3][cc][j];
        }
        __syncthreads();
    }
    if (CS && cb == 0)
        for (int e = t; e < E; e += 256) {
            float sum = 0.f;
            for (int rb = r0; rb < r1; rb += 16) {
                float v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = probs[(size_t)min(rb + u, r1 - 1) * E + e];
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    if (rb + u < r1) sum += v[u];
            }
            CS[(size_t)z * E + e] = sum;
        }
}

// base + sum over z < nz (in order) of P[z n + i], 16 chunks' loads in
// flight at a time.
__device__ inline float sum_chunks(const float *P, int nz, int n, int i, float base) {
    float v = 0.f;
    for (int z0 = 0; z0 < nz; z0 += 16) {
        float q[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) q[u] = P[(size_t)min(z0 + u, nz - 1) * n + i];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            if (z0 + u < nz) v += q[u];
    }
    return base + v;
}

// dwr (+)= sum over z (in order) of P[z] (n = d E floats); with aux, one
// more workgroup adds the column sums CS over z (in order) and takes
// aux = E sum_e f_e P_e, f_e = counts[e] / (T k), P_e = colsum[e] / T.
__global__ __launch_bounds__(256) void router_grad_final_kernel(const float *P, int nz, int n,
                                                                int accumulate, float *dwr,
                                                                const float *CS,
                                                                const int *counts, int T, int E,
                                                                int k, float *aux) {
    __shared__ float cs[kMaxExperts];
    const int nb = (n + 255) / 256;
    if ((int)blockIdx.x < nb) {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if (i < n) dwr[i] = sum_chunks(P, nz, n, i, accumulate ? dwr[i] : 0.f);
        return;
    }
    for (int e = threadIdx.x; e < E; e += 256) cs[e] = sum_chunks(CS, nz, E, e, 0.f);
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
        for (int e = 0; e < E; ++e)
            total = fmaf((float)counts[e] / ((float)T * (float)k), cs[e] / (float)T, total);
        *aux = (float)E * total;
    }
}

// H = silu(G) * U, the forward's SwiGLU.
__global__ __launch_bounds__(256) void act_kernel(const float *G, const float *U, float *H,
                                                  size_t n) {
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        H[i] = swiglu_fast(G[i], U[i]);
}

// In place: G <- dG = dH U silu'(G), U <- dU = dH silu(G).
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(float *G, float *U, const float *dH,
                                                         size_t n) {
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float g = G[i], u = U[i], dh = dH[i];
        const float s = 1.0f / (1.0f + expf(-g));
        G[i] = dh * u * fmaf(g * s, 1.0f - s, s);
        U[i] = dh * g * s;
    }
}

// Where an expert GEMM left its [T k x d] rows: by dispatch position, or by
// slot as ns partials ys apart (summed in order).
// With pieces (a stream-K GEMM): slot a's columns [pcols j, pcols (j + 1))
// hold pieces[a * ceil(d / pcols) + j] partials instead of ns.
struct SlotRows {
    const float *p;
    int by_slot, ns;
    size_t ys;
    const int *pieces = nullptr;
    int pcols = 0;
    __device__ int count(int a, int d, int c) const {
        return pieces ? pieces[(size_t)a * ((d + pcols - 1) / pcols) + c / pcols] : ns;
    }
    // The partials of (row, column c) added in order; the first 8 are
    // loaded together (clamped, masked), so none waits for another.
    __device__ float at(int pos, int a, int d, int c) const {
        const float *r = p + (size_t)(by_slot ? a : pos) * d + c;
        const int n = max(count(a, d, c), 1);
        float q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = r[(size_t)min(u, n - 1) * ys];
        float v = q[0];
#pragma unroll
        for (int u = 1; u < 8; ++u)
            if (u < n) v += q[u];
        for (int s = 8; s < n; ++s) v += r[(size_t)s * ys];
        return v;
    }
    // The same for the four columns c .. c + 3 (16-byte aligned).
    __device__ fx4 at4(int row, int a, int d, int c) const {
        const float *r = p + (size_t)row * d + c;
        const int n = max(count(a, d, c), 1);
        fx4 q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = *reinterpret_cast<const fx4 *>(r + (size_t)min(u, n - 1) * ys);
        fx4 v = q[0];
#pragma unroll
        for (int u = 1; u < 8; ++u)
            if (u < n) v += q[u];
        for (int s = 8; s < n; ++s) v += *reinterpret_cast<const fx4 *>(r + (size_t)s * ys);
        return v;
    }
};

// One wave per dispatch position pos (slot a = perm[pos], token t = a / k):
// dgw[a] = <Y(a), dout[t]> (lane-strided partial sums, then a butterfly),
// dY[pos] = gw[a] dout[t], inv[a] = pos.
__global__ __launch_bounds__(256) void slot_kernel(SlotRows Y, const float *dout,
                                                   const float *gw, const int *perm, int k, int d,
                                                   int n, float *dgw, float *dY, int *inv) {
    const int pos = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (pos >= n) return;
    const int a = perm[pos], t = a / k;
    const float w = gw[a];
    const float *go = dout + (size_t)t * d;
    float *dy = dY + (size_t)pos * d;
    float s = 0.f;
    // Four columns per step, their loads issued together.
    for (int c0 = lane; c0 < d; c0 += 256) {
        float v[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = min(c0 + 64 * u, d - 1);
            v[u] = go[c];
            y[u] = Y.at(pos, a, d, c);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (c0 + 64 * u < d) {
                s = fmaf(y[u], v[u], s);
                dy[c0 + 64 * u] = w * v[u];
            }
    }
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) {
        dgw[a] = s;
        inv[a] = pos;
    }
}

// Eight lanes per token: dlogits [T x E] from dgw through the gate
// renormalisation, the aux term and the softmax.  Every lane of a token
// loads its ids and dgw (kMaxTopK of each, clamped, masked) and the
// probabilities of its experts e = g, g + 8, ... (g = lane % 8) at once, then
// the selected probabilities; S, c and dp(e) are summed in slot order and
// the dot over the experts in expert order (through shuffles), as one thread
// per token would.
// JN experts per lane: 16 up to 128 experts, 32 up to 256.
constexpr int kRbG = 8;
template <int JN>
__global__ __launch_bounds__(256) void router_bwd_kernel(const float *probs, const int *ids,
                                                         const float *dgw,
                                                         const int *counts, int T, int E, int k,
                                                         float aux_coef, float *dlogits) {
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int t = gid / kRbG, g = gid % kRbG;
    const int tc = min(t, T - 1);
    const float *p = probs + (size_t)tc * E;
    int id[kMaxTopK];
    float dg[kMaxTopK], ps[kMaxTopK];
#pragma unroll
    for (int s = 0; s < kMaxTopK; ++s) {
        const size_t q = (size_t)tc * k + min(s, k - 1);
        id[s] = ids[q];
        dg[s] = dgw[q];
    }
    // The aux term's counts enter as differences from a fixed count (the
    // softmax gradient p (dp - sum p dp) does not change when every dp moves
    // by one constant): near-uniform loads then give small exact values, so
    // the subtraction below does not cancel the large common part in fp32.
    const int cref = (int)(((long long)T * k) / E);
    float pv[JN], cn[JN];
#pragma unroll
    for (int j = 0; j < JN; ++j)
        if (kRbG * j < E) {
            const int e = min(g + kRbG * j, E - 1);
            pv[j] = p[e];
            cn[j] = (float)(counts[e] - cref);
        }
#pragma unroll
    for (int s = 0; s < kMaxTopK; ++s) ps[s] = p[id[s]];
    // c = sum over slots of dgw * (p / S), the renormalised weights taken
    // as p / S here: at top-1 that is exactly 1, so the slot term (dgw - c)
    // / S vanishes exactly as its derivative does (the stored gate weight,
    // p * (1 / S), can sit an ulp below 1).
    float S = 0.f, c = 0.f;
#pragma unroll
    for (int s = 0; s < kMaxTopK; ++s)
        if (s < k) S += ps[s];
#pragma unroll
    for (int s = 0; s < kMaxTopK; ++s)
        if (s < k) c = fmaf(dg[s], ps[s] / S, c);
    const float aux_scale = aux_coef * (float)E / ((float)T * (float)T * (float)k);
    float dpv[JN];
#pragma unroll
    for (int j = 0; j < JN; ++j)
        if (kRbG * j < E) {
            const int e = g + kRbG * j;
            float v = aux_scale * cn[j];
#pragma unroll
            for (int s = 0; s < kMaxTopK; ++s)
                if (s < k && id[s] == e) v += (dg[s] - c) / S;
            dpv[j] = v;
        }
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < JN; ++j)
        if (kRbG * j < E)
#pragma unroll
            for (int q = 0; q < kRbG; ++q)
                if (kRbG * j + q < E)
                    dot = fmaf(__shfl(dpv[j], q, kRbG), __shfl(pv[j], q, kRbG), dot);
    if (t >= T) return;
#pragma unroll
    for (int j = 0; j < JN; ++j)
        if (g + kRbG * j < E) dlogits[(size_t)t * E + g + kRbG * j] = pv[j] * (dpv[j] - dot);
}

// dx[t][c..c+3] = sum over slots (in order) of dXr(t k + s), plus
// sum_e dlogits[t][e] wr[c][e] (read from wrT [E x d]); one thread per 4
// columns (d % 4 == 0).
__global__ __launch_bounds__(256) void dx_kernel(SlotRows dXr, const int *inv,
                                                 const float *dlogits, const float *wrT, int T,
                                                 int d, int E, int k, int accumulate, float *dx) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int d4 = d / 4;
    if (i >= (size_t)T * d4) return;
    const int t = (int)(i / d4), c = 4 * (int)(i % d4);
    fx4 v = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < k; ++s) {
        const int a = t * k + s;
        v += dXr.at4(dXr.by_slot ? a : inv[a], a, d, c);
    }
    fx4 rr = {0.f, 0.f, 0.f, 0.f};
    const float *dl = dlogits + (size_t)t * E;
    // Eight experts per step, their loads issued together.
    for (int e0 = 0; e0 < E; e0 += 8) {
        float gv[8];
        fx4 wv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = min(e0 + u, E - 1);
            gv[u] = dl[e];
            wv[u] = *reinterpret_cast<const fx4 *>(wrT + (size_t)e * d + c);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (e0 + u < E)
#pragma unroll
                for (int j = 0; j < 4; ++j) rr[j] = fmaf(gv[u], wv[u][j], rr[j]);
    }
    v += rr;
    fx4 *o = reinterpret_cast<fx4 *>(dx + (size_t)t * d + c);
    *o = accumulate ? *o + v : v;
}

unsigned blocks_for(size_t n) { return (unsigned)std::min<size_t>((n + 255) / 256, 16384); }

#define BWD_TRY(x)                               \
    do {                                         \
        hipError_t e_ = (x);                     \
        if (e_ != hipSuccess) return e_;         \
    } while (0)

}  // namespace

bool backward_engine_ok(int d, int F) { return d % 64 == 0 && F % 64 == 0; }

size_t backward_dh_floats(size_t n, int d, int F, int E) {
    return std::max(n * (size_t)F, (size_t)d * E + E);
}

size_t backward_tail_floats(int d, int F, int max_mtiles, int E) {
    if (!backward_engine_ok(d, F)) return 0;
    const int g = std::max(gateup_tail_groups(2 * F, d, max_mtiles, E),
                           gateup_tail_groups(F, d, max_mtiles, E));
    return (size_t)g * kGemmBM * 256;
}

int backward_slot_splits(int d, int F, int max_mtiles, size_t n, int k) {
    if (!backward_engine_ok(d, F)) return 1;
    return std::max(down_plan(d, F, max_mtiles, n, k).slots, down_plan(d, 2 * F, max_mtiles, n, k).slots);
}

hipError_t launch_moe_backward(const BackwardArgs &b, hipStream_t s) {
    const int d = b.d, F = b.F, E = b.E, k = b.k, T = b.T;
    const size_t n = (size_t)T * k;
    if (T <= 0) return hipSuccess;
    if (d % 16 || F % 16) return hipErrorInvalidValue;   // (dx_kernel: d % 4)
    auto rows = [&](auto gather, auto bt, const float *A, int lda, const float *B, size_t b_e,
                    int ldb, float *C, int K, int N, int accumulate) {
        RowsGemm g{A, lda, b.perm, k, B, b_e, ldb, C, N, b.offsets, b.tile_off, b.tile_expert,
                   E, K, N, b.max_mtiles, accumulate};
        const unsigned grid = (unsigned)(b.max_mtiles * ((N + kRN - 1) / kRN));
        if (K % kMK == 0)
            hipLaunchKernelGGL((rows_mfma_kernel<decltype(gather)::value, decltype(bt)::value>),
                               dim3(grid), dim3(128), 0, s, g);
        else
            hipLaunchKernelGGL((rows_gemm_kernel<decltype(gather)::value, decltype(bt)::value>),
                               dim3(grid), dim3(256), 0, s, g);
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    const size_t nd = n * d;
    const unsigned slot_grid = (unsigned)((n + 3) / 4);
    SlotRows dXr{b.Y, 0, 1, 0};
    if (b.wgu) {
        // The forward's tile engine on the packed weights and their unit
        // transposes; G and U adjacent as GU [n x 2F] in packed column order.
        float *GU = b.G;
        BWD_TRY(launch_transpose_units(b.wdT, b.wdTT, d, F, E, s));
        BWD_TRY(launch_transpose_units(b.wgu, b.wguT, 2 * F, d, E, s));
        GemmArgs g{};
        g.perm = b.perm; g.topk = k; g.offsets = b.offsets; g.tile_off = b.tile_off;
        g.tile_expert = b.tile_expert; g.E = E; g.max_mtiles = b.max_mtiles;
        // Recompute GU and H, then Y by slot (split partials).
        GemmArgs gu = g;
        gu.a = b.x; gu.b = b.wgu; gu.c = GU; gu.K = d; gu.N = 2 * F; gu.ldc = 2 * F;
        gu.c2 = b.H; gu.ldc2 = F;
        if (b.tail_part) {
            gu.tail_groups = gateup_tail_groups(2 * F, d, b.max_mtiles, E);
            gu.tail_part = b.tail_part;
        }
        BWD_TRY(launch_gemm_bwd(gu, 2, s));
        BWD_TRY(launch_tail_fixup(gu, 2, s));
        // (Y and dX: down-projection shapes, by slot with split partials or
        // stream-K pieces, moe::down_plan; one piece-count table serves both
        // in turn.)
        const DownPlan py = down_plan(d, F, b.max_mtiles, n, k);
        GemmArgs gy = g;
        gy.a = b.H; gy.b = b.wdT; gy.c = b.Y; gy.K = F; gy.N = d; gy.ldc = d;
        gy.ksplit = py.slots; gy.split_stride = nd;
        gy.streamk = py.streamk; gy.sk_groups = py.groups; gy.bn = py.bn; gy.pieces = b.pieces;
        BWD_TRY(launch_gemm_down(gy, s));
        hipLaunchKernelGGL(slot_kernel, dim3(slot_grid), dim3(256), 0, s,
                           SlotRows{b.Y, 1, py.slots, nd, py.streamk ? b.pieces : nullptr, py.bn},
                           b.dout, b.gw, b.perm, k, d, (int)n, b.dgw, b.dY, b.inv);
        // dH -> dG, dU in place over GU; dXr = dGU wgu^T by slot (over Y).
        GemmArgs gh = g;
        gh.a = b.dY; gh.b = b.wdTT; gh.c = GU; gh.K = d; gh.N = F; gh.ldc = 2 * F;
        if (b.tail_part) {
            gh.tail_groups = gateup_tail_groups(F, d, b.max_mtiles, E);
            gh.tail_part = b.tail_part;
        }
        BWD_TRY(launch_gemm_bwd(gh, 3, s));
        BWD_TRY(launch_tail_fixup(gh, 3, s));
        const DownPlan px = down_plan(d, 2 * F, b.max_mtiles, n, k);
        GemmArgs gx = g;
        gx.a = GU; gx.b = b.wguT; gx.c = b.Y; gx.K = 2 * F; gx.N = d; gx.ldc = d;
        gx.ksplit = px.slots; gx.split_stride = nd;
        gx.streamk = px.streamk; gx.sk_groups = px.groups; gx.bn = px.bn; gx.pieces = b.pieces;
        BWD_TRY(launch_gemm_down(gx, s));
        dXr = SlotRows{b.Y, 1, px.slots, nd, px.streamk ? b.pieces : nullptr, px.bn};
    } else {
        // Recompute: G, U (gathered x rows), H, Y.
        rows(T_{}, F_{}, b.x, d, b.wg, (size_t)d * F, F, b.G, d, F, 0);
        rows(T_{}, F_{}, b.x, d, b.wu, (size_t)d * F, F, b.U, d, F, 0);
        hipLaunchKernelGGL(act_kernel, dim3(blocks_for(n * F)), dim3(256), 0, s, b.G, b.U, b.H,
                           n * F);
        rows(F_{}, F_{}, b.H, F, b.wd, (size_t)F * d, d, b.Y, F, d, 0);
        // Slots: dgw, dY, the slot -> position map.
        hipLaunchKernelGGL(slot_kernel, dim3(slot_grid), dim3(256), 0, s, SlotRows{b.Y, 0, 1, 0},
                           b.dout, b.gw, b.perm, k, d, (int)n, b.dgw, b.dY, b.inv);
        // Experts: dH, dG and dU (in place over G, U), dXr (over Y).
        rows(F_{}, T_{}, b.dY, d, b.wd, (size_t)F * d, d, b.dH, d, F, 0);
        hipLaunchKernelGGL(swiglu_bwd_kernel, dim3(blocks_for(n * F)), dim3(256), 0, s, b.G,
                           b.U, b.dH, n * F);
        rows(F_{}, T_{}, b.G, F, b.wg, (size_t)d * F, F, b.Y, F, d, 0);
        rows(F_{}, T_{}, b.U, F, b.wu, (size_t)d * F, F, b.Y, F, d, 1);
    }
    // Router and dx.
    {
        const dim3 grid((unsigned)(((size_t)T * kRbG + 255) / 256));
        if (E <= 128)
            hipLaunchKernelGGL(router_bwd_kernel<128 / kRbG>, grid, dim3(256), 0, s, b.probs, b.ids,
                               b.dgw, b.counts, T, E, k, b.aux_coef, b.dlogits);
        else
            hipLaunchKernelGGL(router_bwd_kernel<kMaxExperts / kRbG>, grid, dim3(256), 0, s, b.probs,
                               b.ids, b.dgw, b.counts, T, E, k, b.aux_coef, b.dlogits);
    }
    hipLaunchKernelGGL(dx_kernel, dim3((unsigned)(((size_t)T * (d / 4) + 255) / 256)), dim3(256),
                       0, s, dXr, b.inv,
                       b.dlogits, b.wrT, T, d, E, k, b.accumulate, b.dx);
    // Weight gradients over each expert's rows; the router's over all tokens.
    auto reduce = [&](auto gather, const float *A, int lda, const float *B, int ldb, float *C,
                      size_t c_e, int M, int N, const int *offsets, int nrows, int chunk,
                      int groups, int accumulate) {
        ReduceGemm g{A, lda, b.perm, k, B, ldb, C, c_e, N, offsets, nrows, chunk, M, N,
                     accumulate, M % 4 == 0 && lda % 4 == 0, N % 4 == 0 && ldb % 4 == 0};
        dim3 grid((unsigned)((N + kQN - 1) / kQN), (unsigned)((M + kQM - 1) / kQM),
                  (unsigned)groups);
        hipLaunchKernelGGL((reduce_gemm_kernel<decltype(gather)::value>), grid, dim3(256), 0, s,
                           g);
    };
    if (b.wgu) {
        auto mfma = [&](auto gather, const float *A, int lda, const float *B, int ldb, float *C,
                        float *C_up, int M, int N, int ldc) {
            ReduceGemm g{A, lda, b.perm, k, B, ldb, C, (size_t)M * ldc, ldc, b.offsets, 0, 0, M,
                         N, b.accumulate, 1, 1, C_up};
            // The widest tile that still gives every CU a workgroup.
            const long cus = device_cus();
            auto tiles = [&](int wm, int wn) { return (long)(M / (64 * wm)) * (N / (64 * wn)) * E; };
            // perm / k = the high word of perm * ceil(2^32 / k) (perm k < 2^32:
            // perm < T k <= 2^31 / 64 and k <= 16), or perm itself for k = 1.
            const unsigned magic = k > 1 ? (unsigned)((((unsigned long long)1 << 32) + k - 1) / k) : 0;
            const unsigned one = k > 1 ? 0u : ~0u;
            using I1 = std::integral_constant<int, 1>;
            using I2 = std::integral_constant<int, 2>;
            auto go = [&](auto wm, auto wn) {
                constexpr int WM = decltype(wm)::value, WN = decltype(wn)::value;
                const dim3 grid((unsigned)(N / (64 * WN)), (unsigned)(M / (64 * WM)), (unsigned)E);
                auto launch = [&](auto kg, auto few) {
                    constexpr int KG = decltype(kg)::value;
                    hipLaunchKernelGGL((reduce_split_kernel<decltype(gather)::value, WM, WN, KG,
                                                            decltype(few)::value>),
                                       grid, dim3(256 * KG), 0, s, g, magic, one);
                };
                const bool two = tiles(WM, WN) < 2 * cus, few = n < (size_t)kRedShortRows * E;
                if (few && two) launch(I2{}, T_{});
                else if (few)   launch(I1{}, T_{});
                else if (two)   launch(I2{}, F_{});
                else            launch(I1{}, F_{});
            };
            if (M % 128 == 0 && N % 128 == 0 && tiles(2, 2) >= cus) go(I2{}, I2{});
            else if (M % 128 == 0 && tiles(2, 1) >= cus)           go(I2{}, I1{});
            else if (N % 128 == 0 && tiles(1, 2) >= cus)           go(I1{}, I2{});
            else                                                    go(I1{}, I1{});
        };
        mfma(F_{}, b.H, F, b.dY, d, b.dwd, nullptr, F, d, d);
        // dW_g and dW_u in one launch over GU's 2F packed columns.
        mfma(T_{}, b.x, d, b.G, 2 * F, b.dwg, b.dwu, d, 2 * F, F);
    } else {
        reduce(F_{}, b.H, F, b.dY, d, b.dwd, (size_t)F * d, F, d, b.offsets, 0, 0, E,
               b.accumulate);
        reduce(T_{}, b.x, d, b.G, F, b.dwg, (size_t)d * F, d, F, b.offsets, 0, 0, E,
               b.accumulate);
        reduce(T_{}, b.x, d, b.U, F, b.dwu, (size_t)d * F, d, F, b.offsets, 0, 0, E,
               b.accumulate);
    }
    // The router's over all tokens (and the aux loss's column sums), in row
    // chunks whose partials (in dH, free by now) are then added in chunk
    // order: enough chunks for about one workgroup per CU, as many as dH
    // holds (it holds one chunk's at least: backward_dh_floats).
    const int ncb = (d + 63) / 64;
    const size_t cap = backward_dh_floats(n, d, F, E);
    int R = std::max(16, (int)((T + std::max(1, 256 / ncb) - 1) / std::max(1, 256 / ncb)));
    while (R < T && (size_t)((T + R - 1) / R) * ((size_t)d * E + E) > cap) R *= 2;
    const int nz = (T + R - 1) / R;
    float *P = b.dH, *CS = b.aux ? b.dH + (size_t)nz * d * E : nullptr;
    hipLaunchKernelGGL(router_grad_kernel, dim3((unsigned)ncb, (unsigned)nz), dim3(256), 0, s,
                       b.x, b.dlogits, b.probs, T, d, E, R, P, CS);
    const int nb = (int)((d * E + 255) / 256);
    hipLaunchKernelGGL(router_grad_final_kernel, dim3((unsigned)(nb + (b.aux ? 1 : 0))), dim3(256),
                       0, s, P, nz, d * E, b.accumulate, b.dwr, CS, b.counts, T, E, k, b.aux);
    return hipGetLastError();
}

}  // namespace moe
