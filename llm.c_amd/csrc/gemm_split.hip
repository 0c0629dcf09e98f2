// gemm_split.hip — the grouped expert GEMMs on split operands (gemm_split.h).
//
// Layout of the weights: gemm.hip.  The rows of one expert's m-tile are
// consecutive dispatch positions offsets[e] + m; gate/up gathers them
// straight from x through perm.
//
// Work decomposition: the grid enumerates (m-tile, n-tile) pairs over the
// flat per-expert m-tile list built by the dispatch kernel (tile_off), so a
// hot expert simply owns more tiles; workgroups past the live tiles exit.
#include "gemm_split.h"
#include <algorithm>

namespace moe {
namespace {

using namespace split;

constexpr int BM = kGemmBM;   // 128
constexpr int KT = 32;        // reduction granularity of splits and pieces
constexpr int kThreads = 256;

__device__ __forceinline__ bool any_float_sum(fx16 a) {
    bool any = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) any |= float_sum_needed(a[r]);
    return __ballot(any) != 0;
}

// One tile (m-tile mtg, n-tile nt) over the nk 32-wide K slices from element
// kb; WM x WN waves, operands loaded D steps ahead.  The down projection
// writes its partial to slot `slot` (c + slot * split_stride) and, with
// npieces > 0, records npieces for the tile's rows.
// Every thread of the workgroup calls this together.
template <int MODE, int WM, int WN>
__device__ __forceinline__ void gemm_tile(const GemmArgs &a, char *smem, int mtg, int nt, int kb,
                                          int nk, int slot, int npieces, float *part = nullptr) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int BN = 64 * WN;
    constexpr int MB = 4 / WM;   // 32-row blocks per wave
    // Steps that operands are loaded ahead: one where the sums (128 registers
    // with MB = 4) leave no more, else two (a step is half as long there; the
    // layers of T = 256, d = 512, F = 2048, E = 16, 32 rows per expert
    // and one tile per CU, 95 -> 86 us).
    constexpr int D = MB == 4 ? 1 : 2;
    constexpr int PLANE = kStageBytes / 3, STAGE = kStageBytes;
    const int e = a.tile_expert[mtg];
    const int row0 = a.offsets[e] + (mtg - a.tile_off[e]) * BM;
    const int rows = min(BM, a.offsets[e + 1] - row0);
    const int K = a.K;

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 31, lh = lane >> 5;
    const int n0 = nt * BN + wn * 64;   // the wave's first packed column
    // Valid 32-row blocks of this wave (uniform): rows past the expert's last
    // one and columns past N cost no MFMAs.
    const int nmb = n0 < a.N ? max(0, min(MB, (rows - wm * 32 * MB + 31) / 32)) : 0;

    if (MODE == 1 && npieces > 0)
        for (int r = tid; r < rows; r += kThreads)
            a.pieces[(size_t)a.perm[row0 + r] * ((a.N + BN - 1) / BN) + nt] = npieces;

    auto src_row = [&](int r) -> size_t {   // (rows past the last reuse it)
        const int p = row0 + min(r, rows - 1);
        return MODE == 0 || MODE == 2 ? (size_t)(a.perm[p] / a.topk) : (size_t)p;
    };
    // A: thread t loads k 4 (t % 4) .. + 3 of rows t / 4 and t / 4 + 64.
    const int ar = tid >> 2, aq = tid & 3;
    const float *ap[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) ap[i] = a.a + src_row(ar + 64 * i) * K + kb + 4 * aq;
    // LDS: plane p, 32-row block b: 1 KB at 4 p + b KB, the 16-byte run of
    // (row r, k half h) at 16 (32 h + (r + 8 h) % 32): a fragment read is one
    // contiguous KB, and a store instruction's two halves use other banks.
    const int ah = aq >> 1;
    const int aw = (ar >> 5) * 1024 + 16 * (32 * ah + ((ar + 8 * ah) & 31)) + 8 * (aq & 1);
    const int arow = 16 * (32 * lh + ((li + 8 * lh) & 31)) + wm * MB * 1024;
    // B: lane l holds k 8 (l / 32) .. + 7 of column l % 32 of each 32-column
    // block: two 16-byte pieces of its packed unit.
    const float *bbase = a.b + (size_t)e * a.N * K + (size_t)(n0 < a.N ? n0 : 0) * K +
                         (size_t)(kb / 16) * 256;   // (uniform)
    const unsigned bo0 = ((li >> 4) * (K / 16)) * 256 + lh * 128 + (li & 15) * 4;
    const unsigned bo1 = bo0 + 2 * (K / 16) * 256;

    // Step s's pieces: A in ra[s % D], B in rb[s % D].
    fx4 ra[D][2], rb[D][4];
    const int last = 2 * nk - 1;   // steps of 16 k
    auto load_a = [&](auto set, int s) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            ra[decltype(set)::value][i] =
                *reinterpret_cast<const fx4 *>(ap[i] + 16 * min(s, last));
    };
    auto load_b = [&](auto set, int s) {
        constexpr int S = decltype(set)::value;
        const float *p = bbase + (size_t)min(s, last) * 256;
        rb[S][0] = *reinterpret_cast<const fx4 *>(p + bo0);
        rb[S][1] = *reinterpret_cast<const fx4 *>(p + bo0 + 64);
        rb[S][2] = *reinterpret_cast<const fx4 *>(p + bo1);
        rb[S][3] = *reinterpret_cast<const fx4 *>(p + bo1 + 64);
    };
    auto store_a = [&](auto set, int buf) {
        char *w = smem + buf * STAGE + aw;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const fx4 r = ra[decltype(set)::value][i];
            unsigned t[3][2];
            split2(r[0], r[1], t[0][0], t[1][0], t[2][0]);
            split2(r[2], r[3], t[0][1], t[1][1], t[2][1]);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<ux2 *>(w + p * PLANE + 2048 * i) = ux2{t[p][0], t[p][1]};
        }
    };

    fx16 acc[MB][2];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.0f;

    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, D - 1>;
    load_a(S0{}, 0);
    load_b(S0{}, 0);
    if constexpr (D == 2) { load_a(S1{}, 1); load_b(S1{}, 1); }
    store_a(S0{}, 0);
    load_a(S0{}, D);
    __syncthreads();
    // Step s (parity buf, register set `set`): NM of the wave's row blocks
    // from LDS stage buf; the next step's A rows to the other stage.
    auto step = [&](auto nmc, auto set, auto next, auto bufc, int s) {
        constexpr int NM = decltype(nmc)::value, buf = decltype(bufc)::value;
        constexpr int S = decltype(set)::value;
        if constexpr (NM > 0) {
            ux4 fa[NM][3];
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    fa[m][p] = *reinterpret_cast<const ux4 *>(smem + buf * STAGE + arow +
                                                              p * PLANE + m * 1024);
            const Frag b0 = split8(rb[S][0], rb[S][1]);
            const Frag b1 = split8(rb[S][2], rb[S][3]);
            load_b(set, s + D);
#pragma unroll
            for (int q = 0; q < kPairs; ++q)
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    acc[m][0] = mma(fa[m][kPairA[q]], b0.t[kPairB[q]], acc[m][0]);
                    acc[m][1] = mma(fa[m][kPairA[q]], b1.t[kPairB[q]], acc[m][1]);
                }
        }
        store_a(next, buf ^ 1);
        load_a(next, s + 1 + D);
        __syncthreads();
        // (the next step's splitting stays behind its loads: hoisted up here
        // it waits for them a step early)
        if constexpr (D > 1) __builtin_amdgcn_sched_barrier(0x00c);   // (MFMAs may cross)
    };
    auto loop = [&](auto nmc) {
        using B0 = std::integral_constant<int, 0>;
        using B1 = std::integral_constant<int, 1>;
        for (int s = 0; s < last; s += 2) {
            step(nmc, S0{}, S1{}, B0{}, s);
            step(nmc, S1{}, S0{}, B1{}, s + 1);
        }
    };
    switch (nmb) {
        case 0: loop(std::integral_constant<int, 0>{}); return;
        case 1: loop(std::integral_constant<int, 1>{}); break;
        case 2: if constexpr (MB >= 2) loop(std::integral_constant<int, 2>{}); break;
        case 3: if constexpr (MB >= 3) loop(std::integral_constant<int, 3>{}); break;
        default: if constexpr (MB >= 4) loop(std::integral_constant<int, 4>{}); break;
    }

    // Sums that are not finite, or too small for the split: again as float
    // products (gemm_split.h).
    SumCheck check;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        if (m >= nmb) break;
        check.add(acc[m][0]);
        check.add(acc[m][1]);
    }
    if (!check.fits()) {
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            if (m >= nmb || !(any_float_sum(acc[m][0]) || any_float_sum(acc[m][1]))) continue;
            const float *ax = a.a + src_row((wm * MB + m) * 32 + li) * K + kb + 8 * lh;
            fx16 f[2];
#pragma unroll
            for (int r = 0; r < 16; ++r) f[0][r] = f[1][r] = 0.0f;
#pragma unroll 1
            for (int s = 0; s <= last; ++s) {
                load_b(S0{}, s);
                const fx4 x0 = *reinterpret_cast<const fx4 *>(ax + 16 * s);
                const fx4 x1 = *reinterpret_cast<const fx4 *>(ax + 16 * s + 4);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float x = j < 4 ? x0[j & 3] : x1[j & 3];
                    f[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, rb[0][j >> 2][j & 3], f[0], 0, 0, 0);
                    f[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, rb[0][2 + (j >> 2)][j & 3], f[1], 0, 0, 0);
                }
            }
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[m][n][r] = float_sum_needed(acc[m][n][r]) ? f[n][r] : acc[m][n][r];
        }
    }

    // Accumulator layout of a 32x32 block: lane l, register r holds
    // row 8*(r/4) + 4*(l/32) + (r%4), column l%32.
#define MOE_TILE_ROWS                                                                   \
    _Pragma("unroll") for (int m = 0; m < MB; ++m)                                      \
        _Pragma("unroll") for (int r = 0; r < 16; ++r)                                  \
            if (const int row = (wm * MB + m) * 32 + 8 * (r >> 2) + 4 * lh + (r & 3); row < rows)
    if (MODE != 1 && part) {
        // A piece of a split tile: raw sums, [row][tile column].
        MOE_TILE_ROWS {
            part[row * BN + wn * 64 + li] = acc[m][0][r];
            part[row * BN + wn * 64 + 32 + li] = acc[m][1][r];
        }
    } else if (MODE == 0) {
        const int f = (n0 >> 1) + li;   // feature index
        MOE_TILE_ROWS {
            a.c[(size_t)(row0 + row) * a.ldc + f] = swiglu_fast(acc[m][0][r], acc[m][1][r]);
        }
    } else if (MODE == 2) {
        // Raw gate and up columns (packed order, dispatch-ordered rows) and H.
        const int f = (n0 >> 1) + li;
        MOE_TILE_ROWS {
            const size_t p = (size_t)(row0 + row);
            const float g = acc[m][0][r], u = acc[m][1][r];
            a.c[p * a.ldc + n0 + li] = g;
            a.c[p * a.ldc + n0 + li + 32] = u;
            a.c2[p * a.ldc2 + f] = swiglu_fast(g, u);
        }
    } else if (MODE == 3) {
        // acc = dH for features f = n0 + 32n + li; the gate and up values of
        // f sit at packed columns 64(f/32) + f%32 and 32 past it, and are
        // replaced by dG = dH u silu'(g), dU = dH silu(g).
        MOE_TILE_ROWS {
            float *gu = a.c + (size_t)(row0 + row) * a.ldc;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int col = 2 * n0 + 64 * n + li;
                const float g = gu[col], u = gu[col + 32], dh = acc[m][n][r];
                const float sg = 1.0f / (1.0f + expf(-g));
                gu[col] = dh * u * fmaf(g * sg, 1.0f - sg, sg);
                gu[col + 32] = dh * g * sg;
            }
        }
    } else {
        float *c = a.c + (size_t)slot * a.split_stride;
        MOE_TILE_ROWS {
            const size_t dst = (size_t)a.perm[row0 + row] * a.ldc + n0 + li;
            c[dst] = acc[m][0][r];
            c[dst + 32] = acc[m][1][r];
        }
    }
#undef MOE_TILE_ROWS
}

// The split tail of a gate/up launch: whole tiles [0, dp), a multiple of the
// CUs (tail_groups); r tiles left over (dp .. dp + r - 1), each in s pieces,
// one piece per CU at most; r = s = 0 when the tail is not split.
struct TailLayout { int dp, r, s; };
__device__ __forceinline__ TailLayout tail_layout(const GemmArgs &a, int ntiles, int nks) {
    const int live = a.tile_off[a.E] * ntiles;
    const int r = live % a.tail_groups;
    const int sp = r ? min(min(nks, 4), a.tail_groups / r) : 0;
    if (sp < 2) return TailLayout{live, 0, 0};
    return TailLayout{live - r, r, sp};
}

// Down projection in stream-K form: how `grid` workgroups share `tiles` live
// tiles of nks K slices.  p > 0: every tile in p even pieces, one per
// workgroup; 0: runs of ceil(tiles nks / grid) slices over the flat list of
// (tile, slice) units, most of which touch two tiles.
// Runs load every workgroup alike, but a second tile is a second prologue
// and epilogue, about kSkPass slices' time; so they are taken where even
// pieces would be longer than a run by more than that (T = 4096, d = 256, F =
// 1024, E = 8, top-2: three pieces of 11 slices 111.0 us per layer, runs of 9
// 119.1; T = 139, d = 576, F = 7072, E = 22, top-4: four pieces of 56 slices 297,
// runs of 50 283).
// A piece has four slices or so: fewer cost more in partials than they save
// (T = 59, d = 192, F = 896, E = 7, top-4: 14 pieces 44.2 us, 7 37.7), and the
// combine adds a tile's pieces for each of a token's k slots, eight loads at a
// time: 64 in all at most (T = 24, d = 256, F = 3200, E = 8, top-6: 25 pieces
// 79.3 us, 10 54.0).  Reductions of 6 to 15 slices on few tiles go down to two
// slices for up to four pieces (T = 118, d = 256, F = 256, E = 1: two pieces 37.0
// us, four 35.2; backward T = 71, d = 192, F = 128, E = 12, top-3 92.4, 90.7).
constexpr int kSkPass = 2, kSkFewTiles = 64;
__host__ __device__ constexpr int sk_max_pieces(int tiles, int nks, int topk) {
    const int c = topk < 8 ? 64 / topk : 8;
    int l = (nks + 3) / 4;
    if (tiles <= kSkFewTiles && nks >= 6 && nks < 16) l = nks < 8 ? nks / 2 : 4;
    return c < l ? c : l;
}
__host__ __device__ constexpr int sk_even_pieces(int tiles, int nks, int grid, int topk) {
    const int room = tiles > 0 ? grid / tiles : 0, most = sk_max_pieces(tiles, nks, topk);
    if (room > most) return most;
    if (room < 1) return 0;
    const int run = (int)(((long)tiles * nks + grid - 1) / grid);
    return (nks + room - 1) / room - run > kSkPass ? 0 : room;
}

// Grid: the (m-tile, n-tile) pairs, times the reduction splits.  Down
// projection in stream-K form (a.streamk): a piece of a tile each
// (sk_even_pieces), or workgroup g takes units [g per, (g + 1) per) of the flat
// list of (live tile, K slice) units, per = ceil(units / grid); each tile it
// touches is a piece.  A piece's index within
// the tile (0 for the workgroup holding the tile's first slice) is the
// partial slot it writes, and piece 0 records the tile's piece count for
// the combine.  Slots, pieces and counts follow from the live tile count
// alone, so results are deterministic.
template <int MODE, int WM, int WN>
__global__ __launch_bounds__(kThreads, 2) void grouped_gemm_kernel(GemmArgs a) {
    constexpr int BN = 64 * WN;
    __shared__ __align__(16) char smem[kTileLds];
    const int ntiles = (a.N + BN - 1) / BN;
    const int nks = a.K / KT;
    if (MODE == 1 && a.streamk) {
        const int tiles = a.tile_off[a.E] * ntiles;
        const int pieces = sk_even_pieces(tiles, nks, gridDim.x, a.topk), b = blockIdx.x;
        int tile = 0, k0 = 0, k1 = 0, slot = 0, npieces = pieces;
        long u = 0, uend = 0, per = 0;
        if (pieces) {   // (32-bit divisions only: a piece may be a few slices)
            tile = b / pieces;
            if (tile >= tiles) return;
            slot = b - tile * pieces;
            k0 = slot * nks / pieces;
            k1 = (slot + 1) * nks / pieces;
        } else {
            const long units = (long)tiles * nks;
            per = (units + gridDim.x - 1) / gridDim.x;
            u = b * per;
            uend = u + per < units ? u + per : units;
        }
        do {
            if (!pieces) {
                if (u >= uend) return;
                tile = (int)(u / nks);
                k0 = (int)(u - (long)tile * nks);
                k1 = (int)(k0 + (uend - u) < nks ? k0 + (uend - u) : nks);
                const long tstart = (long)tile * nks;
                const int first = (int)(tstart / per);   // workgroup of the tile's first slice
                slot = b - first;
                npieces = (int)((tstart + nks - 1) / per) - first + 1;
                u += k1 - k0;
            }
            gemm_tile<MODE, WM, WN>(a, smem, tile / ntiles, tile % ntiles, k0 * KT, k1 - k0, slot,
                                    slot == 0 ? npieces : 0);
        } while (!pieces);
        return;
    }
    if (MODE != 1 && a.tail_groups > 0) {
        // Whole tiles in the grid's first dp workgroups, then the pieces of
        // the split tail: piece s of tail tile r covers K slices
        // [s nks / S, (s + 1) nks / S).  (Grid: the m-tile bound's tiles plus
        // tail_groups.)
        const TailLayout tl = tail_layout(a, ntiles, nks);
        const int b = blockIdx.x;
        if (b < tl.dp) {
            gemm_tile<MODE, WM, WN>(a, smem, b / ntiles, b % ntiles, 0, nks, 0, 0);
            return;
        }
        const int j = b - tl.dp;
        if (j >= tl.r * tl.s) return;
        const int r = j / tl.s, sp = j - r * tl.s;
        const int tile = tl.dp + r;
        const int k0 = sp * nks / tl.s, k1 = (sp + 1) * nks / tl.s;
        gemm_tile<MODE, WM, WN>(a, smem, tile / ntiles, tile % ntiles, k0 * KT, k1 - k0, 0, 0,
                            a.tail_part + (size_t)j * BM * BN);
        return;
    }
    const int per_split = a.max_mtiles * ntiles;
    const int ks = blockIdx.x / per_split;       // reduction split (down projection)
    const int nt = (blockIdx.x % per_split) % ntiles;
    int mtg = (blockIdx.x % per_split) / ntiles;
    if (mtg >= a.tile_off[a.E]) return;
    if (a.order) mtg = a.order[mtg];
    const int nk = nks / a.ksplit;   // K steps of this split
    gemm_tile<MODE, WM, WN>(a, smem, mtg, nt, ks * nk * KT, nk, ks, 0);
}

template <int MODE, int WM, int WN>
hipError_t launch_grouped(const GemmArgs &a, hipStream_t s) {
    constexpr int BN = 64 * WN;
    const int ntiles = (a.N + BN - 1) / BN;
    const unsigned grid =
        MODE == 1 && a.streamk
            ? (unsigned)a.sk_groups
            : (unsigned)(a.max_mtiles * ntiles * a.ksplit + (MODE != 1 ? a.tail_groups : 0));
    hipLaunchKernelGGL((grouped_gemm_kernel<MODE, WM, WN>), dim3(grid), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

template <int MODE>
hipError_t launch_mode(const GemmArgs &a, hipStream_t s) {
    const int bn = MODE == 1 ? a.bn : gemm_plan(a.N, a.K, a.max_mtiles, false).bn;
    if (a.K % KT || a.N % 64) return hipErrorInvalidValue;
    if (MODE == 1 && a.streamk) {
        if (!a.pieces || a.sk_groups <= 0) return hipErrorInvalidValue;
        if (bn == 128) return launch_grouped<MODE, 2, 2>(a, s);
        return hipErrorInvalidValue;
    }
    if (a.ksplit < 1 || (a.K / KT) % a.ksplit || (MODE != 1 && a.ksplit != 1)) return hipErrorInvalidValue;
    if (MODE != 1 && a.tail_groups > 0 && (!a.tail_part || a.N % 256 || bn != 256))
        return hipErrorInvalidValue;
    switch (bn) {
        case 256: return launch_grouped<MODE, 1, 4>(a, s);
        case 128: return launch_grouped<MODE, 2, 2>(a, s);
        case 64:  return launch_grouped<MODE, 4, 1>(a, s);
        default:  return hipErrorInvalidValue;
    }
}

// Workgroup 8 r + q: rows 16 q .. 16 q + 15 of tail tile r of a launch with
// a split tail, one thread per (row, 4 columns in each 32-column half of a
// 64-column group).  The sums are the tile's S pieces added in piece order
// (loads of four pieces in flight at a time); the tile engine's epilogue of
// MODE then runs on them.
template <int MODE>
__global__ __launch_bounds__(512) void tail_fixup_kernel(GemmArgs a) {
    constexpr int BN = 256;
    const int ntiles = a.N / BN;
    const TailLayout tl = tail_layout(a, ntiles, a.K / KT);
    const int r = blockIdx.x >> 3;
    if (r >= tl.r) return;
    const int tile = tl.dp + r, mtg = tile / ntiles, nt = tile - mtg * ntiles;
    const int e = a.tile_expert[mtg];
    const int row0 = a.offsets[e] + (mtg - a.tile_off[e]) * BM;
    const int rows = min(BM, a.offsets[e + 1] - row0);
    const int row = 16 * (blockIdx.x & 7) + (threadIdx.x >> 5);
    if (row >= rows) return;
    const int g = (threadIdx.x >> 3) & 3, c = (threadIdx.x & 7) * 4;
    const float *src = a.tail_part + (size_t)r * tl.s * BM * BN + row * BN + 64 * g + c;
    constexpr size_t PS = (size_t)BM * BN;   // floats per piece
    // v0: columns 64 g + c .., v1: 32 further (gate and up, or dH of two
    // feature runs for MODE 3).
    fx4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < tl.s; s0 += 4) {
        fx4 p0[4], p1[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {   // (clamped: every load goes out together)
            const size_t sq = (size_t)min(s0 + q, tl.s - 1) * PS;
            p0[q] = *reinterpret_cast<const fx4 *>(src + sq);
            p1[q] = *reinterpret_cast<const fx4 *>(src + sq + 32);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (s0 + q < tl.s) {
                if (s0 + q == 0) { v0 = p0[0]; v1 = p1[0]; }
                else { v0 += p0[q]; v1 += p1[q]; }
            }
    }
    const size_t p = (size_t)(row0 + row);
    if (MODE == 0 || MODE == 2) {
        // Gate (v0) and up (v1) of features 128 nt + 32 g + c ..
        fx4 h;
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] = swiglu_fast(v0[q], v1[q]);
        if (MODE == 0) {
            *reinterpret_cast<fx4 *>(a.c + p * a.ldc + nt * (BN / 2) + 32 * g + c) = h;
        } else {
            float *gu = a.c + p * a.ldc + nt * BN + 64 * g + c;
            *reinterpret_cast<fx4 *>(gu) = v0;
            *reinterpret_cast<fx4 *>(gu + 32) = v1;
            *reinterpret_cast<fx4 *>(a.c2 + p * a.ldc2 + nt * (BN / 2) + 32 * g + c) = h;
        }
    } else {
        // dH of features 256 nt + 64 g + 32 n + c .. (n = 0: v0, 1: v1); the
        // gate and up values of feature f sit at packed columns
        // 64 (f / 32) + f % 32 and 32 past it, replaced by dG and dU.
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            float *gu = a.c + p * a.ldc + 2 * (nt * BN + 64 * g) + 64 * n + c;
            const fx4 dhv = n ? v1 : v0;
            fx4 gv = *reinterpret_cast<const fx4 *>(gu);
            fx4 uv = *reinterpret_cast<const fx4 *>(gu + 32);
            fx4 dg, du;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float gq = gv[q], uq = uv[q], dh = dhv[q];
                const float sg = 1.0f / (1.0f + expf(-gq));
                dg[q] = dh * uq * fmaf(gq * sg, 1.0f - sg, sg);
                du[q] = dh * gq * sg;
            }
            *reinterpret_cast<fx4 *>(gu) = dg;
            *reinterpret_cast<fx4 *>(gu + 32) = du;
        }
    }
}

}  // namespace

// Compute units of the current device (cached; 256 on MI355X).
int device_cus() {
    static int cus = 0;
    if (cus <= 0) {
        int dev = 0, n = 0;
        cus = hipGetDevice(&dev) == hipSuccess &&
                      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) ==
                          hipSuccess && n > 0
                  ? n : 256;
    }
    return cus;
}

GemmPlan gemm_plan(int N, int K, int max_mtiles, bool allow_split) {
    GemmPlan p{0, 1};
    // A last tile may reach past N: its waves without columns only help
    // staging A, so wide tiles lose nothing while they are few.  (T = 1003,
    // d = 320, F = 1376, E = 12, top-3: 108.5 us, with 64-column tiles 133.)
    if (N % 64) return p;
    p.bn = N % 256 == 0 || N >= 1024 ? 256 : N > 64 ? 128 : 64;
    if (allow_split) {
        // Down projection where stream-K is not taken: wide tiles whole (eight
        // of them per CU and more, or no room for partials); the one 64-column
        // tile of N = 64 splits its reduction until the workgroups cover the
        // CUs (its partials are added by the combine), keeping >= 512
        // reduction elements unless the grid is tiny.
        if (p.bn > 64) return p;
        const long slots = 3L * device_cus(), blocks = max_mtiles;
        const int min_k = blocks * 4 < slots ? 128 : 512;
        while (p.ksplit < 4 && blocks * p.ksplit < slots && K % (2 * p.ksplit * KT) == 0 &&
               K / (2 * p.ksplit) >= min_k)
            p.ksplit *= 2;
        return p;
    }
    // Without a split: 256-column tiles (each column split once per 128 rows)
    // while there is one for every CU, 128-column ones (split by both wave
    // rows) down to a quarter, 64-column ones below.  256 columns from half a
    // tile per CU on against one, us per layer: d = 512, F = 2048, E = 4, top-2 T
    // = 256 88.8 / 75.9; d = 2048, F = 1024, E = 16, top-4 T = 200 197.1 / 151.2; d
    // = 2048, F = 8192, E = 2 T = 64 188.0 / 140.0 (one and a half per CU: even).
    // 128 columns from an eighth or half on: within 2 % either way.
    auto tiles = [&](int bn) { return (long)max_mtiles * ((N + bn - 1) / bn); };
    const long cus = device_cus();
    if (p.bn > 128 && tiles(256) < cus) p.bn = 128;
    if (p.bn == 128 && tiles(128) < cus / 4) p.bn = 64;
    return p;
}

// Stream-K takes 128-column tiles over two workgroups per CU: as many partials
// per slot as 256-column tiles over one per CU, with twice the waves (T =
// 4096, d = 256, F = 1024, E = 8: 115.8 us per layer against 121; 256 columns
// over two per CU 126.5, 128 over four 132; even pieces since, 109.6).
constexpr int kSkBN = 128, kSkPerCu = 2;
DownPlan down_plan(int N, int K, int max_mtiles, size_t n, int k) {
    const GemmPlan g = gemm_plan(N, K, max_mtiles, true);
    DownPlan p{g.bn, g.ksplit, 0, 0};
    if (g.bn < 128 || K % KT) return p;
    // Stream-K when the tiles make fewer than ~4 rounds of two workgroups per
    // CU: every workgroup gets the same number of K slices, where whole tiles
    // (or tiles split a fixed 2 or 4 ways) leave a partial last round.
    const long cus = device_cus();
    if ((long)max_mtiles * ((N + 255) / 256) >= 8 * cus) return p;
    const long nks = K / KT, tn = (N + kSkBN - 1) / kSkBN;
    // As many workgroups as the most tiles the rows can make have pieces (few
    // rows over many experts make an m-tile each: T = 15, d = 192, F = 4768, E =
    // 170, top-7: counted on the fewest, 74 workgroups did the work of 160
    // tiles).
    const long tiles_max = max_mtiles * tn;
    const long few = std::min(tiles_max, (long)kSkFewTiles);
    const int most = sk_max_pieces((int)few, (int)nks, k);
    const long groups = std::max(1L, std::min(kSkPerCu * cus,
                                              std::max(tiles_max * sk_max_pieces((int)tiles_max, (int)nks, k),
                                                       few * most)));
    // Too short to split: whole tiles, no piece counts (T = 60, d = 192, F =
    // 96, E = 30, top-6: 44.4 -> 35.3 us).
    if (most == 1 && tiles_max <= groups) {
        p.bn = gemm_plan(N, K, max_mtiles, false).bn;
        return p;
    }
    // The fewest live tiles n rows can make (all rows in full m-tiles) have
    // the most pieces: `most` or the workgroups there are for each, and where
    // these are at most `most`, runs of a `most + 1`-th of a tile and more.
    // The partials stay bounded: slots n N is about groups tiles at most.
    const long tiles_min = (long)((n + BM - 1) / BM) * tn;
    const long per_min = (tiles_min * nks + groups - 1) / groups;
    const long run_slots = std::min((nks - 1 + per_min - 1) / per_min + 1, (long)most + 2);
    p.bn = kSkBN;
    p.streamk = 1;
    p.groups = (int)groups;
    p.slots = (int)std::max(run_slots, std::min(groups / tiles_min, (long)most));
    return p;
}

int gateup_tail_groups(int N, int K, int max_mtiles, int E) {
    const GemmPlan g = gemm_plan(N, K, max_mtiles, false);
    const long cus = device_cus();
    // Less than one round of whole tiles is not split: the pieces' sums and
    // their own launch cost more than the CUs they fill (T = 512, d = 512, F =
    // 2048, E = 8 through the host drop-in 285 us split, 262 whole; 256 tiles
    // or more: the backward of T = 4096, d = 256, F = 1024 419 against 423).
    const long min_tiles = (long)(max_mtiles - E) * (N / 256);
    if (min_tiles < cus) return 0;
    if (g.bn != 256 || N % 256 || K % KT || K / KT < 2 || (long)max_mtiles * (N / 256) >= 8 * cus) return 0;
    return (int)cus;
}

hipError_t launch_gemm_gateup(const GemmArgs &a, hipStream_t s) { return launch_mode<0>(a, s); }
hipError_t launch_gemm_down(const GemmArgs &a, hipStream_t s) { return launch_mode<1>(a, s); }
hipError_t launch_gemm_bwd(const GemmArgs &a, int mode, hipStream_t s) {
    if (mode == 2) return launch_mode<2>(a, s);
    if (mode == 3) return launch_mode<3>(a, s);
    return hipErrorInvalidValue;
}

hipError_t launch_tail_fixup(const GemmArgs &a, int mode, hipStream_t s) {
    if (a.tail_groups <= 0) return hipSuccess;
    if (!a.tail_part || a.N % 256 || a.ldc % 4 || (mode == 2 && a.ldc2 % 4)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)a.tail_groups * 8);
    switch (mode) {
        case 0: hipLaunchKernelGGL(tail_fixup_kernel<0>, grid, dim3(512), 0, s, a); break;
        case 2: hipLaunchKernelGGL(tail_fixup_kernel<2>, grid, dim3(512), 0, s, a); break;
        case 3: hipLaunchKernelGGL(tail_fixup_kernel<3>, grid, dim3(512), 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_gateup_fixup(const GemmArgs &a, hipStream_t s) { return launch_tail_fixup(a, 0, s); }

}  // namespace moe
