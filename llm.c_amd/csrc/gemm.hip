// gemm.hip — the combine, weight packing, m-tile order, synthetic fill and copy
// kernels around the grouped expert GEMMs (gemm_split.hip).
//
// Layout (device, packed once at upload), per expert a matrix of N packed
// rows by K, stored as 16 x 16 tiles ("units", 1 KB) in MFMA operand order:
//   unit (nb, qb) at ((nb * K/16) + qb) * 256 floats holds rows
//   16nb..16nb+15, k = 16qb..16qb+15; element (row 16nb + j, k = 16qb + 4h + s)
//   sits at h*64 + j*4 + s, so lane 16h + j of a wave loads its 16-byte
//   piece at lane*4 and one wave instruction reads one contiguous unit; the
//   units of one row block follow each other along K.
//   gate/up  wgu [E][2F rows][d]: packed rows 64*fb + c hold gate feature
//            32*fb + c (c < 32) and up feature 32*fb + c - 32 (c >= 32).
//   down     wdT [E][d rows][F]: row n holds W_down[:, n].
#include "moe_internal.h"
#include "moe_math.h"
#include "synth.h"
#include <algorithm>
#include <type_traits>

namespace moe {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BM = kGemmBM;   // 128
// One wave instruction of LDS DMA: lane i's 16 bytes at g go to LDS byte
// address lds + 16 i (lds wave-uniform, passed in M0).  Written as asm: the
// compiler books its own LDS DMA builtin as an LDS access as well as a
// vector load.  The DMA counts on vmcnt only and is waited for explicitly
// (GEMM_WAIT_VMCNT) before the barrier after which its LDS is read.
__device__ __forceinline__ void gemm_dma16(const float *g, unsigned lds) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(g), "{m0}"(lds) : "memory");
}
// s_waitcnt limiting only the vector-memory count (expcnt, lgkmcnt at max).
#define GEMM_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x0F70)

// out[t] = sum over slots of gw * y, one FMA per slot in slot order
// (src/transformer.c:355-358 after contraction), optionally added into out.
// With ksplit > 1 each slot's y is the sum of its split partials, added in
// split order (with pieces: as many as its column block's tile had).  With
// PARTS (ksplit > 1 or pieces) the first 8 partials of a slot are loaded
// together (clamped, masked), and with KS > 0 (k = KS) every slot's loads
// go out before the first sum, so no load waits for another.
template <int KS, bool PARTS>
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a) {
    constexpr int KB = KS > 0 ? KS : 1;   // slots whose loads go out together
    constexpr int NQ = PARTS ? 8 : 1;     // partials loaded together
    const int d4 = a.d >> 2;
    const size_t total = (size_t)a.T * d4;
    const int k = KS > 0 ? KS : a.k;
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const int t = (int)(i / d4), c = (int)(i % d4);
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < k; k0 += KB) {
            floatx4 q[KB][NQ];
            float w[KB];
            int np[KB];
            const float *yp[KB];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const size_t slot = (size_t)t * a.k + k0 + kb;
                w[kb] = a.gw[slot];
                yp[kb] = a.ys + slot * a.d + 4 * c;
                np[kb] = !PARTS ? 1
                         : a.pieces ? a.pieces[slot * ((a.d + a.pieces_cols - 1) / a.pieces_cols) + 4 * c / a.pieces_cols]
                                    : a.ksplit;
                np[kb] = max(np[kb], 1);
#pragma unroll
                for (int u = 0; u < NQ; ++u)
                    q[kb][u] = *reinterpret_cast<const floatx4 *>(
                        yp[kb] + (size_t)min(u, np[kb] - 1) * a.split_stride);
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                floatx4 y = q[kb][0];
#pragma unroll
                for (int u = 1; u < NQ; ++u)
                    if (u < np[kb])
#pragma unroll
                        for (int j = 0; j < 4; ++j) y[j] = y[j] + q[kb][u][j];
                for (int sp = NQ; sp < np[kb]; ++sp) {
                    const floatx4 p = *reinterpret_cast<const floatx4 *>(
                        yp[kb] + (size_t)sp * a.split_stride);
#pragma unroll
                    for (int j = 0; j < 4; ++j) y[j] = y[j] + p[j];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = fmaf(w[kb], y[j], acc[j]);
            }
        }
        floatx4 *o = reinterpret_cast<floatx4 *>(a.out + (size_t)t * a.d + 4 * c);
        if (a.accumulate) {
            floatx4 v = *o;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = v[j] + acc[j];
            *o = v;
        } else {
            *o = acc;
        }
    }
}

// The same for many split-K partials (the fused decode kernel writes one per
// 64 features): G lanes share an output float4, each summing up to 8
// consecutive partials of a slot in split order (PL: 2 for steps of a few
// tokens, so that more workgroups share the loads); lane 0 adds the G group
// sums in a fixed tree order and applies the slot's gate weight.  KS > 0:
// k = KS at compile time, and every load of the lane (partials, gate
// weights, the accumulated output) is issued before the first sum.
template <int G, int KS, int PL = 8>
__global__ __launch_bounds__(256) void combine_groups_kernel(CombineArgs a) {
    constexpr int KB = KS > 0 ? KS : 1;   // slots whose loads go out together
    const int d4 = a.d >> 2;
    const size_t gid = ((size_t)blockIdx.x * 256 + threadIdx.x) / G;
    const int g = threadIdx.x % G;
    const bool valid = gid < (size_t)a.T * d4;
    const int t = valid ? (int)(gid / d4) : 0, c4 = valid ? (int)(gid % d4) : 0;
    const int s0 = PL * g, s1 = min(s0 + PL, a.ksplit);
    const int k = KS > 0 ? KS : a.k;
    floatx4 *o = reinterpret_cast<floatx4 *>(a.out + (size_t)t * a.d + 4 * c4);
    floatx4 prev = {0.f, 0.f, 0.f, 0.f};
    if (KS > 0 && a.accumulate && g == 0) prev = *o;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < k; k0 += KB) {
        floatx4 p[KB][PL];
        float w[KB];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const float *yp = a.ys + ((size_t)t * a.k + k0 + kb) * a.d + 4 * c4;
#pragma unroll
            for (int u = 0; u < PL; ++u)
                p[kb][u] = *reinterpret_cast<const floatx4 *>(
                    yp + (size_t)min(s0 + u, a.ksplit - 1) * a.split_stride);
            w[kb] = a.gw[(size_t)t * a.k + k0 + kb];
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            floatx4 y = {0.f, 0.f, 0.f, 0.f};
            if (s0 < s1) y = p[kb][0];
#pragma unroll
            for (int u = 1; u < PL; ++u)
                if (s0 + u < s1)
#pragma unroll
                    for (int j = 0; j < 4; ++j) y[j] = y[j] + p[kb][u][j];
#pragma unroll
            for (int m = G / 2; m >= 1; m >>= 1)
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = y[j] + __shfl_xor(y[j], m, G);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = fmaf(w[kb], y[j], acc[j]);
        }
    }
    if (valid && g == 0) {
        if (a.accumulate) {
            floatx4 v = KS > 0 ? prev : *o;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = v[j] + acc[j];
            *o = v;
        } else {
            *o = acc;
        }
    }
}

// Packs source matrix src [K x N] (reference layout) into the unit layout
// (unpack != 0: the inverse).  Source column c goes to packed row
// c (mode 0, down), 64*(c/32) + c%32 (mode 1, gate) or that + 32 (mode 2,
// up).  One workgroup moves a 32 x 32 block = 4 units through LDS; grid z
// runs over experts whose matrices are src_e and dst_e floats apart.
__global__ __launch_bounds__(256) void pack_kernel(float *src, float *dst, int K, int N,
                                                    int mode, int unpack, size_t src_e = 0,
                                                    size_t dst_e = 0) {
    __shared__ float tile[32][33];
    src += blockIdx.z * src_e;
    dst += blockIdx.z * dst_e;
    const int c0 = blockIdx.x * 32, k0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int row0 = mode == 0 ? c0 : 64 * (c0 >> 5) + (mode == 2 ? 32 : 0);
    const int t = threadIdx.x;
    const int h = t >> 6, j = (t >> 2) & 15, sx = t & 3;
    if (!unpack) {
        for (int r = ty; r < 32; r += 8) tile[r][tx] = src[(size_t)(k0 + r) * N + c0 + tx];
        __syncthreads();
        for (int u = 0; u < 4; ++u) {
            const int nbl = u >> 1, qbl = u & 1;
            const size_t unit = (size_t)((row0 >> 4) + nbl) * (K / 16) + (k0 >> 4) + qbl;
            dst[unit * 256 + t] = tile[qbl * 16 + 4 * h + sx][nbl * 16 + j];
        }
    } else {
        for (int u = 0; u < 4; ++u) {
            const int nbl = u >> 1, qbl = u & 1;
            const size_t unit = (size_t)((row0 >> 4) + nbl) * (K / 16) + (k0 >> 4) + qbl;
            tile[qbl * 16 + 4 * h + sx][nbl * 16 + j] = dst[unit * 256 + t];
        }
        __syncthreads();
        for (int r = ty; r < 32; r += 8) src[(size_t)(k0 + r) * N + c0 + tx] = tile[r][tx];
    }
}

// dst[e] = the transpose of src[e] in the unit layout: src [E][R rows][C],
// dst [E][C rows][R].  Four 16 x 16 units per workgroup, 64 threads each;
// thread q writes destination floats o = 4q..4q+3 of its unit (row 16rb + j,
// k = 16kb + 4h + s for o = 64h + 4j + s), read from source row
// 16kb + 4h + s, k = 16rb + j.
__global__ __launch_bounds__(256) void transpose_units_kernel(const float *src, float *dst, int R,
                                                              int C) {
    const int units = (R / 16) * (C / 16);
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= units) return;
    const int rb = u % (C / 16), kb = u / (C / 16);
    const size_t base = (size_t)blockIdx.y * R * C;
    const int q = threadIdx.x & 63, h = q >> 4, j = q & 15;
    const float *sp = src + base + ((size_t)kb * (C / 16) + rb) * 256 + (j >> 2) * 64 + (j & 3);
    floatx4 v;
#pragma unroll
    for (int sl = 0; sl < 4; ++sl) v[sl] = sp[(4 * h + sl) * 4];
    *reinterpret_cast<floatx4 *>(dst + base + ((size_t)rb * (R / 16) + kb) * 256 + 4 * q) = v;
}

__global__ __launch_bounds__(256) void fill_normal_kernel(float *dst, size_t n, uint64_t seed,
                                                           uint64_t stream_id, float mean,
                                                           float std) {
    for (size_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = synth_normal(seed, stream_id, i, mean, std);
}

__global__ __launch_bounds__(256) void zero_ints_kernel(int *p, int n) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = 0;
}

// The short-first m-tile order: thread t takes experts [t EPT, (t + 1)
// EPT); the count of short last m-tiles before each expert comes from a
// workgroup scan (wave shuffles, then the wave totals).
constexpr int kOrderThreads = 1024;
__global__ __launch_bounds__(kOrderThreads) void short_first_order_kernel(const int *offsets,
                                                                          const int *tile_off,
                                                                          int E, int *order) {
    __shared__ int wtot[kOrderThreads / 64];
    __shared__ int nshort;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int ept = (E + kOrderThreads - 1) / kOrderThreads;
    const int e0 = min(E, tid * ept), e1 = min(E, e0 + ept);
    auto is_short = [&](int e) {
        const int m = tile_off[e + 1] - tile_off[e];
        return m > 0 && offsets[e + 1] - offsets[e] - BM * (m - 1) <= 96;
    };
    int c = 0;
    for (int e = e0; e < e1; ++e) c += is_short(e);
    int v = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    if (lane == 63) wtot[w] = v;
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        for (int i = 0; i < kOrderThreads / 64; ++i) {
            const int t = wtot[i];
            wtot[i] = run;
            run += t;
        }
        nshort = run;
    }
    __syncthreads();
    int sb = wtot[w] + v - c;   // short m-tiles of the experts before e0
    const int ns = nshort;
    for (int e = e0; e < e1; ++e) {
        const int t0 = tile_off[e], m = tile_off[e + 1] - t0;
        const bool sh = is_short(e);
        for (int j = 0; j < m; ++j) {
            const int mt = t0 + j;
            if (sh && j == m - 1) order[sb] = mt;
            else order[ns + mt - sb] = mt;
        }
        sb += sh;
    }
}

}  // namespace

hipError_t launch_short_first_order(const int *offsets, const int *tile_off, int E, int *order,
                                    hipStream_t s) {
    if (E <= 0 || E > 4 * kOrderThreads || !order) return hipErrorInvalidValue;
    hipLaunchKernelGGL(short_first_order_kernel, dim3(1), dim3(kOrderThreads), 0, s, offsets,
                       tile_off, E, order);
    return hipGetLastError();
}

hipError_t launch_combine(const CombineArgs &a, hipStream_t s) {
    if (a.pieces && (a.pieces_cols <= 0 || a.pieces_cols % 4))
        return hipErrorInvalidValue;
    if (!a.pieces && a.T <= 8 && a.ksplit > 8 && a.ksplit <= 128) {
        // A few tokens: two partials per lane, up to 64 lanes per output.
        const int groups = (a.ksplit + 1) / 2;
        const size_t n = (size_t)a.T * (a.d >> 2);
        if (n == 0) return hipSuccess;
        auto go = [&](auto kern, int G) {
            hipLaunchKernelGGL(kern, dim3((unsigned)((n * G + 255) / 256)), dim3(256), 0, s, a);
        };
        auto by_k = [&](auto gc) {
            constexpr int G = decltype(gc)::value;
            if (a.k == 1)      go(combine_groups_kernel<G, 1, 2>, G);
            else if (a.k == 2) go(combine_groups_kernel<G, 2, 2>, G);
            else               go(combine_groups_kernel<G, 0, 2>, G);
        };
        if (groups <= 8)       by_k(std::integral_constant<int, 8>{});
        else if (groups <= 16) by_k(std::integral_constant<int, 16>{});
        else if (groups <= 32) by_k(std::integral_constant<int, 32>{});
        else                   by_k(std::integral_constant<int, 64>{});
        return hipGetLastError();
    }
    if (!a.pieces && a.ksplit > 8 && a.ksplit <= 128) {
        const int groups = (a.ksplit + 7) / 8;
        const size_t n = (size_t)a.T * (a.d >> 2);
        if (n == 0) return hipSuccess;
        auto go = [&](auto kern, int G) {
            hipLaunchKernelGGL(kern, dim3((unsigned)((n * G + 255) / 256)), dim3(256), 0, s, a);
        };
        auto by_k = [&](auto gc) {
            constexpr int G = decltype(gc)::value;
            if (a.k == 1)      go(combine_groups_kernel<G, 1>, G);
            else if (a.k == 2) go(combine_groups_kernel<G, 2>, G);
            else               go(combine_groups_kernel<G, 0>, G);
        };
        if (groups <= 2)       by_k(std::integral_constant<int, 2>{});
        else if (groups <= 4)  by_k(std::integral_constant<int, 4>{});
        else if (groups <= 8)  by_k(std::integral_constant<int, 8>{});
        else if (groups <= 16) by_k(std::integral_constant<int, 16>{});
        else return hipErrorInvalidValue;
        return hipGetLastError();
    }
    size_t total = (size_t)a.T * (a.d >> 2);
    if (total == 0) return hipSuccess;
    unsigned blocks = (unsigned)std::min<size_t>((total + 255) / 256, 8192);
    auto go = [&](auto parts) {
        constexpr bool P = decltype(parts)::value;
        if (a.k == 1)      hipLaunchKernelGGL((combine_kernel<1, P>), dim3(blocks), dim3(256), 0, s, a);
        else if (a.k == 2) hipLaunchKernelGGL((combine_kernel<2, P>), dim3(blocks), dim3(256), 0, s, a);
        else if (a.k == 4) hipLaunchKernelGGL((combine_kernel<4, P>), dim3(blocks), dim3(256), 0, s, a);
        else               hipLaunchKernelGGL((combine_kernel<0, P>), dim3(blocks), dim3(256), 0, s, a);
    };
    if (a.pieces || a.ksplit > 1) go(std::true_type{});
    else                          go(std::false_type{});
    return hipGetLastError();
}

// dst[r][c] = src[r][c] for c < min(sc, dc), 0 for sc <= c < dc: rows widened
// with zeros, or cut to their first dc columns.
__global__ __launch_bounds__(256) void copy_rows_kernel(const float *src, int rows, int sc,
                                                        float *dst, int dc) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)rows * dc) return;
    const size_t r = i / dc;
    const int c = (int)(i - r * dc);
    dst[i] = c < sc ? src[r * sc + c] : 0.0f;
}

hipError_t launch_copy_rows(const float *src, int rows, int src_cols, float *dst, int dst_cols,
                            hipStream_t s) {
    const size_t n = (size_t)rows * dst_cols;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(copy_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src,
                       rows, src_cols, dst, dst_cols);
    return hipGetLastError();
}

hipError_t launch_pack_gateup(const float *wg, const float *wu, float *dst, int d, int F,
                              hipStream_t s) {
    dim3 grid(F / 32, d / 32);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, const_cast<float *>(wg), dst, d, F, 1, 0);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, const_cast<float *>(wu), dst, d, F, 2, 0);
    return hipGetLastError();
}

hipError_t launch_unpack_gateup(const float *src, float *wg, float *wu, int d, int F,
                                hipStream_t s) {
    dim3 grid(F / 32, d / 32);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, wg, const_cast<float *>(src), d, F, 1, 1);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, wu, const_cast<float *>(src), d, F, 2, 1);
    return hipGetLastError();
}

hipError_t launch_unpack_experts(const float *wgu, const float *wdT, float *wg, float *wu,
                                 float *wd, int E, int d, int F, hipStream_t s) {
    const size_t dF = (size_t)d * F;
    dim3 ggu(F / 32, d / 32, E), gdn(d / 32, F / 32, E);
    hipLaunchKernelGGL(pack_kernel, ggu, dim3(256), 0, s, wg, const_cast<float *>(wgu), d, F, 1, 1,
                       dF, 2 * dF);
    hipLaunchKernelGGL(pack_kernel, ggu, dim3(256), 0, s, wu, const_cast<float *>(wgu), d, F, 2, 1,
                       dF, 2 * dF);
    hipLaunchKernelGGL(pack_kernel, gdn, dim3(256), 0, s, wd, const_cast<float *>(wdT), F, d, 0, 1,
                       dF, dF);
    return hipGetLastError();
}

hipError_t launch_transpose_units(const float *src, float *dst, int R, int C, int E,
                                  hipStream_t s) {
    if (R % 16 || C % 16 || E <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(transpose_units_kernel,
                       dim3((unsigned)(((R / 16) * (C / 16) + 3) / 4), (unsigned)E),
                       dim3(256), 0, s, src, dst, R, C);
    return hipGetLastError();
}

hipError_t launch_pack_down(const float *wd, float *dst, int F, int d, hipStream_t s) {
    dim3 grid(d / 32, F / 32);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, const_cast<float *>(wd), dst, F, d, 0, 0);
    return hipGetLastError();
}

hipError_t launch_unpack_down(const float *src, float *wd, int F, int d, hipStream_t s) {
    dim3 grid(d / 32, F / 32);
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, s, wd, const_cast<float *>(src), F, d, 0, 1);
    return hipGetLastError();
}

hipError_t launch_fill_normal(float *dst, size_t n, uint64_t seed, uint64_t stream_id,
                              float mean, float std, hipStream_t s) {
    if (n == 0) return hipSuccess;
    unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 65536);
    hipLaunchKernelGGL(fill_normal_kernel, dim3(blocks), dim3(256), 0, s, dst, n, seed,
                       stream_id, mean, std);
    return hipGetLastError();
}

// A read of known size through one load path (counter calibration): MODE 0
// LDS DMA (global_load_lds_dwordx4), 1 buffer loads into
// registers with the default cache policy, 2 the same loads non-temporal
// (the decode weight stream).  Workgroup b (4 waves) reads bytes [b span,
// (b + 1) span) in 4 KB steps, eight 1 KB wave instructions in flight; the
// sum of what it read (MODE 0: of its LDS) goes to out[b].
constexpr int kProbeGroups = 1024;
template <int MODE>
__global__ __launch_bounds__(256) void read_probe_kernel(const float *src, size_t span,
                                                         float *out) {
    __shared__ __align__(16) float lds[4][8][256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const char *base = reinterpret_cast<const char *>(src) + (size_t)blockIdx.x * span;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (size_t off = 0; off < span; off += 4096 * 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const char *g = base + off + 4096 * i + 1024 * wave;
            if (MODE == 0) {
                gemm_dma16(reinterpret_cast<const float *>(g) + 4 * lane,
                           (unsigned)(size_t)(const __attribute__((address_space(3))) float *)
                               &lds[wave][i][0]);
            } else {
                const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<char *>(g), (short)0, 1024, 0x00020000);
                acc += __builtin_amdgcn_raw_buffer_load_b128(r, 16 * lane, 0, MODE == 2 ? 2 : 0);
            }
        }
        if (MODE == 0) GEMM_WAIT_VMCNT(0);
    }
    if (MODE == 0) {
        __syncthreads();
        acc[0] = lds[wave][lane & 7][threadIdx.x & 255];
    }
    if (threadIdx.x == 0) out[blockIdx.x] = acc[0] + acc[1] + acc[2] + acc[3];
}

hipError_t launch_read_probe(const float *src, size_t bytes, int mode, float *out,
                             hipStream_t s) {
    const size_t step = (size_t)kProbeGroups * 4096 * 8;
    if (bytes == 0 || bytes % step != 0 || mode < 0 || mode > 2) return hipErrorInvalidValue;
    const size_t span = bytes / kProbeGroups;
    if (mode == 0)
        hipLaunchKernelGGL(read_probe_kernel<0>, dim3(kProbeGroups), dim3(256), 0, s, src, span, out);
    else if (mode == 1)
        hipLaunchKernelGGL(read_probe_kernel<1>, dim3(kProbeGroups), dim3(256), 0, s, src, span, out);
    else
        hipLaunchKernelGGL(read_probe_kernel<2>, dim3(kProbeGroups), dim3(256), 0, s, src, span, out);
    return hipGetLastError();
}

// dst = src, n16 16-byte units; either side may be pinned host memory,
// which the kernel then reads or writes across the bus itself.
__global__ __launch_bounds__(256) void copy16_kernel(const uint4 *src, uint4 *dst, size_t n16) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

hipError_t launch_copy16(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    if (bytes % 16 || reinterpret_cast<uintptr_t>(dst) % 16 || reinterpret_cast<uintptr_t>(src) % 16)
        return hipErrorInvalidValue;
    const size_t n16 = bytes / 16;
    const unsigned blocks = (unsigned)std::min<size_t>((n16 + 255) / 256, 1024);
    hipLaunchKernelGGL(copy16_kernel, dim3(blocks), dim3(256), 0, s, static_cast<const uint4 *>(src),
                       static_cast<uint4 *>(dst), n16);
    return hipGetLastError();
}

hipError_t launch_zero_ints(int *p, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(zero_ints_kernel, dim3((unsigned)std::min(1024, (n + 255) / 256)), dim3(256),
                       0, s, p, n);
    return hipGetLastError();
}

}  // namespace moe
