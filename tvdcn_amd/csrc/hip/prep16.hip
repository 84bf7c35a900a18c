// fp16 / bf16: what a call lays out before its MFMA kernels, in one launch, and the conversions of its
// results after them, in another. The operands need no scales (16-bit values go into the MFMAs as they
// are, checked by nobody), so the jobs do not depend on each other; as launches of their own each cost
// about 4.7 us, most of it the launch. Every job's blocks are consecutive, 256 threads each:
//   cl      X (B, C, S) -> float channels-last: 64 x 64 tiles through LDS, loads of up to 8 values along
//           S, 16-byte stores along C (a channels-last X is only widened)
//   z, ws   Z and the weight as the data gradient's operands (operands.h)
//   w16     the weight as the forward's
//   bias    grad_bias[c] = sum over batch and space of grad_out, a block per channel
//   fill    the float accumulators zeroed
// float16 128 channels, 8 x 1000, k7, training 152 -> 117 us a step; bfloat16 128 channels,
// 2 x 100x152, inference 115 -> 107.
#include <algorithm>
#include <climits>

#include "operands.h"

namespace tvdcn_hip {
namespace {

using namespace win;

constexpr int TT = 64;   // transpose tile

// V consecutive values of T from an address aligned to them (V = 8: 16 bytes)
template <typename T, int V> __device__ __forceinline__ void load_vec(const T *p, float (&v)[V]) {
    if constexpr (V == 8) {
        const uint4 u = *reinterpret_cast<const uint4 *>(p);
        const T *h = reinterpret_cast<const T *>(&u);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = to_acc<float>(h[i]);
    } else if constexpr (V == 4) {
        const Vec4<float> u = load4_t<float, T>(p);
        v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w;
    } else {
        v[0] = to_acc<float>(*p);
    }
}

// tile (s0, c0) of image b: x [B][C][S] -> xcl [B][S][C] (C % 4 == 0; V divides S)
template <typename T, int V>
__device__ __forceinline__ void cl_tile(float *smem, const T *__restrict__ x, float *__restrict__ xcl, int b, int s0, int c0,
                                        int C, int S) {
    float(*tile)[TT + 1] = reinterpret_cast<float(*)[TT + 1]>(smem);   // [c][s]
    const T *xb = x + (size_t)b * C * S;
    float *ob = xcl + (size_t)b * C * S;
    constexpr int PER = TT / V;   // vectors per row
    // (all of a thread's loads before any is stored)
    constexpr int N = TT * PER / 256;
    float v[N][V];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = threadIdx.x + k * 256, c = c0 + i / PER, s = s0 + i % PER * V;
#pragma unroll
        for (int e = 0; e < V; ++e) v[k][e] = 0.f;
        if (c < C && s < S) load_vec<T, V>(xb + (size_t)c * S + s, v[k]);
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int i = threadIdx.x + k * 256;
#pragma unroll
        for (int e = 0; e < V; ++e) tile[i / PER][i % PER * V + e] = v[k][e];
    }
    __syncthreads();
    const int u = threadIdx.x & 15, r0 = threadIdx.x >> 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int sl = r0 + 16 * k, s = s0 + sl, c = c0 + 4 * u;
        if (s < S && c < C)
            *reinterpret_cast<float4 *>(ob + (size_t)s * C + c) =
                make_float4(tile[4 * u][sl], tile[4 * u + 1][sl], tile[4 * u + 2][sl], tile[4 * u + 3][sl]);
    }
}

// tile (s0, c0) of image b: acc [B][S][C] -> y [B][C][S] + bias[c] (C % 4 == 0; V divides S)
template <typename T, int V>
__device__ __forceinline__ void nc_tile(float *smem, const float *__restrict__ acc, T *__restrict__ y,
                                        const T *__restrict__ bias, int b, int s0, int c0, int C, int S) {
    float(*tile)[TT + 1] = reinterpret_cast<float(*)[TT + 1]>(smem);   // [s][c]
    const float *ib = acc + (size_t)b * C * S;
    T *ob = y + (size_t)b * C * S;
    const int u = threadIdx.x & 15, r0 = threadIdx.x >> 4;
    float4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int s = s0 + r0 + 16 * k, c = c0 + 4 * u;
        v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (s < S && c < C) v[k] = *reinterpret_cast<const float4 *>(ib + (size_t)s * C + c);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float *t = &tile[r0 + 16 * k][4 * u];
        t[0] = v[k].x, t[1] = v[k].y, t[2] = v[k].z, t[3] = v[k].w;
    }
    __syncthreads();
    constexpr int PER = TT / V;
#pragma unroll
    for (int k = 0; k < TT * PER / 256; ++k) {
        const int i = threadIdx.x + k * 256, cl = i / PER, sl = i % PER * V, c = c0 + cl, s = s0 + sl;
        if (c >= C || s >= S) continue;
        const float bv = bias != nullptr ? to_acc<float>(bias[c]) : 0.f;
        T *dst = ob + (size_t)c * S + s;
        if constexpr (V == 1) {
            *dst = from_acc<T, float>(tile[sl][cl] + bv);
        } else {
#pragma unroll
            for (int e = 0; e < V; e += 4)
                store4_t<T, float>(dst + e, Vec4<float>{tile[sl + e][cl] + bv, tile[sl + e + 1][cl] + bv,
                                                        tile[sl + e + 2][cl] + bv, tile[sl + e + 3][cl] + bv});
        }
    }
}

// elements [block * 2048, + 2048) of n, T <-> float, eight per thread (x aligned to four values)
template <typename T>
__device__ __forceinline__ void widen_block(unsigned block, const T *__restrict__ x, float *__restrict__ a, size_t n) {
    const size_t i = ((size_t)block * 256 + threadIdx.x) * 8;
    if (i + 8 <= n) {
        const Vec4<float> v0 = load4_t<float, T>(x + i), v1 = load4_t<float, T>(x + i + 4);
        store4<float>(a + i, v0);
        store4<float>(a + i + 4, v1);
    } else {
        for (size_t j = i; j < n; ++j) a[j] = to_acc<float>(x[j]);
    }
}
// (vec: o aligned to four values)
template <typename T>
__device__ __forceinline__ void narrow_block(unsigned block, const float *__restrict__ a, T *__restrict__ o, size_t n, bool vec) {
    const size_t i = ((size_t)block * 256 + threadIdx.x) * 8;
    if (i + 8 <= n && vec) {
        store4_t<T, float>(o + i, load4<float>(a + i));
        store4_t<T, float>(o + i + 4, load4<float>(a + i + 4));
    } else {
        for (size_t j = i; j < min(n, i + 8); ++j) o[j] = from_acc<T, float>(a[j]);
    }
}

// grad_bias of channel c, the block's 256 threads over batch and space (vec: rows of whole aligned quads): four
// sums per thread and row in a fixed order, then a fixed tree (one sum per thread was a chain four times as long
// as the 1024 threads of a launch of its own have)
template <typename T>
__device__ __forceinline__ void bias_block(float *smem, const T *__restrict__ gout, T *__restrict__ gb, int c, int B, int C,
                                           int S, bool vec, bool accumulate) {
    float acc = 0.f;
    for (int b = 0; b < B; ++b) {
        const T *row = gout + ((size_t)b * C + c) * S;
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        if (vec) {
#pragma unroll 4
            for (int s = 4 * threadIdx.x; s < S; s += 1024) {
                const Vec4<float> v = load4_t<float, T>(row + s);
                a[0] += v.x, a[1] += v.y, a[2] += v.z, a[3] += v.w;
            }
        } else {
            // (every load unconditional, past the row's end its last value: one under a condition is waited for alone)
            for (int s0 = threadIdx.x; s0 < S; s0 += 4096) {
                float v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = to_acc<float>(row[min(s0 + 256 * k, S - 1)]);
#pragma unroll
                for (int k = 0; k < 16; ++k) a[k % 4] += s0 + 256 * k < S ? v[k] : 0.f;
            }
        }
        acc += (a[0] + a[1]) + (a[2] + a[3]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float sum = (smem[0] + smem[1]) + (smem[2] + smem[3]);
        gb[c] = from_acc<T, float>(accumulate ? to_acc<float>(gb[c]) + sum : sum);
    }
}

// blocks of each job of a launch, in this order
struct Prep16Blocks {
    unsigned cl, z, ws, w16, bias, fill;
};
struct Prep16Geo {
    int xC, xS, xst, xct;   // X's channels, positions, their 64-tiles
    int zpb, zvec, bvec, accumulate, bias_c, bias_s;
    size_t x_n, zw_plane, fill_n[3];   // (fill_n in floats, rounded up to 4)
};

template <typename T, int V>
__global__ void __launch_bounds__(256)
prep16_kernel(const Geo g, const Prep16Blocks nb, const Prep16Geo pg, const T *__restrict__ x, float *__restrict__ xcl,
              const T *__restrict__ z, uint16_t *__restrict__ zs, uint16_t *__restrict__ zw, const T *__restrict__ w,
              uint16_t *__restrict__ wsp, uint16_t *__restrict__ w16, const int c_tiles, const int ms32, const int slices,
              const int nmb, const int tpp, const int hp, const int pp, const T *__restrict__ gout, T *__restrict__ gb,
              float *__restrict__ f0, float *__restrict__ f1, float *__restrict__ f2, const int first) {
    __shared__ __align__(16) float smem[WL_TK * BC * 33];
    static_assert(WL_TK * BC * 33 >= TT * (TT + 1), "the copy's tile");
    unsigned L = first + blockIdx.x;
    if (L < nb.cl) {
        if constexpr (V == 0) {
            widen_block<T>(L, x, xcl, pg.x_n);
        } else {
            const int st = (int)(L % pg.xst);
            L /= pg.xst;
            cl_tile<T, V>(smem, x, xcl, (int)(L / pg.xct), st * TT, (int)(L % pg.xct) * TT, pg.xC, pg.xS);
        }
        return;
    }
    L -= nb.cl;
    if (L < nb.z) {
        z_split_block<T, 1>(L, smem, z, zs, zw, nullptr, g.G, g.Mg, g.Pn, ms32, pg.zpb, pg.zvec != 0, pg.zw_plane);
        return;
    }
    L -= nb.z;
    if (L < nb.ws) {
        weight_split_block<T, 1>((int)L, smem, w, wsp, nullptr, g.G, g.Mg, g.Cg, g.Kn, c_tiles, ms32);
        return;
    }
    L -= nb.ws;
    if (L < nb.w16) {
        w16_block<T, 1>(L, nb.w16, w, w16, nullptr, g.G, g.Mg, g.Cg, g.Kn, slices, nmb, tpp, hp, pp);
        return;
    }
    L -= nb.w16;
    if (L < nb.bias) {
        bias_block<T>(smem, gout, gb, (int)L, g.B, pg.bias_c, pg.bias_s, pg.bvec != 0, pg.accumulate != 0);
        return;
    }
    L -= nb.bias;
    float *const f[3] = {f0, f1, f2};
#pragma unroll
    for (int k = 0; k < 3; ++k)
        for (size_t i = ((size_t)L * 256 + threadIdx.x) * 4; i < pg.fill_n[k]; i += (size_t)nb.fill * 1024)
            *reinterpret_cast<float4 *>(f[k] + i) = make_float4(0.f, 0.f, 0.f, 0.f);
}

template <typename T, int V>
__global__ void __launch_bounds__(256)
out16_kernel(const float *__restrict__ acc, T *__restrict__ y, const T *__restrict__ bias, const int C, const int S,
             const int st, const int ct, const unsigned n_y, const float *__restrict__ a0, T *__restrict__ o0, const size_t n0,
             const unsigned nb0, const float *__restrict__ a1, T *__restrict__ o1, const size_t n1, const size_t ny,
             const int vec, const int first) {
    __shared__ __align__(16) float smem[TT * (TT + 1)];
    unsigned L = first + blockIdx.x;
    if (L < n_y) {
        if constexpr (V == 0) {
            narrow_block<T>(L, acc, y, ny, vec & 1);
        } else {
            const int s = (int)(L % st);
            L /= st;
            nc_tile<T, V>(smem, acc, y, bias, (int)(L / ct), s * TT, (int)(L % ct) * TT, C, S);
        }
        return;
    }
    L -= n_y;
    if (L < nb0)
        narrow_block<T>(L, a0, o0, n0, vec & 2);
    else
        narrow_block<T>(L - nb0, a1, o1, n1, vec & 4);
}

bool aligned_to(const void *p, size_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }
unsigned flat_blocks(size_t n) { return (unsigned)((n + 2047) / 2048); }

// the widest vector along rows of S values at p: 8, 4 or 1
int row_vec(const void *p, int S) {
    return S % 8 == 0 && aligned_to(p, 16) ? 8 : S % 4 == 0 && aligned_to(p, 8) ? 4 : 1;
}

template <typename T, typename F> hipError_t by_vec(int v, F &&f) {
    switch (v) {
        case 0: return f(T(), std::integral_constant<int, 0>());
        case 1: return f(T(), std::integral_constant<int, 1>());
        case 4: return f(T(), std::integral_constant<int, 4>());
        case 8: return f(T(), std::integral_constant<int, 8>());
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_prep16(int dtype, const Geo &g, const Prep16 &j, hipStream_t s) {
    Prep16Blocks nb{};
    Prep16Geo pg{};
    int v = 1;
    if (j.x != nullptr) {
        pg.xC = g.C;
        pg.xS = g.Sn;
        pg.x_n = (size_t)g.B * g.C * g.Sn;
        // (channels in whole quads: every batch block's base is as aligned)
        if (j.x_cl) {
            if (!aligned_to(j.x, 8)) return hipErrorInvalidValue;
            v = 0;
            nb.cl = flat_blocks(pg.x_n);
        } else {
            v = row_vec(j.x, g.Sn);
            pg.xst = (g.Sn + TT - 1) / TT;
            pg.xct = (g.C + TT - 1) / TT;
            const long long n = (long long)pg.xst * pg.xct * g.B;
            if (n > INT_MAX) return hipErrorInvalidValue;
            nb.cl = (unsigned)n;
        }
    }
    long long total = nb.cl;
    if (j.z != nullptr) {
        if (j.zw != nullptr && g.Pn % 8 != 0) return hipErrorInvalidValue;
        pg.zpb = (g.Pn + 63) / 64;
        pg.zvec = g.Pn % 4 == 0 && aligned_to(j.z, 8);
        pg.zw_plane = (size_t)g.B * g.M * g.Pn;
        const long long nz = (long long)g.B * g.G * j.wt->ms32 * pg.zpb;
        const long long nw = (long long)g.G * j.wt->c_tiles * j.wt->ms32 * ((g.Kn + WL_TK - 1) / WL_TK);
        if (nz > INT_MAX || nw > INT_MAX) return hipErrorInvalidValue;
        nb.z = (unsigned)nz;
        nb.ws = (unsigned)nw;
        total += nz + nw;
    }
    int slices = 0;
    if (j.w16 != nullptr) {
        slices = j.fw->Cg_pad / BC;
        nb.w16 = (unsigned)std::min<size_t>((j.fw->w16_elems / 8 + 255) / 256, 65536);
        total += nb.w16;
    }
    if (j.gb != nullptr) {
        pg.bias_c = j.bias_c;
        pg.bias_s = j.bias_s;
        pg.bvec = j.bias_s % 4 == 0 && aligned_to(j.gout, 8);
        pg.accumulate = j.accumulate;
        nb.bias = (unsigned)j.bias_c;
        total += nb.bias;
    }
    size_t most = 0;
    for (int k = 0; k < 3; ++k) {
        pg.fill_n[k] = j.fill[k] != nullptr ? (j.fill_n[k] + 3) / 4 * 4 : 0;
        most = std::max(most, pg.fill_n[k]);
    }
    // four 16-byte stores per thread on the largest accumulator
    if (most > 0) nb.fill = (unsigned)std::min<size_t>((most + 4095) / 4096, 4096);
    total += nb.fill;
    auto go = [&](auto tv, auto vv) {
        using T = decltype(tv);
        return launch_block_runs(total, 256, [&](int first, unsigned n) {
            hipLaunchKernelGGL((prep16_kernel<T, decltype(vv)::value>), dim3(n), dim3(256), 0, s, g, nb, pg,
                               static_cast<const T *>(j.x), static_cast<float *>(j.xcl), static_cast<const T *>(j.z),
                               static_cast<uint16_t *>(j.zs), static_cast<uint16_t *>(j.zw), static_cast<const T *>(j.w),
                               static_cast<uint16_t *>(j.wsplit), static_cast<uint16_t *>(j.w16), j.wt ? j.wt->c_tiles : 0,
                               j.wt ? j.wt->ms32 : 0, slices, j.fw ? j.fw->Mg_pad / 16 : 0, j.fw ? j.fw->tpp : 0,
                               j.fw ? j.fw->hp : 0, j.fw ? j.fw->pp : 0, static_cast<const T *>(j.gout),
                               static_cast<T *>(j.gb), static_cast<float *>(j.fill[0]), static_cast<float *>(j.fill[1]),
                               static_cast<float *>(j.fill[2]), first);
        });
    };
    switch (dtype) {
        case kF16: return by_vec<__half>(v, go);
        case kBF16: return by_vec<__hip_bfloat16>(v, go);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_out16(int dtype, const Out16 &j, hipStream_t s) {
    const size_t ny = j.acc != nullptr ? (size_t)j.B * j.C * j.S : 0;
    const int st = (j.S + TT - 1) / TT, ct = (j.C + TT - 1) / TT;
    const int v = j.acc == nullptr ? 1 : j.cl ? 0 : row_vec(j.y, j.S);
    const long long n_y = j.acc == nullptr ? 0 : j.cl ? flat_blocks(ny) : (long long)st * ct * j.B;
    const unsigned nb0 = j.a0 != nullptr ? flat_blocks(j.n0) : 0, nb1 = j.a1 != nullptr ? flat_blocks(j.n1) : 0;
    const long long total = n_y + nb0 + nb1;
    const int vec = (aligned_to(j.y, 8) ? 1 : 0) | (aligned_to(j.o0, 8) ? 2 : 0) | (aligned_to(j.o1, 8) ? 4 : 0);
    auto go = [&](auto tv, auto vv) {
        using T = decltype(tv);
        return launch_block_runs(total, 256, [&](int first, unsigned n) {
            hipLaunchKernelGGL((out16_kernel<T, decltype(vv)::value>), dim3(n), dim3(256), 0, s,
                               static_cast<const float *>(j.acc), static_cast<T *>(j.y), static_cast<const T *>(j.bias), j.C,
                               j.S, st, ct, (unsigned)n_y, static_cast<const float *>(j.a0), static_cast<T *>(j.o0), j.n0, nb0,
                               static_cast<const float *>(j.a1), static_cast<T *>(j.o1), j.n1, ny, vec, first);
        });
    };
    switch (dtype) {
        case kF16: return by_vec<__half>(v, go);
        case kBF16: return by_vec<__hip_bfloat16>(v, go);
    }
    return hipErrorInvalidValue;
}

}  // namespace tvdcn_hip
