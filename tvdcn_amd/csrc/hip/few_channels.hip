// Layers of few sampled-side channels (image and label channel counts, toy layers, float64 checks):
// the whole column of a pixel, C * Kn values, fits beside the others of a 64-pixel tile in LDS, so
// one workgroup forms it once and runs every contraction of the call on it.
//
//   forward (and the transposed op's grad_input): Y[m][p] = bias[m] + sum_k W[m][k] S[k][p]
//   data: G[k][p] = sum_m W[m][k] Z[m][p], then per (pixel, tap) the scatter of mask * G into dX, the
//         offset / mask gradients (a thread holds every channel of its pixel and tap: plain stores, no
//         accumulators), dW[m][k] = sum_p Z S, and the bias gradient sum_p Z
//
// Replaces the same reference pairs as the general kernels (tvdcn/csrc/ops/cuda/
// deform_conv2d_kernel.cpp:341-380, 518-626 and the 1D / 3D twins). These calls are a few microseconds
// of work: what bounds them is the chain of dependent loads (offset, corners) of a pixel and the
// launches. So X and Z are read where they are (no channels-last copy, no weight layouts, no operand
// checks: fp32 / fp64 16x16x4 MFMAs on the values themselves), a pixel's taps are spread over the four
// waves, and the forward is one launch, the backward three. 3 -> 5 channels, k3, 4 x 10x10, float32:
// inference 97 -> 12 us a call, training 323 -> 93 (most of it now host time).
#include <algorithm>

#include "kernels.h"

namespace tvdcn_hip {
namespace {

constexpr int BP = 64;    // column pixels per tile
constexpr int NW = 4;     // waves: 16 pixels each in the contractions, every fourth tap in the sampling
// LDS row strides: 16 lanes along a row and 4 rows (forward), or 16 rows and 4 along a row (weight
// gradient) fall on different banks
constexpr int LDF = BP + 16, LDG = BP + 4;

// Sum over the wave, in every lane: a tree (fp32 on the VALU: quad xor 1, quad xor 2, half-row mirror, row mirror,
// then the rows swapped; fp64 through the LDS crossbar)
__device__ __forceinline__ float wave_sum(float v) {
    auto dpp = [&](auto ctrl) {
        v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    dpp(std::integral_constant<int, 0xB1>());
    dpp(std::integral_constant<int, 0x4E>());
    dpp(std::integral_constant<int, 0x141>());
    dpp(std::integral_constant<int, 0x140>());
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// The corners of one (pixel, tap, offset group)
template <int DIM, typename A> struct CornerSet {
    AxisW<DIM, A> aw;
    int idx[1 << DIM];
    bool ok[1 << DIM];
    template <typename T>
    __device__ __forceinline__ CornerSet(const Geo &g, const T *__restrict__ offset, int b, int p, int t, int ogi) {
        aw = axis_weights<DIM, A>(g, sample_point<DIM, A, T>(g, offset, b, p, t, ogi), offset != nullptr);
#pragma unroll
        for (int i = 0; i < (1 << DIM); ++i) corner_at<DIM, A>(g, aw, i, idx[i], ok[i]);
    }
};

// f(c0, c1, corners, mask value) for each run [c0, c1) of channels of one offset and one mask group
template <int DIM, typename A, typename T, typename F>
__device__ __forceinline__ void for_channel_runs(const Geo &g, const T *__restrict__ offset, const T *__restrict__ mask,
                                                 int b, int p, int t, F &&f) {
    const int ro = g.og ? g.cpo : g.C, rm = g.mg ? g.cpm : g.C;
    for (int c0 = 0; c0 < g.C;) {
        const int ogi = c0 / ro, mgi = c0 / rm;
        const int c1 = min((ogi + 1) * ro, (mgi + 1) * rm);
        const CornerSet<DIM, A> cs(g, offset, b, p, t, ogi);
        f(c0, c1, cs, mask_at<A, T>(g, mask, b, mgi, t, p), ogi, mgi);
        c0 = c1;
    }
}

// x: sampled tensor, element (b, c, s) at b * C * Sn + c * xc + s * xp. Workgroup = a tile and every
// gridDim.y-th block of 64 rows
template <int DIM, typename T, typename A>
__global__ void __launch_bounds__(64 * NW)
few_fwd_kernel(const Geo g, const T *__restrict__ x, const int xc, const int xp, const T *__restrict__ w,
               const T *__restrict__ offset, const T *__restrict__ mask, const T *__restrict__ bias, T *__restrict__ y) {
    constexpr int NC = 1 << DIM;
    typedef typename Acc4<A>::type acc4;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    A *S = reinterpret_cast<A *>(smem_raw);   // [C * Kn][LDF]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4;
    const int n0 = blockIdx.x * BP;
    {
        const int n = n0 + lane;
        const bool ok = n < g.NP;
        const int b = fdiv(g.dPn, ok ? n : 0), p = (ok ? n : 0) - b * g.Pn;
        const T *xb = x + (size_t)b * g.C * g.Sn;
        for (int t = wave; t < g.Kn; t += NW)
            for_channel_runs<DIM, A, T>(g, offset, mask, b, p, t, [&](int c0, int c1, const CornerSet<DIM, A> &cs, A mk, int, int) {
                A cw[NC];
#pragma unroll
                for (int i = 0; i < NC; ++i) cw[i] = cs.aw.inside && ok ? corner_weight<DIM, A>(cs.aw, i) : A(0);
#pragma unroll 4
                for (int c = c0; c < c1; ++c) {
                    A v = A(0);
#pragma unroll
                    for (int i = 0; i < NC; ++i)
                        if (cs.ok[i] && cs.aw.inside) v += cw[i] * to_acc<A>(xb[c * xc + cs.idx[i] * xp]);
                    S[(c * g.Kn + t) * LDF + lane] = ok ? v * mk : A(0);
                }
            });
    }
    __syncthreads();
    const int px = wave * 16 + (lane & 15), n = n0 + px;
    const int b = fdiv(g.dPn, n < g.NP ? n : 0), p = n - b * g.Pn;
    const int Kg = g.Cg * g.Kn;
    const A zero = A(0);
    for (int grp = 0; grp < g.G; ++grp) {
        const A *Sg = S + (size_t)grp * Kg * LDF + px;
        for (int m0 = blockIdx.y * 64; m0 < g.Mg; m0 += gridDim.y * 64) {
            acc4 acc[4];
            const int nb = min(4, (g.Mg - m0 + 15) / 16);
            const T *wr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[r] = acc4{zero, zero, zero, zero};
                // (rows past Mg repeat its last one: they are not stored)
                wr[r] = w + ((size_t)grp * g.Mg + min(m0 + 16 * r + (lane & 15), g.Mg - 1)) * Kg;
            }
#pragma unroll 4
            for (int k0 = 0; k0 < Kg; k0 += 4) {
                const int k = k0 + q;
                const A bv = k < Kg ? Sg[k * LDF] : zero;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < nb) acc[r] = mfma16x16x4(k < Kg ? to_acc<A>(wr[r][k]) : zero, bv, acc[r]);
            }
            if (n < g.NP)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int m = m0 + 16 * r + mfma_row<A>(lane, v);
                        if (r < nb && m < g.Mg) {
                            const int mg = grp * g.Mg + m;
                            A o = acc[r][v];
                            if (bias != nullptr) o += to_acc<A>(bias[mg]);
                            y[((size_t)b * g.M + mg) * g.Pn + p] = from_acc<T, A>(o);
                        }
                    }
        }
    }
}

// gx (accumulation type, x's order, or null: no scatter); goff / gmask (null: not wanted); part (null: no
// weight gradient): this workgroup's [M][Kg + 1] partial sums, the last column the bias gradient's.
// Workgroup = a run of `chunks` tiles.
template <int DIM, typename T, typename A>
__global__ void __launch_bounds__(64 * NW)
few_data_kernel(const Geo g, const T *__restrict__ z, const T *__restrict__ x, const int xc, const int xp,
                const T *__restrict__ w, const T *__restrict__ offset, const T *__restrict__ mask, A *__restrict__ gx,
                T *__restrict__ goff, T *__restrict__ gmask, A *__restrict__ part, const int chunks) {
    constexpr int NC = 1 << DIM;
    typedef typename Acc4<A>::type acc4;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int K = g.C * g.Kn, Kg = g.Cg * g.Kn;
    A *Gs = reinterpret_cast<A *>(smem_raw);      // [K][LDG]
    A *S = Gs + (size_t)K * LDG;                  // [K][LDG] (part)
    int *zo = reinterpret_cast<int *>(S + (part != nullptr ? (size_t)K * LDG : 0));   // [BP] offsets of the pixels in z
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4;
    const A zero = A(0);
    const bool coord = goff != nullptr || gmask != nullptr;
    if (part != nullptr) part += (size_t)blockIdx.x * g.M * (Kg + 1);

    for (int ch = 0; ch < chunks; ++ch) {
        const int n0 = (blockIdx.x * chunks + ch) * BP;
        if (n0 >= g.NP) break;
        const int nl = n0 + lane;
        const bool ok = nl < g.NP;
        const int b = fdiv(g.dPn, ok ? nl : 0), p = (ok ? nl : 0) - b * g.Pn;
        if (wave == 0) zo[lane] = ok ? b * g.M * g.Pn + p : -1;
        __syncthreads();
        // ---- G[k][px]
        {
            const int px = wave * 16 + (lane & 15);
            const int o = zo[px];
            for (int grp = 0; grp < g.G; ++grp) {
                const T *zg = z + (size_t)grp * g.Mg * g.Pn + max(o, 0);
                for (int k0 = 0; k0 < Kg; k0 += 64) {
                    acc4 acc[4];
                    const int nb = min(4, (Kg - k0 + 15) / 16);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[r] = acc4{zero, zero, zero, zero};
                    const T *wg = w + (size_t)grp * g.Mg * Kg;
#pragma unroll 4
                    for (int m0 = 0; m0 < g.Mg; m0 += 4) {
                        const int m = m0 + q;
                        const A bv = m < g.Mg && o >= 0 ? to_acc<A>(zg[(size_t)m * g.Pn]) : zero;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int k = k0 + 16 * r + (lane & 15);
                            if (r < nb) acc[r] = mfma16x16x4(m < g.Mg && k < Kg ? to_acc<A>(wg[(size_t)m * Kg + k]) : zero, bv, acc[r]);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int k = k0 + 16 * r + mfma_row<A>(lane, v);
                            if (r < nb && k < Kg) Gs[(grp * Kg + k) * LDG + px] = acc[r][v];
                        }
                }
            }
        }
        __syncthreads();
        // ---- per (pixel, tap): scatter, offset / mask gradients, the column for the weight gradient
        const T *xb = x != nullptr ? x + (size_t)b * g.C * g.Sn : nullptr;
        A *gxb = gx != nullptr ? gx + (size_t)b * g.C * g.Sn : nullptr;
        for (int t = wave; t < g.Kn; t += NW) {
            A qo[DIM], qm = zero;   // sums of the offset group's directions and of the mask group
#pragma unroll
            for (int a = 0; a < DIM; ++a) qo[a] = zero;
            for_channel_runs<DIM, A, T>(g, offset, mask, b, p, t, [&](int c0, int c1, const CornerSet<DIM, A> &cs, A mk, int ogi, int mgi) {
#pragma unroll 2
                for (int c = c0; c < c1; ++c) {
                    const int k = c * g.Kn + t;
                    const A gv = Gs[k * LDG + lane];
                    if (xb != nullptr) {
                        A xv[NC], s = zero;
#pragma unroll
                        for (int i = 0; i < NC; ++i) xv[i] = cs.ok[i] && ok ? to_acc<A>(xb[c * xc + cs.idx[i] * xp]) : zero;
                        if (cs.aw.inside) {
#pragma unroll
                            for (int i = 0; i < NC; ++i)
                                if (cs.ok[i]) s += corner_weight<DIM, A>(cs.aw, i) * xv[i];
                        }
                        if (coord) {
#pragma unroll
                            for (int a = 0; a < DIM; ++a) {
                                A d = zero;
#pragma unroll
                                for (int i = 0; i < NC; ++i)
                                    if (cs.ok[i]) d += corner_dweight<DIM, A>(cs.aw, i, a) * xv[i];
                                qo[a] += gv * d * mk;
                            }
                            qm += gv * s;
                        }
                        if (part != nullptr) S[k * LDG + lane] = ok ? s * mk : zero;
                    }
                    if (gxb != nullptr && ok) {
                        const A val = gv * mk;
#pragma unroll
                        for (int i = 0; i < NC; ++i)
                            if (cs.ok[i]) atomic_add(gxb + c * xc + cs.idx[i] * xp, corner_weight<DIM, A>(cs.aw, i) * val);
                    }
                }
                if (goff != nullptr && c1 == (ogi + 1) * g.cpo) {
#pragma unroll
                    for (int a = 0; a < DIM; ++a) {
                        if (ok) goff[((((size_t)b * g.og + ogi) * g.Kn + t) * DIM + a) * g.Pn + p] = from_acc<T, A>(qo[a]);
                        qo[a] = zero;
                    }
                }
                if (gmask != nullptr && c1 == (mgi + 1) * g.cpm) {
                    if (ok) gmask[(((size_t)b * g.mg + mgi) * g.Kn + t) * g.Pn + p] = from_acc<T, A>(qm);
                    qm = zero;
                }
            });
        }
        if (part != nullptr) {
            __syncthreads();
            // ---- bias gradient: the tile's sum of a row of Z by a tree over the lanes, then the tiles in turn (a column
            //      of ones beside dW's had a chain of all the workgroup's pixels: error 7.4e-7 on 8 x 224x224, 1.5e-7
            //      so). Lane i keeps row i of the wave's 64, so that a tile reads and writes its partial sums once.
            for (int m0 = 0; m0 < g.M; m0 += 64 * NW) {
                const int ml = m0 + wave + NW * lane;
                A *dst = part + (size_t)ml * (Kg + 1) + Kg;
                const A before = ch > 0 && ml < g.M ? *dst : zero;
                const int rows = min(64, (g.M - m0 - wave + NW - 1) / NW);
                const T *zr = z + (size_t)b * g.M * g.Pn + (size_t)(m0 + wave) * g.Pn + p;
                A sum = zero;
#pragma unroll 8
                for (int i = 0; i < rows; ++i) {
                    const A v = wave_sum(ok ? to_acc<A>(zr[(size_t)i * NW * g.Pn]) : zero);
                    sum = lane == i ? v : sum;
                }
                if (ml < g.M) *dst = before + sum;
            }
            // ---- dW[m][k]: 16 x 16 blocks dealt to the waves; each is added to the workgroup's partial sums of its
            //      earlier tiles
            const int mb = (g.Mg + 15) / 16, kb = (Kg + 15) / 16;
            for (int i = wave; i < g.G * mb * kb; i += NW) {
                const int k = i % kb * 16 + (lane & 15), r = i / kb;
                const int m0 = r % mb * 16, grp = r / mb;
                const int m = min(m0 + (lane & 15), g.Mg - 1);   // (rows past Mg: not stored)
                const T *zr = z + ((size_t)grp * g.Mg + m) * g.Pn;
                const A *Sr = S + (size_t)(grp * Kg + min(k, Kg - 1)) * LDG;   // (columns past Kg: not stored)
                acc4 acc;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int mr = m0 + mfma_row<A>(lane, v);
                    acc[v] = ch > 0 && mr < g.Mg && k < Kg ? part[((size_t)grp * g.Mg + mr) * (Kg + 1) + k] : zero;
                }
#pragma unroll
                for (int s = 0; s < BP; s += 4) {
                    const int o = zo[s + q];
                    acc = mfma16x16x4(o >= 0 ? to_acc<A>(zr[max(o, 0)]) : zero, Sr[s + q], acc);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int mr = m0 + mfma_row<A>(lane, v);
                    if (mr < g.Mg && k < Kg) part[((size_t)grp * g.Mg + mr) * (Kg + 1) + k] = acc[v];
                }
            }
        }
        __syncthreads();   // the tables are free for the next tile
    }
}

// gw[m][k] = (accumulate: gw +) sum over the splits of part[split][m][k], gbias[m] the same of column Kg.
// Block = 32 columns x 8 runs of splits, four sums each; added in a fixed tree.
template <typename T, typename A>
__global__ void __launch_bounds__(256) few_reduce_kernel(const A *__restrict__ part, T *__restrict__ gw, T *__restrict__ gb,
                                                         int M, int Kg, int splits, bool accumulate) {
    __shared__ A sums[8][32];
    const int e = blockIdx.x * 32 + (threadIdx.x & 31), r = threadIdx.x >> 5;
    const int n = M * (Kg + 1);
    A a[4] = {A(0), A(0), A(0), A(0)};
    if (e < n) {
        const int per = (splits + 7) / 8, s1 = min(splits, (r + 1) * per);
        int s = r * per;
        for (; s + 8 <= s1; s += 8)
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i % 4] += part[(size_t)(s + i) * n + e];
#pragma unroll
        for (int i = 0; i < 7; ++i)
            if (s + i < s1) a[i % 4] += part[(size_t)(s + i) * n + e];
    }
    sums[r][threadIdx.x & 31] = (a[0] + a[1]) + (a[2] + a[3]);
    __syncthreads();
    if (r != 0 || e >= n) return;
    auto at = [&](int i) { return sums[i][threadIdx.x]; };
    const A v = ((at(0) + at(1)) + (at(2) + at(3))) + ((at(4) + at(5)) + (at(6) + at(7)));
    const int m = e / (Kg + 1), k = e - m * (Kg + 1);
    if (k == Kg && gb == nullptr) return;
    T *dst = k < Kg ? gw + (size_t)m * Kg + k : gb + m;
    *dst = from_acc<T, A>(accumulate ? to_acc<A>(*dst) + v : v);
}

// acc[b][c][s] = bias[c] (the transposed forward's output before the scatter), element order as x's
template <typename T, typename A>
__global__ void __launch_bounds__(256) few_init_kernel(A *__restrict__ y, const T *__restrict__ bias, int C, int Sn, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = bias != nullptr ? to_acc<A>(bias[(i / Sn) % C]) : A(0);
}

template <typename F> hipError_t by_type(int dtype, int dim, F &&f) {
    auto d = [&](auto tv, auto av) {
        switch (dim) {
            case 1: return f(std::integral_constant<int, 1>(), tv, av);
            case 2: return f(std::integral_constant<int, 2>(), tv, av);
            case 3: return f(std::integral_constant<int, 3>(), tv, av);
        }
        return hipErrorInvalidValue;
    };
    switch (dtype) {
        case kF32: return d(float(), float());
        case kF64: return d(double(), double());
        case kF16: return d(__half(), float());
        case kBF16: return d(__hip_bfloat16(), float());
    }
    return hipErrorInvalidValue;
}

size_t acc_bytes(int dtype) { return dtype == kF64 ? sizeof(double) : sizeof(float); }
size_t fwd_lds(const Geo &g, int dtype) { return (size_t)g.C * g.Kn * LDF * acc_bytes(dtype); }
// (weight: the columns beside G, for the weight gradient)
size_t data_lds(const Geo &g, int dtype, bool weight) {
    return (size_t)(weight ? 2 : 1) * g.C * g.Kn * LDG * acc_bytes(dtype) + BP * sizeof(int);
}

}  // namespace

FewPlan plan_few(const Geo &g, int dtype, int dim) {
    FewPlan f{};
    // Columns of up to 128 values, or 200 on grids of up to a tile per CU, and weights of up to 24576: beyond
    // either the general kernels' wider tiles win (float32, us a training step, general -> here: 3 -> 64 k3 on 8 x 224x224 5476 ->
    // 1535, 5 -> 512 k3 on 4 x 64x64 652 -> 280, 10 -> 512 666 -> 679, 14 -> 512 668 -> 882, 21 -> 30 on
    // 20x20 459 -> 214, 30 -> 30 on 16 x 128x128 4406 -> 9081). A fused mask
    // activation's gradient is finished in the accumulation type, which 16-bit gradients here never are (the
    // forward of such a layer follows its backward; not timed apart).
    // Fewer than 2^30 pixels: four threads each stay below HIP's 2^32 of a launch, and a run of tiles that
    // ends past the last pixel below 2^31.
    const long long column = (long long)g.C * g.Kn;
    f.ok = g.NP < 1 << 30 && (column <= 128 || (column <= 200 && g.NP <= 256 * BP)) &&
           (long long)g.M * g.Cg * g.Kn <= 24576 && data_lds(g, dtype, true) <= WIN_LDS_TARGET &&
           (g.mask_act == 0 || dtype == kF32 || dtype == kF64);
    if (!f.ok || g.NP == 0) return f;
    // The scatter alone (the transposed forward): a lane per pixel, so that an atomic instruction reaches up to 64
    // lines for one channel, where the general kernel's covers the channels of a pixel's corner, one line. Its cost
    // grows with the channels, the general kernel's hardly. float32, us a call, general -> here: 1D k16 on
    // 8 x 65536, 3 / 5 / 7 channels 1591 -> 928, 1542 -> 1506, 1594 -> 2087; 2D k4 on 8 x 128x128, 1 / 2 / 3
    // channels 649 -> 280, 595 -> 548, 655 -> 835; 3D k4 on 2 x 8x28x28, 1 / 2 channels 399 -> 250, 366 -> 486.
    // Small layers have a launch less here: 1D k3 on 4 x 4096, 9 channels 30 -> 22, 2D k4 on 2 x 32x32, 3 / 5
    // channels 33 -> 28, 33 -> 43. Several offset or mask groups in a conv group take the general kernel's per-lane
    // path: 1D k3 on 12 x 258, float16, 32 channels in 2 conv and 4 offset groups 56 -> 28.
    const long long work = (long long)g.NP * g.Kn;
    const bool small = work <= 65536;
    f.scatter = g.C <= (dim == 1 ? (small ? 9 : 5) : dim == 2 ? (small ? 3 : 2) : 1) ||
                (dim == 1 && (g.og > g.G || g.mg > g.G) && work <= 16384);
    const int tiles = (g.NP + BP - 1) / BP;
    // one tile per workgroup up to one per CU, then runs of tiles (each workgroup's partial sums of dW are
    // read back by the reduction)
    f.chunks = (tiles + 255) / 256;
    f.splits = (tiles + f.chunks - 1) / f.chunks;
    f.part_elems = (size_t)f.splits * g.M * (g.Cg * g.Kn + 1);
    return f;
}

hipError_t launch_few_fwd(int dtype, int dim, const Geo &g, const void *x, bool x_cl, const void *w, const void *offset,
                          const void *mask, const void *bias, void *y, hipStream_t s) {
    return by_type(dtype, dim, [&](auto dv, auto tv, auto av) {
        using T = decltype(tv);
        using A = decltype(av);
        auto kern = few_fwd_kernel<decltype(dv)::value, T, A>;
        static std::atomic<unsigned long long> lds_raised{0};
        const hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(kern), lds_raised);
        if (e != hipSuccess) return e;
        // row blocks on workgroups of their own, each sampling the tile again, until the chip holds
        // three workgroups per CU
        const int tiles = (g.NP + BP - 1) / BP, rows = (g.Mg + 63) / 64;
        const dim3 grid((unsigned)tiles, (unsigned)std::max(1, std::min(rows, 768 / tiles)));
        hipLaunchKernelGGL(kern, grid, dim3(64 * NW), fwd_lds(g, dtype), s, g,
                           static_cast<const T *>(x), x_cl ? 1 : g.Sn, x_cl ? g.C : 1, static_cast<const T *>(w),
                           static_cast<const T *>(offset), static_cast<const T *>(mask), static_cast<const T *>(bias),
                           static_cast<T *>(y));
        return hipGetLastError();
    });
}

hipError_t launch_few_data(int dtype, int dim, const Geo &g, const FewPlan &f, const void *z, const void *x, bool x_cl,
                           const void *w, const void *offset, const void *mask, void *gx, void *goff, void *gmask,
                           void *part, hipStream_t s) {
    return by_type(dtype, dim, [&](auto dv, auto tv, auto av) {
        using T = decltype(tv);
        using A = decltype(av);
        auto kern = few_data_kernel<decltype(dv)::value, T, A>;
        static std::atomic<unsigned long long> lds_raised{0};
        const hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(kern), lds_raised);
        if (e != hipSuccess) return e;
        // without a weight gradient (the transposed forward) there are no partial sums to read back, and a tile needs
        // half the LDS: a workgroup per tile, as many on a CU as fit (64 -> 1 channel k4 on 8 x 128x128 294 -> 285 us
        // against runs of tiles, 1D k16 on 8 x 65536 542 -> 509)
        const bool weight = part != nullptr;
        const int tiles = (g.NP + BP - 1) / BP;
        hipLaunchKernelGGL(kern, dim3((unsigned)(weight ? f.splits : tiles)), dim3(64 * NW), data_lds(g, dtype, weight), s, g,
                           static_cast<const T *>(z), static_cast<const T *>(x), x_cl ? 1 : g.Sn, x_cl ? g.C : 1,
                           static_cast<const T *>(w), static_cast<const T *>(offset), static_cast<const T *>(mask),
                           static_cast<A *>(gx), static_cast<T *>(goff), static_cast<T *>(gmask), static_cast<A *>(part),
                           weight ? f.chunks : 1);
        return hipGetLastError();
    });
}

hipError_t launch_few_reduce(int dtype, const Geo &g, const FewPlan &f, const void *part, void *gw, void *gb,
                             bool accumulate, hipStream_t s) {
    return by_type(dtype, 1, [&](auto, auto tv, auto av) {
        using T = decltype(tv);
        using A = decltype(av);
        const int n = g.M * (g.Cg * g.Kn + 1);
        hipLaunchKernelGGL((few_reduce_kernel<T, A>), dim3((unsigned)((n + 31) / 32)), dim3(256), 0, s,
                           static_cast<const A *>(part), static_cast<T *>(gw), static_cast<T *>(gb), g.M, g.Cg * g.Kn,
                           f.splits, accumulate);
        return hipGetLastError();
    });
}

hipError_t launch_few_init(int dtype, const Geo &g, void *y, const void *bias, hipStream_t s) {
    return by_type(dtype, 1, [&](auto, auto tv, auto av) {
        using T = decltype(tv);
        using A = decltype(av);
        const size_t n = (size_t)g.B * g.C * g.Sn;
        hipLaunchKernelGGL((few_init_kernel<T, A>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                           static_cast<A *>(y), static_cast<const T *>(bias), g.C, g.Sn, n);
        return hipGetLastError();
    });
}

}  // namespace tvdcn_hip
