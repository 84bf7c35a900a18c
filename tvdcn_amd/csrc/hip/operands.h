// The 16-bit MFMA operand layouts, as the work of one 256-thread block each: the kernels that write them
// run several in one launch (bwd_data_win.hip, fwd_win.hip, prep16.hip).
#pragma once

#include "window.h"

namespace tvdcn_hip {
namespace win {

// Z (B, G * Mg, Pn) -> zs [B][G][ms32][NP][Pn][32]: per 32-channel step and piece, every pixel's
// 32 channels (zero past Mg) as 4 lane groups of 8 (the 16x16x32 B-operand layout), so that a
// wave's fragment load of one piece for 16 consecutive pixels reads 1 KB of whole lines.
// Block = 64 pixels of one (image, group, step), transposed through LDS.
// (zvec: Pn % 4 == 0 and z aligned to 4 elements: the tile is read in 4-pixel vectors)
template <typename T, int NP>
__device__ __forceinline__ void z_split_block(long long bid, float *smem, const T *__restrict__ z,
                                              uint16_t *__restrict__ zs, uint16_t *__restrict__ zw, int *flag, int G,
                                              int Mg, int Pn, int ms32, int pblocks, bool zvec, size_t zw_plane) {
    float(*tile)[65] = reinterpret_cast<float(*)[65]>(smem);   // [32][65]
    const int sz = NP == 2 ? operand_scale(flag, AMAX_Z) : 0;   // (every lane: before any returns)
    // (the block index is a grid index: 32-bit division, not the 64-bit sequence)
    const unsigned ub = (unsigned)bid;
    const int pb = (int)(ub % (unsigned)pblocks);
    const unsigned bgs = ub / (unsigned)pblocks;   // (b * G + grp) * ms32 + step
    const int st = (int)(bgs % (unsigned)ms32);
    const unsigned bg = bgs / (unsigned)ms32;
    const int grp = (int)(bg % (unsigned)G);
    const unsigned b = bg / (unsigned)G;
    const int p0 = pb * 64;
    const T *src = z + ((size_t)b * G + grp) * (size_t)Mg * Pn;
    if (zvec) {
        for (int i = threadIdx.x; i < 32 * 16; i += 256) {
            const int ml = i >> 4, pl = 4 * (i & 15);
            const int m = st * 32 + ml, p = p0 + pl;
            Vec4<float> v{0.f, 0.f, 0.f, 0.f};
            if (m < Mg && p < Pn) v = load4_t<float, T>(src + (size_t)m * Pn + p);   // all four inside
            tile[ml][pl] = v.x;
            tile[ml][pl + 1] = v.y;
            tile[ml][pl + 2] = v.z;
            tile[ml][pl + 3] = v.w;
        }
    } else {
        for (int i = threadIdx.x; i < 32 * 64; i += 256) {
            const int ml = i >> 6, pl = i & 63;
            const int m = st * 32 + ml, p = p0 + pl;
            float v = 0.f;
            if (m < Mg && p < Pn) v = to_acc<float>(src[(size_t)m * Pn + p]);
            tile[ml][pl] = v;
        }
    }
    __syncthreads();
    if (zw != nullptr) {
        // the same values for the weight gradient, in 8-pixel column blocks: element (image b, row
        // m of Z's M, pixel p) at ((b * Pn / 8 + p / 8) * M + m) * 8 + p % 8 of each piece's plane
        // (Pn % 8 == 0), so that a wave's A fragment (16 rows x 4 blocks of 8 pixels) reads whole
        // lines. Thread = (row ml, 8-pixel block px / 8): consecutive threads, consecutive rows.
        const int ml = threadIdx.x & 31, px = 8 * (threadIdx.x >> 5);
        const int m = st * 32 + ml, pw = p0 + px;
        if (m < Mg && pw < Pn) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = tile[ml][px + e];
            uint4 out[NP];
            pack8_16<T, NP>(v, sz, out);
            const size_t M = (size_t)G * Mg;
            uint16_t *dst = zw + ((size_t)b * (Pn / 8) + pw / 8) * M * 8 + ((size_t)grp * Mg + m) * 8;
#pragma unroll
            for (int k = 0; k < NP; ++k) *reinterpret_cast<uint4 *>(dst + k * zw_plane) = out[k];
        }
    }
    const int pl = threadIdx.x >> 2, q = threadIdx.x & 3, p = p0 + pl;
    if (p >= Pn) return;
    float v[8];
    bool bad = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        v[e] = tile[q * 8 + e][pl];
        bad = bad || split_bad(v[e]);
    }
    uint4 out[NP];
    pack8_16<T, NP>(v, sz, out);
    uint16_t *dst = zs + ((size_t)bgs * NP * Pn + p) * 32 + q * 8;
#pragma unroll
    for (int k = 0; k < NP; ++k) *reinterpret_cast<uint4 *>(dst + (size_t)k * Pn * 32) = out[k];
    if (NP == 2 && bad) atomicOr(flag, 1);
}

// taps per block of the weight's layouts (17 KB of LDS)
constexpr int WL_TK = 8;

// weight (M, Cg, Kn) -> split chunks [G][c_tiles][ms32][Kn][NP][4 q][16 c][8 e]: per (step, tap)
// and piece, the 16x16x32 A-operand fragment of 16 channels x 32 GEMM-side channels (lane
// q * 16 + c holds rows 8q .. 8q + 7 of channel c; zero past Mg / Cg). Block = (group, channel
// slice, step, run of up to WL_TK taps), transposed through LDS.
template <typename T, int NP>
__device__ __forceinline__ void weight_split_block(int L, float *smem, const T *__restrict__ w,
                                                   uint16_t *__restrict__ out, int *flag, int G, int Mg, int Cg,
                                                   int Kn, int c_tiles, int ms32) {
    float(*tile)[BC][33] = reinterpret_cast<float(*)[BC][33]>(smem);   // [tap][c][m]
    const int tchunks = (Kn + WL_TK - 1) / WL_TK;
    const int tc = L % tchunks;
    L /= tchunks;
    const int st = L % ms32;
    L /= ms32;
    const int ct = L % c_tiles;
    const int grp = L / c_tiles;
    const int t0 = tc * WL_TK, nt = min(WL_TK, Kn - t0);
    const int n = 32 * BC * nt;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const int tt = e % nt, r = e / nt;   // (m, c, tap), taps fastest
        const int ci = r % BC, mi = r / BC;
        const int m = st * 32 + mi, c = ct * BC + ci;
        float v = 0.f;
        if (m < Mg && c < Cg) v = to_acc<float>(w[(((size_t)grp * Mg + m) * Cg + c) * Kn + t0 + tt]);
        tile[tt][ci][mi] = v;
    }
    __syncthreads();
    uint16_t *dst = out + ((((size_t)grp * c_tiles + ct) * ms32 + st) * Kn + t0) * (NP * 512);
    const int sw = NP == 2 ? operand_scale(flag, AMAX_W) : 0;
    bool bad = false;
    for (int u = threadIdx.x; u < nt * 64; u += blockDim.x) {
        const int tt = u >> 6, l = u & 63, q = l >> 4, c = l & 15;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = tile[tt][c][q * 8 + e];
            bad = bad || split_bad(v[e]);
        }
        uint4 o[NP];
        pack8_16<T, NP>(v, sw, o);
#pragma unroll
        for (int k = 0; k < NP; ++k) *reinterpret_cast<uint4 *>(dst + (size_t)tt * (NP * 512) + k * 512 + l * 8) = o[k];
    }
    if (NP == 2 && bad) atomicOr(flag, 1);
}

// weight (M, Cg, Kn) -> W16[G][slices][pp][Mg_pad / 16][NP][64 lanes][8]: per (slice, tap pair j
// of pass p, 16-row block) the 16x16x32 A fragments: lane l = m % 16 + 16 q holds at e = 0..7
// W[m][slice * 16 + 4 q + e % 4] at tap p * tpp + 2 j + e / 4 (zero past the pass, Mg, Cg); fp32
// as two fp16 pieces at the weight's scale (*flag set for a value bad for the split), fp16 / bf16
// as they are
template <typename T, int NP>
__device__ __forceinline__ void w16_block(unsigned block, unsigned blocks, const T *__restrict__ w, uint16_t *__restrict__ out,
                                          int *flag, int G, int Mg, int Cg, int Kn, int slices, int nmb, int tpp, int hp,
                                          int pp) {
    const unsigned total = (unsigned)G * slices * pp * nmb * 64;
    const int sw = NP == 2 ? operand_scale(flag, AMAX_W) : 0;
    bool bad = false;
    for (unsigned i = block * 256 + threadIdx.x; i < total; i += blocks * 256) {
        const int l = (int)(i & 63);
        unsigned r = i >> 6;
        const int mb = (int)(r % nmb);
        r /= nmb;
        const int pq = (int)(r % pp);
        r /= pp;
        const int cs = (int)(r % slices);
        const int grp = (int)(r / slices);
        const int pass = pq / hp, j = pq - pass * hp;
        const int tf = pass * tpp, ntp = min(tpp, Kn - tf);
        const int m = mb * 16 + (l & 15), q = l >> 4;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tl = 2 * j + (e >> 2), c = cs * BC + 4 * q + (e & 3);
            v[e] = (tl < ntp && m < Mg && c < Cg) ? to_acc<float>(w[(((size_t)grp * Mg + m) * Cg + c) * Kn + tf + tl]) : 0.f;
            bad = bad || split_bad(v[e]);
        }
        uint4 o[NP];
        pack8_16<T, NP>(v, sw, o);
        uint16_t *dst = out + ((((size_t)grp * slices + cs) * pp + pq) * nmb + mb) * (NP * 512) + l * 8;
#pragma unroll
        for (int k = 0; k < NP; ++k) *reinterpret_cast<uint4 *>(dst + k * 512) = o[k];
    }
    if (NP == 2 && bad) atomicOr(flag, 1);
}

}  // namespace win
}  // namespace tvdcn_hip
