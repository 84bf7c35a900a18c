// Family F, windowed variant: the forward gather-GEMM with the sampled columns formed
// from an LDS window of the sampled tensor.
//
//   Y[b][m][p] = bias[m] + sum_{t, c in group} W[m][c][t] * mask * bilinear(X[b][c], pos(b, og(c), t, p))
//
// Replaces the reference's im2col kernel + addmm_ pair
// (tvdcn/csrc/ops/cuda/deform_conv2d_common_kernels.cu:138-256 and
// deform_conv2d_kernel.cpp:341-380; 1D/3D twins); the columns are never written
// to HBM. Also computes the transposed op's input gradient.
//
// Workgroup = (spatial tile of 256 column pixels, 128 or 64 GEMM-side rows, a share of the (pass,
// channel slice) units: grids too small to fill the chip take several shares); eight
// waves, wave w owning 32 pixels x all rows (64 or 32 accumulators per lane; 64-row
// tiles serve small GEMM sides and grids too small to fill the chip). The reduction runs
// over 16-channel slices x taps; per step (slice, tap) every lane forms its own MFMA
// B fragment -- the sampled values of 4 channels of one of its pixels -- straight from
// the X window (LDS) and the sampling table, one step ahead, while the MFMAs of the
// current step run with A = W[m][c] (16-byte fragments of the re-laid-out weight, each
// reloaded for the next step right after its last use). Waves own disjoint pixels, so
// nothing is exchanged between them inside a slice: barriers only where the X window
// of the next slice (prefetched into registers during the last step of the current
// one) replaces the current one, and where the sampling table is rebuilt (when the
// offset / mask group changes). See window.h for the tile / window machinery.
#include "operands.h"

namespace tvdcn_hip {
namespace {

using namespace win;

constexpr int NW = 8;               // waves per workgroup
constexpr int NT = 64 * NW;
constexpr int PB = 2;               // 16-pixel blocks per wave
constexpr int TM = WIN_TMAX;
constexpr int PF = 3;               // X window prefetch distance, steps
// MB = 16-row blocks per wave (rows per workgroup 16 * MB); XQ = X window quads
// prefetched per thread (cells * 4 <= XQ * NT): the 64-row variant spends the
// registers its smaller accumulator frees on a larger window
constexpr int xq_of(int mb) { return mb == 8 ? 8 : 12; }
static_assert(NW * PB * 16 == BPX, "one tile of pixels per workgroup");

constexpr int GEO_WORDS = TM * BPX * 4;

// lanes 4a .. 4a + 3 hold r[v] of row v at pixels 4a .. 4a + 3: on return lane 4a + i holds row i's four
// pixels (two exchanges within lane quads)
__device__ __forceinline__ void transpose_quad(acc4 &r, int lane) {
    auto swap = [&](auto ctrl, bool hi, int lo_v, int hi_v) {
        const float send = hi ? r[lo_v] : r[hi_v];
        const float got = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), decltype(ctrl)::value, 0xF, 0xF, true));
        r[lo_v] = hi ? got : r[lo_v];
        r[hi_v] = hi ? r[hi_v] : got;
    };
    const std::integral_constant<int, 0xB1> x1;   // lane ^ 1
    const std::integral_constant<int, 0x4E> x2;   // lane ^ 2
    swap(x1, lane & 1, 0, 1);
    swap(x1, lane & 1, 2, 3);
    swap(x2, lane & 2, 0, 2);
    swap(x2, lane & 2, 1, 3);
}

// 16 rows (m0 .. m0 + 15 of the group's rows at yg) x 16 pixels, lane (pixel l % 16 = p, rows 4 (l / 16) ..):
// vec (P_x % 4 == 0: the lane quad's pixels are consecutive, all inside the grid or all outside, and 4-aligned):
// one row's four pixels per lane, else four single values
template <typename T>
__device__ __forceinline__ void store_frag(const Geo &g, T *yg, int m0, int p, bool vec, acc4 r) {
    const int lane = threadIdx.x & 63;
    const int m = m0 + 4 * (lane >> 4);
    if (vec) {
        transpose_quad(r, lane);
        const int mi = m + (lane & 3);
        if (p >= 0 && mi < g.Mg)
            store4_t<T, float>(yg + (size_t)mi * g.Pn + (p - (lane & 3)), Vec4<float>{r[0], r[1], r[2], r[3]});
    } else if (p >= 0) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (m + v < g.Mg) yg[(size_t)(m + v) * g.Pn + p] = from_acc<T, float>(r[v]);
    }
}

// STAGE: the 16-bit loop's weight blocks are staged in LDS (1D / 2D, fw.stage_bytes > 0). LOOP: the 16x16x32 MFMA
// loop, the fp32 one, or both, of which the operand flag selects one. ONE: a single pass of taps. Either loop
// beside the other, or beside a loop over the passes, cost the 2D kernel 75 registers and 226 spilled scalars (174
// and none without), the compiler keeping both loops' and all phases' values live. fp16 / bf16 run the 16-bit
// loop alone; a long fp32 call launches either loop's kernel and the flag has one return at once, a short one both
// in one kernel (launch_k). (always_inline: at this size the inliner otherwise leaves the lambdas as calls.)
// bfloat16 128 channels, 2 x 100x152 inference 107 -> 103 us.
constexpr int LOOP_F32 = 0, LOOP_16 = 1, LOOP_BOTH = 2;
template <int DIM, typename T, int MB, bool STAGE, int LOOP, bool ONE>
__global__ void __launch_bounds__(NT)
fwd_win_kernel(const Geo g, const WinTiles wt, const FwdWin fw, const float *__restrict__ xcl,
               const float *__restrict__ wf, const uint16_t *__restrict__ w16, const int *flag,
               const T *__restrict__ offset, const T *__restrict__ mask, const T *__restrict__ bias,
               T *__restrict__ y, float *__restrict__ y32) {
    constexpr int NC = 1 << DIM;
    constexpr int BMR = MB * 16;
    constexpr int XQ = xq_of(MB);
    extern __shared__ float smem[];
    acc4 *geo = reinterpret_cast<acc4 *>(smem);     // [TM][BPX]
    float *xwin = smem + GEO_WORDS;                 // [cells][XS]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int q = lane >> 4;

    int L = xcd_remap(blockIdx.x, gridDim.x);
    const int mt = L % fw.m_tiles;
    L /= fw.m_tiles;
    const int ks = L % fw.ksplit;   // share of the (pass, channel slice) units (fw.ksplit > 1: fp32 partials)
    L /= fw.ksplit;
    const int n_sp = g.B * wt.ntile[0] * wt.ntile[1] * wt.ntile[2];
    const int sp = L % n_sp;
    const int grp = L / n_sp;
    const bool deformable = offset != nullptr;
    const int slices = (g.Cg + BC - 1) / BC;
    const bool flagged = npiece_of<T>() == 2 && flag != nullptr && *flag != 0;
    if (LOOP != LOOP_BOTH && npiece_of<T>() == 2 && flag != nullptr && flagged != (LOOP == LOOP_F32)) return;   // the other launch's
    const bool use16 = LOOP == LOOP_16 || (LOOP == LOOP_BOTH && w16 != nullptr && !flagged);
    // fp32 as fp16 pieces: the sampled columns' scale, and the one back out (the weight's with it)
    const int s_b = npiece_of<T>() == 2 && use16 ? sampled_scale(g, flag, mask != nullptr) : 0;
    const int s_back = npiece_of<T>() == 2 && use16 ? -(s_b + operand_scale(flag, AMAX_W)) : 0;
    // the sampling table's masks carry 2^s_b, so that the B fragments come out of the sampling at
    // their pieces' scale
    const float mscale_b = ldexpf(1.f, s_b);
    // this share's units u = pass * slices + slice, u in [u_lo, u_lo + fw.units_per); per pass the slices
    // [cs_lo, cs_hi) of them
    const int u_lo = ks * fw.units_per;
    int cs_lo = 0, cs_hi = 0;
    auto pass_slices = [&](int pass) __attribute__((always_inline)) {
        cs_lo = max(u_lo - pass * slices, 0);
        cs_hi = min(u_lo + fw.units_per - pass * slices, slices);
        return cs_lo < cs_hi;
    };
    auto passes = [&](auto &&body) __attribute__((always_inline)) {
        if constexpr (ONE) {
            if (pass_slices(0)) body(0, g.Kn);
        } else {
            for (int t0 = 0, pass = 0; t0 < g.Kn; t0 += wt.tpp, ++pass)
                if (pass_slices(pass)) body(t0, min(wt.tpp, g.Kn - t0));
        }
    };

    Tile tile;
    tile.init(g, wt, sp, 0, grp);
    if constexpr (DIM == 3) {
        if (tid < XS) xwin[wt.cells * XS + tid] = 0.f;   // zero cell of the 3D corner reads
    }
    const float *xg = xcl + (size_t)tile.b * g.Sn * g.C + (size_t)grp * g.Cg;   // group's channel 0


    // X window prefetch: quad e = tid + j * NT of the window (cell e / 4, quad e % 4). The
    // cells (and their grid indices) are the same for every slice: resolved once.
    // (3D resolves them at each fill: its registers are taken by the B fragments of a tap group)
    int xsi[XQ];   // flat sampled-grid index of the thread's cells (-1: outside the grid / window)
    auto resolve_cells = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < XQ; ++j) {
            const int e = tid + j * NT;
            xsi[j] = e < wt.cells * 4 ? tile.cell_index(g, wt, e >> 2) : -1;
        }
    };
    if constexpr (DIM != 3) resolve_cells();
    acc4 xpre[XQ];
    auto prefetch_x = [&](int cs) __attribute__((always_inline)) {
        const float *xb = xg + cs * BC + 4 * (tid & 3);
        const bool q_ok = cs * BC + 4 * (tid & 3) < g.Cg;   // quad of thread tid + j * NT is tid % 4
#pragma unroll
        for (int j = 0; j < XQ; ++j) {
            xpre[j] = acc4{0.f, 0.f, 0.f, 0.f};
            if (xsi[j] >= 0 && q_ok) xpre[j] = *reinterpret_cast<const acc4 *>(xb + (size_t)xsi[j] * g.C);
        }
    };
    auto store_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < XQ; ++j) {
            const int e = tid + j * NT;
            if (e < wt.cells * 4) *reinterpret_cast<acc4 *>(xwin + (e >> 2) * XS + 4 * (e & 3)) = xpre[j];
        }
    };

    // B fragment of pixel block pb for (slice cs, tap tl of the pass): the sampled values of
    // channels cs * 16 + 4 * (lane / 16) .. + 3 at pixel wave * 32 + pb * 16 + lane % 16
    auto build_b = [&](int cs, int tl, acc4 (&bv)[PB]) __attribute__((always_inline)) {
        const int qd = q;
        const bool q_ok = cs * BC + 4 * qd < g.Cg;
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            const acc4 r = geo[tl * BPX + wave * (PB * 16) + pb * 16 + (lane & 15)];
            const int fc = fast_cell<DIM>(r);
            const float mk = rec_mask<DIM>(r);
            acc4 sv;
            if (fc >= 0) {
                sv = window_sample_masked<DIM>(wt, xwin, fc, 4 * qd, r, mk);
            } else {
                Point<DIM, float> pt;
#pragma unroll
                for (int a = 0; a < DIM; ++a) {
                    pt.pos[a] = r[a];
                    pt.base[a] = (int)r[a];
                }
                const AxisW<DIM, float> aw = axis_weights<DIM, float>(g, pt, deformable);
                sv = acc4{0.f, 0.f, 0.f, 0.f};
                if (aw.inside) {
#pragma unroll
                    for (int kk = 0; kk < NC; ++kk) {
                        int idx;
                        bool v;
                        corner_at<DIM, float>(g, aw, kk, idx, v);
                        if (!v) continue;
                        const int cell = tile.corner_cell<DIM>(wt, aw, kk);
                        // LDS read unconditional (clamped), global read in its own branch: the two
                        // address spaces are never merged into one pointer
                        acc4 x = *reinterpret_cast<const acc4 *>(xwin + max(cell, 0) * XS + 4 * qd);
                        if (cell < 0) {
                            x = acc4{0.f, 0.f, 0.f, 0.f};
                            if (q_ok) x = *reinterpret_cast<const acc4 *>(xg + cs * BC + (size_t)idx * g.C + 4 * qd);
                        }
                        sv += corner_weight<DIM, float>(aw, kk) * x;
                    }
                }
                sv *= mk;
            }
            bv[pb] = sv;
        }
    };

    // A operand: W[m][c] fragments, rows m = mt * BMR + mb * 16 + lane % 16, channels
    // 4 * (lane / 16) .. + 3 of the slice. Layout Wp[grp][slice][t][Mg_pad / 16][16 m][16 c]
    // (fwd_win_weight_kernel): the row blocks of one (slice, tap) are 1 KB apart and each
    // is one contiguous 1 KB wave load; consecutive taps of a slice are adjacent.
    const size_t step_elems = (size_t)fw.Mg_pad * BC;
    const float *wlane = wf + (size_t)grp * slices * g.Kn * step_elems + (size_t)mt * MB * 256 + (lane & 15) * BC + 4 * q;
    auto wptr = [&](int cs, int t) __attribute__((always_inline)) { return wlane + ((size_t)cs * g.Kn + t) * step_elems; };
    auto load_w = [&](const float *p, acc4 (&wr)[MB]) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) wr[mb] = *reinterpret_cast<const acc4 *>(p + mb * 256);
    };

    acc4 acc[MB][PB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) acc[mb][pb] = acc4{0.f, 0.f, 0.f, 0.f};

    // MFMAs of one step with B fragments bv and A fragments wr; each row block's fragment
    // is reloaded from pn (the next step's, or this step's own at the end of a pass) right
    // after its last use (issue order pinned)
    auto mfma_step = [&](const acc4 (&bv)[PB], acc4 (&wr)[MB], const float *pn) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) acc[mb][pb] = mfma16x16x4(wr[mb][kk], bv[pb][kk], acc[mb][pb]);
            wr[mb] = *reinterpret_cast<const acc4 *>(pn + mb * 256);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // switch the tables to slice cs: X window from the prefetch registers, sampling
    // table rebuilt when the slice's offset / mask group differs from the last one
    int geo_og = -1, geo_mg = -1;
    auto open_slice = [&](int cs, int t0, int ntaps) __attribute__((always_inline)) {
        if constexpr (DIM == 3) {
            resolve_cells();
            prefetch_x(cs);
        }
        store_x();
        const int c_first = grp * g.Cg + cs * BC;
        const int og_s = g.og ? c_first / g.cpo : 0, mg_s = g.mg ? c_first / g.cpm : 0;
        if (og_s != geo_og || mg_s != geo_mg) {
            tile.ogu = og_s;
            tile.mgu = mg_s;
            // (the sampled values' piece scale folded into the records' masks)
            fill_geo<DIM, T, 3, true>(g, wt, tile, offset, mask, t0, ntaps, geo, tid, NT, mscale_b);
            geo_og = og_s;
            geo_mg = mg_s;
        }
    };

    // ---- 16-bit pass (1D / 2D): steps of (slice, tap pair) on 16x16x32 MFMAs. Lane (row
    //      l % 16, K group q = l / 16) holds at e = 0..7 the value of channel 4q + e % 4 at tap
    //      2j + e / 4 of the pair: its B fragment is the pair's two sampled quads (zero past the
    //      pass), split into pieces for fp32 and rounded to T otherwise (the reference's columns
    //      of a half-precision input are half). W16 holds the A fragments in the same K order.
    //      The weight blocks are staged in LDS (below).
    auto pass16 = [&](int t0, int ntaps) __attribute__((always_inline)) {
        if constexpr (DIM < 3) {
            constexpr int NP = npiece_of<T>();
            const int npair = (ntaps + 1) >> 1;
            const int nsteps = (cs_hi - cs_lo) * npair;
            geo_og = geo_mg = -1;   // a new pass of taps: the table must be rebuilt
            const int nmb = fw.Mg_pad / 16;
            const int pp0 = (t0 / wt.tpp) * fw.hp;
            // (the step's block: wave-uniform; lanes add their offsets when they load)
            const uint16_t *wl = w16 + (size_t)mt * MB * (NP * 512);
            auto wptr16 = [&](int cs, int j) __attribute__((always_inline)) {
                return wl + (((size_t)grp * slices + cs) * fw.pp + pp0 + j) * nmb * (NP * 512);
            };
            auto build_pair = [&](int cs, int j, uint4 (&bp)[PB][NP]) __attribute__((always_inline)) {
                acc4 b0[PB], b1[PB];
                build_b(cs, 2 * j, b0);
                if (2 * j + 1 < ntaps) {
                    build_b(cs, 2 * j + 1, b1);
                } else {
#pragma unroll
                    for (int pb = 0; pb < PB; ++pb) b1[pb] = acc4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) {
                    const float v[8] = {b0[pb][0], b0[pb][1], b0[pb][2], b0[pb][3],
                                        b1[pb][0], b1[pb][1], b1[pb][2], b1[pb][3]};
                    pack8_16<T, NP>(v, 0, bp[pb]);   // (already at scale 2^s_b)
                }
            };
            if constexpr (STAGE) {
                // The weight blocks (per step MB row blocks x NP pieces, 1 KB each, contiguous in W16)
                // are staged in LDS, double-buffered, in units of U = 8 / MB steps (64-row tiles take
                // two steps per unit, so that a unit's MFMAs cover the loads of the next): the
                // global-to-LDS loads of unit u + 1 are issued at the top of unit u (one 1 KB wave
                // instruction per piece, spread over the waves), and every wave reads its A fragments
                // from LDS. Loaded straight from global memory each wave fetched the same blocks:
                // eight times the bytes through the vector memory path, which then bounded the MFMAs.
                constexpr int U = 8 / MB;            // steps per staging unit
                constexpr int NI = MB * NP;          // 1 KB pieces per step
                constexpr int WBLK = NI * 512;       // 16-bit values per step
                uint16_t *wst = reinterpret_cast<uint16_t *>(xwin + (size_t)wt.cells * XS);   // [2][U][WBLK]
                // (slice, pair) of the next step to stage, advanced step by step (no divisions)
                int s_cs = cs_lo, s_j = 0;
                auto stage_unit = [&](int u, int buf) __attribute__((always_inline)) {
#pragma unroll
                    for (int su = 0; su < U; ++su) {
                        const int k = u * U + su;
                        if (k >= nsteps) break;
                        const uint16_t *blk = wptr16(s_cs, s_j);
                        if (++s_j == npair) {
                            s_j = 0;
                            ++s_cs;
                        }
                        uint16_t *dst = wst + (buf * U + su) * WBLK;
                        for (int i = wave; i < NI; i += NW)
                            __builtin_amdgcn_global_load_lds(blk + i * 512 + lane * 8, dst + i * 512, 16, 0, 0);
                    }
                };
                auto load_w16 = [&](const uint16_t *blk, int mb, uint4 (&f)[NP]) __attribute__((always_inline)) {
                    const uint16_t *p = blk + mb * (NP * 512) + lane * 8;
#pragma unroll
                    for (int k = 0; k < NP; ++k) f[k] = *reinterpret_cast<const uint4 *>(p + k * 512);
                };
                // MFMAs of one step on its staged block; block mb + 1's fragments are read before
                // block mb's MFMAs
                auto mfma_pair = [&](const uint4 (&bv)[PB][NP], uint4 (&wa)[2][NP], const uint16_t *blk) __attribute__((always_inline)) {
                    load_w16(blk, 0, wa[0]);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        if (mb + 1 < MB) load_w16(blk, mb + 1, wa[(mb + 1) & 1]);
#pragma unroll
                        for (int pb = 0; pb < PB; ++pb)
                            acc[mb][pb] = mfma16x16x32_np<T, NP>(wa[mb & 1], bv[pb], acc[mb][pb]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                // the staged unit's loads done, then the workgroup barrier that publishes it
                auto publish = [&]() __attribute__((always_inline)) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    __syncthreads();
                };
                // step k: its B fragments are built, then its MFMAs run (the LDS latency of the
                // sampling is covered by the other wave of the SIMD)
                uint4 wa[2][NP], bv[PB][NP];
                prefetch_x(cs_lo);
                __syncthreads();   // previous pass done with the tables and the staging buffers
                stage_unit(0, 0);
                open_slice(cs_lo, t0, ntaps);
                publish();
                // the next slice's X window is requested two pair steps before it is needed
                const int pf_j = max(npair - 2, 0);
                // (slice, pair) of step k, advanced step by step
                int cs = cs_lo, j = 0;
                for (int k = 0; k < nsteps; ++k) {
                    const bool more = k + 1 < nsteps;
                    const int u = k / U, su = k - u * U;
                    const int jn = j + 1 == npair ? 0 : j + 1;
                    if (su == 0 && (u + 1) * U < nsteps) stage_unit(u + 1, (u + 1) & 1);
                    if (j == pf_j && cs + 1 < cs_hi) prefetch_x(cs + 1);
                    build_pair(cs, j, bv);
                    mfma_pair(bv, wa, wst + ((u & 1) * U + su) * WBLK);
                    // the unit's end: every wave done with its buffer (and, at a slice change, with
                    // the window), the next unit's blocks visible
                    const bool unit_end = su == U - 1 || !more;
                    if (unit_end) publish();
                    if (more && jn == 0) {
                        if (!unit_end) __syncthreads();   // every wave done reading the window
                        open_slice(cs + 1, t0, ntaps);
                        __syncthreads();
                    }
                    j = jn;
                    if (jn == 0) ++cs;
                }
            } else {
                // (the weight's staging would cost the window its margin: fragments straight from
                // global memory, each row block's loaded one block ahead)
                auto load_w16g = [&](const uint16_t *p, uint4 (&f)[NP]) __attribute__((always_inline)) {
#pragma unroll
                    for (int k = 0; k < NP; ++k) f[k] = *reinterpret_cast<const uint4 *>(p + lane * 8 + k * 512);
                };
                // MFMAs of one step; block mb + 1's fragments (the next step's block 0 at the end)
                // are loaded before block mb's MFMAs
                auto mfma_pair_g = [&](const uint4 (&bv)[PB][NP], uint4 (&wa)[2][NP], const uint16_t *pcur,
                                       const uint16_t *pnext) __attribute__((always_inline)) {
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        load_w16g(mb + 1 < MB ? pcur + (size_t)(mb + 1) * (NP * 512) : pnext, wa[(mb + 1) & 1]);
#pragma unroll
                        for (int pb = 0; pb < PB; ++pb)
                            acc[mb][pb] = mfma16x16x32_np<T, NP>(wa[mb & 1], bv[pb], acc[mb][pb]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                static_assert(MB % 2 == 0, "row blocks in pairs: the next step's block 0 lands in slot 0");
                uint4 wa[2][NP], bv[PB][NP];
                prefetch_x(cs_lo);
                load_w16g(wptr16(cs_lo, 0), wa[0]);
                __syncthreads();   // previous pass done with the tables
                open_slice(cs_lo, t0, ntaps);
                __syncthreads();
                const int pf_j = max(npair - 2, 0);
                int cs = cs_lo, j = 0;   // step k's (slice, pair), advanced step by step
                for (int k = 0; k < nsteps; ++k) {
                    const bool more = k + 1 < nsteps;
                    const int jn = j + 1 == npair ? 0 : j + 1;
                    const int csn = jn == 0 ? cs + 1 : cs;
                    if (j == pf_j && cs + 1 < cs_hi) prefetch_x(cs + 1);
                    build_pair(cs, j, bv);
                    const uint16_t *pcur = wptr16(cs, j);
                    mfma_pair_g(bv, wa, pcur, more ? wptr16(csn, jn) : pcur);
                    if (more && jn == 0) {
                        __syncthreads();   // every wave done reading the current window
                        open_slice(csn, t0, ntaps);
                        __syncthreads();
                    }
                    cs = csn;
                    j = jn;
                }
            }
        }
    };

    if constexpr (DIM == 3) {
        // 3D: taps in groups of four, lane row q sampling tap 4 * group + q at its pixel for
        // all 16 channels of the slice (the corner geometry formed once per (pixel, tap)
        // rather than once per channel quad); a row transpose then gives every lane its
        // channel quad of the group's four taps, the B fragments of four steps.
        auto build_group = [&](int cs, int tg, int ntaps, acc4 (&bq)[4][PB]) __attribute__((always_inline)) {
            const int tl = tg * 4 + q;
            const int nq = min(4, (g.Cg - cs * BC) >> 2);   // channel quads of the slice in the group
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) {
                acc4 sv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) sv[j] = acc4{0.f, 0.f, 0.f, 0.f};
                if (tl < ntaps) {
                    const acc4 r = geo[tl * BPX + wave * (PB * 16) + pb * 16 + (lane & 15)];
                    if (nq == 4)
                        sample3_all<true>(g, wt, tile, xwin, xg + cs * BC, 4, r, deformable, sv);
                    else
                        sample3_all<false>(g, wt, tile, xwin, xg + cs * BC, nq, r, deformable, sv);
                }
                transpose_rows4(sv);
#pragma unroll
                for (int j = 0; j < 4; ++j) bq[j][pb] = sv[j];
            }
        };
        if (use16) {
            // 16x16x32 steps: a group's four taps are two tap pairs, each pair's B fragment its
            // two sampled quads (the 16-bit loop's K order, W16 below), split into pieces (fp32)
            // or rounded to T; the pair's A fragments come from global memory, each row block's
            // loaded one block ahead
            constexpr int NP = npiece_of<T>();
            const int nmb = fw.Mg_pad / 16;
            const uint16_t *wl = w16 + (size_t)mt * MB * (NP * 512);
            auto load_w16g = [&](const uint16_t *p, uint4 (&f)[NP]) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < NP; ++k) f[k] = *reinterpret_cast<const uint4 *>(p + lane * 8 + k * 512);
            };
            static_assert(MB % 2 == 0, "row blocks in pairs: the next step's block 0 lands in slot 0");
            passes([&](int t0, int ntaps) __attribute__((always_inline)) {
                const int ngr = (ntaps + 3) >> 2;
                const int ngroups = (cs_hi - cs_lo) * ngr;
                geo_og = geo_mg = -1;
                const int pp0 = (t0 / wt.tpp) * fw.hp;
                auto wptr16 = [&](int cs, int j) __attribute__((always_inline)) {
                    return wl + (((size_t)grp * slices + cs) * fw.pp + pp0 + j) * nmb * (NP * 512);
                };
                uint4 wa[2][NP];
                load_w16g(wptr16(cs_lo, 0), wa[0]);
                __syncthreads();   // previous pass done with the tables
                open_slice(cs_lo, t0, ntaps);
                __syncthreads();
                int cs = cs_lo, tg = 0;
                for (int k = 0; k < ngroups; ++k) {
                    const bool more = k + 1 < ngroups;
                    const int tgn = tg + 1 == ngr ? 0 : tg + 1;
                    const int csn = tgn == 0 ? cs + 1 : cs;
                    acc4 bq[4][PB];
                    build_group(cs, tg, ntaps, bq);
                    const int npr = (min(4, ntaps - tg * 4) + 1) >> 1;   // tap pairs of the group
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (h < npr) {
                            uint4 bv[PB][NP];
#pragma unroll
                            for (int pb = 0; pb < PB; ++pb) {
                                const float v[8] = {bq[2 * h][pb][0],     bq[2 * h][pb][1],     bq[2 * h][pb][2],
                                                    bq[2 * h][pb][3],     bq[2 * h + 1][pb][0], bq[2 * h + 1][pb][1],
                                                    bq[2 * h + 1][pb][2], bq[2 * h + 1][pb][3]};
                                pack8_16<T, NP>(v, 0, bv[pb]);   // (already at scale 2^s_b)
                            }
                            const uint16_t *pcur = wptr16(cs, 2 * tg + h);
                            const uint16_t *pnext =
                                h + 1 < npr ? wptr16(cs, 2 * tg + h + 1) : (more ? wptr16(csn, 2 * tgn) : pcur);
#pragma unroll
                            for (int mb = 0; mb < MB; ++mb) {
                                load_w16g(mb + 1 < MB ? pcur + (size_t)(mb + 1) * (NP * 512) : pnext, wa[(mb + 1) & 1]);
#pragma unroll
                                for (int pb = 0; pb < PB; ++pb)
                                    acc[mb][pb] = mfma16x16x32_np<T, NP>(wa[mb & 1], bv[pb], acc[mb][pb]);
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        }
                    }
                    if (more && tgn == 0) {
                        __syncthreads();   // every wave done reading the current window
                        open_slice(csn, t0, ntaps);
                        __syncthreads();
                    }
                    cs = csn;
                    tg = tgn;
                }
            });
        } else {
            passes([&](int t0, int ntaps) __attribute__((always_inline)) {
                const int ngr = (ntaps + 3) >> 2;   // tap groups per slice
                const int ngroups = (cs_hi - cs_lo) * ngr;
                geo_og = geo_mg = -1;   // a new pass of taps: the table must be rebuilt

                // group k = (slice cs_lo + k / ngr, taps 4 * (k % ngr) ..): its B fragments are
                // built at its start (the sampling's LDS latency is covered by the other wave of
                // the SIMD), then its steps run; wa holds the weight fragments of the next step.
                // The X window of a slice is loaded at the slice switch (the registers a prefetch
                // would hold across the steps are taken by the group's B fragments).
                acc4 wa[MB];
                load_w(wptr(cs_lo, t0), wa);
                __syncthreads();   // previous pass done with the tables
                open_slice(cs_lo, t0, ntaps);
                __syncthreads();
                int cs = cs_lo, tg = 0;   // group k's (slice, tap group), advanced group by group
                for (int k = 0; k < ngroups; ++k) {
                    const bool more = k + 1 < ngroups;
                    const int tgn = tg + 1 == ngr ? 0 : tg + 1;
                    const int csn = tgn == 0 ? cs + 1 : cs;
                    acc4 bq[4][PB];
                    build_group(cs, tg, ntaps, bq);
                    const int nt = min(4, ntaps - tg * 4);
                    const int tb = t0 + tg * 4;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (j < nt) {
                            // weight fragments of the step after this one (this step's own at the end)
                            const float *pn = j + 1 < nt ? wptr(cs, tb + j + 1)
                                                         : (more ? wptr(csn, t0 + tgn * 4) : wptr(cs, tb + j));
                            mfma_step(bq[j], wa, pn);
                        }
                    }
                    if (more && tgn == 0) {
                        __syncthreads();   // every wave done reading the current window
                        open_slice(csn, t0, ntaps);
                        __syncthreads();
                    }
                    cs = csn;
                    tg = tgn;
                }
            });
        }
    } else if (use16) {
        passes(pass16);
    } else {
        passes([&](int t0, int ntaps) __attribute__((always_inline)) {
            const int nsteps = (cs_hi - cs_lo) * ntaps;
            geo_og = geo_mg = -1;   // a new pass of taps: the table must be rebuilt

            // step k = (slice cs_lo + k / ntaps, tap k % ntaps). Invariant at the top of step k:
            // its B fragments are in bcur, its weight fragments in wa.
            acc4 wa[MB], bcur[PB], bnxt[PB];
            prefetch_x(cs_lo);
            load_w(wptr(cs_lo, t0), wa);
            __syncthreads();   // previous pass done with the tables
            open_slice(cs_lo, t0, ntaps);
            __syncthreads();
            build_b(cs_lo, 0, bcur);
            // the next slice's X window is requested PF steps before it is needed (memory
            // latency exceeds one step's MFMAs), or at the slice's first step when shorter
            const int pf_tl = max(ntaps - PF, 0);
            int cs = cs_lo, tl = 0;   // step k's (slice, tap), advanced step by step
            for (int k = 0; k < nsteps; ++k) {
                const bool more = k + 1 < nsteps;
                const int tln = tl + 1 == ntaps ? 0 : tl + 1;
                const int csn = tln == 0 ? cs + 1 : cs;
                const bool new_slice = more && tln == 0;
                if (tl == pf_tl && cs + 1 < cs_hi) prefetch_x(cs + 1);
                if (more && !new_slice) build_b(csn, tln, bnxt);
                mfma_step(bcur, wa, more ? wptr(csn, t0 + tln) : wptr(cs, t0 + tl));
                if (new_slice) {
                    __syncthreads();   // every wave done reading the current window
                    open_slice(csn, t0, ntaps);
                    __syncthreads();
                    build_b(csn, 0, bnxt);
                }
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) bcur[pb] = bnxt[pb];
                cs = csn;
                tl = tln;
            }
        });
    }

    // ---- epilogue: + bias, store NC<spatial>. With several shares each stores its fp32 partial to
    //      its own plane of y32 in the accumulators' order (whole 1 KB wave stores; in y's order the
    //      partials of 128 rows x 256 pixels took half of a one-slice workgroup's 36 us), bias with
    //      the first share; share_sum_kernel adds the planes in order, so the result is deterministic.
    const size_t tile_id = ((size_t)grp * n_sp + sp) * fw.m_tiles + mt;
    float *frag = nullptr;
    if (fw.ksplit > 1)
        frag = y32 + ((((size_t)ks * g.G * n_sp * fw.m_tiles + tile_id) * NW + wave) * (MB * PB)) * 256 + lane * 4;
    int pix[PB];
#pragma unroll
    for (int pb = 0; pb < PB; ++pb) pix[pb] = tile.pixel(g, wt, wave * (PB * 16) + pb * 16 + (lane & 15));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m0 = mt * BMR + mb * 16;
        acc4 bv = acc4{0.f, 0.f, 0.f, 0.f};
        if (bias != nullptr && ks == 0)
#pragma unroll
            for (int v = 0; v < 4; ++v) bv[v] = to_acc<float>(bias[grp * g.Mg + min(m0 + 4 * q + v, g.Mg - 1)]);
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) {
            acc4 r = acc[mb][pb];
#pragma unroll
            for (int v = 0; v < 4; ++v) r[v] = (s_back != 0 ? ldexpf(r[v], s_back) : r[v]) + bv[v];
            if (fw.ksplit > 1)
                *reinterpret_cast<acc4 *>(frag + (mb * PB + pb) * 256) = r;
            else
                store_frag<T>(g, y + ((size_t)tile.b * g.M + (size_t)grp * g.Mg) * g.Pn, m0, pix[pb], fw.vec, r);
        }
    }
}

// The fragments of share_sum: wave = 16 rows x 16 pixels of one tile, summed over the shares in order and
// stored in y's order. Bound by the partials' bytes, read once each.
template <typename T, int MB>
__global__ void __launch_bounds__(256) share_sum_kernel(const Geo g, const WinTiles wt, const FwdWin fw,
                                                        const float *__restrict__ part, T *__restrict__ y, size_t frags) {
    const int lane = threadIdx.x & 63;
    const size_t f = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);   // ((tile * NW + wave) * MB + mb) * PB + pb
    if (f >= frags) return;
    const float *src = part + f * 256 + lane * 4;
    acc4 v = *reinterpret_cast<const acc4 *>(src);
#pragma unroll 4
    for (int k = 1; k < fw.ksplit; ++k) v += *reinterpret_cast<const acc4 *>(src + (size_t)k * frags * 256);
    const int i = (int)(f % (NW * MB * PB));
    const int pb = i % PB, mb = i / PB % MB, wave = i / (PB * MB);
    int L = (int)(f / (NW * MB * PB));
    const int mt = L % fw.m_tiles;
    L /= fw.m_tiles;
    const int n_sp = g.B * wt.ntile[0] * wt.ntile[1] * wt.ntile[2];
    const int grp = L / n_sp;
    Tile tile;
    tile.init(g, wt, L % n_sp, 0, grp);
    store_frag<T>(g, y + ((size_t)tile.b * g.M + (size_t)grp * g.Mg) * g.Pn, (mt * MB + mb) * 16,
                  tile.pixel(g, wt, wave * (PB * 16) + pb * 16 + (lane & 15)), fw.vec, v);
}

// weight (M, Cg, Kn) -> Wp[G][slices][Kn][Mg_pad / 16][16 m][16 c], zero padded (grid-stride loop
// over the calling grid)
template <typename T>
__device__ __forceinline__ void fwd_weight_f32(const T *__restrict__ w, float *__restrict__ wp, int G, int Mg, int Cg,
                                               int Kn, int slices, int Mg_pad) {
    // 32-bit index arithmetic (the launcher refuses layouts of 2^31 elements or more)
    const unsigned total = (unsigned)G * slices * Kn * Mg_pad * BC;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int ci = (int)(i % BC);
        unsigned r = i / BC;
        const int m = (int)(r % Mg_pad);   // row blocks of 16 are consecutive: m = block * 16 + row
        r /= Mg_pad;
        const int t = (int)(r % Kn);
        r /= Kn;
        const int cs = (int)(r % slices);
        const int grp = (int)(r / slices);
        const int c = cs * BC + ci;
        float v = 0.f;
        if (m < Mg && c < Cg) v = to_acc<float>(w[(((size_t)grp * Mg + m) * Cg + c) * Kn + t]);
        wp[i] = v;
    }
}

template <typename T>
__global__ void fwd_win_weight_kernel(const T *__restrict__ w, float *__restrict__ wp, int G, int Mg, int Cg, int Kn,
                                      int slices, int Mg_pad) {
    fwd_weight_f32<T>(w, wp, G, Mg, Cg, Kn, slices, Mg_pad);
}

// the weight as W16 (w16_block) and, wp, in the fp32 loop's layout, in one launch
template <typename T, int NP>
__global__ void __launch_bounds__(256)
fwd_w16_kernel(const T *__restrict__ w, uint16_t *__restrict__ out, int *flag, int G, int Mg, int Cg, int Kn, int slices,
               int nmb, int tpp, int hp, int pp, float *__restrict__ wp) {
    if (wp != nullptr) fwd_weight_f32<T>(w, wp, G, Mg, Cg, Kn, slices, nmb * 16);
    w16_block<T, NP>(blockIdx.x, gridDim.x, w, out, flag, G, Mg, Cg, Kn, slices, nmb, tpp, hp, pp);
}

template <int DIM, typename T, int MB, bool STAGE, int LOOP, bool ONE>
hipError_t launch_k1(const Geo &g, const WinTiles &wt, const FwdWin &fw, const void *xcl, const void *wf,
                    const void *w16, const int *flag, const void *offset, const void *mask, const void *bias, void *y,
                    void *y32, hipStream_t s) {
    auto kern = fwd_win_kernel<DIM, T, MB, STAGE, LOOP, ONE>;
    const size_t lds = ((size_t)GEO_WORDS + (size_t)(wt.cells + (DIM == 3)) * XS) * sizeof(float) + fw.stage_bytes;
    static std::atomic<unsigned long long> lds_raised{0};   // per device, see raise_lds_limit
    if (const hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(kern), lds_raised); e != hipSuccess)
        return e;
    const long long blocks = (long long)g.G * g.B * wt.ntile[0] * wt.ntile[1] * wt.ntile[2] * fw.m_tiles * fw.ksplit;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NT), lds, s, g, wt, fw, static_cast<const float *>(xcl),
                       static_cast<const float *>(wf), static_cast<const uint16_t *>(w16), flag,
                       static_cast<const T *>(offset), static_cast<const T *>(mask),
                       static_cast<const T *>(bias), static_cast<T *>(y), static_cast<float *>(y32));
    return hipGetLastError();
}

// fp16 / bf16: the 16-bit loop. fp32: both loops, as kernels of their own where that pays for the launch that is not
// selected (fw.split, 2D / 3D: see split_loops)
template <int DIM, typename T, int MB, bool STAGE>
hipError_t launch_k(const Geo &g, const WinTiles &wt, const FwdWin &fw, const void *xcl, const void *wf,
                    const void *w16, const int *flag, const void *offset, const void *mask, const void *bias, void *y,
                    void *y32, hipStream_t s) {
    if constexpr (npiece_of<T>() == 2) {
        if (DIM == 1 || w16 == nullptr || flag == nullptr || !fw.split)
            return launch_k1<DIM, T, MB, STAGE, LOOP_BOTH, false>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
    }
    if constexpr (npiece_of<T>() == 1 || DIM > 1) {
        const hipError_t e =
            g.Kn <= wt.tpp
                ? launch_k1<DIM, T, MB, STAGE, LOOP_16, true>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s)
                : launch_k1<DIM, T, MB, STAGE, LOOP_16, false>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
        if (e != hipSuccess || npiece_of<T>() == 1) return e;
        if constexpr (npiece_of<T>() == 2)
            return launch_k1<DIM, T, MB, STAGE, LOOP_F32, false>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
    }
    return hipErrorInvalidValue;
}

template <int DIM, typename T>
hipError_t launch_m(const Geo &g, const WinTiles &wt, const FwdWin &fw, const void *xcl, const void *wf,
                    const void *w16, const int *flag, const void *offset, const void *mask, const void *bias, void *y,
                    void *y32, hipStream_t s) {
    // 3D: 64-row tiles only (the trilinear sampler needs the registers), no weight staging
    if constexpr (DIM < 3) {
        if (fw.stage_bytes > 0) {
            if (fw.mb == 8) return launch_k<DIM, T, 8, true>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
            if (fw.mb == 4) return launch_k<DIM, T, 4, true>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
            return hipErrorInvalidValue;
        }
        if (fw.mb == 8) return launch_k<DIM, T, 8, false>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
    }
    if (fw.mb == 4) return launch_k<DIM, T, 4, false>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_d(int dim, const Geo &g, const WinTiles &wt, const FwdWin &fw, const void *xcl, const void *wf,
                    const void *w16, const int *flag, const void *offset, const void *mask, const void *bias, void *y,
                    void *y32, hipStream_t s) {
    switch (dim) {
        case 1: return launch_m<1, T>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
        case 2: return launch_m<2, T>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
        case 3: return launch_m<3, T>(g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

size_t x_window_cell_bytes() { return XS * sizeof(float); }

// Rows per workgroup and shares of the (pass, channel slice) units, from a model of the launch's time:
// one workgroup per CU at a time (the window takes most of the LDS), so `rounds` of the chip, each a
// start and a table fill plus the share's units, then the sum of the partials. Microseconds, measured
// on one to eight units of 5 tap pairs and 16 to 256 workgroups: a unit takes about the same with 64
// rows as with 128, so the larger tile wins unless the GEMM side is small, and a grid that leaves
// CUs idle takes more shares instead. Inference, us a call, against 64-row tiles in at most two
// shares: float16 256 -> 256 channels k3 on one 25 x 38 image (48 workgroups of 8 units -> 192 of
// 1) 110 -> 58; bfloat16 128 -> 128 on 2 x 100 x 152 (280 of 8, two rounds -> 140 of 128 rows)
// 177 -> 127; float16 3D 32 -> 32 k3 on 9 x 28 x 30 (96 of 4 passes -> 192 of 2) 91 -> 61.
namespace {
constexpr double SHARE_US = 8.0, PAIR_US = 2.0, SUM_US = 5.0, SUM_BYTES_PER_US = 4e6;
constexpr size_t SHARE_BYTES_MAX = (size_t)64 << 20;   // partials of one call
// Whether a float32 launch of `us` modelled microseconds runs its two loops as kernels of their own: fewer registers
// for the launch that is not selected, 4 us. Inference, us a call, one kernel against two: 1D never (512 channels k5 on
// 16 x 4096 773 / 774, 16 on 100 24 / 27); 2D from 100 (256 channels k3 on 8 x 64x64 222 / 220, 128 on 2 x 100x152
// 131.4 / 130.0, but 256 on 2 x 64x64 84.7 / 85.3, 16 on 8x8 24 / 27); 3D, whose sampler spills beside a second loop,
// from 15 (64 channels k3 on 2 x 16x56x56 599 / 542, on 8x20x20 67 / 64, but 16 channels k1 on 4x4x4 28 / 31).
bool split_loops(int dim, double us) { return dim == 2 ? us >= 100.0 : dim == 3 && us >= 15.0; }
void split_shares(FwdWin &f, const Geo &g, int dim, int mb_max, long long spatial, int slices, int tpp, int npiece, bool lean) {
    const int npass = (g.Kn + tpp - 1) / tpp, units = npass * slices;
    double best = 0.0;
    for (int mb = mb_max; mb >= 4; mb -= 4) {
        const int m_tiles = (g.Mg + 16 * mb - 1) / (16 * mb);
        const double out_bytes = 4.0 * spatial * m_tiles * (16 * mb * BPX);   // a share's partials
        const double unit_us = (tpp + 1) / 2 * PAIR_US * (mb == 8 ? (npiece == 2 ? 1.3 : 1.1) : 1.0);
        for (int ks = 1; ks <= (lean ? 1 : std::min(units, 64)); ++ks) {
            const int per = (units + ks - 1) / ks;
            if ((units + per - 1) / per != ks) continue;   // the same units per share with fewer shares
            if (ks > 1 && out_bytes * ks > (double)SHARE_BYTES_MAX) break;
            const long long rounds = (spatial * m_tiles * ks + 255) / 256;
            const double us = rounds * (SHARE_US + per * unit_us) + (ks > 1 ? SUM_US + 2 * ks * out_bytes / SUM_BYTES_PER_US : 0.0);
            if (best == 0.0 || us < best) {
                best = us;
                f.mb = mb;
                f.ksplit = ks;
                f.units_per = per;
                f.split = split_loops(dim, us);
            }
        }
    }
}
}  // namespace

FwdWin plan_fwd_win(const Geo &g, const WinTiles &base, int dim, WinTiles &wt, bool lean) {
    FwdWin f{};
    f.ok = false;
    wt = base;
    if (!base.ok || g.Mg < 16) return f;
    // 3D samples taps in groups of four: passes of eight taps fill their groups (27 taps:
    // 8, 8, 8, 3 = seven groups, where passes of nine would take nine)
    const int tpp = dim == 3 && g.Kn > WIN_TMAX ? 8 : base.tpp;
    const long long spatial = (long long)g.G * g.B * base.ntile[0] * base.ntile[1] * base.ntile[2];
    const int slices = (g.Cg + BC - 1) / BC;
    // (3D: one more cell, the zero cell)
    const int zc = dim == 3 ? 1 : 0;
    // window of a tile of mb row blocks beside `extra` bytes of LDS (XQ quads prefetched per thread)
    auto window = [&](int mb, int extra) {
        return win_resize(base, g, dim, (size_t)(GEO_WORDS + zc * XS) * sizeof(float) + extra, XS * sizeof(float),
                          (long long)xq_of(mb) * NT / 4 - zc);
    };
    // 128-row tiles prefetch fewer window cells: not where that costs the window its margin (strided
    // layers, whose samples outside it would go to global memory)
    const bool wide = dim < 3 && g.Mg > 64 && window(8, 0).R[2] >= std::min(window(4, 0).R[2], 4);
    split_shares(f, g, dim, wide ? 8 : 4, spatial, slices, tpp, base.npiece, lean);
    const int rows = 16 * f.mb;
    const long long max_cells = (long long)xq_of(f.mb) * NT / 4;
    wt = window(f.mb, 0);
    if (wt.cells == 0) return f;   // no window fits: the unwindowed forward
    // 1D / 2D: two staging buffers of the 16-bit loop's weight blocks (8 row blocks x npiece KB
    // each: one step of 128-row tiles or two of 64-row tiles) when the window keeps a margin of
    // min(R, 4) cells beside them (a smaller window sends samples to global memory)
    f.stage_bytes = 0;
    if (dim < 3) {
        const int stage = 2 * 8 * base.npiece * 1024;
        const WinTiles ws = window(f.mb, stage);
        const int e = 2;   // the last axis: used in every rank
        if (ws.cells > 0 && ws.R[e] >= std::min(wt.R[e], 4)) {
            wt = ws;
            f.stage_bytes = stage;
        }
    }
    const size_t lds = ((size_t)GEO_WORDS + (size_t)(wt.cells + zc) * XS) * sizeof(float) + f.stage_bytes;
    if (lds > WIN_LDS_TARGET || wt.cells > max_cells) return f;
    f.m_tiles = (g.Mg + rows - 1) / rows;
    f.Mg_pad = f.m_tiles * rows;
    f.Cg_pad = (g.Cg + BC - 1) / BC * BC;
    wt.tpp = tpp;
    f.part_elems = f.ksplit > 1 ? (size_t)f.ksplit * spatial * f.m_tiles * rows * BPX : 0;
    f.vec = g.P[2] % 4 == 0 && wt.box[2] % 4 == 0;
    // 16-bit weight fragments
    f.npiece = base.npiece;
    f.tpp = wt.tpp;
    f.hp = (wt.tpp + 1) / 2;
    f.pp = (g.Kn + wt.tpp - 1) / wt.tpp * f.hp;
    f.w16_elems = (size_t)g.G * slices * f.pp * (f.Mg_pad / 16) * f.npiece * 512;
    // the layout kernels index in 32 bits
    if ((size_t)g.G * slices * g.Kn * f.Mg_pad * BC > (size_t)INT_MAX || f.w16_elems / 8 > (size_t)INT_MAX) return f;
    f.ok = true;
    return f;
}

hipError_t launch_fwd_win_layout(int dtype, const Geo &g, const FwdWin &fw, const void *w, void *wp, hipStream_t s) {
    const int slices = fw.Cg_pad / BC;
    const size_t n = (size_t)g.G * slices * g.Kn * fw.Mg_pad * BC;
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
#define TVDCN_FWL(T)                                                                                             \
    hipLaunchKernelGGL((fwd_win_weight_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, s, static_cast<const T *>(w), \
                       static_cast<float *>(wp), g.G, g.Mg, g.Cg, g.Kn, slices, fw.Mg_pad);                      \
    return hipGetLastError();
    switch (dtype) {
        case kF32: { TVDCN_FWL(float) }   // (fp16 / bf16 run no fp32 loop)
    }
#undef TVDCN_FWL
    return hipErrorInvalidValue;
}

hipError_t launch_fwd_win_layout16(int dtype, const Geo &g, const FwdWin &fw, const void *w, void *w16, int *flag,
                                   hipStream_t s, void *wp) {
    if (fw.w16_elems == 0) return wp != nullptr ? launch_fwd_win_layout(dtype, g, fw, w, wp, s) : hipSuccess;
    const int slices = fw.Cg_pad / BC;
    size_t n = fw.w16_elems / (fw.npiece * 8);   // threads: one per lane fragment
    if (wp != nullptr) n = std::max(n, (size_t)g.G * slices * g.Kn * fw.Mg_pad * BC);
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
#define TVDCN_FW16(T, NP)                                                                                              \
    hipLaunchKernelGGL((fwd_w16_kernel<T, NP>), dim3((unsigned)blocks), dim3(256), 0, s, static_cast<const T *>(w),    \
                       static_cast<uint16_t *>(w16), flag, g.G, g.Mg, g.Cg, g.Kn, slices, fw.Mg_pad / 16, fw.tpp,    \
                       fw.hp, fw.pp, static_cast<float *>(wp));                                                        \
    return hipGetLastError();
    switch (dtype) {
        case kF32: { TVDCN_FW16(float, npiece_of<float>()) }   // (fp16 / bf16: launch_prep16)
    }
#undef TVDCN_FW16
    return hipErrorInvalidValue;
}

static hipError_t launch_share_sum(int dtype, const Geo &g, const WinTiles &wt, const FwdWin &fw, const void *y32, void *y,
                                   hipStream_t s) {
    const size_t frags = fw.part_elems / fw.ksplit / 256;
    const dim3 grid((unsigned)((frags + 3) / 4));
    auto go = [&](auto tv, auto mv) {
        using T = decltype(tv);
        hipLaunchKernelGGL((share_sum_kernel<T, decltype(mv)::value>), grid, dim3(256), 0, s, g, wt, fw,
                           static_cast<const float *>(y32), static_cast<T *>(y), frags);
        return hipGetLastError();
    };
    auto by_mb = [&](auto tv) {
        return fw.mb == 8 ? go(tv, std::integral_constant<int, 8>()) : go(tv, std::integral_constant<int, 4>());
    };
    switch (dtype) {
        case kF32: return by_mb(float());
        case kF16: return by_mb(__half());
        case kBF16: return by_mb(__hip_bfloat16());
    }
    return hipErrorInvalidValue;
}

hipError_t launch_fwd_win(int dtype, int dim, const Geo &g, const WinTiles &wt, const FwdWin &fw_, const void *xcl,
                          const void *wf, const void *w16, const int *flag, const void *offset, const void *mask,
                          const void *bias, void *y, void *y32, hipStream_t s) {
    if (fw_.ksplit != 1 && y32 == nullptr) return hipErrorInvalidValue;
    if (dtype != kF32 && w16 == nullptr) return hipErrorInvalidValue;
    if (g.B == 0) return hipSuccess;
    // (a batch block's output may be less aligned than the caller's)
    const size_t quad = 4 * (dtype == kF32 ? sizeof(float) : sizeof(uint16_t));
    FwdWin fw = fw_;
    fw.vec = fw.vec && reinterpret_cast<uintptr_t>(y) % quad == 0;
    hipError_t e = hipErrorInvalidValue;
    switch (dtype) {
        case kF32: e = launch_d<float>(dim, g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s); break;
        case kF16: e = launch_d<__half>(dim, g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s); break;
        case kBF16:
            e = launch_d<__hip_bfloat16>(dim, g, wt, fw, xcl, wf, w16, flag, offset, mask, bias, y, y32, s);
            break;
    }
    return e != hipSuccess || fw.ksplit == 1 ? e : launch_share_sum(dtype, g, wt, fw, y32, y, s);
}

}  // namespace tvdcn_hip
