// ib3d_sor_march.h -- two red-black sweeps in one pass over a large grid, FP64
// and FP32.  Included by ib3d_sor.hip after ib3d_sor_block.h.
#pragma once

// Two whole sweeps, src -> dst, bit for bit four half-sweeps (k_sor's update,
// operand for operand; see k_sor_block about the two buffers, TRACK, FIRST and
// APPLY).  A workgroup owns a tile of colour slots and rows and a chunk of
// planes, and marches through the planes with four updates in flight: on the step
// that brings plane k in, it updates red at k-1 and black at k-2 for the first
// time, red at k-3 and black at k-4 for the second.  What an update reads in its
// own column (the planes below and above, the other colour's cell, its own old
// value) the thread holds in registers, in rings of three planes; the
// neighbouring columns' values come from LDS, written one step earlier (two
// buffers, one barrier per step).  The tile is loaded with a halo of four cells
// (two slots, four rows) on the sides that do not end the grid, and a chunk of
// planes starts and ends four planes outside.
//
// A thread owns one slot (a red and a black cell of every plane).  Rows of one
// parity share waves, so which neighbour is the slot's own other cell (q) is
// uniform: it is the same for all four updates of a step and alternates from
// step to step.  The loop is unrolled over twelve steps, so that q, the rings'
// entries and the LDS buffer are compile-time constants; the two parities run
// copies of the loop that differ in q.
//
// Of the four updates of a step each needs the one before as its plane above,
// but that is the last of the six subtractions: all that precedes it is done
// for the four together, and only the last subtraction, the quotient and the
// relaxation chain.  The FP64 quotients are block_div's; whether one of them was
// out of its range is asked once per chunk, which is then marched again with
// divisions.
//
// The first eight planes of a chunk only feed the ones above them, by one more
// update every two planes, so their steps do none to three of the four: 20 of the
// 160 updates per slot of a chunk of 32 planes (FP64 with TRACK 38.0 -> 35.4 us per
// sweep at 256x192x192, FP32 17.3 -> 16.5).
//
// What bounds it: vector arithmetic (58% of the issue slots in FP32, 69% in FP64;
// the rest is the four updates' chain, 15 LDS reads per step and the barrier, at four
// waves per SIMD), of which the halo is 1.65 times at 256x192x192.  us per sweep, k_sor_pz
// (FP32: k_sweep2_pz) -> here: FP64 with TRACK 66.8 -> 35.4 at 256x192x192, 180 ->
// 92 at 384x256x256 (the half-sweeps' atomicMax and, from 384x256x256 on, an
// Infinity Cache that no longer holds the arrays); FP32 25-28 -> 16.5 at
// 256x192x192, 63.7 -> 43.3 at 384x256x256 (half-sweeps), level 1 of 256x192x192
// (128x96x96) 9.2 -> 6.1.
//
// Measured and dropped: one step at a time with every update in a branch of its
// own (FP64 48 us per sweep, FP32 28.5); the four updates together but the rings
// moved on every step (FP32 24.5); 64 registers and two workgroups per CU with
// chunks of half the planes (FP32 24.2); 24 x 42 tiles (20.4), 36 x 20 (21.7),
// 36 x 14 (31.2).
// HX slots x EY rows; half of the threads for the rows of either parity
template <int HX, int EY> struct MarchShape {
    static constexpr int HALF = HX * (EY / 2), HP = (HALF + 63) / 64 * 64, NT = 2 * HP;
    static_assert(EY % 2 == 0 && NT <= 1024, "march shape");
};

// The workgroup's barrier, for waves that run different copies of a loop: the
// hardware counts waves, each of which passes the same number of barriers.
__device__ __forceinline__ void wave_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <typename T, int HX, int EY, bool FIRST, bool TRACK, bool APPLY>
__global__ void __launch_bounds__((MarchShape<HX, EY>::NT))
k_sor_march(const T *__restrict__ s0, const T *__restrict__ s1, T *__restrict__ d0, T *__restrict__ d1,
            const T *__restrict__ b0, const T *__restrict__ b1, const T *__restrict__ axc, const T *__restrict__ ayc,
            const T *__restrict__ azc, SorGeom g, int ntx, int nty, int tz, T omega, T omm, const double *gate,
            double thr, const double *prev, double *slot, double *__restrict__ acc0, double *__restrict__ acc1) {
    using S = MarchShape<HX, EY>;
    constexpr int HALF = S::HALF, HP = S::HP, NT = S::NT, PAD = HX + 1;
    __shared__ T L[2][4][PAD + EY * HX + PAD];
    __shared__ T X[2][3][sizeof(T) == 8 ? HX : 1];
    __shared__ int stop;
    if (!TRACK && gated(gate, thr)) return;
    const int tid = (int)threadIdx.x;
    const int blk = xcd_block();
    const int bz = blk / (ntx * nty), br = blk - bz * (ntx * nty), by = br / ntx, bx = br - by * ntx;
    // own slots [o0, o1) and rows [r0, r1); the tile covers HX slots from h0 and
    // EY rows from j0
    const int NS = (g.sx - 2) / 2 + 1;
    const int o0 = bx == 0 ? 0 : (HX - 2) + (bx - 1) * (HX - 4), o1 = bx == ntx - 1 ? NS : (HX - 2) + bx * (HX - 4);
    const int h0 = bx == 0 ? 0 : o0 - 2;
    const int r0 = by == 0 ? 1 : (EY - 4) + (by - 1) * (EY - 8),
              r1 = by == nty - 1 ? g.sy - 1 : (EY - 4) + by * (EY - 8);
    const int j0 = by == 0 ? 0 : r0 - 4;
    const int k0 = 1 + bz * tz, k1 = min(k0 + tz, g.sz - 1);
    const int par = __builtin_amdgcn_readfirstlane(tid >= HP ? 1 : 0);   // parity of the rows of this wave
    const int w = tid - par * HP;
    const int wc = min(w, HALF - 1);
    const int ly = 2 * (wc / HX) + ((par + j0) & 1), h = wc % HX;
    const int hs = h0 + h, jj = j0 + ly;
    const bool in = w < HALF && hs < g.H && jj < g.sy;
    const bool own = in && hs >= o0 && hs < o1 && jj >= r0 && jj < r1;
    const int hc = min(hs, g.H - 1), jc = min(jj, g.sy - 1);
    const uint32_t base = (uint32_t)(jc * g.H + hc);
    const int li = PAD + ly * HX + h;
    auto at = [](const T *p, uint32_t i) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (uint32_t)sizeof(T));
    };
    typedef __attribute__((address_space(4))) T CT;
    const CT *az = (const CT *)azc;
    // x coefficients of the tile's slots: parity q, then west, diagonal, east; in
    // FP64 read from LDS on every step, in FP32 held in registers
    constexpr bool XLDS = sizeof(T) == 8;
    if (XLDS && tid < 6 * HX) {
        const int a = tid / HX % 3, i = min(2 * (h0 + tid % HX) + tid / (3 * HX), g.sxp - 1);
        X[tid / (3 * HX)][a][tid % HX] = axc[a * g.sxp + i];
    }
    T xr[2][3] = {};
    if (!XLDS)
#pragma unroll
        for (int a = 0; a < 6; a++) xr[a / 3][a % 3] = axc[a % 3 * g.sxp + min(2 * hc + a / 3, (int)g.sxp - 1)];
    const T y1 = ayc[jc], y2 = ayc[g.sy + jc], y3 = ayc[2 * g.sy + jc];
    if (TRACK) {
        if (tid < 64) {
            const double pv = prev && tid < 2 * kBlockSub ? prev[tid] : 0.0;
            const unsigned long long hot = __ballot(pv >= thr);
            bool done = false;
            for (int q = 0; q < 2; q++) done |= ((hot >> (q * kBlockSub)) & ((1u << kBlockSub) - 1u)) == 0;
            if (tid == 0) stop = prev && done;
        }
        __syncthreads();
        if (stop) return;
    }
    for (int i = tid; i < 8 * (PAD + EY * HX + PAD); i += NT) (&L[0][0][0])[i] = T(0);
    __syncthreads();
    constexpr int A = PAD + EY * HX + PAD;
    constexpr int AHEAD = sizeof(T) == 8 ? 1 : 2;   // steps that the loads run ahead
    bool hot[2];   // a live owned cell moved by thr or more in sweep 1, 2
    // the whole march; fast: block_div's quotients, true when one of them may
    // not be the division's
    auto march = [&](auto fast, auto q0c) {
        constexpr bool F = decltype(fast)::value;
        constexpr int q0 = decltype(q0c)::value;
        // Rings of three planes: entry (k mod 3) of bo is old black of plane k, of
        // ra and ba red and black after the first sweep, of rc red after the
        // second, rb and bb the right-hand sides (0 where dead) and lr, lb whether
        // the cells are live
        T bo[3] = {}, ra[3] = {}, ba[3] = {}, rc[3] = {}, rb[3] = {}, bb[3] = {};
        bool lvr[3] = {}, lvb[3] = {};
        T za[4] = {}, zd[4] = {}, zc[4] = {};   // z coefficients, entry (plane mod 4)
        struct In {
            T bo, ro, rb, bb, er, eb;
        };
        In in_[AHEAD + 1];
        hot[0] = hot[1] = false;
        DivRange range;
        uint32_t o1 = 0, o2 = 0;   // offsets of planes k-1, k-2 of the loads
        auto plane_off = [&](int p) { return (uint32_t)(min(max(p, 0), g.sz - 1) * g.plane); };
        const int ka = k0 - 4, kb = k1 + 3;   // planes loaded
        o1 = plane_off(ka - 1);
        o2 = plane_off(ka - 2);
        auto load = [&](int k, In &n) {
            const uint32_t o0 = plane_off(k);
            n.bo = FIRST ? T(0) : at(s1, base + o0);
            n.ro = FIRST ? T(0) : at(s0, base + o1);
            n.rb = at(b0, base + o1);
            n.bb = at(b1, base + o2);
            if (APPLY) {
                n.er = at(s0, base + o1);
                n.eb = at(s1, base + o2);
            }
            o2 = o1;
            o1 = o0;
        };
        // ph = (k - ka) mod 12; the first U of the four updates
        auto step = [&](auto phc, auto uc, int k) {
            constexpr int ph = decltype(phc)::value, q = (q0 + ph) & 1, U = decltype(uc)::value;
            // ring entries of planes k .. k-5, with plane k at entry ph mod 3
            constexpr int e0 = ph % 3, e1 = (ph + 2) % 3, e2 = (ph + 1) % 3, e3 = e0, e4 = e1, e5 = e2;
            constexpr int f1 = (ph + 3) % 4, f2 = (ph + 2) % 4, f3 = (ph + 1) % 4, f4 = ph % 4;
            const T *lr = &L[(ph + 1) & 1][0][0];
            T *lw = &L[ph & 1][0][0];
            const In n = in_[ph % (AHEAD + 1)];
            // z coefficients of plane k-1
            const int pz = min(max(k - 1, 0), g.sz - 1);
            za[f1] = az[pz];
            zd[f1] = az[g.sz + pz];
            zc[f1] = az[2 * g.sz + pz];
            load(k + AHEAD + 1, in_[ph % (AHEAD + 1)]);
            // (the entries of plane k-3 and before are still the rings' oldest)
            const T ro = n.ro, rhs3 = rb[e3], old1 = ra[e3], bo2 = bo[e2], bo1 = bo[e1];
            const bool live3 = lvr[e3], live4 = lvb[e4];
            const T rhs4 = bb[e4], rc5 = rc[e5], rc4 = rc[e4], ba4 = ba[e4], ba3 = ba[e3], ra2 = ra[e2];
            const bool live1 = in && k - 1 >= 1 && k - 1 <= g.sz - 2 && n.rb == n.rb;
            const bool live2 = in && k - 2 >= 1 && k - 2 <= g.sz - 2 && n.bb == n.bb;
            const T rhs1 = live1 ? n.rb : T(0), rhs2 = live2 ? n.bb : T(0);
            if (APPLY && own) {
                if (k - 1 >= k0 && k - 1 < k1 && live1) acc0[base + (uint32_t)((k - 1) * g.plane)] += (double)n.er;
                if (k - 2 >= k0 && k - 2 < k1 && live2) acc1[base + (uint32_t)((k - 2) * g.plane)] += (double)n.eb;
            }
            const T x1 = XLDS ? X[q][0][h] : xr[q][0], xy = (XLDS ? X[q][1][h] : xr[q][1]) + y2,
                    x3 = XLDS ? X[q][2][h] : xr[q][2];
            // the four updates: everything but the plane above is known before the
            // first of them, so only the last subtraction, the quotient and the
            // relaxation chain
            auto part = [&](int a, T rhs, T ctr, T below, T z) {
                const T *l = lr + a * A;
                const T side = l[q ? li + 1 : li - 1];
                return ((((rhs - x1 * (q ? ctr : side)) - x3 * (q ? side : ctr)) - y1 * l[li - HX]) -
                        y3 * l[li + HX]) - z * below;
            };
            auto relax = [&](T v, T above, T z, T d, T pold, bool live) {
                v = v - z * above;
                const T den = xy + d;
                if (F) range.add(v);
                const T pnew = omm * pold + omega * (F ? block_div(v, den, block_rcp(den)) : sor_div(v, den));
                return live ? pnew : pold;
            };
            T g1 = 0, g2 = 0, g3 = 0, g4 = 0, v1 = ro, v2 = bo2, v3 = old1, v4 = ba4;
            if (U > 0) g1 = part(0, rhs1, bo1, bo2, za[f1]);
            if (U > 1) g2 = part(1, rhs2, ra2, old1, za[f2]);
            if (U > 2) g3 = part(2, rhs3, ba3, ba4, za[f3]);
            if (U > 3) g4 = part(3, rhs4, rc4, rc5, za[f4]);
            if (U > 0) v1 = relax(g1, n.bo, zc[f1], zd[f1], ro, live1);
            if (U > 1) v2 = relax(g2, v1, zc[f2], zd[f2], bo2, live2);
            if (U > 2) v3 = relax(g3, v2, zc[f3], zd[f3], old1, live3);
            if (U > 3) v4 = relax(g4, v3, zc[f4], zd[f4], ba4, live4);
            if (TRACK) {
                if (k - 1 >= k0 && k - 1 < k1) hot[0] |= (double)fabs(v1 - ro) >= thr;
                if (k - 2 >= k0 && k - 2 < k1) hot[0] |= (double)fabs(v2 - bo2) >= thr;
                if (k - 3 >= k0 && k - 3 < k1) hot[1] |= (double)fabs(v3 - old1) >= thr;
                if (k - 4 >= k0) hot[1] |= (double)fabs(v4 - ba4) >= thr;
            }
            if (own) {
                if (k - 3 >= k0 && k - 3 < k1) d0[base + (uint32_t)((k - 3) * g.plane)] = v3;
                if (k - 4 >= k0) d1[base + (uint32_t)((k - 4) * g.plane)] = v4;
            }
            if (w < HALF) {
                lw[li] = n.bo;
                lw[A + li] = v1;
                lw[2 * A + li] = v2;
                lw[3 * A + li] = v3;
            }
            bo[e0] = n.bo;
            ra[e1] = v1;
            rb[e1] = rhs1;
            lvr[e1] = live1;
            ba[e2] = v2;
            bb[e2] = rhs2;
            lvb[e2] = live2;
            rc[e3] = v3;
            wave_barrier();
        };
#pragma unroll
        for (int q = 0; q <= AHEAD; q++) load(ka + q, in_[q]);
        // the first planes only feed the updates above them: plane k0 - 3 is the
        // first to need one update, k0 - 2 two, k0 - 1 three, k0 four
#define IB3D_STEP(P, U) step(std::integral_constant<int, P>{}, std::integral_constant<int, U>{}, ka + P);
        IB3D_STEP(0, 0) IB3D_STEP(1, 0) IB3D_STEP(2, 1) IB3D_STEP(3, 1) IB3D_STEP(4, 2) IB3D_STEP(5, 2) IB3D_STEP(6, 3)
        IB3D_STEP(7, 3)
#undef IB3D_STEP
        for (int k = ka; k + 8 <= kb; k += 12) {
#define IB3D_STEP(P)                                                                                                \
    if (k + P > kb) break;                                                                                          \
    step(std::integral_constant<int, P % 12>{}, std::integral_constant<int, 4>{}, k + P);
            IB3D_STEP(8) IB3D_STEP(9) IB3D_STEP(10) IB3D_STEP(11) IB3D_STEP(12) IB3D_STEP(13) IB3D_STEP(14)
            IB3D_STEP(15) IB3D_STEP(16) IB3D_STEP(17) IB3D_STEP(18) IB3D_STEP(19)
#undef IB3D_STEP
        }
        return F && range.unsafe();
    };
    // q of the red cells of plane ka-1 in this wave's rows
    const bool odd = (par + k0 - 4 + 1) & 1;
    bool unsafe;
    if (odd)
        unsafe = march(std::true_type{}, std::integral_constant<int, 1>{});
    else
        unsafe = march(std::true_type{}, std::integral_constant<int, 0>{});
    if (sizeof(T) == 8 && __syncthreads_or(unsafe)) {   // again, with divisions
        if (odd)
            march(std::false_type{}, std::integral_constant<int, 1>{});
        else
            march(std::false_type{}, std::integral_constant<int, 0>{});
    }
    if (TRACK) {
        for (int q = 0; q < 2; q++) {
            if (__syncthreads_or(own && hot[q]) && tid == 0)
                atomicMax(reinterpret_cast<unsigned long long *>(slot + q * kBlockSub + (blk & (kBlockSub - 1))),
                          (unsigned long long)__double_as_longlong(thr));
        }
    }
}
