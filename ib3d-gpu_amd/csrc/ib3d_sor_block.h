// ib3d_sor_block.h -- several red-black sweeps of a block of cells in one
// launch (temporal blocking), FP64 and FP32.  Included by ib3d_sor.hip, which
// defines SorGeom, xcd_block, gated and wave_max.
#pragma once

// M whole sweeps, src -> dst, of the OX x OY x OZ cells a workgroup owns.
//
// The block is loaded with a halo of 2M cells on every side.  Half-sweep m
// (1..2M) updates its colour's cells at positions [m, E-m) of each axis, whose
// neighbours were exact after half-sweep m-1, so the owned cells are exact
// after the last one: bit for bit 2M half-sweep launches, since every update
// is k_sor's, operand for operand.  src is only read, so no workgroup sees
// another one's results; the owned interior cells (updated or not) go to dst,
// and cells never written (walls, padding) must already agree in both buffers.
//
// A thread holds one (i, j) column of the block in registers, its cells split
// by colour.  The columns are split by the parity of i + j + (first plane), one
// half of the waves each: in a wave of parity par, red entry t is plane
// 2t + par and black entry t plane 2t + 1 - par.  So every lane has work in
// every half-sweep, a global load is one colour array at consecutive slots, the
// z neighbours are registers of the thread, and the x and y neighbours are
// entry t of columns of the other parity, read from LDS: four reads and one
// write per update.
//
// Cells outside the arrays and cells with a NaN right-hand side are not updated
// (live); cells outside the arrays hold 0 and are read only by lanes whose
// result is not kept.
//
// What bounds it: a launch cannot take less than about 4.5 us (the gap to the
// launch it depends on, about 2.4 us, and the loads, which come from the
// Infinity Cache because another XCD wrote them); above that FP64 arithmetic,
// at 6 clocks per instruction and wave on this part, times the updates that
// the halo repeats (on 24 x 16 x 8 blocks the waves execute 2.75 updates per
// owned one).  The kernel replaces two k_sor_pz launches per sweep, each of
// which walks eight planes through two dependent loads (7-9 us whatever the
// grid).  us per FP64 sweep with TRACK, k_sor_pz -> here: 14.9 -> 3.5 at
// 32x24x24, 17.6 -> 4.1 at 48x32x32, 17.8 -> 6.0 at 64x48x48, 16.5 -> 8.2 at
// 128x64x64; FP32: 14.4 -> 3.1 at 48x32x32, 14.8 -> 3.3, 12.7 -> 4.8.
//
// Measured and dropped: one sweep per launch (28 x 12 x 8 blocks: 9.1 us at
// 128x64x64, 7.2 at 48x32x32), three (6.1 at 48x32x32), columns of both
// parities in one wave (the z neighbours and coefficients then need selects and
// three more LDS reads per update: 10.2 us per launch at 48x32x32 against 8.8),
// the z coefficients as scalar loads (their waits also drain the LDS reads:
// 11.4 us), and the compiler's division (below).
//
// FIRST: the sweep starts from zero, as k_sor's FIRST.  APPLY (with FIRST):
// the previous increment, still in src, is first added to the FP64 unknown
// (acc0, acc1) of the owned live cells.
//
// TRACK (the reference's stopping rule): max |new - old| of sweep q over the
// owned cells goes to slot[q * kBlockSub + (workgroup % kBlockSub)], spread over
// kBlockSub addresses because atomics on one address serialise; a value at or
// above thr is recorded as thr.  The launch does nothing when any sweep of the
// launch before (`prev`, same layout, or null) was below thr, and a launch that
// did nothing leaves its slots at zero and so stops all that follow.
static constexpr int kBlockSub = 16;

template <int M, int OX, int OY, int OZ> struct BlockShape {
    static constexpr int R = 2 * M, EX = OX + 2 * R, EY = OY + 2 * R, EZ = OZ + 2 * R;
    static constexpr int HX = EX / 2, HALF = HX * EY, HP = (HALF + 63) / 64 * 64, NT = 2 * HP, N2 = EZ / 2;
    static_assert(M <= 2 && 2 * N2 <= 32 && OX % 2 == 0 && OZ % 2 == 0 && NT <= 1024, "block shape");
};

// a / b in two parts: the reciprocal, once per cell and launch, and the
// quotient.  They are the steps the compiler emits for an FP64 division (two
// Newton steps on v_rcp_f64, a quotient and one residual correction, v_div_fixup
// for zeros and special values) without its scaling of extreme operands, which
// DivRange and the caller's check of the denominators (|b| in [2^-64, 2^64])
// make unnecessary; so the result is the division's.  The compiler's own
// sequence runs its steps through VCC, which keeps the divisions of
// neighbouring cells from overlapping: 28 ns per wave and division against 13.
// FP32 multiplies by the hardware reciprocal, as sor_div.
__device__ __forceinline__ double block_rcp(double b) {
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    return y;
}
__device__ __forceinline__ float block_rcp(float b) { return __builtin_amdgcn_rcpf(b); }

// numerators whose quotient block_div may round differently from a division
// (subnormal steps or an overflow on the way): nonzero below 2^-900, or 2^900
// and above (with infinities and NaN).  lo collects the smallest key - 1 (zero
// wraps to the largest), hi the largest key.
struct DivRange {
    uint32_t lo = 0xffffffffu, hi = 0;
    __device__ __forceinline__ void add(double a) {
        const uint32_t key = ((uint32_t)__double2hiint(a) << 1) | min((uint32_t)__double2loint(a), 1u);
        lo = min(lo, key - 1u);
        hi = max(hi, key);
    }
    __device__ __forceinline__ void add(float) {}
    __device__ __forceinline__ bool unsafe() const {
        return lo < ((1023u - 900u) << 21) - 1u || hi >= ((1023u + 900u) << 21);
    }
};
// (the fixup reads only the sign and range of its denominator: y serves)
__device__ __forceinline__ double block_div(double a, double b, double y) {
    const double q = a * y;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), y, q), y, a);
}
__device__ __forceinline__ float block_div(float a, float, float y) { return a * y; }

static constexpr int kBlockGroup = 4;   // updates of a column in flight together (2 and 8: the same or slower)
template <typename T, int M, int OX, int OY, int OZ, bool FIRST, bool TRACK, bool APPLY>
__global__ void __launch_bounds__((BlockShape<M, OX, OY, OZ>::NT))
k_sor_block(const T *__restrict__ s0, const T *__restrict__ s1, T *__restrict__ d0, T *__restrict__ d1,
            const T *__restrict__ b0, const T *__restrict__ b1, const T *__restrict__ axc, const T *__restrict__ ayc,
            const T *__restrict__ azc, SorGeom g, int nbx, int nby, T omega, T omm, const double *gate, double thr,
            const double *prev, double *slot, double *__restrict__ acc0, double *__restrict__ acc1) {
    using S = BlockShape<M, OX, OY, OZ>;
    constexpr int R = S::R, EX = S::EX, EY = S::EY, EZ = S::EZ, HX = S::HX, HALF = S::HALF, HP = S::HP, N2 = S::N2,
                  NT = S::NT, G = kBlockGroup;
    __shared__ T L[2][N2][2][HALF];
    __shared__ T zt[EZ][2];   // z coefficients (below, above) of the block's planes
    __shared__ T zd[EZ];      // and their diagonal part
    __shared__ int stop;
    __shared__ double dmax[TRACK ? M : 1][NT / 64];
    if (!TRACK && gated(gate, thr)) return;
    const int tid = (int)threadIdx.x;
    const int blk = xcd_block();
    const int bz = blk / (nbx * nby), br = blk - bz * (nbx * nby), by = br / nbx, bx = br - by * nbx;
    const int i0 = 1 + OX * bx - R, j0 = 1 + OY * by - R, k0 = 1 + OZ * bz - R;
    const int par = __builtin_amdgcn_readfirstlane(tid >= HP ? 1 : 0);
    const int w = tid - par * HP;
    const bool col_ok = w < HALF;
    const int ly = w / HX, h = w - ly * HX;
    const int e = (par + i0 + j0 + ly + k0) & 1;
    const int lx = 2 * h + e;
    const int ii = i0 + lx, jj = j0 + ly;
    const bool in_xy = col_ok && ii >= 0 && ii < g.sx && jj >= 0 && jj < g.sy;
    const int ic = min(max(ii, 0), g.sx - 1), jc = min(max(jj, 0), g.sy - 1);
    const bool own = in_xy && lx >= R && lx < EX - R && ly >= R && ly < EY - R && ii <= g.sx - 2 && jj <= g.sy - 2;
    const uint32_t base = (uint32_t)(jc * g.H + (ic >> 1));
    const T nan = (T)__builtin_nanf("");
    auto at = [](const T *p, uint32_t i) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (uint32_t)sizeof(T));
    };
    double pv = 0.0;
    if (TRACK && prev && tid < M * kBlockSub) pv = prev[tid];
    uint32_t live = 0;   // bit c * N2 + t: the cell is updated
    T X[2][N2], B[2][N2], Y[2][N2], D[2][N2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int q = c ? 1 - par : par;
#pragma unroll
        for (int t = 0; t < N2; t++) {
            const uint32_t f = base + (uint32_t)(min(max(k0 + 2 * t + q, 0), g.sz - 1) * g.plane);
            X[c][t] = (FIRST && !APPLY) ? T(0) : at(c ? s1 : s0, f);
            B[c][t] = at(c ? b1 : b0, f);
        }
    }
    const T a1x = axc[ic], a2x = axc[g.sxp + ic], a3x = axc[2 * g.sxp + ic];
    const T a1y = ayc[jc], a2y = ayc[g.sy + jc], a3y = ayc[2 * g.sy + jc];
    if (tid < EZ) zd[tid] = azc[g.sz + min(max(k0 + tid, 0), g.sz - 1)];
    if (tid < 2 * EZ) {
        const int k = tid >> 1;
        zt[k][tid & 1] = azc[(tid & 1) * 2 * g.sz + min(max(k0 + k, 0), g.sz - 1)];
    }
    if (TRACK && tid < 64) {
        // a sweep of the launch before that left every sub-slot below thr
        const unsigned long long hot = __ballot(pv >= thr);
        bool done = false;
        for (int q = 0; q < M; q++) done |= ((hot >> (q * kBlockSub)) & ((1u << kBlockSub) - 1u)) == 0;
        if (tid == 0) stop = prev && done;
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int q = c ? 1 - par : par;
#pragma unroll
        for (int t = 0; t < N2; t++) {
            const int kk = k0 + 2 * t + q;
            if (!(in_xy && kk >= 0 && kk < g.sz)) {
                X[c][t] = T(0);
                B[c][t] = nan;
            }
            const bool on = B[c][t] == B[c][t];
            live |= on ? 1u << (c * N2 + t) : 0u;
            if (APPLY && t >= R / 2 && t < N2 - R / 2) {
                if (own && kk <= g.sz - 2 && on)
                    (c ? acc1 : acc0)[base + (uint32_t)(kk * g.plane)] += (double)X[c][t];
            }
            if (FIRST) X[c][t] = on ? T(0) : X[c][t];
            B[c][t] = on ? B[c][t] : T(0);
            if (col_ok) L[c][t][par][w] = X[c][t];
        }
    }
    __syncthreads();
    if (TRACK && stop) return;
    const T axy = a2x + a2y;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int q = c ? 1 - par : par;
#pragma unroll
        for (int t = 0; t < N2; t++) {
            D[c][t] = axy + zd[2 * t + q];
            Y[c][t] = block_rcp(D[c][t]);
        }
    }
    // my row's other-parity columns: west and east neighbours
    const int nw = ly * HX + h - 1 + e, ne = nw + 1, ns = w - HX, nn = w + HX, op = 1 - par;
    auto half = [&](auto mc, auto qc) {
        constexpr int m = decltype(mc)::value, q = decltype(qc)::value;
        constexpr int c = (m - 1) & 1, o = 1 - c;
        // entries with a plane in [m, EZ-m)
        constexpr int tlo = (m - q + 1) / 2, thi = (EZ - m - q + 1) / 2;
        double d = 0.0;
#pragma unroll
        for (int t0 = tlo; t0 < thi; t0 += G) {
            T gs[G], pw[G], pe[G], ps[G], pn[G];
#define IB3D_STAGE(stmt)                                                                                             \
    _Pragma("unroll") for (int u = 0; u < G; u++) {                                                                  \
        const int t = t0 + u;                                                                                        \
        if (t < thi) { stmt; }                                                                                       \
    }
            constexpr bool z = FIRST && m == 1;
            IB3D_STAGE(pw[u] = z ? T(0) : L[o][t][op][nw]; pe[u] = z ? T(0) : L[o][t][op][ne];
                       ps[u] = z ? T(0) : L[o][t][op][ns]; pn[u] = z ? T(0) : L[o][t][op][nn];)
            IB3D_STAGE(gs[u] = B[c][t] - a1x * pw[u])
            IB3D_STAGE(gs[u] = gs[u] - a3x * pe[u])
            IB3D_STAGE(gs[u] = gs[u] - a1y * ps[u])
            IB3D_STAGE(gs[u] = gs[u] - a3y * pn[u])
            IB3D_STAGE(gs[u] = gs[u] - zt[2 * t + q][0] * (z ? T(0) : (q ? X[o][t] : X[o][t - 1 + q])))
            IB3D_STAGE(gs[u] = gs[u] - zt[2 * t + q][1] * (z ? T(0) : (q ? X[o][t + q] : X[o][t])))
            DivRange range;
            IB3D_STAGE(range.add(gs[u]))
            if (__builtin_expect(__any(range.unsafe()), 0)) {
                IB3D_STAGE(gs[u] = gs[u] / D[c][t])
            } else {
                IB3D_STAGE(gs[u] = block_div(gs[u], D[c][t], Y[c][t]))
            }
            IB3D_STAGE(
                const T pnew = omm * X[c][t] + omega * gs[u];
                const T pset = (live >> (c * N2 + t)) & 1 ? pnew : X[c][t];
                if (TRACK && 2 * t + q >= R && 2 * t + q < EZ - R) d = fmax(d, (double)fabs(pset - X[c][t]));
                X[c][t] = pset;
                if (m < 2 * M) L[c][t][par][w] = X[c][t];)
#undef IB3D_STAGE
        }
        return d;
    };
    double dall[M];
    auto sweep_half = [&](auto mc) {
        constexpr int m = decltype(mc)::value;
        constexpr int c = (m - 1) & 1;
        double d = 0.0;
        if (lx >= m && lx < EX - m && ly >= m && ly < EY - m) {
            if ((c ? 1 - par : par) == 0)
                d = half(mc, std::integral_constant<int, 0>{});
            else
                d = half(mc, std::integral_constant<int, 1>{});
        }
        if (TRACK) dall[(m - 1) / 2] = c ? fmax(dall[(m - 1) / 2], d) : d;
        if (m < 2 * M) __syncthreads();
    };
    sweep_half(std::integral_constant<int, 1>{});
    sweep_half(std::integral_constant<int, 2>{});
    if constexpr (M >= 2) {
        sweep_half(std::integral_constant<int, 3>{});
        sweep_half(std::integral_constant<int, 4>{});
    }
    if (own) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int q = c ? 1 - par : par;
#pragma unroll
            for (int t = R / 2; t < N2 - R / 2; t++) {
                const int kk = k0 + 2 * t + q;
                if (kk <= g.sz - 2) (c ? d1 : d0)[base + (uint32_t)(kk * g.plane)] = X[c][t];
            }
        }
    }
    if (TRACK) {
        // a value at or above thr is recorded as thr: only "not yet" matters
        // there, and it needs no reduction over the wave
#pragma unroll
        for (int q = 0; q < M; q++) {
            const double v = own ? dall[q] : 0.0;
            const double wv = __any(v >= thr) ? thr : wave_max(v);
            if ((tid & 63) == 0) dmax[q][tid >> 6] = wv;
        }
        __syncthreads();
    }
    if (TRACK && tid < M) {
        double v = 0.0;
        for (int q = 0; q < NT / 64; q++) v = fmax(v, dmax[tid][q]);
        if (v > 0.0)
            atomicMax(reinterpret_cast<unsigned long long *>(slot + tid * kBlockSub + (blockIdx.x & (kBlockSub - 1))),
                      (unsigned long long)__double_as_longlong(v));
    }
}
