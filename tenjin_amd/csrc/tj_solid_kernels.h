// Kernels of the elastoplastic path (SOLID = 1): directional 5-wave flux
// passes and the fused update / post-step kernel.
#pragma once
#include "tj_kernels.h"
#include "tj_solid.h"

namespace tj {
inline namespace TJ_VIEW_NS {

template <int NM, typename R>
__device__ __forceinline__ SSt<NM, R> shfl_state(const SSt<NM, R>& S, int src) {
    SSt<NM, R> T;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        T.al[m] = shfl_any(S.al[m], src);
        T.ar[m] = shfl_any(S.ar[m], src);
        T.are[m] = shfl_any(S.are[m], src);
    }
    T.rho = shfl_any(S.rho, src);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        T.u[q] = shfl_any(S.u[q], src);
        T.sig[q] = shfl_any(S.sig[q], src);
    }
    T.E = shfl_any(S.E, src);
    T.p = shfl_any(S.p, src);
    T.a = shfl_any(S.a, src);
#pragma unroll
    for (int q = 0; q < 9; ++q) T.V[q] = shfl_any(S.V[q], src);
    return T;
}

// lane - 1's state (lane 0 keeps its own) by DPP row moves, as lane_dn
template <int NM, typename R>
__device__ __forceinline__ SSt<NM, R> state_dn(const SSt<NM, R>& S) {
    SSt<NM, R> T;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        T.al[m] = lane_dn(S.al[m]);
        T.ar[m] = lane_dn(S.ar[m]);
        T.are[m] = lane_dn(S.are[m]);
    }
    T.rho = lane_dn(S.rho);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        T.u[q] = lane_dn(S.u[q]);
        T.sig[q] = lane_dn(S.sig[q]);
    }
    T.E = lane_dn(S.E);
    T.p = lane_dn(S.p);
    T.a = lane_dn(S.a);
#pragma unroll
    for (int q = 0; q < 9; ++q) T.V[q] = lane_dn(S.V[q]);
    return T;
}

// The left image of a reconstructed state across a reflective face:
// reflect_odd flips the normal velocity and momentum only (boundary.cpp:3-42).
template <int NM, typename R>
__device__ __forceinline__ void flip_s(SSt<NM, R>& S, int d) { S.u[d] = -S.u[d]; }

// The flux planes of direction D hold what the update reads of wave5's flux:
// alpha, alpha rho, rho u, E, the two rows of V other than D (row D's flux is
// V_D u_D - V_D u_D = 0 and its jumps are 0), alpha rho epsilon, S* and row D
// of V*.  20 of 23 components: 72 of the 984 and 1208 bytes a cell that the
// FP64 update stages moved at the device's copy rate.
template <int NM>
struct SFace {
    static constexpr int N = 3 * NM + 14;
    static constexpr int ARE = 2 * NM + 10, SS = 3 * NM + 10, VS = 3 * NM + 11;
    // component of V row r (r != d), column c
    static constexpr int v(int d, int r, int c) { return 2 * NM + 4 + 3 * (r > d ? r - 1 : r) + c; }
};
// put(q, x) for each plane q of direction D, from wave5's flux
template <int NM, int D, typename R, typename Put>
__device__ __forceinline__ void put_face(const R* Fv, Put put) {
    using S = SFace<NM>;
    constexpr int NC = 3 * NM + 13;
#pragma unroll
    for (int q = 0; q < 2 * NM + 4; ++q) put(q, Fv[q]);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (r != D) put(S::v(D, r, c), Fv[2 * NM + 4 + r * 3 + c]);
#pragma unroll
    for (int m = 0; m < NM; ++m) put(S::ARE + m, Fv[2 * NM + 13 + m]);
    put(S::SS, Fv[NC]);
#pragma unroll
    for (int c = 0; c < 3; ++c) put(S::VS + c, Fv[NC + 1 + c]);
}

// Flux passes of the solid path, one reconstruction per cell: a lane
// reconstructs one cell (MUSCL, then p2c + sound speed of both face states)
// and face f takes its left state UR(f-1) from lane - 1, the cell one below
// along D, so a segment of LN lanes gives LN - 1 faces.  The domain's end
// faces take the image of the edge cell's own state.
//
// Bound by VALU issue: 3100 to 3200 instructions a wave in FP64 (two waves per
// SIMD; 144^3: x 417 us, y 437, z 442), 1900 in FP32 (four).  A march of one
// wave along D, with the rows in registers, keeps one wave per SIMD in flight
// and gives a small level few waves: y and z passes of 144^3 in FP64 780 us
// against 490 in these tiles (512^2: 102 against 54), both with an IEEE division
// for every quotient, and of 203 x 160 x 131 in FP32 430 against 285.  Blocks
// run in XCD order: tiles side by side share the cache lines of rows whose pitch
// is no multiple of the line (the same FP32 y pass 395 us in round-robin order).
// The face of a lane: c its lower face along D, PL / PR the reconstructed
// primitives of its cell, LN lanes to a segment (ld the lane within it).
// The right state moves up before the left one is built, so two face states
// are live at a time.
template <int NM, int D, bool RW, typename R>
__device__ __forceinline__ void face_s(const Level& lv, const SPrim<NM, R>& PL, const SPrim<NM, R>& PR, int c, bool face,
                                       R* Fv, unsigned& st) {
    const int nd = lv.n[D];
    SSt<NM, R> Lf;
    {
        SSt<NM, R> SRs;
        p2c_sound_s<NM, RW, R>(lv, PR, D, SRs);
        Lf = state_dn<NM, R>(SRs);
        if (c == 0) {
            Lf = SRs;
            if (lv.bc_lo[D]) flip_s<NM, R>(Lf, D);
        }
    }
    SSt<NM, R> Rf;
    p2c_sound_s<NM, RW, R>(lv, PL, D, Rf);
    if (c == nd && lv.bc_hi[D]) flip_s<NM, R>(Rf, D);
    if (face) wave5<NM, RW, R>(lv, Lf, Rf, D, Fv, st);
}

// x pass: waves of 64 / LN rows by LN lanes along x (144^3 FP64, an IEEE division
// for every quotient: 555 us with segments of 64, 467 with 32; 203 x 160 x 131
// FP32: 340 and 309, and 381 with 16, whose loads fall into four row pieces).
template <int NM, int LN, bool RW, typename R>
__global__ __launch_bounds__(256) void k_flux_x_s(Level lv, MF U, FacesT<R> F, Clock* clk) {
    if (clk->done) return;
    constexpr int PER = LN - 1;
    const int lane = threadIdx.x & 63, ld = lane % LN;
    const long long wave = xcd_block(blockIdx.x, gridDim.x, 2) * (blockDim.x >> 6) + wave_in_block();
    const int nx = lv.n[0], ny = lv.n[1];
    const int nseg = (nx + 1 + PER - 1) / PER;
    const long long rows = (long long)ny * lv.n[2];
    if (wave >= nseg * ((rows + 64 / LN - 1) / (64 / LN))) return;
    const int seg = (int)(wave % nseg);
    const long long row0 = wave / nseg * (64 / LN) + lane / LN;
    const bool act = row0 < rows;
    const long long row = act ? row0 : rows - 1;
    const int j = (int)(row % ny), k = (int)(row / ny);
    const int c = seg * PER - 1 + ld;
    bool fl;
    const int s = bcmap(c, nx, lv.bc_lo[0], lv.bc_hi[0], fl);
    SPrim<NM, R> PL, PR;
    {
        SPrim<NM, R> Pm, Pc, Pp;
        load_sprim<NM, R>(lv, U, s - 1, j, k, Pm);
        load_sprim<NM, R>(lv, U, s, j, k, Pc);
        load_sprim<NM, R>(lv, U, s + 1, j, k, Pp);
        muscl_s<NM, R>(Pm, Pc, Pp, PL, PR);
    }
    unsigned st = 0;
    R Fv[3 * NM + 17];
    const bool face = act && ld >= 1 && c >= 0 && c <= nx;
    face_s<NM, 0, RW, R>(lv, PL, PR, c, face, Fv, st);
    if (face) {
        const long long id = ((long long)k * F.ny + j) * F.nx + c;
        put_face<NM, 0>(Fv, [&](int q, R x) { F.p[q * F.cs + id] = x; });
    }
    if (st) atomicOr(&clk->status, st);
}

// y / z pass: a block of four waves owns 16 columns along x by one segment of
// 16 cells along D.  The primitives of the tile and its two halo rows are
// staged in LDS (rows of 16 cells, coalesced); lanes then run along D, four
// columns to a wave, and the fluxes go back through LDS to rows of 16.  Lanes
// that load and store their own 4 x 16 tile in memory order instead, without
// LDS, take 505 us against 490 (144^3 FP64) and 860 against 285 (FP32), whose
// row pieces are then 32 and 16 bytes.
template <int NM, typename R>
struct STile {
    static constexpr int TC = 16, LN = 16;       // columns, lanes along D
    static constexpr int PER = LN - 1;           // faces per segment
    static constexpr int ROWS = LN + 2;          // rows c0 - 1 .. c0 + LN
    static constexpr int NP = 3 * NM + 13;       // primitives
    static constexpr int NF = SFace<NM>::N;      // flux planes
    static constexpr int FR = PER + 2;           // column pitch of the staged fluxes
    static constexpr int WORDS = NP * TC * ROWS > NF * TC * FR ? NP * TC * ROWS : NF * TC * FR;
};
// The fluxes of faces c0 + 1 .. c0 + 15 along D of columns i0 .. i0 + 15, o the
// other index: left in lds, plane q of column col and face c0 + 1 + f at
// (q * TC + col) * FR + f, with a barrier at the end.
template <int NM, int D, bool RW, typename R>
__device__ __forceinline__ void tile_faces_s(const Level& lv, const MF& U, R* lds, int i0, int c0, int o, unsigned& st) {
    using T = STile<NM, R>;
    constexpr int TC = T::TC, LN = T::LN, ROWS = T::ROWS, FR = T::FR;
    const int nx = lv.n[0], nd = lv.n[D];
    const int tid = threadIdx.x;
    auto P = [&](int q, int col, int t) -> R& { return lds[(q * TC + col) * ROWS + t]; };
    // one cell of the first 16 rows per thread; then the two rows left, their
    // components dealt out over the block, so that all loads are in flight
    // together (a second round of whole cells leaves 7 threads in 8 idle)
    {
        const int col = tid % TC, t = tid / TC, r = c0 - 1 + t;
        SPrim<NM, R> Pq;
        load_sprim<NM, R>(lv, U, i0 + col, D == 1 ? r : o, D == 2 ? r : o, Pq);
        const int hc = tid % TC, ht = LN + (tid / TC & 1), hr = c0 - 1 + ht;
        int hi = i0 + hc, hj = D == 1 ? hr : o, hk = D == 2 ? hr : o;
        bool f[3];
        map3(lv, hi, hj, hk, f);
        constexpr int HN = (T::NP + 7) / 8;
        R hv[HN];
#pragma unroll
        for (int n = 0; n < HN; ++n) {
            const int q = tid / 32 + 8 * n;
            if (q < T::NP) {
                const bool ep = q >= 2 * NM && q < 3 * NM;
                const int u = q - 3 * NM;
                const int comp = q < NM ? lv.cs[ALPHA] + q
                               : q < 2 * NM ? lv.cs[RHO_K] + q - NM
                               : ep ? (lv.plastic ? lv.cs[EPSILON] + q - 2 * NM : 0)
                               : u < 3 ? lv.cs[VELOCITY] + u
                               : u == 3 ? lv.cs[PRESSURE] : lv.cs[V_TENSOR] + u - 4;
                const R v = (R)U.at(comp, hi, hj, hk);
                hv[n] = ep && !lv.plastic ? R(0) : ((u == 0 && f[0]) || (u == 1 && f[1]) || (u == 2 && f[2]) ? -v : v);
            }
        }
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            P(m, col, t) = Pq.a[m];
            P(NM + m, col, t) = Pq.r[m];
            P(2 * NM + m, col, t) = Pq.e[m];
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) P(3 * NM + q, col, t) = Pq.u[q];
        P(3 * NM + 3, col, t) = Pq.p;
#pragma unroll
        for (int q = 0; q < 9; ++q) P(3 * NM + 4 + q, col, t) = Pq.V[q];
#pragma unroll
        for (int n = 0; n < HN; ++n) {
            const int q = tid / 32 + 8 * n;
            if (q < T::NP) P(q, hc, ht) = hv[n];
        }
    }
    __syncthreads();
    const int ld = tid % LN, col = tid / LN;
    const int c = c0 + ld;  // the lane's cell along D
    bool fl;
    const int s = bcmap(c, nd, lv.bc_lo[D], lv.bc_hi[D], fl);
    SPrim<NM, R> PL, PR;
    {
        // row s of the tile (lanes beyond the domain hold no face: clamped)
        const int t = min(max(s - c0 + 1, 1), ROWS - 2);
        auto get = [&](int tt, SPrim<NM, R>& Pq) {
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                Pq.a[m] = P(m, col, tt);
                Pq.r[m] = P(NM + m, col, tt);
                Pq.e[m] = P(2 * NM + m, col, tt);
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) Pq.u[q] = P(3 * NM + q, col, tt);
            Pq.p = P(3 * NM + 3, col, tt);
#pragma unroll
            for (int q = 0; q < 9; ++q) Pq.V[q] = P(3 * NM + 4 + q, col, tt);
        };
        SPrim<NM, R> Pm, Pc, Pp;
        get(t - 1, Pm);
        get(t, Pc);
        get(t + 1, Pp);
        muscl_s<NM, R>(Pm, Pc, Pp, PL, PR);
    }
    R Fv[3 * NM + 17];
    const bool face = i0 + col < nx && ld >= 1 && c >= 0 && c <= nd;
    face_s<NM, D, RW, R>(lv, PL, PR, c, face, Fv, st);
    __syncthreads();  // every wave has read its primitives: the fluxes may overwrite them
    if (face) put_face<NM, D>(Fv, [&](int q, R x) { lds[(q * TC + col) * FR + ld - 1] = x; });
    __syncthreads();
}
template <int NM, int D, bool RW, typename R>
__global__ __launch_bounds__(256) void k_flux_yz_s(Level lv, MF U, FacesT<R> F, Clock* clk) {
    using T = STile<NM, R>;
    constexpr int TC = T::TC, PER = T::PER, NF = T::NF, FR = T::FR;
    __shared__ R lds[T::WORDS];
    if (clk->done) return;  // uniform: the clock does not change during the launch
    const int nx = lv.n[0], nd = lv.n[D];
    const int nxt = (nx + TC - 1) / TC, nseg = (nd + 1 + PER - 1) / PER;
    const long long tile = xcd_block(blockIdx.x, gridDim.x, 2);
    const int xt = (int)(tile % nxt);
    const int rest = (int)(tile / nxt);
    const int seg = rest % nseg, o = rest / nseg;
    const int i0 = xt * TC, c0 = seg * PER - 1;
    const int tid = threadIdx.x;
    unsigned st = 0;
    tile_faces_s<NM, D, RW, R>(lv, U, lds, i0, c0, o, st);
    const int cc = tid % TC, f = tid / TC;  // column, face of the segment
    const int ii = i0 + cc, cf = c0 + 1 + f;
    if (f < PER && ii < nx && cf <= nd) {
        const int fj = D == 1 ? cf : o, fk = D == 2 ? cf : o;
        const long long id = ((long long)fk * F.ny + fj) * F.nx + ii;
#pragma unroll
        for (int q = 0; q < NF; ++q) F.p[q * F.cs + id] = lds[(q * TC + cc) * FR + f];
    }
    if (st) atomicOr(&clk->status, st);
}

// Per-cell solid state held by the update kernel.
template <int NM>
struct SCell {
    double al[NM], ar[NM], rk[NM], e[NM], are[NM], rho, ru[3], u[3], E, p, V[9], hj2;
};

template <bool NT>
__device__ __forceinline__ double ld(const double& src) {
    if constexpr (NT) return get_base(src);
    else return src;
}
// NT: non-temporal loads (get_base), for the update's input and, in stage 2,
// the step's starting state (256^3 plate: the update stages 0.3-0.8 % faster)
template <int NM, bool NT = false>
__device__ __forceinline__ void load_scell(const Level& lv, const MF& U, int i, int j, int k, SCell<NM>& C) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        C.al[m] = ld<NT>(U.at(lv.cs[ALPHA] + m, i, j, k));
        C.ar[m] = ld<NT>(U.at(lv.cs[ALPHARHO] + m, i, j, k));
        C.rk[m] = ld<NT>(U.at(lv.cs[RHO_K] + m, i, j, k));
        C.e[m] = lv.plastic ? ld<NT>(U.at(lv.cs[EPSILON] + m, i, j, k)) : 0.0;
        C.are[m] = lv.plastic ? ld<NT>(U.at(lv.cs[ALPHARHOEPSILON] + m, i, j, k)) : 0.0;
    }
    C.rho = ld<NT>(U.at(lv.cs[RHO], i, j, k));
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        C.ru[q] = ld<NT>(U.at(lv.cs[RHOU] + q, i, j, k));
        C.u[q] = ld<NT>(U.at(lv.cs[VELOCITY] + q, i, j, k));
    }
    C.E = ld<NT>(U.at(lv.cs[TOTAL_E], i, j, k));
    C.p = ld<NT>(U.at(lv.cs[PRESSURE], i, j, k));
#pragma unroll
    for (int q = 0; q < 9; ++q) C.V[q] = ld<NT>(U.at(lv.cs[V_TENSOR] + q, i, j, k));
    C.hj2 = ld<NT>(U.at(lv.cs[HJ2], i, j, k));
}
// NT: non-temporal stores (put_state), for the end-of-step state
template <int NM, bool NT = false>
__device__ __forceinline__ void store_scell(const Level& lv, const MF& U, int i, int j, int k, const SCell<NM>& C) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        put_state<NT>(U.at(lv.cs[ALPHA] + m, i, j, k), C.al[m]);
        put_state<NT>(U.at(lv.cs[ALPHARHO] + m, i, j, k), C.ar[m]);
        put_state<NT>(U.at(lv.cs[RHO_K] + m, i, j, k), C.rk[m]);
        if (lv.plastic) {
            put_state<NT>(U.at(lv.cs[EPSILON] + m, i, j, k), C.e[m]);
            put_state<NT>(U.at(lv.cs[ALPHARHOEPSILON] + m, i, j, k), C.are[m]);
        }
    }
    put_state<NT>(U.at(lv.cs[RHO], i, j, k), C.rho);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        put_state<NT>(U.at(lv.cs[RHOU] + q, i, j, k), C.ru[q]);
        put_state<NT>(U.at(lv.cs[VELOCITY] + q, i, j, k), C.u[q]);
    }
    put_state<NT>(U.at(lv.cs[TOTAL_E], i, j, k), C.E);
    put_state<NT>(U.at(lv.cs[PRESSURE], i, j, k), C.p);
#pragma unroll
    for (int q = 0; q < 9; ++q) put_state<NT>(U.at(lv.cs[V_TENSOR] + q, i, j, k), C.V[q]);
    put_state<NT>(U.at(lv.cs[HJ2], i, j, k), C.hj2);
}

// geometricSourceTerm (radial.cpp:5-31, flux.cpp:51-77) of a solid cell
// whose stored stress is that of its own state, as it is after the
// conservativeToPrimitive that ends plasticUpdate: sigma from p and the
// deviatoric Hencky strain dH (stressTensor, boxaccesscellarray.cpp:176-203).
// V rows 0 and 1 take +1/3 V u_x, row 2 -2/3 V u_x.
template <int NM, bool RW>
__device__ __forceinline__ void radial_solid(const Level& lv, double f, SCell<NM>& C, const double* dH) {
    double s0[3], s1[3], s2[3];
    stress_col<NM, RW>(lv, C.al, C.rk, C.p, dH, 0, s0);
    stress_col<NM, RW>(lv, C.al, C.rk, C.p, dH, 1, s1);
    stress_col<NM, RW>(lv, C.al, C.rk, C.p, dH, 2, s2);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        C.ar[m] += f * (C.ar[m] * C.u[0]);
        // a select, not a conditional store: the latter put C.are in scratch
        C.are[m] = lv.plastic ? C.are[m] + f * (C.are[m] * C.u[0]) : C.are[m];
    }
    radial_momentum_energy(f, C.u, s0, s1[0], s2[0], s2[2], C.ru, C.E);
#pragma unroll
    for (int q = 0; q < 6; ++q) C.V[q] += f * ((1.0 / 3.0) * C.V[q] * C.u[0]);
#pragma unroll
    for (int q = 6; q < 9; ++q) C.V[q] += f * (-(2.0 / 3.0) * C.V[q] * C.u[0]);
}
// plasticUpdate's conservativeToPrimitive leaves p and dH of the state; a
// stand-alone source recomputes dH from V (hencky does what getHenckyJ2 does).
template <int NM, bool RW>
__device__ __forceinline__ void radial_solid_c2p(const Level& lv, double f, SCell<NM>& C, double* dH, bool have_dH) {
    if (!have_dH) hencky(C.V, dH);
    radial_solid<NM, RW>(lv, f, C, dH);
    C.hj2 = c2p_s<NM, RW>(lv, C.al, C.ar, C.are, C.ru, C.E, C.V, C.rk, C.e, C.rho, C.u, C.p, dH);
}

// update_cell_s: update (hllc.cpp:493-523, with the V rows of :511-514) in x, y, z order,
// then conservativeToPrimitive.  Stage 2 adds the RK average (hllc.cpp:705),
// plasticUpdate (main.cpp:154-157, plastic.cpp:227-244), the geometric source
// (main.cpp:159-162), cleanUpV (main.cpp:164-167), cleanUpAlpha
// (main.cpp:169-171), the NaN scan and the next getTimeStep.
// fa(d, q, hi): plane q of the cell's low (0) or high (1) face along d < ND.
template <int NM, int STAGE, bool RW, typename T, int ND = 3, typename Face>
__device__ __forceinline__ void update_cell_s(const Level& lv, const MF& Uin, const MF& Ub, const MF& Uo, int i, int j,
                                              int k, double dt, unsigned ops, Face fa, double& cand, unsigned& st) {
    using S = SFace<NM>;
    SCell<NM> C;
    load_scell<NM, true>(lv, Uin, i, j, k, C);
    double a0[NM], V0[9], u0[3];
#pragma unroll
    for (int m = 0; m < NM; ++m) a0[m] = C.al[m];
#pragma unroll
    for (int q = 0; q < 9; ++q) V0[q] = C.V[q];
#pragma unroll
    for (int q = 0; q < 3; ++q) u0[q] = C.u[q];
    // unrolled over the directions (a loop to lv.dim kept C.are in scratch
    // memory: the plastic-only update made its index dynamic)
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        if (d >= lv.dim) break;
        const double dtdx = dt / lv.dx[d];
        const double s0 = (double)fa(d, S::SS, 0), s1 = (double)fa(d, S::SS, 1);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            C.al[m] += dtdx * ((double)fa(d, m, 0) - (double)fa(d, m, 1) - a0[m] * (s0 - s1));
            C.ar[m] += dtdx * ((double)fa(d, NM + m, 0) - (double)fa(d, NM + m, 1));
            if (lv.plastic) {
                const double fl = (double)fa(d, S::ARE + m, 0), fh = (double)fa(d, S::ARE + m, 1);
                C.are[m] += dtdx * (fl - fh);
            }
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) C.ru[q] += dtdx * ((double)fa(d, 2 * NM + q, 0) - (double)fa(d, 2 * NM + q, 1));
        C.E += dtdx * ((double)fa(d, 2 * NM + 3, 0) - (double)fa(d, 2 * NM + 3, 1));
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double vs0 = (double)fa(d, S::VS + c, 0), vs1 = (double)fa(d, S::VS + c, 1);
                const double jump = r == d ? 0.0 : (double)fa(d, S::v(d, r, c), 0) - (double)fa(d, S::v(d, r, c), 1);
                C.V[r * 3 + c] += dtdx * (jump - (2.0 / 3.0) * V0[r * 3 + c] * (s0 - s1) + u0[r] * (vs0 - vs1));
            }
    }
    double dH[9];
    // Stage 2 with the plastic relaxation: the conservativeToPrimitive that
    // ends it rewrites rho, u, p, HJ2 and dH, so this one forms only what
    // the relaxation reads (rho_k and epsilon, as c2p_s does).  The values
    // are those of the full sequence.
    const bool relax = STAGE == 2 && (ops & 1u) != 0;
    SCell<NM> B;
    if (STAGE == 2) load_scell<NM, true>(lv, Ub, i, j, k, B);  // in flight across the branch
    if (relax) {  // nor are these averages read (156 VGPRs, three waves per SIMD; 171 with them)
        B.rho = B.p = B.hj2 = 0.0;
#pragma unroll
        for (int q = 0; q < 3; ++q) B.u[q] = 0.0;
    }
    if (relax) {
        c2p_rk_e<NM>(lv, C.al, C.ar, C.are, C.rk, C.e);
        C.rho = C.p = C.hj2 = 0.0;  // rewritten after the relaxation (no loads of Uin's values)
    } else C.hj2 = c2p_s<NM, RW>(lv, C.al, C.ar, C.are, C.ru, C.E, C.V, C.rk, C.e, C.rho, C.u, C.p, dH);
    if (STAGE == 2) {
        // U1 = (U * 1/2) + (U2 * 1/2) over every component
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            C.al[m] = B.al[m] * (1.0 / 2.0) + C.al[m] * (1.0 / 2.0);
            C.ar[m] = B.ar[m] * (1.0 / 2.0) + C.ar[m] * (1.0 / 2.0);
            C.rk[m] = B.rk[m] * (1.0 / 2.0) + C.rk[m] * (1.0 / 2.0);
            C.e[m] = B.e[m] * (1.0 / 2.0) + C.e[m] * (1.0 / 2.0);
            C.are[m] = B.are[m] * (1.0 / 2.0) + C.are[m] * (1.0 / 2.0);
        }
        C.rho = B.rho * (1.0 / 2.0) + C.rho * (1.0 / 2.0);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            C.ru[q] = B.ru[q] * (1.0 / 2.0) + C.ru[q] * (1.0 / 2.0);
            C.u[q] = B.u[q] * (1.0 / 2.0) + C.u[q] * (1.0 / 2.0);
        }
        C.E = B.E * (1.0 / 2.0) + C.E * (1.0 / 2.0);
        C.p = B.p * (1.0 / 2.0) + C.p * (1.0 / 2.0);
#pragma unroll
        for (int q = 0; q < 9; ++q) C.V[q] = B.V[q] * (1.0 / 2.0) + C.V[q] * (1.0 / 2.0);
        C.hj2 = B.hj2 * (1.0 / 2.0) + C.hj2 * (1.0 / 2.0);
        if (relax) {  // plastic relaxation, then conservativeToPrimitive
            st |= plastic_cell<NM, RW>(lv, C.al, C.ar, C.rk, C.e, C.are, C.V);
            C.hj2 = c2p_s<NM, RW>(lv, C.al, C.ar, C.are, C.ru, C.E, C.V, C.rk, C.e, C.rho, C.u, C.p, dH);
        }
        if (ops & 32u) radial_solid_c2p<NM, RW>(lv, radial_factor(lv, i, dt), C, dH, (ops & 1u) != 0);
        if (ops & 2u) cleanup_v<NM, T>(lv, C.al, C.V);  // FP32 in the mixed form
        if (ops & 4u) st |= cleanup_alpha<NM>(C.al);
        if (ops & 16u) {
            bool bad = false;
#pragma unroll
            for (int m = 0; m < NM; ++m)
                bad |= __builtin_isnan(C.al[m]) || __builtin_isnan(C.ar[m]) || __builtin_isnan(C.rk[m]) ||
                       (lv.plastic && (__builtin_isnan(C.e[m]) || __builtin_isnan(C.are[m])));
#pragma unroll
            for (int q = 0; q < 3; ++q) bad |= __builtin_isnan(C.ru[q]) || __builtin_isnan(C.u[q]);
#pragma unroll
            for (int q = 0; q < 9; ++q) bad |= __builtin_isnan(C.V[q]);
            bad |= __builtin_isnan(C.E) || __builtin_isnan(C.p);
            if (bad) st |= 1u;
        }
        if (ops & 8u) {
            const double a = sound_s<NM, RW>(lv, C.al, C.ar, C.rk, C.rho, C.p, C.hj2);
            put_state<STAGE == 2>(Uo.at(lv.cs[SOUNDSPEED], i, j, k), a);
            #pragma unroll
            for (int d = 0; d < 3; ++d)  // unrolled: constant indices keep the state in registers
                if (d < lv.dim) cand = dmin(cand, qdiv(lv.dx[d], a + __builtin_fabs(C.u[d])));
        }
    }
    store_scell<NM, STAGE == 2>(lv, Uo, i, j, k, C);
}

// Bound by HBM: with 20 flux planes a direction in place of 23, stage 1 of
// 144^3 FP64 takes 543 us (23 planes: 605), stage 2 700 (760).
template <int NM, int STAGE, bool RW, typename T>
__global__ __launch_bounds__(256) void k_update_s(Level lv, MF Uin, MF Ub, MF Uo, FacesT<T> F0, FacesT<T> F1, FacesT<T> F2,
                                                  Clock* clk, unsigned ops) {
    if (clk->done) return;
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = xcd_block(blockIdx.x, gridDim.x, lv.dim) * blockDim.x + threadIdx.x;
    const long long ncell = (long long)nx * ny * nz;
    double cand = __builtin_huge_val();
    unsigned st = 0;
    if (id < ncell) {
        const int i = (int)(id % nx);
        const int j = (int)((id / nx) % ny);
        const int k = (int)(id / ((long long)nx * ny));
        update_cell_s<NM, STAGE, RW, T>(lv, Uin, Ub, Uo, i, j, k, clk->dt, ops, [&](int d, int q, int hi) {
            const FacesT<T>& F = d == 0 ? F0 : (d == 1 ? F1 : F2);
            return F.at(q, i + (d == 0 && hi), j + (d == 1 && hi), k + (d == 2 && hi));
        }, cand, st);
    }
    if (STAGE == 2 && (ops & 8u)) {
        block_min_to(cand, dt_slot(lv, clk));
    }
    if (st) atomicOr(&clk->status, st);
}

// The y flux pass and the update of stage 1 in one launch: the tile's y faces
// stay in LDS and the update takes the other directions' faces from their
// planes.  A tile gives 15 faces and completes the 14 cells between them, lanes
// along x again.  The update alone is bound by HBM and the pass by VALU issue:
// 144^3 FP64 433 + 543 us as two launches, 839 as one; 512^2 49 + 30 and 69.
// Stage 2 stays apart: its update has as much arithmetic as a pass and takes
// three waves per SIMD alone, two here (144^3 FP64 1363 against 1135 us, FP32
// fluxes on 203 x 160 x 131 1640 against 1010).  With the z pass in the place
// of y, whose tile rows lie whole planes apart, stage 1 takes 800 and 890 us
// against 781 and 826.  DIM: the level's dimensions.  For levels without
// Romenskii or Wilkins materials (use_stage1_solid).
template <int NM, int DIM, typename R>
__global__ __launch_bounds__(256) void k_stage1_s(Level lv, MF U, MF Uo, FacesT<R> F0, FacesT<R> F2, Clock* clk) {
    using T = STile<NM, R>;
    constexpr int TC = T::TC, FR = T::FR, PER = T::PER - 1;
    __shared__ R lds[T::WORDS];
    if (clk->done) return;  // uniform: the clock does not change during the launch
    const int nx = lv.n[0], ny = lv.n[1];
    const int nxt = (nx + TC - 1) / TC, nseg = (ny + PER - 1) / PER;
    const long long tile = xcd_block(blockIdx.x, gridDim.x, 2);
    const int xt = (int)(tile % nxt);
    const int rest = (int)(tile / nxt);
    const int seg = rest % nseg, k = rest / nseg;
    const int i0 = xt * TC, c0 = seg * PER - 1;
    const int tid = threadIdx.x;
    double cand = __builtin_huge_val();
    unsigned st = 0;
    tile_faces_s<NM, 1, false, R>(lv, U, lds, i0, c0, k, st);
    const int cc = tid % TC, f = tid / TC;
    const int i = i0 + cc, j = c0 + 1 + f;
    if (f < PER && i < nx && j < ny) {
        update_cell_s<NM, 1, false, R, DIM>(lv, U, U, Uo, i, j, k, clk->dt, 0u, [&](int d, int q, int hi) {
            if (d == 1) return lds[(q * TC + cc) * FR + f + hi];
            return d == 0 ? F0.at(q, i + hi, j, k) : F2.at(q, i, j, k + hi);
        }, cand, st);
    }
    if (st) atomicOr(&clk->status, st);
}

template <int NM, bool RW>
__global__ __launch_bounds__(256) void k_sound_dt_s(Level lv, MF U, Clock* clk) {
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long ncell = (long long)nx * ny * nz;
    double cand = __builtin_huge_val();
    if (id < ncell) {
        const int i = (int)(id % nx);
        const int j = (int)((id / nx) % ny);
        const int k = (int)(id / ((long long)nx * ny));
        SCell<NM> C;
        load_scell<NM>(lv, U, i, j, k, C);
        const double a = sound_s<NM, RW>(lv, C.al, C.ar, C.rk, C.rho, C.p, C.hj2);
        U.at(lv.cs[SOUNDSPEED], i, j, k) = a;
        #pragma unroll
        for (int d = 0; d < 3; ++d)  // unrolled: constant indices keep the state in registers
            if (d < lv.dim) cand = dmin(cand, qdiv(lv.dx[d], a + __builtin_fabs(C.u[d])));
    }
    block_min_to(cand, dt_slot(lv, clk));
}

// setInitialConditions for solid levels: thermal -> total pressure shift
// (initialise.cpp:104, with the HJ2 component as given) then
// primitiveToConservative (which computes HJ2 and devH).
template <int NM, bool RW>
__global__ __launch_bounds__(256) void k_init_p2c_s(Level lv, MF U, int shift) {
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (long long)nx * ny * nz) return;
    const int i = (int)(id % nx);
    const int j = (int)((id / nx) % ny);
    const int k = (int)(id / ((long long)nx * ny));
    SPrim<NM> P;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        P.a[m] = U.at(lv.cs[ALPHA] + m, i, j, k);
        P.r[m] = U.at(lv.cs[RHO_K] + m, i, j, k);
        P.e[m] = lv.plastic ? U.at(lv.cs[EPSILON] + m, i, j, k) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) P.u[q] = U.at(lv.cs[VELOCITY] + q, i, j, k);
    P.p = U.at(lv.cs[PRESSURE], i, j, k);
#pragma unroll
    for (int q = 0; q < 9; ++q) P.V[q] = U.at(lv.cs[V_TENSOR] + q, i, j, k);
    if (shift) {
        double ar[NM], G, Ent, Pnt;
#pragma unroll
        for (int m = 0; m < NM; ++m) ar[m] = P.a[m] * P.r[m];
        eos_sums_s<NM, RW>(lv, P.a, ar, P.r, U.at(lv.cs[HJ2], i, j, k), G, Ent, Pnt);
        P.p += Pnt / G;
        U.at(lv.cs[PRESSURE], i, j, k) = P.p;
    }
    SSt<NM> S;
    p2c_sound_s<NM, RW>(lv, P, 0, S);
    double dH[9];
    const double hj2 = hencky(P.V, dH);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        U.at(lv.cs[ALPHARHO] + m, i, j, k) = S.ar[m];
        if (lv.plastic) U.at(lv.cs[ALPHARHOEPSILON] + m, i, j, k) = S.are[m];
    }
    U.at(lv.cs[RHO], i, j, k) = S.rho;
#pragma unroll
    for (int q = 0; q < 3; ++q) U.at(lv.cs[RHOU] + q, i, j, k) = S.u[q] * S.rho;
    U.at(lv.cs[TOTAL_E], i, j, k) = S.E;
    U.at(lv.cs[HJ2], i, j, k) = hj2;
#pragma unroll
    for (int q = 0; q < 9; ++q) U.at(lv.cs[DEVH] + q, i, j, k) = dH[q];
}

// derived components of a solid state: devH, HJ2 from V and sigma
// (boxaccesscellarray.cpp:176-216, 326-380)
template <int NM, bool RW>
__global__ __launch_bounds__(256) void k_derive_s(Level lv, MF U) {
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (long long)nx * ny * nz) return;
    const int i = (int)(id % nx);
    const int j = (int)((id / nx) % ny);
    const int k = (int)(id / ((long long)nx * ny));
    double V[9], dH[9], al[NM], rk[NM];
#pragma unroll
    for (int q = 0; q < 9; ++q) V[q] = U.at(lv.cs[V_TENSOR] + q, i, j, k);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        al[m] = U.at(lv.cs[ALPHA] + m, i, j, k);
        rk[m] = U.at(lv.cs[RHO_K] + m, i, j, k);
    }
    const double hj2 = hencky(V, dH);
    const double p = U.at(lv.cs[PRESSURE], i, j, k);
    U.at(lv.cs[HJ2], i, j, k) = hj2;
#pragma unroll
    for (int q = 0; q < 9; ++q) U.at(lv.cs[DEVH] + q, i, j, k) = dH[q];
    for (int d = 0; d < 3; ++d) {
        double sig[3];
        stress_col<NM, RW>(lv, al, rk, p, dH, d, sig);
        for (int r = 0; r < 3; ++r) U.at(lv.cs[SIGMA] + 3 * r + d, i, j, k) = sig[r];
    }
}

}  // inline namespace TJ_VIEW_NS
}  // namespace tj

namespace tj {
inline namespace TJ_VIEW_NS {

// conservativeToPrimitive over the valid cells of a solid level.
template <int NM, bool RW>
__global__ __launch_bounds__(256) void k_c2p_s(Level lv, MF U) {
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (long long)nx * ny * nz) return;
    const int i = (int)(id % nx);
    const int j = (int)((id / nx) % ny);
    const int k = (int)(id / ((long long)nx * ny));
    SCell<NM> C;
    load_scell<NM>(lv, U, i, j, k, C);
    double dH[9];
    C.hj2 = c2p_s<NM, RW>(lv, C.al, C.ar, C.are, C.ru, C.E, C.V, C.rk, C.e, C.rho, C.u, C.p, dH);
    store_scell<NM>(lv, U, i, j, k, C);
}

// The post-step chain of main.cpp:154-171 on a state, stand-alone
// (tj_post_step): plastic + c2p, the geometric source + c2p (with the clock's
// dt), cleanUpV, cleanUpAlpha, NaN scan, sound speed and the CFL minimum, each
// when its bit is set.
template <int NM, bool RW>
__global__ __launch_bounds__(256) void k_post_s(Level lv, MF U, Clock* clk, unsigned ops) {
    const int nx = lv.n[0], ny = lv.n[1], nz = lv.n[2];
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long ncell = (long long)nx * ny * nz;
    double cand = __builtin_huge_val();
    unsigned st = 0;
    if (id < ncell) {
        const int i = (int)(id % nx);
        const int j = (int)((id / nx) % ny);
        const int k = (int)(id / ((long long)nx * ny));
        SCell<NM> C;
        load_scell<NM>(lv, U, i, j, k, C);
        double dH[9];
        if (ops & 1u) {
            st |= plastic_cell<NM, RW>(lv, C.al, C.ar, C.rk, C.e, C.are, C.V);
            C.hj2 = c2p_s<NM, RW>(lv, C.al, C.ar, C.are, C.ru, C.E, C.V, C.rk, C.e, C.rho, C.u, C.p, dH);
        }
        if (ops & 32u) radial_solid_c2p<NM, RW>(lv, radial_factor(lv, i, clk->dt), C, dH, (ops & 1u) != 0);
        if (ops & 2u) cleanup_v<NM>(lv, C.al, C.V);
        if (ops & 4u) st |= cleanup_alpha<NM>(C.al);
        if (ops & 16u) {
            bool bad = false;
#pragma unroll
            for (int m = 0; m < NM; ++m)
                bad |= __builtin_isnan(C.al[m]) || __builtin_isnan(C.ar[m]) || __builtin_isnan(C.rk[m]) ||
                       (lv.plastic && (__builtin_isnan(C.e[m]) || __builtin_isnan(C.are[m])));
#pragma unroll
            for (int q = 0; q < 3; ++q) bad |= __builtin_isnan(C.ru[q]) || __builtin_isnan(C.u[q]);
#pragma unroll
            for (int q = 0; q < 9; ++q) bad |= __builtin_isnan(C.V[q]);
            bad |= __builtin_isnan(C.E) || __builtin_isnan(C.p);
            if (bad) st |= 1u;
        }
        if (ops & 8u) {
            const double a = sound_s<NM, RW>(lv, C.al, C.ar, C.rk, C.rho, C.p, C.hj2);
            U.at(lv.cs[SOUNDSPEED], i, j, k) = a;
            #pragma unroll
            for (int d = 0; d < 3; ++d)  // unrolled: constant indices keep the state in registers
                if (d < lv.dim) cand = dmin(cand, qdiv(lv.dx[d], a + __builtin_fabs(C.u[d])));
        }
        store_scell<NM>(lv, U, i, j, k, C);
    }
    if (ops & 8u) {
        block_min_to(cand, dt_slot(lv, clk));
    }
    if (st) atomicOr(&clk->status, st);
}

}  // inline namespace TJ_VIEW_NS
}  // namespace tj
