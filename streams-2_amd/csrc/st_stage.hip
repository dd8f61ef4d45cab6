// st_stage.hip -- the one-pass stage: the kernels st_rk_sync / st_advance run
// for the KEEP split (nkeep = 0) of a calorically perfect gas with the Roe
// WENO split, three ghost layers and a periodic span (one_pass_stage below);
// every other solve runs the separate sweeps of st_kernels.hip.
//
// One stage is
//   flux     x, y and z central fluxes and the viscous terms of every cell in
//            one march along z, the bulk sums of force_rhs, the CFL radii where
//            the step recomputes dt, and at the third stage the Ducros sensor
//   items    WENO faces of the flagged cells; the last workgroup finishes the
//            bulk sums (dpdx) and, at the first stage, the CFL step
//   update   grad(div/3) terms, w += fln with the forcing, wall ghosts, and
//            the viscosity of the new state
// and at the first stage of a step two kernels turn the sensor into bit masks
// and into the list of WENO work items, which the three stages share (the
// reference switches on the sensor of the previous step's last stage).  All of
// them form the primitives from w; of w_aux they read the viscosity (its power
// law is the one costly primitive, and whoever changes w stores it), the sensor
// and div/3.  The aux pass (w -> w_aux(1:7) over the ghosted box,
// st_kernels.hip) runs at the last stage of a call alone, whose w_aux the
// caller can read, and at the first, for the viscosity of a w that anyone may
// have set.
#include "st_device.h"
#include "st_flux.h"
#include "st_items.h"
#include "st_solver.h"

namespace st {

// ============================================================ sensor masks
// Bit masks of the switch: the sensor of the ghosted box as one bit per point
// (k_hot_bits), then per interior cell and direction whether its lower and
// its upper face are WENO faces.  A face i of direction d takes the WENO flux
// when a point i-ws+1 .. i+ws along d is above the threshold (the switch
// window of the reference kernels, kernels_cpu.F90:466-470).
//
// Layouts: hot bits, ceil(rx/64) words per ghosted row, bit e of a row the
// point i = e + 1 - ng.  Cell records and list segments: st_items.h.
constexpr int kItemBlocks = 512;     // workgroups of the item kernel at most (two per CU)

__host__ __device__ __forceinline__ int hot_words(const Geo &g) { return (g.rx + 63) / 64; }

// the cells with a WENO face, 32 cells of a row per entry, one word a direction
__host__ __device__ __forceinline__ int dirty_per_row(const Geo &g) { return (g.nx + 31) / 32; }

size_t hot_dirty_bytes(const Geo &g) { return sizeof(uint3) * (size_t)dirty_per_row(g) * g.ny * g.nz; }
size_t hot_bits_bytes(const Geo &g) { return sizeof(uint64_t) * (size_t)hot_words(g) * g.sy * g.sz; }
size_t hot_rec_bytes(const Geo &g) { return sizeof(uint64_t) * kRecWords * (size_t)rec_per_row(g) * g.ny * g.nz; }

// One wave per word, bound by the read of the sensor (8 B a point).
template <typename R>
__device__ __forceinline__ void k_hot_bits_body(const dim3 blockIdx, const dim3 gridDim, Geo g, KPar P,
                                                const R *__restrict__ wa, uint64_t *__restrict__ hot) {
    const int lane = threadIdx.x & 63;
    const int nwg = hot_words(g);
    const int tot = nwg * g.sy * g.sz;
    const R thr = R(P.sensor_threshold);
    const R *S = wa + 7 * (size_t)g.nvol;
    // four consecutive words a wave: their loads are in flight together
    const int w0 = 4 * (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    R v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int wd = w0 + q;
        const int row = wd / nwg, e = 64 * (wd - row * nwg) + lane;
        v[q] = wd < tot && e < g.rx ? S[(size_t)row * g.sx + e] : thr;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const unsigned long long m = __ballot(v[q] > thr);
        if (lane == 0 && w0 + q < tot) hot[w0 + q] = m;
    }
}
template <typename R>
__global__ __launch_bounds__(256) void k_hot_bits(Geo g, KPar P, const R *__restrict__ wa,
                                                  uint64_t *__restrict__ hot) {
    k_hot_bits_body<R>(dim3(blockIdx.x, blockIdx.y, blockIdx.z), dim3(gridDim.x, gridDim.y, gridDim.z), g, P, wa, hot);
}

// Record of 64 cells per thread (all directions by word operations), then the
// work items of the block's segment of `256 * wpt` records, in cell order, x
// before y before z of one cell.  An item is one flagged cell and direction:
//   bits 0-23 cell, relative to the segment's first cell; 24-25 direction;
//   26 lower face WENO; 27 upper face WENO.
// The list of a segment starts at its first cell's index, so it has room for
// one item per cell; a segment with more writes none and reports -3 * cells:
// its items are then all (cell, direction) pairs, read from the records.
__device__ __forceinline__ void k_hot_items_body(const dim3 blockIdx, const dim3 gridDim, Geo g, KPar P,
                                                 const uint64_t *__restrict__ hot, uint64_t *__restrict__ rec,
                                                 uint3 *__restrict__ dirty, int wpt, int *__restrict__ list, int *__restrict__ counts) {
    __shared__ int wsum[4];
    const int nwx = rec_per_row(g), nwg = hot_words(g);
    const int nwords = nwx * g.ny * g.nz;
    const int segw = 256 * wpt;
    const int W0 = blockIdx.x * segw;
    const int S0 = seg_first_cell(g, nwx, W0, nwords), S1 = seg_first_cell(g, nwx, W0 + segw, nwords);
    const int ws = P.weno_scheme;
    const int wa0 = W0 + (int)threadIdx.x * wpt, wa1 = min(wa0 + wpt, nwords);
    int c = 0;
    for (int wd = wa0; wd < wa1; wd++) {
        const int q = wd % nwx, r = wd / nwx;
        const int j = r % g.ny + 1, k = r / g.ny + 1;
        // bits of the points 64q+1-3+s .. of ghosted row (j, k)
        auto row = [&](int jj, int kk, int s) {
            const size_t b = ((size_t)(kk + g.ng - 1) * g.sy + (jj + g.ng - 1)) * nwg + q;
            const uint64_t lo = hot[b], hi = q + 1 < nwg ? hot[b + 1] : 0ull;
            return s == 0 ? lo : (lo >> s) | (hi << (64 - s));
        };
        const int nc = g.nx - 64 * q;
        const uint64_t in = nc >= 64 ? ~0ull : (1ull << nc) - 1ull;
        uint64_t lh[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int o = -3; o <= 3; o++) {
            const bool lower = o >= -ws && o <= ws - 1, upper = o >= -ws + 1 && o <= ws;
            if (!lower && !upper) continue;
            const uint64_t x = row(j, k, 3 + o), y = row(j + o, k, 3), z = row(j, k + o, 3);
            if (lower) { lh[0] |= x; lh[2] |= y; lh[4] |= z; }
            if (upper) { lh[1] |= x; lh[3] |= y; lh[5] |= z; }
        }
        // cells outside the Euler range of a direction get no flux there
        uint64_t rx = in;
        for (int d = 0; d < 2; d++) {
            const int f = d == 0 ? P.eul_lo[0] - 1 - 64 * q : P.eul_hi[0] - 64 * q;  // cells below / up to f
            const uint64_t below = f <= 0 ? 0ull : (f >= 64 ? ~0ull : (1ull << f) - 1ull);
            rx &= d == 0 ? ~below : below;
        }
        const uint64_t msk[3] = {rx, j >= P.eul_lo[1] && j <= P.eul_hi[1] ? in : 0ull,
                                 k >= P.eul_lo[2] && k <= P.eul_hi[2] ? in : 0ull};
        uint64_t *o = rec + (size_t)kRecWords * wd;
        uint64_t dd[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const uint64_t a = lh[2 * d] & msk[d], b = lh[2 * d + 1] & msk[d];
            o[2 * d] = a;
            o[2 * d + 1] = b;
            dd[d] = a | b;
            c += __popcll(dd[d]);
        }
        uint3 *dr = dirty + (size_t)r * dirty_per_row(g) + 2 * q;
        dr[0] = make_uint3((unsigned)dd[0], (unsigned)dd[1], (unsigned)dd[2]);
        if (nc > 32) dr[1] = make_uint3((unsigned)(dd[0] >> 32), (unsigned)(dd[1] >> 32), (unsigned)(dd[2] >> 32));
    }
    int total;
    int off = block_excl_scan256(c, wsum, &total);
    const int report = segment_report(total, S1 - S0);
    if (threadIdx.x == 0) counts[blockIdx.x] = report;
    if (c == 0 || report < 0) return;
    int *seg = list + S0;
    for (int wd = wa0; wd < wa1; wd++) {
        const uint64_t *o = rec + (size_t)kRecWords * wd;
        uint64_t lh[6], any = 0;
#pragma unroll
        for (int d = 0; d < 6; d++) {
            lh[d] = o[d];
            any |= lh[d];
        }
        const int cell0 = seg_first_cell(g, nwx, wd, nwords) - S0;
        while (any) {
            const int b = __ffsll((unsigned long long)any) - 1;
            any &= any - 1ull;
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int lo = (int)(lh[2 * d] >> b) & 1, hi = (int)(lh[2 * d + 1] >> b) & 1;
                if (lo | hi) seg[off++] = (cell0 + b) | d << 24 | lo << 26 | hi << 27;
            }
        }
    }
}
__global__ __launch_bounds__(256) void k_hot_items(Geo g, KPar P, const uint64_t *__restrict__ hot,
                                                   uint64_t *__restrict__ rec, uint3 *__restrict__ dirty, int wpt, int *__restrict__ list,
                                                   int *__restrict__ counts) {
    k_hot_items_body(dim3(blockIdx.x, blockIdx.y, blockIdx.z), dim3(gridDim.x, gridDim.y, gridDim.z), g, P, hot, rec, dirty, wpt, list, counts);
}

// ============================================================ one-pass fluxes
// A value the optimizer cannot see through: address arithmetic of the rare
// branches (edges, ghost images) built on it stays inside them instead of
// being hoisted out of the march, where it would hold registers.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A value that is the same in every lane, held in scalar registers: what FP64
// arithmetic makes of kernel arguments would otherwise fill vector ones.
__device__ __forceinline__ double uniform(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
__device__ __forceinline__ float uniform(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }

// A point's stencil values: rho, u, v, w, T, mu, and in the mixed form the
// stored deviation p - p_ref (in FP64 the pressure is rho*T*R).
constexpr int VR = 0, VU = 1, VT = 4, VM = 5, VP_ = 6;
template <typename R>
constexpr int kNP = sizeof(R) == sizeof(double) ? 6 : 7;
template <typename R>
struct SP {
    R a[kNP<R>];
};
// p/R in FP64, p - p_ref in the mixed form
template <typename R>
__device__ __forceinline__ R sp_press(const SP<R> &p) {
    if constexpr (sizeof(R) == sizeof(double)) return p.a[VR] * p.a[VT];
    else return p.a[VP_];
}

// What the three directions add up for one cell.  Every term of the right-hand
// side has the form f_k = (u_k m + mk[k]) / 4 for the momenta (the pressure
// and mu Laplacian terms ride in mk) and the energy takes u_k mk[k] / 4 of the
// same sums, so five accumulators serve the convective, pressure, diffusion
// and conduction terms of all directions.
template <typename R>
struct CellAcc {
    R m, mk[3];  // sums of U = c (un_i + un_j)(rho_i + rho_j) and of U u_j, metric included; + 4 grad p - 4 mu lap u
    R e;         // energy terms that are no u_k mk[k] / 4: U e_j / 4, p div u, conduction
};

// Velocity and viscosity derivatives along one direction.
template <typename R>
struct Grad {
    R u[3], m;
};

// Uniform values of the flux arithmetic.
template <typename R>
struct FluxConst {
    R c[H], c2[H + 1];  // first- and second-derivative weights (the viscous terms; Euler along z)
    R rg, pref;         // pressure = rg * sp_press + pref
    R ea, eb;           // internal energy = ea + eb T
    R rg4, ea2, eb4;    // 4 rg, 2 ea, eb / 4
    R cpr;              // cp / Pr
    R gamr, prm1;       // c^2 = gamr T, 1 / Pr
    double ta, tb;      // T = ta + tb e
    double rgas, p0;    // stored p - p_ref of the mixed form = rgas rho T - p0
};

// The central flux difference of the cell along direction D, and its viscous
// derivatives.  The flux of the reference (kernels_cpu.F90:466-618, 1109-1257,
// 1854-2004) at a face is a sum of pair terms G_l(a, b) over the pairs that
// straddle it with b - a = l.  Between two faces of equal stencil order the
// sums telescope: the difference is sum_l c_l (G_l(i, i+l) - G_l(i-l, i)), six
// pairs that all hold the cell's own point i.  What depends on point i alone
// then factors out of the sums (e.g. sum U (u_i + u_j) = u_i sum U + sum U u_j),
// the pressure and velocity parts of the energy flux become the p and u_d
// derivatives, and the internal energy, affine in T, needs only sum U T_j.
// That is ~11 operations a pair and no face values to carry between cells or
// lanes; the face form with its register march and lane moves issued ~2.5x
// the instructions.  am is the metric of the Euler term (0: direction not
// taken here), w the first-derivative weights of its stencil order (per lane
// along x and y, see edge_cell), a1, s1, q1 the viscous metrics, pr the cell's
// pressure.
// The neighbours of a direction in the order +1, -1, +2, -2, +3, -3, each
// read from LDS (D < 2) one step ahead of its use; a scheduler free to start
// every read of a direction at once would hold 72 registers of them.
template <typename R, int D, typename Get, typename Use>
__device__ __forceinline__ void each_neighbour(const Get &at, const Use &use) {
    SP<R> nb[2];
    nb[0] = at(1);
#pragma unroll
    for (int q = 0; q < 2 * H; q++) {
        if (q + 1 < 2 * H) nb[(q + 1) & 1] = at(q & 1 ? (q + 3) / 2 : -(q + 2) / 2);
        if (D != 2) __builtin_amdgcn_sched_barrier(0);
        use(nb[q & 1], q / 2, (q & 1) != 0);
        if (D != 2) __builtin_amdgcn_sched_barrier(0);
    }
}

template <typename R, int D, typename Get>
__device__ __forceinline__ R flux_dir(const FluxConst<R> &K, const SP<R> &o, const Get &at, const R (&w)[H], R pr, R am,
                                      R a1, R s1, R q1, CellAcc<R> &A, Grad<R> &G) {
    R m = R(0), mu_ = R(0), mv = R(0), mw = R(0), mt = R(0), ps = R(0);
    R gu = R(0), gv = R(0), gw = R(0), gt = R(0), gm = R(0), gn = R(0);
    R lu = K.c2[0] * o.a[VU], lv = K.c2[0] * o.a[VU + 1], lw = K.c2[0] * o.a[VU + 2], lt = K.c2[0] * o.a[VT];
    each_neighbour<R, D>(at, [&](const SP<R> &p, int l, bool neg) {
        const R c = neg ? -K.c[l] : K.c[l], c2 = K.c2[l + 1], cw = neg ? -w[l] : w[l];
        const R U = (cw * (o.a[VU + D] + p.a[VU + D])) * (o.a[VR] + p.a[VR]);
        m += U;
        mu_ += U * p.a[VU];
        mv += U * p.a[VU + 1];
        mw += U * p.a[VU + 2];
        mt += U * p.a[VT];
        ps += cw * sp_press(p);
        if (D != 2) gn += cw * p.a[VU + D];
        gu += c * p.a[VU];
        gv += c * p.a[VU + 1];
        gw += c * p.a[VU + 2];
        gt += c * p.a[VT];
        gm += c * p.a[VM];
        lu += c2 * p.a[VU];
        lv += c2 * p.a[VU + 1];
        lw += c2 * p.a[VU + 2];
        lt += c2 * p.a[VT];
    });
    const R mu4 = R(-4) * o.a[VM];
    (D == 0 ? mu_ : (D == 1 ? mv : mw)) += K.rg4 * ps;
    A.e += am * (K.eb4 * mt + pr * (D == 2 ? gw : gn));
    gu *= a1; gv *= a1; gw *= a1; gt *= a1; gm *= a1;
    A.m += am * m;
    A.mk[0] += am * mu_ + mu4 * (lu * s1 + gu * q1);
    A.mk[1] += am * mv + mu4 * (lv * s1 + gv * q1);
    A.mk[2] += am * mw + mu4 * (lw * s1 + gw * q1);
    A.e -= K.cpr * (gm * gt + o.a[VM] * (lt * s1 + gt * q1));
    G.u[0] = gu; G.u[1] = gv; G.u[2] = gw;
    G.m = gm;
    return gt;
}

// The same with the viscous terms of the second-order conservative form
// (visflx_reduced_ord2 and visflx_x/y/z, kernels_cpu.F90:4623-4721, 4779-4999):
// hc = 1/(x_{i+1} - x_{i-1}), hm = 1/(x_i - x_{i-1}), hp = 1/(x_{i+1} - x_i).
// The face fluxes mu du/dx of the momenta go to mk, their kinetic part
// mu d(|u|^2/2)/dx to e less the u_k mk[k] / 4 that the sums already carry:
// (|u_p|^2 - |u_o|^2)/2 - u_o.(u_p - u_o) = |u_p - u_o|^2 / 2.
template <typename R, int D, typename Get>
__device__ __forceinline__ R flux_dir_cons(const FluxConst<R> &K, const SP<R> &o, const Get &at, const R (&w)[H], R pr, R am,
                                           R hc, R hm, R hp, CellAcc<R> &A, Grad<R> &G) {
    R m = R(0), mu_ = R(0), mv = R(0), mw = R(0), mt = R(0), ps = R(0), gn = R(0), gt = R(0);
    G.u[0] = G.u[1] = G.u[2] = G.m = R(0);
    each_neighbour<R, D>(at, [&](const SP<R> &p, int l, bool neg) {
        const R c = neg ? -w[l] : w[l];
        const R U = (c * (o.a[VU + D] + p.a[VU + D])) * (o.a[VR] + p.a[VR]);
        m += U;
        mu_ += U * p.a[VU];
        mv += U * p.a[VU + 1];
        mw += U * p.a[VU + 2];
        mt += U * p.a[VT];
        ps += c * sp_press(p);
        gn += c * p.a[VU + D];
        if (l == 0) {
            const R h = neg ? -hc : hc;
            const R f = (o.a[VM] + p.a[VM]) * ((neg ? hm : hp) * hc);
            G.m += h * p.a[VM];
            gt += h * p.a[VT];
            R k2 = R(0);
#pragma unroll
            for (int x = 0; x < 3; x++) {
                const R d = p.a[VU + x] - o.a[VU + x];
                G.u[x] += h * p.a[VU + x];
                A.mk[x] -= R(4) * f * d;
                k2 += d * d;
            }
            A.e -= f * ((p.a[VT] - o.a[VT]) * K.cpr + R(0.5) * k2);
        }
    });
    (D == 0 ? mu_ : (D == 1 ? mv : mw)) += K.rg4 * ps;
    A.e += am * (K.eb4 * mt + pr * gn);
    A.m += am * m;
    A.mk[0] += am * mu_;
    A.mk[1] += am * mv;
    A.mk[2] += am * mw;
    return gt;
}

// Beside a non-periodic boundary the two faces of a cell can have different
// half widths, or one is a zero-flux wall face.  flux_dir then works with the
// weights d_l of the wider face, and this adds the difference at the other
// one: sum_l (d_l - c_l) S_l, S_l the pairs that straddle it (zero flux: c_l
// = 0, but the pressure part stays).  side is -1 (lower face) or +1; points
// are taken at side * offset, so that both sides run the same code.  Only the
// point pairs in flight are held in registers.
template <typename R>
struct EdgeW {
    R e[H], p[H];  // d_l - c_l, for the convective and the pressure part
};
template <typename R, int D, typename Get>
__device__ __forceinline__ void edge_cell(const Get &at, const SP<R> &o, unsigned edge, const R (*cd)[H],
                                          const FluxConst<R> &K, R am, R f[5]) {
    const int lo = (int)(edge & 15u), hi = (int)(edge >> 4) & 15;
    const bool upper = (edge >> 9) & 1u || lo > hi;
    const bool zero = upper ? (edge >> 9) & 1u : (edge >> 8) & 1u;
    const int side = upper ? 1 : -1, small = upper ? hi : lo, big = max(lo, hi);
    EdgeW<R> W;
    am = upper ? -am : am;
#pragma unroll
    for (int l = 0; l < H; l++) {
        const R d = am * cd[big - 1][l], c = am * cd[small - 1][l];
        W.e[l] = d - (zero ? R(0) : c);
        W.p[l] = d - c;
    }
    auto pair = [&](const SP<R> &A, const SP<R> &B, int l) {
        const R una = A.a[VU + D], unb = B.a[VU + D];
        const R pA = sp_press(A) * K.rg, pB = sp_press(B) * K.rg;
        const R uv = R(0.25) * W.e[l - 1] * (una + unb) * (A.a[VR] + B.a[VR]);
        f[0] += R(2) * uv;
#pragma unroll
        for (int x = 0; x < 3; x++) f[1 + x] += uv * (A.a[VU + x] + B.a[VU + x]);
        f[1 + D] += W.p[l - 1] * (pA + pB);
        f[4] += uv * (K.ea2 + K.eb * (A.a[VT] + B.a[VT]) + A.a[VU] * B.a[VU] + A.a[VU + 1] * B.a[VU + 1] +
                      A.a[VU + 2] * B.a[VU + 2]) +
                W.e[l - 1] * (una * (pB + K.pref) + unb * (pA + K.pref));
    };
    {
        const SP<R> m1 = at(side);
        pair(m1, o, 1);
        __builtin_amdgcn_sched_barrier(0);
        pair(m1, at(-side), 2);
        __builtin_amdgcn_sched_barrier(0);
        pair(m1, at(-2 * side), 3);
        __builtin_amdgcn_sched_barrier(0);
    }
    {
        const SP<R> m2 = at(2 * side);
        pair(m2, o, 2);
        __builtin_amdgcn_sched_barrier(0);
        pair(m2, at(-side), 3);
        __builtin_amdgcn_sched_barrier(0);
    }
    pair(at(3 * side), o, 3);
    __builtin_amdgcn_sched_barrier(0);
}

template <typename R>
constexpr int kFluxWaves = sizeof(R) == sizeof(double) ? 2 : 3;

constexpr int kFluxMaxChunk = 32;
// FP64 also takes the CFL radii, from the point it holds; the mixed form's
// points are rounded, and it takes them from w in FP64, where w was last written
// or in the aux pass
template <typename R>
constexpr bool kFluxDt = sizeof(R) == sizeof(double);

struct FluxArgs {
    const double *dx1, *dxs, *dx2, *dy1, *dys, *dy2, *dz1, *dzs, *dz2;  // metrics
    const double *xc, *yc, *zc, *yn;                                    // node coordinates, y faces
    const int *eocx, *eocy;
    const uint3 *dirty;   // cells with a WENO face (k_hot_items)
    const double *w;
    double *wallprop;
    double *dtpart;       // block maxima of the CFL radii (null: no new dt)
    double *partials;     // 5 block sums of force_rhs (SUMS)
    int chunk;
    int last;             // third stage: |omega| and the sensor are written
};

// One workgroup marches a TX x TY column tile along z over `chunk` planes:
// each lane keeps its 7-plane z stencil in registers, the x and y stencils
// come from an LDS copy of the current plane with a 3-point halo (two
// buffers, one barrier a plane).  All three directions read the same six
// values of a point, so the state is read once a stage and the right-hand side
// is written once; the separate passes (aux, x + y sweep, viscous march, z
// march) moved 96 + 96 + 120 + 152 B a cell, this one 48 + 48.  Two waves per SIMD: the z
// window, the look-ahead and the accumulators fill 256 registers, so what a
// lane can re-read (offsets, metrics, running sums) stays in LDS, and what is
// uniform in scalar registers; a spilled look-ahead load (waited for at once to
// be stored) cost 2x.
// The primitives are formed from w as a point enters the window or the halo,
// about 20 operations each for two points a lane and plane: 512 x 256 x 256
// 1.25 -> 1.36 ms, for the aux pass of 0.60 ms and half of the reads.
// Bound by vector issue and what two waves cannot hide of the waits: ~770
// vector instructions a wave and plane with the start-up planes (77 % of them
// FP64), which keep the vector units busy for 57 % of the cycles at the 2.0 GHz
// of a loaded chip; the waves wait for 30 % of theirs (counters on
// 512 x 256 x 256).  There, with the bulk sums: 1.36 to 1.41 ms, where the
// passes it replaces took 0.64 + 0.85 + 0.99 + 1.37; 128 x 96 x 64: 52 us for
// 20 + 38 + 35 + 41.  Mixed, 256 x 192 x 128: 203 us for 131 + 124 + 115 + 175.
template <typename T>
__device__ __forceinline__ T at_off(const T *__restrict__ base, unsigned bytes) {
    return *(const T *)((const char *)base + bytes);
}
template <typename T>
__device__ __forceinline__ void put_off(T *__restrict__ base, unsigned bytes, T v) {
    *(T *)((char *)base + bytes) = v;
}
// a point of one plane of w and of the viscosity: `plane` and `mu` their
// (uniform) starts, `off` the lane's byte offset in w's (a plane is far below
// 4 GiB)
template <typename R>
struct Raw {
    double c[5];
    R mu;
};
template <typename R>
__device__ __forceinline__ Raw<R> load_raw(const double *__restrict__ plane, const R *__restrict__ mu, size_t nv,
                                           unsigned off) {
    Raw<R> p;
#pragma unroll
    for (int m = 0; m < 5; m++) p.c[m] = at_off(plane + m * nv, off);
    p.mu = at_off(mu, sizeof(R) == sizeof(double) ? off : off >> 1);
    return p;
}
// eval_aux (kernels_cpu.F90:6960-7011) for a calorically perfect gas
template <typename R>
__device__ __forceinline__ SP<R> primitives(const FluxConst<R> &K, const Raw<R> &x) {
    SP<R> p;
    const double ri = 1.0 / x.c[0], u = x.c[1] * ri, v = x.c[2] * ri, w = x.c[3] * ri;
    const double t = K.ta + K.tb * (x.c[4] * ri - 0.5 * (u * u + v * v + w * w));
    p.a[VR] = R(x.c[0]);
    p.a[VU] = R(u);
    p.a[VU + 1] = R(v);
    p.a[VU + 2] = R(w);
    p.a[VT] = R(t);
    p.a[VM] = x.mu;
    if constexpr (sizeof(R) != sizeof(double)) p.a[VP_] = R(x.c[0] * t * K.rgas - K.p0);
    return p;
}

template <typename R, bool CONS, bool SUMS>
__device__ __forceinline__ void k_flux_body(const dim3 blockIdx, const dim3 gridDim, Geo g, KPar P, R *__restrict__ wa,
                                            R *__restrict__ fl, FluxArgs F) {
    constexpr int TX = 32, TY = 8, NP = kNP<R>;
    static_assert(TX * TY >= 2 * H * (TX + TY), "fewer lanes than halo points");
    __shared__ R tiles[2][NP][TY + 2 * H][TX + 2 * H];
    // metrics of the tile: Euler, then the three viscous ones (read from memory
    // inside the march they would wait behind the previous plane's stores)
    __shared__ R smx[4][TX], smy[4][TY], smz[4][kFluxMaxChunk];
    __shared__ double sred[SUMS ? 5 : 1][SUMS ? TX * TY : 1];
    __shared__ double lds[4][5];
    // byte offsets of this lane: its point and its halo point in a plane of
    // w_aux, its cell in a plane of the right-hand side, its mask entry.  (A
    // spilled register would come back through the vector memory counter,
    // behind the look-ahead loads.)
    __shared__ unsigned soff[4][TX * TY];
    __shared__ unsigned sedge[2][TX * TY];  // edge_cell's face orders along x and y
    __shared__ R scd[H][H];
    __shared__ R swx[H][TX], swy[H][TY];    // Euler weights of the tile's columns and rows
    __shared__ double sdt[kFluxDt<R> ? TX * TY : 1];  // running CFL maximum of each lane
    const int tx = threadIdx.x, ty = threadIdx.y;
    // band of whole tile rows per XCD (workgroups are dealt round-robin to the
    // 8 XCDs): the halo points then mostly come from the XCD's own L2
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    const int flat = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    if (gridDim.y % 8 == 0) {
        const int band = gridDim.y / 8;
        const int per = gridDim.x * band;
        const int r = (flat >> 3) % per;
        bz = (flat >> 3) / per;
        bx = r % gridDim.x;
        by = (flat & 7) * band + r / gridDim.x;
    }
    const int i = bx * TX + tx + 1, j = by * TY + ty + 1;
    const int k0 = bz * F.chunk + 1, k1 = min(k0 + F.chunk - 1, g.nz);
    const bool act = i <= g.nx && j <= g.ny;
    const int ic = min(i, g.nx), jc = min(j, g.ny);
    const int ng = g.ng;
    const size_t nv = g.nvol, ni = g.nint;
    const int tid = ty * TX + tx;
    // offsets in a plane: this lane's point, its halo point (lanes 0 ..
    // 2H*TX-1 the y halo rows, the next 2H*TY lanes the x halo columns, the
    // rest none) and its cell of the right-hand side
    // (ghost points of periodic directions at their images, which are what
    // bcswap would have copied there)
    auto source = [&](int x, int y) {
        x = min(x, g.nx + H);
        y = min(y, g.ny + H);
        if (P.periodic[0]) x = x < 1 ? x + g.nx : (x > g.nx ? x - g.nx : x);
        if (P.periodic[1]) y = y < 1 ? y + g.ny : (y > g.ny ? y - g.ny : y);
        return (unsigned)sizeof(double) * (unsigned)((x + ng - 1) + g.sx * (y + ng - 1));
    };
    soff[0][tid] = source(i, j);
    soff[2][tid] = (unsigned)sizeof(R) * (unsigned)((ic - 1) + g.nx * (jc - 1));
    const bool hl = tid < 2 * H * (TX + TY);
    int hlx = tx + H, hly = ty + H;
    if (tid < 2 * H * TX) {
        const int r = tid / TX;
        hly = r < H ? r : r + TY;
        hlx = tid % TX + H;
    } else if (hl) {
        const int q = tid - 2 * H * TX, c6 = q % (2 * H);
        hly = q / (2 * H) + H;
        hlx = c6 < H ? c6 : c6 + TX;
    }
    soff[1][tid] = source(bx * TX + 1 - H + hlx, by * TY + 1 - H + hly);
    const int hslot = hly * (TX + 2 * H) + hlx;
    // (indices for the rare branches, formed there)
    auto li = [&]() { return bx * TX + opaque(tx) + 1; };
    auto lj = [&]() { return by * TY + opaque(ty) + 1; };
    auto plane = [&](int k) { return wa + (ptrdiff_t)(k + ng - 1) * g.sxy; };
    auto load = [&](int k, unsigned off) {  // z is periodic
        const ptrdiff_t z = (ptrdiff_t)((k < 1 ? k + g.nz : (k > g.nz ? k - g.nz : k)) + ng - 1) * g.sxy;
        return load_raw(F.w + z, (const R *)(wa + 6 * nv + z), nv, off);
    };
    // cells beside a non-periodic boundary: faces of lowered order or zero flux
    const int lb = P.lmax_base;
    const bool inx = i >= P.eul_lo[0] && i <= P.eul_hi[0], iny = j >= P.eul_lo[1] && j <= P.eul_hi[1];
    bool edx, edy;
    {
        auto edge = [&](const int *eoc, int c, int n, int zlo, int zhi) {
            return (unsigned)max(lb + eoc[c - 1], 1) | (unsigned)max(lb + eoc[c], 1) << 4 |
                   (c == 1 && zlo == 1 ? 1u << 8 : 0u) | (c == n && zhi == 1 ? 1u << 9 : 0u);
        };
        const unsigned plain = (unsigned)(lb | lb << 4);
        const unsigned ex = edge(F.eocx, ic, g.nx, P.fzf[0], P.fzf[1]), ey = edge(F.eocy, jc, g.ny, P.fzf[2], P.fzf[3]);
        edx = act && inx && ex != plain;
        edy = act && iny && ey != plain;
        sedge[0][tid] = ex;
        sedge[1][tid] = ey;
    }
    if (tid < H * H) scd[tid / H][tid % H] = R(P.cd1tab[tid / H][tid % H]);
    if (tid < H * TX) {
        const int c = min(bx * TX + tid % TX + 1, g.nx);
        swx[tid / TX][tid % TX] = R(P.cd1tab[max(max(lb + F.eocx[c - 1], lb + F.eocx[c]), 1) - 1][tid / TX]);
    } else if (tid >= 128 && tid < 128 + H * TY) {
        const int q = tid - 128, c = min(by * TY + q % TY + 1, g.ny);
        swy[q / TY][q % TY] = R(P.cd1tab[max(max(lb + F.eocy[c - 1], lb + F.eocy[c]), 1) - 1][q / TY]);
    }
    // ghost images of div/3 (and the sensor) are written from this column
    const bool wall = j == 1;
    const bool imgc = i <= ng || i > g.nx - ng || j <= ng || j > g.ny - ng;
    FluxConst<R> K;
#pragma unroll
    for (int l = 0; l < H; l++) K.c[l] = R(P.vd1[l]);
#pragma unroll
    for (int l = 0; l <= H; l++) K.c2[l] = R(P.vd2[l]);
    K.rg = R(sizeof(R) == sizeof(double) ? P.rgas0 : 1.0);
    K.pref = R(sizeof(R) == sizeof(double) ? 0.0 : P.p_ref);
    // e_from_temperature of a calorically perfect gas
    K.eb = R(cvc(P, 0));
    K.ea = uniform(R(P.t0 * (cvc(P, P.indx_cp_r + 1) - cvc(P, 0))));
    K.ea2 = uniform(R(2) * K.ea);
    K.eb4 = uniform(R(0.25) * K.eb);
    K.rg4 = uniform(R(4) * K.rg);
    K.cpr = uniform(R(cpc(P, 0) / P.prandtl));
    K.tb = uniform(1.0 / cvc(P, 0));
    K.ta = uniform(P.t0 - cvc(P, P.indx_cp_r + 1) * P.t0 * K.tb);
    K.gamr = uniform(R(cpc(P, 0) / (cpc(P, 0) - P.rgas0) * P.rgas0));
    K.prm1 = uniform(R(1.0 / P.prandtl));
    K.rgas = P.rgas0;
    K.p0 = P.p_ref;
    if (tid < TX) {
        const int q = min(bx * TX + tid + 1, g.nx);
        smx[0][tid] = R(F.dx1[q - 1]);
        if (CONS) {
            smx[1][tid] = R(1.0 / (F.xc[q + ng] - F.xc[q + ng - 2]));
            smx[2][tid] = R(1.0 / (F.xc[q + ng - 1] - F.xc[q + ng - 2]));
            smx[3][tid] = R(1.0 / (F.xc[q + ng] - F.xc[q + ng - 1]));
        } else {
            smx[1][tid] = R(F.dxs[q - 1]);
            smx[2][tid] = R(F.dx2[q - 1]);
        }
    } else if (tid >= 64 && tid < 64 + TY) {
        const int q = min(by * TY + tid - 64 + 1, g.ny);
        smy[0][tid - 64] = R(F.dy1[q - 1]);
        if (CONS) {
            smy[1][tid - 64] = R(1.0 / (F.yc[q + ng] - F.yc[q + ng - 2]));
            smy[2][tid - 64] = R(1.0 / (F.yc[q + ng - 1] - F.yc[q + ng - 2]));
            smy[3][tid - 64] = R(1.0 / (F.yc[q + ng] - F.yc[q + ng - 1]));
        } else {
            smy[1][tid - 64] = R(F.dys[q - 1]);
            smy[2][tid - 64] = R(F.dy2[q - 1]);
        }
    }
    else if (tid >= 128 && tid < 128 + min(F.chunk, kFluxMaxChunk)) {
        const int z = tid - 128, q = min(k0 + z, g.nz);
        smz[0][z] = R(F.dz1[q - 1]);
        if (CONS) {
            smz[1][z] = R(1.0 / (F.zc[q + ng] - F.zc[q + ng - 2]));
            smz[2][z] = R(1.0 / (F.zc[q + ng - 1] - F.zc[q + ng - 2]));
            smz[3][z] = R(1.0 / (F.zc[q + ng] - F.zc[q + ng - 1]));
        } else {
            smz[1][z] = R(F.dzs[q - 1]);
            smz[2][z] = R(F.dz2[q - 1]);
        }
    }
    if (SUMS) {
#pragma unroll
        for (int q = 0; q < 5; q++) sred[q][tid] = 0.0;
    }
    // masks of this lane's 32 cells (a tile row is 32 cells from a multiple of 32)
    const int dpr = dirty_per_row(g);
    soff[3][tid] = (unsigned)sizeof(uint3) * (unsigned)((jc - 1) * dpr + ((ic - 1) >> 5));
    const size_t dirtyplane = (size_t)g.ny * dpr;
    auto load_masks = [&](int k) { return at_off(F.dirty + (size_t)(k - 1) * dirtyplane, soff[3][tid]); };
    // bit d: direction d of the cell has a WENO face
    auto masks_of = [&](const uint3 &m) {
        return ((m.x >> tx) & 1u) | (((m.y >> tx) & 1u) << 1) | (((m.z >> tx) & 1u) << 2);
    };
    auto fill = [&](int b, const SP<R> &centre, const SP<R> &halo) {
#pragma unroll
        for (int q = 0; q < NP; q++) {
            tiles[b][q][ty + H][tx + H] = centre.a[q];
            if (hl) (&tiles[b][q][0][0])[hslot] = halo.a[q];
        }
    };
    SP<R> win[2 * H + 1], hv;  // planes k-3 .. k+3; the halo
    Raw<R> nxt, hnx;           // the look-ahead
    if (kFluxDt<R>) sdt[tid] = 0.0;
    uint3 mk;
    unsigned wm;
#pragma unroll
    for (int q = 0; q < 2 * H + 1; q++) win[q] = primitives(K, load(min(k0 - H + q, g.nz + H), soff[0][tid]));
    hv = primitives(K, load(k0, soff[1][tid]));
    mk = load_masks(k0);
    wm = masks_of(mk);
    fill(0, win[H], hv);
    int buf = 0;
    for (int k = k0; k <= k1; k++, buf ^= 1) {
        const SP<R> &o = win[H];
        R(*tile)[TY + 2 * H][TX + 2 * H] = tiles[buf];
        __syncthreads();
        auto at_x = [&](int l) {
            SP<R> p;
#pragma unroll
            for (int q = 0; q < NP; q++) p.a[q] = tile[q][ty + H][tx + H + l];
            return p;
        };
        auto at_y = [&](int l) {
            SP<R> p;
#pragma unroll
            for (int q = 0; q < NP; q++) p.a[q] = tile[q][ty + H + l][tx + H];
            return p;
        };
        auto at_z = [&](int l) { return win[H + l]; };
        CellAcc<R> A;
        A.m = A.e = R(0);
#pragma unroll
        for (int q = 0; q < 3; q++) A.mk[q] = R(0);
        const R pr = K.rg * sp_press(o) + K.pref;
        const R az = smz[0][k - k0], ax = smx[0][tx], ay = smy[0][ty];
        const R amx = inx && !(wm & 1u) ? ax : R(0), amy = iny && !(wm & 2u) ? ay : R(0),
                amz = (wm & 4u) ? R(0) : az;
        // loads of plane k+1 (halo, masks) and k+1+H (centre): issued once the
        // z terms are done and taken up before this plane's stores are issued
        // (memory counters retire in order: a load waited for behind a store
        // waits for the store), they overlap the x and y work
        auto look_ahead = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            // (clamped, not skipped, behind the last plane: a load left in
            // flight by one iteration only would make every iteration wait
            // for its stores)
            nxt = load(min(k + 1 + H, g.nz + H), soff[0][tid]);
            hnx = load(k + 1, soff[1][tid]);
            mk = load_masks(min(k + 1, g.nz));
            __builtin_amdgcn_sched_barrier(0);
        };
        // The stress terms of a pair of directions are added as soon as both
        // have their derivatives (kernels_cpu.F90:3996-4180; in the
        // conservative form their mu-gradient part, sig_xy = d(u_y)/dx_x):
        // momentum in mk, dissipation in e, and the vorticity for the sensor.
        R om2 = R(0);
        auto cross = [&](int x, int y, const Grad<R> &X, const Grad<R> &Y) {
            const R a = Y.u[x], b = X.u[y];  // d u_x / dy, d u_y / dx
            om2 += (b - a) * (b - a);
            if (CONS) {
                A.mk[x] -= R(4) * (Y.m * b);
                A.mk[y] -= R(4) * (X.m * a);
                A.e -= R(2) * o.a[VM] * (a * b);
            } else {
                const R sxy = a + b;
                A.mk[x] -= R(4) * (Y.m * sxy);
                A.mk[y] -= R(4) * (X.m * sxy);
                A.e -= o.a[VM] * (sxy * sxy);
            }
        };
        R gty;
        Grad<R> GX, GY, GZ;
        auto weights = [&](const R *sw, int stride, R (&w)[H]) {
#pragma unroll
            for (int l = 0; l < H; l++) w[l] = sw[l * stride];
        };
        R ew[H];
        if constexpr (CONS) {
            flux_dir_cons<R, 2>(K, o, at_z, K.c, pr, amz, smz[1][k - k0], smz[2][k - k0], smz[3][k - k0], A, GZ);
            look_ahead();
            weights(&swx[0][tx], TX, ew);
            flux_dir_cons<R, 0>(K, o, at_x, ew, pr, amx, smx[1][tx], smx[2][tx], smx[3][tx], A, GX);
            cross(0, 2, GX, GZ);
            weights(&swy[0][ty], TY, ew);
            gty = flux_dir_cons<R, 1>(K, o, at_y, ew, pr, amy, smy[1][ty], smy[2][ty], smy[3][ty], A, GY);
        } else {
            flux_dir<R, 2>(K, o, at_z, K.c, pr, amz, az, smz[1][k - k0], smz[2][k - k0], A, GZ);
            look_ahead();
            weights(&swx[0][tx], TX, ew);
            flux_dir<R, 0>(K, o, at_x, ew, pr, amx, ax, smx[1][tx], smx[2][tx], A, GX);
            cross(0, 2, GX, GZ);
            weights(&swy[0][ty], TY, ew);
            gty = flux_dir<R, 1>(K, o, at_y, ew, pr, amy, ay, smy[1][ty], smy[2][ty], A, GY);
        }
        cross(0, 1, GX, GY);
        cross(1, 2, GY, GZ);
        const R u = o.a[VU], v = o.a[VU + 1], w = o.a[VU + 2], t = o.a[VT], mu = o.a[VM];
        const R uy = GY.u[0], wy = GY.u[2];
        const R d3 = (GX.u[0] + GY.u[1] + GZ.u[2]) * R(1.0 / 3.0);
        {
            // 2 (du_x/dx - div/3); the conservative form has its first half in the face fluxes
            const R two = R(2);
            const R s11 = CONS ? GX.u[0] - two * d3 : two * (GX.u[0] - d3);
            const R s22 = CONS ? GY.u[1] - two * d3 : two * (GY.u[1] - d3);
            const R s33 = CONS ? GZ.u[2] - two * d3 : two * (GZ.u[2] - d3);
            A.mk[0] -= R(4) * (GX.m * s11);
            A.mk[1] -= R(4) * (GY.m * s22);
            A.mk[2] -= R(4) * (GZ.m * s33);
            A.e -= mu * (s11 * GX.u[0] + s22 * GY.u[1] + s33 * GZ.u[2]);
        }
        R f[5];
        f[0] = R(0.5) * A.m;
        f[1] = R(0.25) * (u * A.m + A.mk[0]);
        f[2] = R(0.25) * (v * A.m + A.mk[1]);
        f[3] = R(0.25) * (w * A.m + A.mk[2]);
        f[4] = R(0.25) * ((K.ea2 + K.eb * t) * A.m + u * A.mk[0] + v * A.mk[1] + w * A.mk[2]) + A.e;
        if (edx && !(wm & 1u)) edge_cell<R, 0>(at_x, o, sedge[0][tid], scd, K, ax, f);
        if (edy && !(wm & 2u)) edge_cell<R, 1>(at_y, o, sedge[1][tid], scd, K, ay, f);
        if (SUMS && act) {
            // force_rhs: the grad(div/3) part of the rho*u sum by parts
            // along the uniform periodic x: -sum mu d(D)/dx = +sum D d(mu)/dx
            sred[0][tid] += double(f[0]);
            sred[1][tid] += double(f[1]) + double(d3) * double(GX.m);
            double w1, w2;
            if constexpr (sizeof(R) == sizeof(double)) {
                w1 = o.a[VR];
                w2 = o.a[VR] * u;
            } else {
                const int c = gidx(g, li(), lj(), k);
                w1 = F.w[c];
                w2 = F.w[nv + c];
            }
            sred[2][tid] += w1;
            sred[3][tid] += w2;
            sred[4][tid] += w2 * double(t);
        }
        if constexpr (kFluxDt<R>) {
            if (F.dtpart && act) {
                // the spectral radii of compute_dt (kernels_cpu.F90:6814-6880)
                const int ii = li() - 1, jj = lj() - 1;
                const R nu = o.a[VM] / o.a[VR], cs = sqrt(K.gamr * t);
                const R sm = fmax(fmax(F.dxs[ii], F.dys[jj]), F.dzs[k - 1]);
                R mx = fmax((fabs(u) + cs) * ax, (fabs(v) + cs) * ay);
                mx = fmax(mx, (fabs(w) + cs) * az);
                sdt[tid] = fmax(sdt[tid], fmax(mx, fmax(nu, nu * K.prm1) * sm));
            }
        }
        hv = primitives(K, hnx);
        fill(buf ^ 1, win[H + 1], hv);
        wm = masks_of(mk);
#pragma unroll
        for (int q = 0; q < 2 * H; q++) win[q] = win[q + 1];
        win[2 * H] = primitives(K, nxt);
        __builtin_amdgcn_sched_barrier(0);
        if (act) {
            const unsigned oc = sizeof(R) == sizeof(double) ? soff[0][tid] : soff[0][tid] >> 1, of = soff[2][tid];
            R *fk = fl + (size_t)(k - 1) * g.nx * g.ny;
#pragma unroll
            for (int q = 0; q < 5; q++) put_off(fk + q * ni, of, f[q]);
            put_off(plane(k) + 9 * nv, oc, d3);
            const bool img = imgc || k <= ng || k > g.nz - ng;
            if (img) write_images(g, P, wa + 9 * nv, li(), lj(), k, d3, true);
            if (F.last) {
                // visflx(3): the sensor from the stored |omega| and div/3
                // (sensor_subroutine, kernels_cpu.F90:4726-4744); the switch
                // of this step works from the masks, so it can go in place
                const R om = sqrt(om2);
                put_off(plane(k) + 8 * nv, oc, om);
                const R dv = R(3.0) * d3, ul = R(P.u0 / P.l0);
                R sv = -dv / sqrt(om * om + dv * dv + ul * ul);
                sv = fmax(sv, R(0.0));
                put_off(plane(k) + 7 * nv, oc, sv * sv);
                if (img) write_images(g, P, wa + 7 * nv, li(), lj(), k, sv * sv, false);
            }
            if (wall) {
                const size_t wsz = (size_t)g.sx * g.sz;
                const size_t wp = (size_t)(li() + ng - 1) + (size_t)g.sx * (k + ng - 1);
                F.wallprop[wp] = double(mu * uy);
                F.wallprop[wsz + wp] = double(mu * wy);
                F.wallprop[2 * wsz + wp] = double(mu * gty * K.cpr);
            }
        }
    }
    if (kFluxDt<R> && F.dtpart) {
        const double mx = wave_max(sdt[tid]);
        if ((tid & 63) == 0) lds[tid >> 6][0] = mx;
        __syncthreads();
        if (tid == 0) F.dtpart[flat] = fmax(fmax(lds[0][0], lds[1][0]), fmax(lds[2][0], lds[3][0]));
        __syncthreads();
    }
    if (SUMS) {
        const int jy = min(lj(), g.ny);
        const double dy = F.yn[jy] - F.yn[jy - 1];
        double red[5];
#pragma unroll
        for (int q = 0; q < 5; q++) red[q] = sred[q][tid] * dy;
        block_sum<5>(red, lds);
        if (tid == 0) {
#pragma unroll
            for (int q = 0; q < 5; q++) F.partials[(size_t)flat * 5 + q] = red[q];
        }
    }
}
template <typename R, bool CONS, bool SUMS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kFluxWaves<R>))) void k_flux(Geo g, KPar P, R *__restrict__ wa, R *__restrict__ fl, FluxArgs F) {
    k_flux_body<R, CONS, SUMS>(dim3(blockIdx.x, blockIdx.y, blockIdx.z), dim3(gridDim.x, gridDim.y, gridDim.z), g, P, wa, fl, F);
}

// ============================================================ WENO items
// A stencil point in direction-aligned velocities: n normal, a and b the
// tangential ones in the order of the eigenvector routines, so that one code
// serves all directions and the direction is a property of the lane.
struct IP {
    double r, n, a, b, t;
};
struct ItemConst {
    double ea, eb, rg, gam;  // e = ea + eb T, gas constant, cp/(cp - R)
    double ta, tb;           // T = ta + tb (h - |u|^2/2) of the Roe average
    __device__ __forceinline__ double enthalpy(const IP &q) const {
        return ea + (eb + rg) * q.t + 0.5 * (q.n * q.n + q.a * q.a + q.b * q.b);
    }
};

// Reconstruction from five values, v[2] the upwind cell (wenorec_1d,
// kernels_cpu.F90:2526-2667, one side; orders 3 with Jiang-Shu or Z weights, 2,
// 1).  The normalized weights alpha_k / sum alpha of alpha_k = d_k / (eps +
// beta_k)^2 are taken over their common denominator, which leaves one
// division of the eleven the quotients ask for.
__device__ __forceinline__ double weno_side(double v0, double v1, double v2, double v3, double v4, int ord,
                                            int version, double scale) {
    if (ord >= 3) {
        const double s0 = v0 - 2.0 * v1 + v2, s1 = v1 - 2.0 * v2 + v3, s2 = v2 - 2.0 * v3 + v4;
        const double g0 = v0 - 4.0 * v1 + 3.0 * v2, g1 = v1 - v3, g2 = 3.0 * v2 - 4.0 * v3 + v4;
        const double t = 13.0 / 12.0;
        const double b0 = scale * (t * s0 * s0 + 0.25 * g0 * g0), b1 = scale * (t * s1 * s1 + 0.25 * g1 * g1),
                     b2 = scale * (t * s2 * s2 + 0.25 * g2 * g2);
        double n0, n1, n2;
        if (version == 0) {
            const double q0 = 0.000001 + b0, q1 = 0.000001 + b1, q2 = 0.000001 + b2;
            const double m0 = q1 * q2, m1 = q0 * q2, m2 = q0 * q1;
            n0 = 0.1 * m0 * m0;
            n1 = 0.6 * m1 * m1;
            n2 = 0.3 * m2 * m2;
        } else {
            // eps40 is the single-precision literal 1.e-35 of the reference
            const double eps40 = (double)1.e-35f, tau = fabs(b0 - b2) + eps40;
            const double q0 = b0 + eps40, q1 = b1 + eps40, q2 = b2 + eps40;
            n0 = 0.1 * (b0 + tau) * (q1 * q2);
            n1 = 0.6 * (b1 + tau) * (q0 * q2);
            n2 = 0.3 * (b2 + tau) * (q0 * q1);
        }
        const double c0 = 2.0 * v0 - 7.0 * v1 + 11.0 * v2, c1 = -v1 + 5.0 * v2 + 2.0 * v3, c2 = 2.0 * v2 + 5.0 * v3 - v4;
        return (n0 * c0 + n1 * c1 + n2 * c2) / (6.0 * (n0 + n1 + n2));
    }
    if (ord == 2) {
        const double d0 = v2 - v1, d1 = v3 - v2;
        const double q0 = 0.000001 + scale * (d0 * d0), q1 = 0.000001 + scale * (d1 * d1);
        const double n0 = q1 * q1, n1 = 2.0 * (q0 * q0);
        return (n0 * (3.0 * v2 - v1) + n1 * (v2 + v3)) / (2.0 * (n0 + n1));
    }
    return v2;
}

// Characteristic WENO flux of the face between q[2] and q[3] (Roe average,
// eigenvectors and local Lax-Friedrichs split of kernels_cpu.F90:619-682,
// 2728-2782, 3013-3089).  The projections of a point on the two acoustic
// fields and the entropy field share K = (b1 - b2 u.u_l + b2 H_l)/2: they are
// K +- (un - un_l)/(2c) and 1 - 2K; wc = rho s - e p and gc = rho un s + n p then
// give the conserved and the flux component of any field.
__device__ __forceinline__ void weno_face(const KPar &P, const ItemConst &C, const IP (&q)[6], int eoc, double fh[5]) {
    const double hA = C.enthalpy(q[2]), hB = C.enthalpy(q[3]);
    const double r = sqrt(q[3].r / q[2].r), rp1 = 1.0 / (r + 1.0);
    const double un = (r * q[3].n + q[2].n) * rp1, ta = (r * q[3].a + q[2].a) * rp1, tb = (r * q[3].b + q[2].b) * rp1;
    const double h = (r * hB + hA) * rp1;
    const double qq = 0.5 * (un * un + ta * ta + tb * tb);
    const double tt = C.ta + C.tb * (h - qq);
    const double gm1 = C.gam - 1.0, prho = tt * C.rg, cc = C.gam * prho;
    const double c = sqrt(cc), ci = 1.0 / c;
    const double etot = h - prho;
    const double b2 = gm1 * ci * ci, b3 = etot - prho / gm1, b1 = prho * ci * ci - b2 * (etot - 2.0 * qq);
    double ev0 = -1.0, ev1 = -1.0, ev4 = -1.0;
    double K[6];
    const int ws = P.weno_scheme;
#pragma unroll
    for (int l = 0; l < 6; l++) {
        K[l] = 0.5 * (b1 + b2 * (C.enthalpy(q[l]) - (un * q[l].n + ta * q[l].a + tb * q[l].b)));
        if (l < 3 - ws || l > 2 + ws) continue;
        const double cl = sqrt(C.gam * C.rg * q[l].t);
        ev0 = fmax(fabs(q[l].n - cl), ev0);
        ev1 = fmax(fabs(q[l].n), ev1);
        ev4 = fmax(fabs(q[l].n + cl), ev4);
    }
    int ord = ws + eoc;
    if (ord < 1) ord = 1;
    const double u0_2 = P.u0 * P.u0, r2u2 = P.rho0 * P.rho0 * u0_2;
    const double sc1 = 1.0 / r2u2, sc2 = 1.0 / (r2u2 * u0_2);
#pragma unroll
    for (int m = 0; m < 5; m++) fh[m] = 0.0;
    // one field per iteration, not unrolled (instruction cache): its
    // projection is al + be K + la un_l + xa a_l + xb b_l
#pragma unroll 1
    for (int m = 0; m < 5; m++) {
        double al, be, la = 0.0, xa = 0.0, xb = 0.0, en, ee, ev = ev1, scale = sc1;
        double e0 = 1.0, e1 = un, e2 = ta, e3 = tb, e4;  // right eigenvector
        if (m == 0 || m == 4) {
            const double sg = m == 0 ? 0.5 : -0.5;
            al = sg * ci * un;
            be = 1.0;
            la = -sg * ci;
            en = -0.5 * b2 * un - sg * ci;
            ee = 0.5 * b2;
            ev = m == 0 ? ev0 : ev4;
            e1 = un - 2.0 * sg * c;
            e4 = h - 2.0 * sg * un * c;
        } else if (m == 1) {
            al = 1.0;
            be = -2.0;
            en = b2 * un;
            ee = -b2;
            e4 = b3;
        } else {
            al = m == 2 ? -ta : -tb;
            be = 0.0;
            en = ee = 0.0;
            xa = m == 2 ? 1.0 : 0.0;
            xb = m == 2 ? 0.0 : 1.0;
            scale = sc2;
            e0 = e1 = 0.0;
            e2 = xa;
            e3 = xb;
            e4 = m == 2 ? ta : tb;
        }
        double gp[6], gn[6];
#pragma unroll
        for (int l = 0; l < 6; l++) {
            const IP &x = q[l];
            const double s = al + be * K[l] + la * x.n + xa * x.a + xb * x.b;
            const double pp = x.r * x.t * C.rg;
            const double wc = x.r * s - ee * pp, gc = x.r * x.n * s + en * pp;
            gp[l] = 0.5 * (gc + ev * wc);
            gn[l] = gc - gp[l];
        }
        const double fi = weno_side(gp[0], gp[1], gp[2], gp[3], gp[4], ord, P.weno_version, scale) +
                          weno_side(gn[5], gn[4], gn[3], gn[2], gn[1], ord, P.weno_version, scale);
        fh[0] += e0 * fi;
        fh[1] += e1 * fi;
        fh[2] += e2 * fi;
        fh[3] += e3 * fi;
        fh[4] += e4 * fi;
    }
}

// Central KEEP flux of the same face with half width lm (kernels_cpu.F90:466-618).
__device__ __forceinline__ void central_face(const KPar &P, const ItemConst &C, const IP (&q)[6], int lm, bool zero,
                                             double fh[5]) {
    double f0 = 0.0, f1 = 0.0, f2 = 0.0, f3 = 0.0, f4 = 0.0, f5 = 0.0;
#pragma unroll
    for (int l = 1; l <= 3; l++) {
        const double v3 = P.cd1tab[2][l - 1], v2 = P.cd1tab[1][l - 1], v1 = P.cd1tab[0][l - 1];
        const double c = l > lm ? 0.0 : (lm >= 3 ? v3 : (lm == 2 ? v2 : v1));
#pragma unroll
        for (int m = 0; m < l; m++) {
            const IP &A = q[2 - m], &B = q[2 - m + l];
            const double pA = A.r * A.t * C.rg, pB = B.r * B.t * C.rg;
            const double uv = c * (A.n + B.n) * (A.r + B.r);
            f0 += uv;
            f1 += uv * (A.n + B.n);
            f2 += uv * (A.a + B.a);
            f3 += uv * (A.b + B.b);
            f4 += uv * (2.0 * C.ea + C.eb * (A.t + B.t) + A.n * B.n + A.a * B.a + A.b * B.b) +
                  4.0 * c * (A.n * pB + B.n * pA);
            f5 += c * (pA + pB);
        }
    }
    const double w = zero ? 0.0 : 0.25;
    fh[0] = 2.0 * w * f0;
    fh[1] = w * f1 + f5;
    fh[2] = w * f2;
    fh[3] = w * f3;
    fh[4] = w * f4;
}

struct ItemArgs {
    const int *eoc[3];
    const double *metric[3];
    const uint64_t *rec;
    const int *list, *counts;
    int nseg, wpt;
    // finish of the stage's reductions
    const double *partials;  // 5 sums of each of nblk workgroups of k_flux
    int nblk;
    const double *dtpart;    // ndt block maxima of the CFL radii (ndt = 0: no new dt)
    int ndt;
    double *stage2;
    int *ticket;
    DevScalars *ds;
    const double *yn;
    double rkr, rkg;
    int channel, first;
};

// The WENO work items of the stage: item (cell, direction) evaluates the two
// faces of the cell along the direction, WENO or central as the masks say,
// and gives the cell (fhat_hi - fhat_lo) * metric.  The items of one cell are
// neighbours in the list: the lane of the first one adds them up in direction
// order and stores, so a cell is written once and the result does not depend
// on the schedule.  A wave takes 64 items and owns the cells that start in
// the first 62.  All directions share one launch, and every face is hybrid
// per lane; bound by the latency of the scattered stencil loads and, where
// WENO cells are many, by the arithmetic of the faces.  On 384 x 128 x 96 with
// a shock (1.6 % WENO faces) 71 us a stage, with the general characteristic
// routines of st_flux.h at one wave per SIMD 125; on 512 x 256 x 256 0.29 ms
// after 25 steps (0.54 % of the faces; 0.54 ms averaged over them).
//
// The workgroups then finish the reductions of the stage (two levels, fixed
// order): the bulk sums of k_flux with the items' changes, giving b1, b2,
// dpdx and the bulk values of force_rhs (singleideal_cpu.F90:845-889), and
// the CFL step (:1507-1514).  The sums of the previous stage's right-hand
// side are those it finished with (DevScalars::rhs_sum).
template <typename R>
__device__ __forceinline__ void k_weno_items_body(const dim3 blockIdx, const dim3 gridDim, Geo g, KPar P,
                                                  const double *__restrict__ w, R *__restrict__ fl, ItemArgs A) {
    __shared__ pair_t pre[kItemSeg + 1];
    __shared__ pair_t wsum[4];
    __shared__ double lds[4][6];
    __shared__ bool last;
    const int t = threadIdx.x, lane = t & 63;
    double red[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    pair_t total;
    {
        pair_t cs[16], sum = 0;
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int sgi = 16 * t + q;
            cs[q] = sgi < A.nseg ? segment_pairs(A.counts[sgi]) : 0;
            sum += cs[q];
        }
        pair_t run = block_excl_scan256(sum, wsum, &total);
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int sgi = 16 * t + q;
            if (sgi < A.nseg) pre[sgi] = run;
            run += cs[q];
        }
        if (t == 0) pre[A.nseg] = total;
        __syncthreads();
    }
    const size_t nv = g.nvol, ni = g.nint;
    const int nwx = rec_per_row(g), nwords = nwx * g.ny * g.nz;
    // item `odd` of pair e: its cell (linear) and code, both left alone for a
    // blank; in a segment without a list the (cell, direction) pairs in order,
    // their masks from the records
    auto item = [&](pair_t e, int odd, int &cell, int &code) {
        const int lo = pair_segment(pre, A.nseg, e);
        const int S0 = seg_first_cell(g, nwx, lo * 256 * A.wpt, nwords);
        const int x = 2 * (int)(e - pre[lo]) + odd, report = A.counts[lo];
        if (x >= segment_items(report)) return;
        if (report >= 0) {
            code = A.list[S0 + x];
            cell = S0 + (code & 0xffffff);
        } else {
            cell = S0 + x / 3;
            const int d = x % 3, i0 = cell % g.nx;
            const uint64_t *rc = A.rec + kRecWords * ((size_t)(cell / g.nx) * nwx + (i0 >> 6)) + 2 * d;
            code = d << 24 | (int)((rc[0] >> (i0 & 63)) & 1ull) << 26 | (int)((rc[1] >> (i0 & 63)) & 1ull) << 27;
        }
    };
    ItemConst C;
    C.eb = cvc(P, 0);
    C.ea = uniform(P.t0 * (cvc(P, P.indx_cp_r + 1) - C.eb));
    C.rg = P.rgas0;
    C.gam = uniform(cpc(P, 0) / (cpc(P, 0) - P.rgas0));
    C.tb = uniform(1.0 / cpc(P, 0));
    C.ta = uniform(P.t0 - cpc(P, P.indx_cp_r + 1) * P.t0 * C.tb);
    const double te = uniform(1.0 / C.eb), t0e = uniform(P.t0 - cvc(P, P.indx_cp_r + 1) * P.t0 * te);  // T = t0e + te e
    const unsigned wave = (blockIdx.x * blockDim.x + t) >> 6;
    const unsigned nwaves = (gridDim.x * blockDim.x) >> 6;
    for (pair_t base = wave * 31; base < total; base += nwaves * 31) {
        const pair_t e = base + (lane >> 1);
        int cell = -1, code = 0;
        if (e < total) item(e, lane & 1, cell, code);
        const bool lo_hot = (code >> 26) & 1, hi_hot = (code >> 27) & 1;
        const bool work = cell >= 0 && (lo_hot || hi_hot);
        double d[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (work) {
            const int dir = (code >> 24) & 3;
            const int i = cell % g.nx + 1, jk = cell / g.nx;
            const int j = jk % g.ny + 1, k = jk / g.ny + 1;
            const int c = dir == 0 ? i : (dir == 1 ? j : k);
            const int n = dir == 0 ? g.nx : (dir == 1 ? g.ny : g.nz);
            const int *eoc = dir == 0 ? A.eoc[0] : (dir == 1 ? A.eoc[1] : A.eoc[2]);
            const double *met = dir == 0 ? A.metric[0] : (dir == 1 ? A.metric[1] : A.metric[2]);
            const size_t on = (size_t)(1 + dir) * nv, o1 = (dir == 0 ? 2 : 1) * nv, o2 = (dir == 2 ? 2 : 3) * nv;
            // every load of the stencil before any arithmetic; periodic
            // neighbours at their images
            IP q[7];
            double re[7];
#pragma unroll
            for (int s = 0; s < 7; s++) {
                int pi = i, pj = j, pk = k;
                if (dir == 0) pi += s - 3;
                else if (dir == 1) pj += s - 3;
                else pk += s - 3;
                if (P.periodic[0]) pi = pi < 1 ? pi + g.nx : (pi > g.nx ? pi - g.nx : pi);
                if (P.periodic[1]) pj = pj < 1 ? pj + g.ny : (pj > g.ny ? pj - g.ny : pj);
                if (P.periodic[2]) pk = pk < 1 ? pk + g.nz : (pk > g.nz ? pk - g.nz : pk);
                const int src = gidx(g, pi, pj, pk);
                q[s].r = w[src];
                q[s].n = w[on + src];
                q[s].a = w[o1 + src];
                q[s].b = w[o2 + src];
                re[s] = w[4 * nv + src];
            }
#pragma unroll
            for (int s = 0; s < 7; s++) {
                const double ri = 1.0 / q[s].r;
                q[s].n *= ri;
                q[s].a *= ri;
                q[s].b *= ri;
                const double qq = 0.5 * (q[s].n * q[s].n + q[s].a * q[s].a + q[s].b * q[s].b);
                q[s].t = t0e + te * (re[s] * ri - qq);
            }
            const int elo = eoc[c - 1], ehi = eoc[c];
            const double mt = met[c - 1];
            const int zlo = dir == 0 ? P.fzf[0] : (dir == 1 ? P.fzf[2] : P.fzf[4]);
            const int zhi = dir == 0 ? P.fzf[1] : (dir == 1 ? P.fzf[3] : P.fzf[5]);
            // WENO face first (the lower one where it has one): the lanes of a
            // wave then run the WENO branch together
            const bool alo = lo_hot || !hi_hot;
            auto sel = [](bool c, const IP &x, const IP &y) {
                return IP{c ? x.r : y.r, c ? x.n : y.n, c ? x.a : y.a, c ? x.b : y.b, c ? x.t : y.t};
            };
            // the window of the first face and the point the other one adds
            IP qw[6], ex = sel(alo, q[6], q[0]);
#pragma unroll
            for (int s = 0; s < 6; s++) qw[s] = sel(alo, q[s], q[s + 1]);
            double x[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
            for (int s2 = 0; s2 < 2; s2++) {
                const bool lo = (s2 == 0) == alo;
                double fh[5];
                const int eo = lo ? elo : ehi;
                if (lo ? lo_hot : hi_hot) weno_face(P, C, qw, eo, fh);
                else
                    central_face(P, C, qw, max(P.lmax_base + eo, 1),
                                 lo ? c == 1 && zlo == 1 : c == n && zhi == 1, fh);
                const double sg = lo ? -mt : mt;
#pragma unroll
                for (int m = 0; m < 5; m++) x[m] += sg * fh[m];
                IP nw[6];
#pragma unroll
                for (int s = 0; s < 6; s++) nw[s] = sel(alo, s < 5 ? qw[s + 1] : ex, s > 0 ? qw[s - 1] : ex);
#pragma unroll
                for (int s = 0; s < 6; s++) qw[s] = nw[s];
            }
            d[0] = x[0];
            d[4] = x[4];
            d[1] = dir == 0 ? x[1] : x[2];
            d[2] = dir == 0 ? x[2] : (dir == 1 ? x[1] : x[3]);
            d[3] = dir == 2 ? x[1] : x[3];
        }
        // the cell's first item adds its other ones (at most two) and stores
        const int c1 = __shfl_down(cell, 1, 64), c2 = __shfl_down(cell, 2, 64);
        int cm = __shfl_up(cell, 1, 64);
        if (lane == 0) {
            cm = -1;
            int cd;
            if (base > 0) item(base - 1, 1, cm, cd);
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
            const double a = __shfl_down(d[m], 1, 64), b = __shfl_down(d[m], 2, 64);
            if (c1 == cell) d[m] += a;
            if (c2 == cell) d[m] += b;
        }
        const bool lead = lane < 62 && cell >= 0 && cm != cell;
        if (lead && (d[0] != 0.0 || d[1] != 0.0 || d[2] != 0.0 || d[3] != 0.0 || d[4] != 0.0)) {
            R fo[5], fn[5];
#pragma unroll
            for (int m = 0; m < 5; m++) fo[m] = fl[m * ni + cell];
#pragma unroll
            for (int m = 0; m < 5; m++) {
                fn[m] = R(double(fo[m]) + d[m]);
                fl[m * ni + cell] = fn[m];
            }
            if (A.channel) {
                const int jj = (cell / g.nx) % g.ny + 1;
                const double dy = A.yn[jj] - A.yn[jj - 1];
                red[0] += (double(fn[0]) - double(fo[0])) * dy;
                red[1] += (double(fn[1]) - double(fo[1])) * dy;
            }
        }
    }
    if (!A.channel && A.ndt == 0) return;
    // this workgroup's slices of the block sums and of the CFL maxima
    double mx = 0.0;
    if (A.channel) {
        const int per = (A.nblk + (int)gridDim.x - 1) / (int)gridDim.x;
        const int b0 = (int)blockIdx.x * per, b1 = min(b0 + per, A.nblk);
        for (int b = b0 + t; b < b1; b += 256) {
#pragma unroll
            for (int q = 0; q < 5; q++) red[q] += A.partials[(size_t)b * 5 + q];
        }
    }
    if (A.ndt) {
        const int per = (A.ndt + (int)gridDim.x - 1) / (int)gridDim.x;
        const int b0 = (int)blockIdx.x * per, b1 = min(b0 + per, A.ndt);
        for (int b = b0 + t; b < b1; b += 256) mx = fmax(mx, A.dtpart[b]);
    }
    auto block_reduce = [&]() {  // totals in every thread
#pragma unroll
        for (int q = 0; q < 5; q++) red[q] = wave_total(red[q]);
        mx = wave_max(mx);
        if (lane == 63) {
#pragma unroll
            for (int q = 0; q < 5; q++) lds[t >> 6][q] = red[q];
        }
        if (lane == 0) lds[t >> 6][5] = mx;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 5; q++) red[q] = (lds[0][q] + lds[1][q]) + (lds[2][q] + lds[3][q]);
        mx = fmax(fmax(lds[0][5], lds[1][5]), fmax(lds[2][5], lds[3][5]));
    };
    block_reduce();
    if (gridDim.x > 1) {
        if (t == 0) {
#pragma unroll
            for (int q = 0; q < 5; q++) A.stage2[blockIdx.x * 6 + q] = red[q];
            A.stage2[blockIdx.x * 6 + 5] = mx;
            __threadfence();
            last = atomicAdd(A.ticket, 1) == (int)gridDim.x - 1;
        }
        __syncthreads();
        if (!last) return;
        __threadfence();
        // the second-level values, past the non-coherent caches, by the same tree
        mx = 0.0;
#pragma unroll
        for (int q = 0; q < 5; q++) red[q] = 0.0;
        for (int b = t; b < (int)gridDim.x; b += 256) {
#pragma unroll
            for (int q = 0; q < 5; q++)
                red[q] += __hip_atomic_load(&A.stage2[b * 6 + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            mx = fmax(mx, __hip_atomic_load(&A.stage2[b * 6 + 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        block_reduce();  // (the barrier after the ticket separates the two uses of lds)
        if (t == 0) *A.ticket = 0;
    }
    if (t == 0) {
        DevScalars *ds = A.ds;
        if (A.ndt) {
            const double dt_min = 1.0 / mx;
            ds->dt = P.cfl * dt_min;
        }
        if (A.channel) {
            const double rhodt = A.rkr * ds->dt, gamdt = A.rkg * ds->dt;
            double b1 = -gamdt * red[0], b2 = -gamdt * red[1];
            if (A.rkr != 0.0) {
                b1 -= rhodt * ds->rhs_sum[0];
                b2 -= rhodt * ds->rhs_sum[1];
            }
            b1 = b1 / P.volchan;
            b2 = b2 / P.volchan;
            ds->rhs_sum[0] = red[0];
            ds->rhs_sum[1] = red[1];
            const double b3 = red[2] / P.volchan, b4 = red[3] / P.volchan, b5 = red[4] / P.volchan;
            ds->dpdx = (A.first ? 0.0 : ds->dpdx) + b2;
            ds->rhobulk = b3;
            ds->ubulk = b4 / b3;
            ds->tbulk = b5 / b3 / ds->ubulk;
            ds->b1 = b1;
            ds->b2 = b2;
        }
    }
}
// two waves per SIMD: the scattered loads of one batch overlap the other's work
template <typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_weno_items(
    Geo g, KPar P, const double *__restrict__ w, R *__restrict__ fl, ItemArgs A) {
    k_weno_items_body<R>(dim3(blockIdx.x, blockIdx.y, blockIdx.z), dim3(gridDim.x, gridDim.y, gridDim.z), g, P, w, fl, A);
}

// ============================================================ update
struct UpdArgs {
    const double *dx1, *dy1, *dz1, *xc, *yc, *zc, *yn;
    const double *dxs, *dys, *dzs;  // viscous metrics of the CFL radii
    DevScalars *ds;
    double rkr, rkg;
    int channel;
    int keep;          // something reads the finished right-hand side again: store it
    int mu;            // the next stage reads the viscosity of the new state: store it
    int step_end;      // third stage of st_advance: icyc += 1, time += dt
    double *partials;  // block sums of rho u T dy (FV)
    double *dtpart;    // block maxima of the CFL radii of the new state (with mu; null: not wanted)
};

// visflx_div (kernels_cpu.F90:3484-3532, or its second-order form with O2,
// :3446-3480) on the completed right-hand side, then update_flux +
// force_rhs_2 + update_field (:3400-3442, 3092-3116) and the staggered
// isothermal-wall ghosts; with FV, force_var_1 (:3241-3278) and the block sums
// of rho*u*T*dy.  The grad(div/3) terms cost two more reads here (mu, div/3:
// 16 B a cell) where the pass of their own re-read and re-wrote the
// right-hand side (152 B).  The velocities of the energy term are formed from
// w as eval_aux forms them.  With U.mu the viscosity of the new state follows:
// here its power law hides behind the memory, in k_flux, which evaluates every
// point about twice, it would not.  One cell a lane: with a few planes to a
// lane the constants of that power law were kept in registers across them, one
// wave per SIMD less and 4 % slower (and without it no faster, 1379 against
// 1371 us).  Bound by HBM: 40 + 40 + 40 + 8 + 8 B read and 32 + 40 + 8 B
// written a cell (the third stage mostly without the 32), 1.33 ms a stage on
// 512 x 256 x 256 (5.1 TB/s in the bytes moved, where k_aux moves 5.6; 112
// registers leave four waves per SIMD, whose vector units are busy for 37 % of
// the cycles), 34 us on 128 x 96 x 64.  The right-hand sides are
// read with the non-temporal hint: neither is read again before a full stage of
// traffic has passed.
template <typename R, bool FV, bool O2>
__device__ __forceinline__ void k_update_div_body(const dim3 blockIdx, const dim3 gridDim, Geo g, KPar P,
                                                  double *__restrict__ w, R *__restrict__ wa,
                                                  const R *__restrict__ flp, R *__restrict__ fl, UpdArgs U) {
    __shared__ double lds[4][1];
    const int i = blockIdx.x * 64 + threadIdx.x + 1;
    const int j = blockIdx.y * 4 + threadIdx.y + 1;
    const int k = blockIdx.z + 1;
    constexpr int HW = O2 ? 1 : 3;
    double acc[1] = {0.0};
    const double dt = U.ds->dt;
    if (i <= g.nx && j <= g.ny) {
        const size_t nv = g.nvol, ni = g.nint;
        const double rhodt = U.rkr * dt, gamdt = U.rkg * dt;
        const double b1 = U.channel ? U.ds->b1 : 0.0, b2 = U.channel ? U.ds->b2 : 0.0;
        const int ng = g.ng;
        const R *D = wa + 9 * nv;
        R ax, ay;
        if (O2) {
            ax = R(1.0) / R(U.xc[i + ng] - U.xc[i + ng - 2]);
            ay = R(1.0) / R(U.yc[j + ng] - U.yc[j + ng - 2]);
        } else {
            ax = R(U.dx1[i - 1]);
            ay = R(U.dy1[j - 1]);
        }
        const int c = gidx(g, i, j, k), oi = iidx(g, i, j, k);
        R fo[5], fp[5];
#pragma unroll
        for (int m = 0; m < 5; m++) fo[m] = __builtin_nontemporal_load(&fl[m * ni + oi]);
        if (U.rkr != 0.0) {
#pragma unroll
            for (int m = 0; m < 5; m++) fp[m] = __builtin_nontemporal_load(&flp[m * ni + oi]);
        }
        double wo[5];
#pragma unroll
        for (int m = 0; m < 5; m++) wo[m] = w[m * nv + c];
        const R mu = wa[6 * nv + c];
        R gx = R(0), gy = R(0), gz = R(0);
#pragma unroll
        for (int l = 1; l <= HW; l++) {
            const R cl = O2 ? R(1) : R(P.vd1[l - 1]);
            gx += cl * (D[c + l] - D[c - l]);
            gy += cl * (D[c + l * g.sx] - D[c - l * g.sx]);
            gz += cl * (D[c + l * g.sxy] - D[c - l * g.sxy]);
        }
        const R az = O2 ? R(1.0) / R(U.zc[k + ng] - U.zc[k + ng - 2]) : R(U.dz1[k - 1]);
        const R sx = mu * (gx * ax), sy = mu * (gy * ay), sz = mu * (gz * az);
        const double ri = 1.0 / wo[0];
        const double uo = wo[1] * ri, vo = wo[2] * ri, wwo = wo[3] * ri;
        fo[1] -= sx;
        fo[2] -= sy;
        fo[3] -= sz;
        fo[4] -= sx * R(uo) + sy * R(vo) + sz * R(wwo);
        if (U.keep) {
#pragma unroll
            for (int m = 1; m < 5; m++) fl[m * ni + oi] = fo[m];
        }
        double fln[5];
#pragma unroll
        for (int m = 0; m < 5; m++) {
            fln[m] = -gamdt * double(fo[m]);
            if (U.rkr != 0.0) fln[m] = -rhodt * double(fp[m]) + fln[m];
        }
        if (U.channel) {
            fln[0] = fln[0] - b1;
            fln[1] = fln[1] - b2;
            fln[4] = fln[4] - uo * b2;
        }
        double wn[5];
#pragma unroll
        for (int m = 0; m < 5; m++) {
            wn[m] = wo[m] + fln[m];
            w[m * nv + c] = wn[m];
        }
        if (FV) {
            const double dy = U.yn[j] - U.yn[j - 1];
            const double rn = 1.0 / wn[0];
            const double uu = wn[1] * rn, vv = wn[2] * rn, ww = wn[3] * rn;
            const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
            const double ee = wn[4] / wn[0] - qq;
            const double tt = temperature_from_e(P, ee, 0.0);
            wa[5 * nv + c] = R(tt);
            acc[0] += wn[1] * tt * dy;
        } else {
            double mu_new = 0.0;
            // the cell's viscosity, and bcwall_staggered (kernels_cpu.F90:
            // 6612-6678) with the ghosts' at either wall
#pragma unroll 1
            for (int o = U.mu ? 0 : 1; o < 3; o++) {
                double x[5];
                int d = c;
                if (o == 0) {
#pragma unroll
                    for (int m = 0; m < 5; m++) x[m] = wn[m];
                } else {
                    if (!P.wall_stag[o - 1] || (o == 1 ? j > g.ng : j <= g.ny - g.ng)) continue;
                    wall_ghost_of(P, wn, 0.0, x);
                    d = gidx(g, i, o == 1 ? 1 - j : 2 * g.ny + 1 - j, k);
#pragma unroll
                    for (int m = 0; m < 5; m++) w[m * nv + d] = x[m];
                }
                if (!U.mu) continue;
                const double m = mu_of(P, x);
                wa[6 * nv + d] = R(m);
                if (o == 0) mu_new = m;
            }
            if (!kFluxDt<R> && U.dtpart) {
                const double a[3] = {U.dx1[i - 1], U.dy1[j - 1], U.dz1[k - 1]};
                const double s[3] = {U.dxs[i - 1], U.dys[j - 1], U.dzs[k - 1]};
                acc[0] = cfl_radius(P, wn, mu_new, a, s);
            }
        }
    }
    if (FV) {
        block_sum<1>(acc, lds);
        if (flat_thread() == 0)
            U.partials[(int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z))] = acc[0];
    }
    if (!FV && !kFluxDt<R> && U.dtpart) {
        const int ft = flat_thread();
        const double mx = wave_max(acc[0]);
        if ((ft & 63) == 0) lds[ft >> 6][0] = mx;
        __syncthreads();
        if (ft == 0)
            U.dtpart[(int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z))] =
                fmax(fmax(lds[0][0], lds[1][0]), fmax(lds[2][0], lds[3][0]));
    }
    // run()'s loop end (singleideal_cpu.F90:1604,1642); nothing else of this
    // launch reads time or icyc
    if (U.step_end && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && flat_thread() == 0) {
        U.ds->icyc = U.ds->icyc + 1;
        U.ds->time = U.ds->time + dt;
    }
}
template <typename R, bool FV, bool O2>
__global__ __launch_bounds__(256) void k_update_div(Geo g, KPar P, double *__restrict__ w, R *__restrict__ wa,
                                                    const R *__restrict__ flp, R *__restrict__ fl, UpdArgs U) {
    k_update_div_body<R, FV, O2>(dim3(blockIdx.x, blockIdx.y, blockIdx.z), dim3(gridDim.x, gridDim.y, gridDim.z), g, P, w, wa, flp, fl, U);
}

// ================================================================ launchers
#define ST_DISPATCH(call)                         \
    do {                                          \
        if (s->mixed) {                           \
            using R = float;                      \
            call;                                 \
        } else {                                  \
            using R = double;                     \
            call;                                 \
        }                                         \
    } while (0)

// The one-pass stage covers the KEEP split of a calorically perfect gas with
// the Roe split on the fused kernels' three ghost layers.  The span must be
// periodic (the z stencils sit in registers, where a face of lowered order
// has no cheap form) and, where force_rhs needs the bulk sums, x periodic
// and uniform (its grad(div/3) sum is taken by parts along x).
bool one_pass_stage(const st_solver *s) {
    const st_params &p = s->p;
    return p.ng == H && p.nkeep == 0 && p.calorically_perfect == 1 && p.flux_splitting == 0 && s->kp.ndim == 3 &&
           s->kp.periodic[2] && s->kp.eul_lo[0] <= s->kp.eul_hi[0] && s->kp.eul_lo[1] <= s->kp.eul_hi[1] &&
           (!p.channel_case || (s->kp.periodic[0] && s->x_uniform));
}

// With the bulk sums launch_flux fixes the chunk by the grid, without them
// visc_chunk sets it; the separate sweeps take both.
int launch_shapes(const st_solver *s) {
    if (!one_pass_stage(s)) return kShapeVisc | kShapeMarch;
    return s->p.channel_case ? 0 : kShapeVisc;
}

static const int kFluxTX = 32, kFluxTY = 8;

// Planes per workgroup of k_flux.  The chip holds two (FP64) or three (mixed)
// workgroups a CU, and a round of them takes about chunk + 1.3 plane times
// (4.9 us a plane and 6.4 us for the stencil's first planes and the launch, on
// 512 x 256 x 256 at chunks 1 to 32; with a CU to itself a workgroup takes
// 3.8 us a plane).  Long chunks spare the start-up, short ones fill the chip
// and its last round: the chunk with the least rounds x round time.  On
// 128 x 96 x 64 chunks 2, 4, 8, 16 took 57, 54, 56, 73 us (7 is taken: 53).
static int flux_chunk(const Geo &g, bool mixed) {
    const long tiles = (long)((g.nx + kFluxTX - 1) / kFluxTX) * ((g.ny + kFluxTY - 1) / kFluxTY);
    const int cus = 256, slots = cus * (mixed ? 3 : 2);
    int best = 1;
    double least = 0.0;
    for (int c = 1; c <= kFluxMaxChunk && c <= g.nz; c++) {
        const long blocks = tiles * ((g.nz + c - 1) / c);
        const double t = blocks <= cus ? 1.3 + 0.77 * c : (double)((blocks + slots - 1) / slots) * (1.3 + c);
        if (c == 1 || t < least) {
            least = t;
            best = c;
        }
    }
    return best;
}
static dim3 flux_grid(const Geo &g, int chunk) {
    return dim3((g.nx + kFluxTX - 1) / kFluxTX, (g.ny + kFluxTY - 1) / kFluxTY, (g.nz + chunk - 1) / chunk);
}
static dim3 update_grid(const Geo &g) { return dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz); }
static int nblocks(const dim3 &d) { return (int)(d.x * d.y * d.z); }

// Doubles of the reduction scratch: [0, flux) the block sums of k_flux (or of
// k_update_div), [dt, dt + blocks) the CFL maxima of k_flux (of the aux pass
// elsewhere), then the second-level values of k_weno_items.
int one_pass_flux_slots(const Geo &g, bool mixed) { return 5 * nblocks(flux_grid(g, flux_chunk(g, mixed))); }
int one_pass_update_blocks(const Geo &g) { return nblocks(update_grid(g)); }
int one_pass_dt_slots(const Geo &g) {
    const int f = nblocks(flux_grid(g, 1)), a = aux_dt_blocks(g), u = one_pass_update_blocks(g);
    return f > a ? (f > u ? f : u) : (a > u ? a : u);
}

hipError_t launch_hot_items(st_solver *s) {
    const Geo &g = s->g;
    const long words = (long)hot_words(g) * g.sy * g.sz;
    ST_DISPATCH(ST_GO(k_hot_bits, ST_T(R), 256, 0, dim3((unsigned)((words + 15) / 16)), dim3(256), g, s->kp,
                      (const R *)s->w_aux, s->hot));
    int wpt;
    const int nseg = item_segments(g, &wpt);
    ST_GO(k_hot_items, , 256, 0, dim3((unsigned)nseg), dim3(256), g, s->kp, (const uint64_t *)s->hot, s->hot_rec, s->hot_dirty, wpt,
          s->fixlist, s->counters + 8);
    return hipGetLastError();
}

hipError_t launch_flux(st_solver *s, void *fl, int stage, bool dt) {
    const Geo &g = s->g;
    const bool sums = s->p.channel_case != 0, cons = s->p.conservative_viscous == 1;
    // with the bulk sums the chunk is a function of the grid alone: they are
    // grouped by workgroup, and a tuned chunk must not change results
    const int chunk = s->visc_chunk > 0 && !sums ? (s->visc_chunk < kFluxMaxChunk ? s->visc_chunk : kFluxMaxChunk)
                                               : flux_chunk(g, s->mixed);
    const dim3 grid = flux_grid(g, chunk);
    FluxArgs F{};
    F.dx1 = s->dcsidx; F.dxs = s->dcsidxs; F.dx2 = s->dcsidx2;
    F.dy1 = s->detady; F.dys = s->detadys; F.dy2 = s->detady2;
    F.dz1 = s->dzitdz; F.dzs = s->dzitdzs; F.dz2 = s->dzitdz2;
    F.xc = s->x; F.yc = s->y; F.zc = s->z; F.yn = s->yn;
    F.eocx = s->eoc[0]; F.eocy = s->eoc[1];
    F.dirty = s->hot_dirty;
    F.w = s->w;
    F.wallprop = s->wallprop;
    F.partials = s->partials;
    F.chunk = chunk;
    F.last = stage == 2;
    if (sums) s->force_nblk = nblocks(grid);
    F.dtpart = dt && !s->mixed ? s->dtpart : nullptr;
    if (F.dtpart) s->dt_nblk = nblocks(grid);
#define ST_LAUNCH_FX(C_, S_) \
    ST_DISPATCH(ST_GO(k_flux, ST_T(R, C_, S_), 256, kFluxWaves<R>, grid, dim3(kFluxTX, kFluxTY), g, s->kp, (R *)s->w_aux, (R *)fl, F))
    if (cons && sums) ST_LAUNCH_FX(true, true);
    else if (cons) ST_LAUNCH_FX(true, false);
    else if (sums) ST_LAUNCH_FX(false, true);
    else ST_LAUNCH_FX(false, false);
#undef ST_LAUNCH_FX
    return hipGetLastError();
}

hipError_t launch_weno_items(st_solver *s, void *fl, int stage, bool dt) {
    const Geo &g = s->g;
    ItemArgs A{};
    for (int d = 0; d < 3; d++) A.eoc[d] = s->eoc[d];
    A.metric[0] = s->dcsidx;
    A.metric[1] = s->detady;
    A.metric[2] = s->dzitdz;
    A.rec = s->hot_rec;
    A.list = s->fixlist;
    A.counts = s->counters + 8;
    A.nseg = item_segments(g, &A.wpt);
    A.partials = s->partials;
    A.nblk = s->force_nblk;
    A.dtpart = s->dtpart;
    A.ndt = dt ? s->dt_nblk : 0;
    A.stage2 = s->stage2;
    A.ticket = s->counters + 1;
    A.ds = s->ds;
    A.yn = s->yn;
    A.rkr = s->rhork[stage];
    A.rkg = s->gamrk[stage];
    A.channel = s->p.channel_case != 0;
    A.first = stage == 0;
    // one workgroup per 8192 cells, at most what the chip holds at once
    long nb = (long)((g.nint + 8191) / 8192);
    nb = nb < 1 ? 1 : (nb > kItemBlocks ? kItemBlocks : nb);
    ST_DISPATCH(ST_GO(k_weno_items, ST_T(R), 256, 2, dim3((unsigned)nb), dim3(256), g, s->kp, s->w, (R *)fl, A));
    return hipGetLastError();
}

hipError_t launch_update_div(st_solver *s, const void *fl_prev, void *fl, int stage, bool step_end, bool last, bool mu, bool dt) {
    const Geo &g = s->g;
    const bool fv = s->p.channel_case && s->p.theta_wall >= -1.0, o2 = s->p.conservative_viscous == 1;
    UpdArgs U{};
    U.dx1 = s->dcsidx; U.dy1 = s->detady; U.dz1 = s->dzitdz;
    U.xc = s->x; U.yc = s->y; U.zc = s->z; U.yn = s->yn;
    U.ds = s->ds;
    U.rkr = s->rhork[stage];
    U.rkg = s->gamrk[stage];
    U.channel = s->p.channel_case;
    // the first two stages' are F[prev] of the next; the third's has no reader
    // but the caller, and is left out (32 of 216 B a cell) while further steps
    // of the call follow: 512x256x256 1380 -> 1307 us a stage over three stages
    U.keep = stage < 2 || last;
    U.mu = mu && !fv;
    U.dxs = s->dcsidxs; U.dys = s->detadys; U.dzs = s->dzitdzs;
    U.dtpart = dt ? s->dtpart : nullptr;
    if (dt) s->dt_nblk = one_pass_update_blocks(g);
    U.step_end = step_end ? 1 : 0;
    U.partials = s->partials;
    const dim3 grid = update_grid(g);
#define ST_LAUNCH_UD(F_, O_)                                                                                  \
    ST_DISPATCH(ST_GO(k_update_div, ST_T(R, F_, O_), 256, 0, grid, dim3(64, 4), g, s->kp, s->w, (R *)s->w_aux, \
                      (const R *)fl_prev, (R *)fl, U))
    if (fv && o2) ST_LAUNCH_UD(true, true);
    else if (fv) ST_LAUNCH_UD(true, false);
    else if (o2) ST_LAUNCH_UD(false, true);
    else ST_LAUNCH_UD(false, false);
#undef ST_LAUNCH_UD
    return hipGetLastError();
}

}  // namespace st
