// moments.hip -- the collide and stream step on 13 moments per node instead of 19
// populations, for the reference's relaxation rates.
//
// With rate 1 on rows 0, 1, 3, 5, 7, 10, 12 and 16..18 the collision reads of the
// pulled populations only the density, the momentum (rows 3, 5, 7) and the nine rows
// 2, 4, 6, 8, 9, 11, 13, 14, 15.  Within a run of steps these are what a step hands to
// the next: the density array and 12 moments per node.  The last step of a call also
// writes the populations, the state that the rest of the library reads and writes; a step
// after any of these has written them starts from the populations.  Every variant forms a
// node's moments from its 19 pulled values with the same operations, and floating
// contraction is limited to single expressions (below), so a run rounds the same however
// it is split.
#pragma clang fp contract(on)

#include "internal.h"
#include "lbm_math.h"
#include "device_common.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace cpmp {

namespace {

// stored moments: j, then the rows that relax
constexpr int kMom = kMomentFields;
CPMP_HD constexpr int mom_row(int k) {
    return k == 0 ? 3 : k == 1 ? 5 : k == 2 ? 7 : k == 3 ? 2 : k == 4 ? 4 : k == 5 ? 6 : k == 6 ? 8 : k == 7 ? 9
         : k == 8 ? 11 : 6 + (k - 9) + 7;
}
static_assert(mom_row(9) == 13 && mom_row(10) == 14 && mom_row(11) == 15, "moment rows");

template <class TC>
struct __align__(2 * sizeof(TC)) Pair {
    TC r, m;   // rho, mu
};

// Tile of a workgroup: TY x TZ columns it advances, one ring of neighbours whose
// collisions it repeats, and the frame of 3 more that their force stencils read.
// TY = 1 is the lattice of one row in y, which is its own y neighbour.
template <int TY_, int TZ_>
struct Tile {
    static constexpr int TY = TY_, TZ = TZ_;
    static constexpr bool flat = TY == 1;
    static constexpr int HY = flat ? 0 : 1;
    static constexpr int RY = TY + 2 * HY, RZ = TZ + 2, NN = RY * RZ;   // colliding nodes of a plane
    // waves: the own nodes, the rows above and below, the columns at the z ends
    static constexpr int own = TY * TZ, rows = flat ? 0 : 2 * TZ, ends = 2 * RY;
    static constexpr int NT = own + (rows + 63) / 64 * 64 + 64;
    static constexpr int EY = flat ? 1 : TY + 8, EZ = TZ + 8, ES = EZ | 1, EP = EY * ES;   // rho and mu of a plane, odd row stride
    static constexpr int HE = (EP + NT - 1) / NT;
    static_assert(own % 64 == 0 && rows <= 64 && ends <= 64, "one wave each for the rows and the z ends");
};

// Isotropic 6th-order gradients of rho and mu (Gradx7/y7/z7, Common.h:222-241) from the
// LDS ring: nine directional differences, each face diagonal serving two components.
template <class TC, class TL>
struct RingStencil {
    const Pair<TC> (*a)[TL::EP];
    const int *slot;   // ring slot of plane x + dx, dx = -3..3
    int base;
    __device__ __forceinline__ Pair<TC> at(int dx, int dy, int dz) const {
        return a[slot[dx + 3]][base + (TL::flat ? 0 : dy * TL::ES) + dz];
    }
    __device__ __forceinline__ void dd(int ux, int uy, int uz, TC &dr, TC &dm) const {
        const Pair<TC> m3 = at(-3 * ux, -3 * uy, -3 * uz), m2 = at(-2 * ux, -2 * uy, -2 * uz), m1 = at(-ux, -uy, -uz);
        const Pair<TC> p1 = at(ux, uy, uz), p2 = at(2 * ux, 2 * uy, 2 * uz), p3 = at(3 * ux, 3 * uy, 3 * uz);
        dr = TC(45) * (p1.r - m1.r) - TC(9) * (p2.r - m2.r) + (p3.r - m3.r);
        dm = TC(45) * (p1.m - m1.m) - TC(9) * (p2.m - m2.m) + (p3.m - m3.m);
    }
    __device__ __forceinline__ void grad(TC (&gr)[3], TC (&gm)[3]) const {
        const TC s = TC(1.0 / 360.0);
        TC rx, mx, ry, my, rz, mz, rxy, mxy, rxn, mxn, rxz, mxz, rxm, mxm, ryz, myz, ryn, myn;
        dd(1, 0, 0, rx, mx);
        dd(0, 1, 0, ry, my);
        dd(0, 0, 1, rz, mz);
        dd(1, 1, 0, rxy, mxy);
        dd(1, -1, 0, rxn, mxn);
        dd(1, 0, 1, rxz, mxz);
        dd(1, 0, -1, rxm, mxm);
        dd(0, 1, 1, ryz, myz);
        dd(0, 1, -1, ryn, myn);
        gr[0] = (TC(2) * rx + rxz + rxm + rxy + rxn) * s;
        gr[1] = (TC(2) * ry + ryz + ryn + rxy - rxn) * s;
        gr[2] = (TC(2) * rz + rxz - rxm + ryz - ryn) * s;
        gm[0] = (TC(2) * mx + mxz + mxm + mxy + mxn) * s;
        gm[1] = (TC(2) * my + myz + myn + mxy - mxn) * s;
        gm[2] = (TC(2) * mz + mxz - mxm + myz - myn) * s;
    }
};

// Moment k of node (x, y, z) is at (x * 12 + k) * ny * nz + mom_site(y, z): within a
// plane the tiles are contiguous runs (the last tiles of a row or column are narrower),
// so a workgroup streams whole lines.
template <class TL>
__device__ __forceinline__ unsigned mom_site(const DevParams &P, int y, int z) {
    const int y0 = y / TL::TY * TL::TY, z0 = z / TL::TZ * TL::TZ;
    const int h = min(TL::TY, P.ny - y0), w = min(TL::TZ, P.nz - z0);
    return (unsigned)(y0 * P.nz + h * z0 + (y - y0) * w + (z - z0));
}
// The first and last column of every tile are kept a second time, as runs of TY values:
// moment k of row r of side s (0 first, 1 last) of a tile at
// (((x * tiles + tile) * 2 + s) * 12 + k) * TY + r.  A neighbour in z reads its halo there
// instead of one value from each of 12 * TY lines.

template <class TF, class TS, class TC>
struct StepArgs {
    const TF *fin;        // populations (IN_P) or
    const TC *min;        // moments of the state before the step
    TF *fout;             // and after it (OUT_P: populations)
    TC *mout;
    const TC *ein;        // edge columns of min and mout
    TC *eout;
    const TS *rho, *mu;
    TS *rho_out;
    TS *mv;               // u + F / (2 rho) (DIAG, may be null)
    TS *uout;             // adjoint tape: u, grad mu, grad rho (DIAG, may be null)
    int ntz, nty, xc;
};

enum { kPlain, kQp, kGuo };   // force term: exact difference, with Qp, Guo (Qp if on)

// One step.  A workgroup owns a tile of columns and marches along x over xc planes.  It
// collides every node of its tile and of the ring of neighbours around it, posts the 16
// populations that leave their column in an LDS mailbox, and each own node collects what
// arrives: after the plane behind it has collided, a node holds its 19 pulled values and
// writes their moments (OUT_P: its post-collision populations too).  Nothing is exchanged between workgroups within a
// step, so any lattice size works and no density completion follows; the price is the
// ring: 476 collisions for 384 nodes, and two more planes per chunk.
//
// Bound: memory.  At 256^3 FP32 a launch moves 2.18 GB (1.74 GB of state) in 0.453 ms, 4.8
// TB/s, what a large copy reaches; the VALU is busy 71 % of it.  FP64 0.89 ms, 4.7 TB/s.  The
// population march with its density completion took 0.62 (FP32) and 1.24 ms (FP64).
// Tile: 12 x 32 fills 8 waves, 2 per SIMD, and two workgroups a CU (8 x 32: 5.3 waves
// unevenly over the SIMDs, step 0.623 against 0.604 ms at 256^3 FP32; 12 x 64 with one
// workgroup of 15 waves per CU 0.568 against 0.579, but its tail grows on other sizes).
// 4 waves per SIMD (128 VGPRs) keep the second workgroup: at 136 the step took 0.689 ms.
template <class TF, class TS, class TC, class TL, bool IN_P, bool OUT_P, bool DIAG, bool NW, int FC>
__global__ void __launch_bounds__(TL::NT, sizeof(TC) == 4 ? 4 : 2) k_moment_step(const DevParams P, const StepArgs<TF, TS, TC> A) {
    __shared__ Pair<TC> s_rm[7][TL::EP];       // planes x-3 .. x+3
    __shared__ TC s_mail[Q - 3][TL::NN];       // populations 3..18 of plane x
    __shared__ TC s_edge[2 * kMom * TL::TY];   // edge columns of a finished plane
    int t = blockIdx.x;
    {
        // workgroup b runs on XCD b % 8: each XCD takes a contiguous range of tiles (z
        // fastest, then y), so neighbouring tiles read their common lines from one L2
        const int n = gridDim.x, k = t & 7;
        t = k * (n >> 3) + min(k, n & 7) + (t >> 3);
    }
    const int tzi = t % A.ntz;
    t /= A.ntz;
    const int tyi = t % A.nty, ch = t / A.nty, tile = tyi * A.ntz + tzi;
    constexpr int TZ = TL::TZ;
    const int y0 = tyi * TL::TY, z0 = tzi * TZ;
    const int xa = ch * A.xc, xb = min(xa + A.xc, P.nx);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool inner = wave < TL::own / 64;            // the waves of the own nodes
    const bool ends = wave == TL::NT / 64 - 1;         // the wave of the z ends
    // position (ly, lz) in the frame of colliding nodes
    int ly, lz;
    if (inner) {
        ly = tid / TZ + TL::HY;
        lz = tid % TZ + 1;
    } else if (!ends) {
        ly = tid - TL::own < TZ ? 0 : TL::RY - 1;
        lz = (tid - TL::own) % TZ + 1;
    } else {
        const int r = min(tid - (TL::NT - 64), TL::ends - 1);
        ly = r % TL::RY;
        lz = r < TL::RY ? 0 : TL::RZ - 1;
    }
    const int pos = ly * TL::RZ + lz;
    const int yu = y0 + ly - TL::HY, zu = z0 + lz - 1;      // before the periodic wrap
    const int y = wrapc(yu, P.ny), z = wrapc(zu, P.nz);
    const bool own = inner && yu < P.ny && zu < P.nz;
    const bool fluid = NW || !is_solid(P, z);
    const bool post = (!ends || tid - (TL::NT - 64) < TL::ends) && fluid;
    const bool bb_lo = !NW && is_solid(P, wrap_off(z, -1, P.nz));   // z - 1 solid: c_z > 0 arrives bounced
    const bool bb_hi = !NW && is_solid(P, wrap_off(z, 1, P.nz));
    const int pl = P.ny * P.nz;
    const unsigned node = (unsigned)(y * P.nz + z);
    // lane part of the moments' address and the step from one moment to the next: the z
    // ends read the neighbouring tile's edge column (a tile whose z end is the lattice's
    // holds its wrapped neighbour among its own lanes and does not use the far end)
    const int tiles = A.ntz * A.nty;
    const unsigned site = ends ? (unsigned)((y / TL::TY * A.ntz + z / TZ) * 2 + (lz == 0 ? 1 : 0)) * (kMom * TL::TY) + y % TL::TY
                               : mom_site<TL>(P, y, z);
    const int zlast = min(z0 + TZ, P.nz) - 1;
    const bool edge = zu == z0 || zu == zlast;
    const int eslot = (zu == z0 ? 0 : kMom * TL::TY) + ly - TL::HY;

    auto wrap_x = [&](int x) { return P.nx >= 8 ? (x < 0 ? x + P.nx : (x >= P.nx ? x - P.nx : x)) : wrapc(x, P.nx); };

    // rho and mu of one plane: frame entries e = tid + h NT of this thread
    unsigned eoff[TL::HE];
#pragma unroll
    for (int h = 0; h < TL::HE; ++h) {
        const int e = min(tid + h * TL::NT, TL::EP - 1), ey = e / TL::ES, ez = min(e - ey * TL::ES, TL::EZ - 1);
        eoff[h] = (unsigned)((TL::flat ? 0 : wrapc(y0 - 4 + ey, P.ny)) * P.nz + wrapc(z0 - 4 + ez, P.nz));
    }
    TC er[TL::HE], em[TL::HE];
    auto fetch_plane = [&](int x, TC (&r)[TL::HE], TC (&m)[TL::HE]) {
        const size_t b = (size_t)wrap_x(x) * pl;
        const TS *rp = A.rho + b, *mp = A.mu + b;
#pragma unroll
        for (int h = 0; h < TL::HE; ++h) { r[h] = (TC)*lane_at(rp, eoff[h]); m[h] = (TC)*lane_at(mp, eoff[h]); }
    };
    auto store_plane = [&](int slot, const TC (&r)[TL::HE], const TC (&m)[TL::HE]) {
#pragma unroll
        for (int h = 0; h < TL::HE; ++h)
            if ((h + 1) * TL::NT <= TL::EP || tid + h * TL::NT < TL::EP) s_rm[slot][tid + h * TL::NT] = Pair<TC>{r[h], m[h]};
    };

    // the state before the step at this thread's node of plane x
    constexpr int NI = IN_P ? Q : kMom;
    TC next[NI];
    Nbr nb;
    if constexpr (IN_P) {
        nb = make_nbr(P, 0, y, z);
        if (NW) nb.sb[0] = nb.sb[2] = false;
    }
    const unsigned psite = IN_P || OUT_P ? pop_site(P, 0, y, z) : 0u;
    auto fetch_state = [&](int x) {
        const int xw = wrap_x(x);
        if constexpr (IN_P) {
            nb.site = (unsigned)xw * (unsigned)pl + psite;
            nb.ox[0] = (wrap_off(xw, -1, P.nx) - xw) * pl;
            nb.ox[2] = (wrap_off(xw, 1, P.nx) - xw) * pl;
#pragma unroll
            for (int q = 0; q < Q; ++q) next[q] = (TC)A.fin[pull_index(nb, (unsigned)P.N, q)];
        } else {
            const TC *b = ends ? A.ein + (size_t)xw * tiles * (2 * kMom * TL::TY) : A.min + (size_t)xw * kMom * pl;
            const size_t st = ends ? TL::TY : pl;   // uniform over a wave
#pragma unroll
            for (int k = 0; k < kMom; ++k) next[k] = *lane_at(b + k * st, site);
        }
    };

    {   // the first seven planes, all loads in flight at once
        TC r7[7][TL::HE], m7[7][TL::HE];
#pragma unroll
        for (int k = 0; k < 7; ++k) fetch_plane(xa - 4 + k, r7[k], m7[k]);
        if constexpr (!IN_P) fetch_state(xa - 1);
#pragma unroll
        for (int k = 0; k < 7; ++k) store_plane(k, r7[k], m7[k]);
    }
    fetch_plane(xa + 3, er, em);
    int s0 = 0;   // ring slot of plane x - 3
    const int one = z0 == zlast ? kMom * TL::TY : TL::NT;
    // a finished plane's edge columns, from LDS to memory
    auto flush_edges = [&](int xp) {
        static_assert(2 * kMom * TL::TY <= TL::NT, "one value per thread");
        TC *b = A.eout + ((size_t)xp * tiles + tile) * (2 * kMom * TL::TY);
        // a tile of one column keeps it as its first
        if (tid < 2 * kMom * TL::TY) *lane_at(b, (unsigned)tid) = s_edge[tid - (tid >= one ? kMom * TL::TY : 0)];
    };
    const int base = (TL::flat ? 0 : (ly + 3) * TL::ES) + lz + 3;

    // arrivals: fa[] of plane x (its c_x = 0 and c_x > 0 values; c_x < 0 follows with plane
    // x + 1), and the c_x > 0 values of plane x + 1
    TC fa[Q], fb[5];
    TC sv[2];   // bounced c_x < 0 arrivals (12, 14) of plane x
#pragma unroll
    for (int q = 0; q < Q; ++q) fa[q] = TC(0);
#pragma unroll
    for (int i = 0; i < 5; ++i) fb[i] = TC(0);
    sv[0] = sv[1] = TC(0);
    auto bounced = [&](int q) { return !NW && (cz(q) > 0 ? bb_lo : cz(q) < 0 ? bb_hi : false); };
    __syncthreads();

    for (int x = xa - 1; x <= xb; ++x) {
        // moments are loaded a plane ahead (past the chunk wrapped, and not used); the
        // populations of a run's first step at the start of their own plane, behind the
        // stencils, which keeps 19 registers free and a second workgroup on the CU
        TC m[Q];
        if constexpr (IN_P) {
            fetch_state(x);
        } else {
#pragma unroll
            for (int k = 0; k < kMom; ++k) m[mom_row(k)] = next[k];
            fetch_state(x + 1);
        }
        if (x > xa + 1) flush_edges(x - 2);
        TC out[Q];
        if (fluid) {
            int slot[7];
#pragma unroll
            for (int d = 0; d < 7; ++d) slot[d] = s0 + d >= 7 ? s0 + d - 7 : s0 + d;
            const RingStencil<TC, TL> st{s_rm, slot, base};
            TC gr[3], gm[3], u[3];
            st.grad(gr, gm);
            if constexpr (IN_P) moments(next, m);
            const TC r = st.at(0, 0, 0).r, third = TC(1.0 / 3.0);
            const TC Fx = gr[0] * third - gm[0] * r, Fy = gr[1] * third - gm[1] * r, Fz = gr[2] * third - gm[2] * r;
            if (FC != kPlain && P.qp_on) {
                TC qp[Q];
                qp_terms(gr[0], gr[1], gr[2], (TC)P.K1, (TC)P.K2, qp);
                collide_moments<TC, true, FC == kGuo>(m, r, Fx, Fy, Fz, rates<TC>(P), qp, out, u);
            } else {
                collide_moments<TC, true, FC == kGuo>(m, r, Fx, Fy, Fz, rates<TC>(P), (const TC *)nullptr, out, u);
            }
            if (post) {
#pragma unroll
                for (int q = 3; q < Q; ++q) s_mail[q - 3][pos] = out[q];
            }
            if (DIAG && own && x >= xa && x < xb) {
                const size_t I = (size_t)x * pl + node, N = (size_t)P.N;
                if (A.uout) {
                    const TC t9[9] = {u[0], u[1], u[2], gm[0], gm[1], gm[2], gr[0], gr[1], gr[2]};
#pragma unroll
                    for (int a = 0; a < 9; ++a) A.uout[a * N + I] = (TS)t9[a];
                }
                if (A.mv) {
                    const TC h = TC(0.5) / r;
                    A.mv[I] = (TS)(u[0] + Fx * h);
                    A.mv[N + I] = (TS)(u[1] + Fy * h);
                    A.mv[2 * N + I] = (TS)(u[2] + Fz * h);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < Q; ++q) out[q] = TC(0);
        }
        if constexpr (OUT_P) {
            // solid nodes' own slots read zero after a step, stored with their row
            if (own && x >= xa && x < xb) {
                const unsigned b = (unsigned)x * (unsigned)pl + psite;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    // whole lines in the tiled layout; elsewhere the L2 has to merge them
                    // (150x117x83: 136 us a step with streaming stores, 79 without)
                    TF *p = &A.fout[(unsigned)q * (unsigned)P.N + b];
                    if (P.tiled) __builtin_nontemporal_store((TF)out[q], p);
                    else *p = (TF)out[q];
                }
            }
        }
        __syncthreads();                       // mailbox of plane x posted, plane x - 3 no longer read
        store_plane(s0, er, em);               // plane x + 4
        fetch_plane(x + 5, er, em);
        s0 = s0 == 6 ? 0 : s0 + 1;
        if (inner) {
            // what arrives along q: the neighbour's value, or the node's own along opp(q)
            // where the neighbour is solid (half-way bounce-back)
            auto kept = [&](int q) { return s_mail[q - 3][pos]; };
            auto mail = [&](int q) {
                const int from = (q - 3) * TL::NN + pos - (TL::flat ? 0 : cy(q) * TL::RZ) - cz(q);
                return (&s_mail[0][0])[bounced(q) && cx(q) == 0 ? (opp(q) - 3) * TL::NN + pos : from];
            };
            // c_x < 0 completes plane x - 1
            fa[2] = out[2];
            fa[8] = mail(8);
            fa[10] = mail(10);
            fa[12] = bounced(12) ? sv[0] : mail(12);
            fa[14] = bounced(14) ? sv[1] : mail(14);
            if (x > xa && own) {
                TC n[Q];
                moments(fa, n);
                const int xp = x - 1;
                TC *b = A.mout + (size_t)xp * kMom * pl;
#pragma unroll
                for (int k = 0; k < kMom; ++k) {
                    const TC v = fluid ? n[mom_row(k)] : TC(0);
                    __builtin_nontemporal_store(v, lane_at(b + (size_t)k * pl, site));
                    if (edge) s_edge[k * TL::TY + eslot] = v;
                }
                if (fluid) {
                    // FP32 arithmetic on FP64 storage: the density is summed in its own
                    // precision from the sums of two and four that the moments form (all 19
                    // terms in FP64: steps 3 % slower at 20 us, 1 to 2 % at 90 us)
                    TS d = (TS)n[0];
                    if constexpr (sizeof(TS) > sizeof(TC)) {
                        auto pair = [&](int q) { return fa[q] + fa[q + 1]; };
                        auto four = [&](int q) { return (fa[q] + fa[q + 3]) + (fa[q + 1] + fa[q + 2]); };
                        d = (TS)fa[0] + (((TS)pair(1) + (TS)pair(3)) + (TS)pair(5)) + (((TS)four(7) + (TS)four(11)) + (TS)four(15));
                    }
                    *lane_at(A.rho_out + (size_t)xp * pl, node) = d;
                }
            }
            // keeps the other arrivals out of the registers that the moments need
            __builtin_amdgcn_sched_barrier(0);
            // c_x = 0 and the c_x > 0 values of plane x - 1 make plane x
            fa[0] = out[0];
            fa[1] = fb[0];
            fa[7] = fb[1];
            fa[9] = fb[2];
            fa[11] = bounced(11) ? kept(opp(11)) : fb[3];
            fa[13] = bounced(13) ? kept(opp(13)) : fb[4];
#pragma unroll
            for (int q = 3; q < Q; ++q)
                if (cx(q) == 0) fa[q] = mail(q);
            fb[0] = out[1];
            fb[1] = mail(7);
            fb[2] = mail(9);
            fb[3] = mail(11);
            fb[4] = mail(13);
            if (!NW) {
                sv[0] = kept(opp(12));
                sv[1] = kept(opp(14));
            }
        }
        __syncthreads();                       // mailbox free, ring plane x + 4 and edge columns in place
    }
    flush_edges(xb - 1);
}

using TileRow = Tile<1, 192>;
using TileBox = Tile<12, 32>;

template <class TF, class TS, class TC>
hipError_t launch_form(cpmp_ctx *c, bool in_p, bool out_p, void *mv, TS *uout) {
    const DevParams &P = c->dp;
    StepArgs<TF, TS, TC> a;
    // moments alternate between c->mom and the population set that is not current; the
    // populations of the last step replace the current ones, which nothing reads any
    // more unless this step starts from them
    const void *in = c->mom_at == 1 ? c->mom : c->f[c->cur ^ 1];
    void *out = c->mom_at == 1 ? c->f[c->cur ^ 1] : c->mom;
    a.fin = (const TF *)c->f[c->cur];
    a.fout = (TF *)c->f[in_p ? c->cur ^ 1 : c->cur];
    a.min = (const TC *)in;
    a.mout = (TC *)out;
    a.ein = a.min + (size_t)kMom * c->N;   // the edge columns follow the moments
    a.eout = a.mout + (size_t)kMom * c->N;
    a.rho = (const TS *)c->rho;
    a.mu = (const TS *)c->mu;
    a.rho_out = (TS *)c->rho_next;
    a.mv = (TS *)mv;
    a.uout = uout;
    const bool nw = P.lo == 0 && P.hi == 0, diag = mv || uout;
    const int fc = P.forcing == 1 ? kGuo : P.qp_on ? kQp : kPlain;
    auto go = [&](auto tl, auto ip, auto op, auto dg) {
        using TL = decltype(tl);
        a.ntz = (P.nz + TL::TZ - 1) / TL::TZ;
        a.nty = (P.ny + TL::TY - 1) / TL::TY;
        a.xc = c->step_chunk;
        const dim3 grid((unsigned)(a.ntz * a.nty * ((P.nx + a.xc - 1) / a.xc)));
        auto run = [&](auto nw_t, auto fc_t) {
            hipLaunchKernelGGL((k_moment_step<TF, TS, TC, TL, decltype(ip)::value, decltype(op)::value, decltype(dg)::value,
                                              decltype(nw_t)::value, decltype(fc_t)::value>),
                               grid, dim3(TL::NT), 0, c->stream, P, a);
        };
        auto force = [&](auto nw_t) {
            if (fc == kPlain) run(nw_t, std::integral_constant<int, kPlain>{});
            else if (fc == kQp) run(nw_t, std::integral_constant<int, kQp>{});
            else run(nw_t, std::integral_constant<int, kGuo>{});
        };
        if (nw) force(std::true_type{});
        else force(std::false_type{});
        return hipGetLastError();
    };
    using Y = std::true_type;
    using N = std::false_type;
    auto io = [&](auto tl) {
        if (in_p) return out_p ? go(tl, Y{}, Y{}, Y{}) : go(tl, Y{}, N{}, Y{});
        if (out_p) return go(tl, N{}, Y{}, Y{});
        return diag ? go(tl, N{}, N{}, Y{}) : go(tl, N{}, N{}, N{});
    };
    return P.ny == 1 ? io(TileRow{}) : io(TileBox{});
}

}  // namespace

// Planes per workgroup.  A chunk of n planes collides n + 2 and loads 7 planes of rho and
// mu before its first (together about 4 planes' time), and the launch takes as many
// rounds as its workgroups need places on the device (2 per CU with 4-byte arithmetic,
// 1 with 8-byte: LDS; twice as many of the one-row tiles' 4 waves), so the chunk length that
// minimises rounds * (n + 4) is taken.  In a sweep over 1..128 planes on 14 lattices in three
// forms, kept under profiles/, it is the best in 34 of 42 runs and within 9 % of it in all (us
// per step: 64^3 FP64 4: 32.7, 2: 43.5, 8: 46.6; 128^3 FP32 12: 77, 4: 90, 24: 118; 256^3 FP32
// 32: 491, 16: 520, 43: 562; 3001x1x501 FP64 18: 101, 8: 112, 32: 142).  CPMP_XC overrides.
int moment_chunk(int nx, int ny, int nz, int form) {
    if (const char *e = std::getenv("CPMP_XC")) {
        const int v = std::atoi(e);
        if (v >= 1 && v <= 1024) return v;
    }
    const bool flat = ny == 1;
    const int ty = 12;
    const long long tiles = flat ? (nz + 191) / 192 : (long long)((ny + ty - 1) / ty) * ((nz + 31) / 32);
    const long long places = (form == CPMP_FORM_FP64 ? 256 : 512) * (flat ? 2 : 1);
    int best = 32;
    double cost = 1e300;
    for (int n = 1; n <= 128; ++n) {
        const long long wg = tiles * ((nx + n - 1) / n);
        const double rounds = (double)((wg + places - 1) / places);
        const double t = rounds * (n + 4);
        if (t < cost) { cost = t; best = n; }
    }
    return best;
}

// values of a moment set: 12 per node and the edge columns of every tile
size_t moment_bytes(int nx, int ny, int nz, int form) {
    const int ty = ny == 1 ? TileRow::TY : TileBox::TY, tz = ny == 1 ? TileRow::TZ : TileBox::TZ;
    const size_t tiles = (size_t)((ny + ty - 1) / ty) * ((nz + tz - 1) / tz);
    return (size_t)nx * kMom * ((size_t)ny * nz + tiles * 2 * ty) * (form == CPMP_FORM_FP64 ? 8 : 4);
}

hipError_t launch_moment_step(cpmp_ctx *c, bool out_pops, bool want_mv, void *uout) {
    void *mv = want_mv ? c->mv : nullptr;
    const bool in_pops = c->mom_at == 0;
    hipError_t e = hipErrorInvalidValue;
    switch (c->form) {
    case CPMP_FORM_FP64: e = launch_form<double, double, double>(c, in_pops, out_pops, mv, (double *)uout); break;
    case CPMP_FORM_FP32: e = launch_form<float, float, float>(c, in_pops, out_pops, mv, (float *)uout); break;
    case CPMP_FORM_FP32A: e = launch_form<double, double, float>(c, in_pops, out_pops, mv, (double *)uout); break;
    }
    if (in_pops && out_pops) c->cur ^= 1;
    c->mom_at = c->mom_at == 1 ? 2 : 1;
    return e;
}

}  // namespace cpmp
