// mu.hip -- the chemical potential of the step.
#include "internal.h"
#include "lbm_math.h"
#include "device_common.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace cpmp {

namespace {

// ---------------------------------------------------------------------------
// Chemical potential (ChemPotential, FluidCuda.cu:444-463):
//   mu = K^2 mu_eos(clamp(rho)) - Ka * Laplacian(rho).
// FP64 form: all in FP64, the Laplacian as the reference writes it.
// FP32 storage forms (mu is stored in FP32): the Laplacian is summed over the
// differences rho_k - rho_0 (its coefficients sum to zero, so this is the same
// operator, and the differences carry no cancellation), and mu_eos is evaluated
// in FP32 with the hardware log2 and reciprocal (relative error of a few ulp,
// below the FP32 rounding of the stored mu).

// mu_eos in FP32 with v_log_f32 / v_rcp_f32; same closed forms as mu_eos_t
__device__ __forceinline__ float ln_hw(float x) { return __builtin_amdgcn_logf(x) * 0.693147180559945f; }
__device__ __forceinline__ float rcp_hw(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float mu_eos_fast(int eos, int form, float A, float B, float T, float d) {
    const float s2 = 1.41421356f;
    const float bd = B * d, rom = rcp_hw(1.0f - bd);
    if (form == 1 || eos == EOS_PRW || eos == EOS_PRM) {
        return T * ln_hw(d * rom) - A * rcp_hw(s2 * 2.0f * B) * ln_hw((s2 - 1.0f + bd) * rcp_hw(s2 + 1.0f - bd))
               + T * rom - A * d * rcp_hw(1.0f + bd * 2.0f - bd * bd);
    }
    if (eos == EOS_VDW) return T * ln_hw(d * rom) + T * rom - 2.0f * A * d;
    if (eos == EOS_RKE || eos == EOS_RKS) {
        const float op = 1.0f + bd;
        return T * ln_hw(d * rom) + T * rom - A * rcp_hw(B) * ln_hw(op) - A * d * rcp_hw(op);
    }
    return T * (ln_hw(d) + (8.0f * bd - 9.0f * bd * bd + 3.0f * bd * bd * bd) * rom * rom * rom) - 2.0f * A * d;
}

// mu_eos in FP64 with ln64 and one reciprocal for all the quotients of an EOS (the closed
// forms of mu_eos_t; for Peng-Robinson (sqrt2 - 1 + bd)(sqrt2 + 1 - bd) = 1 + 2 bd - bd^2,
// so the quotient in its second logarithm is (sqrt2 - 1 + bd)^2 over the same denominator)
// TIGHT: ln64's
template <bool TIGHT>
__device__ __forceinline__ double mu_eos_fast(const DevParams &P, double d) {
    auto ln = [](double x) { return ln64<TIGHT>(x); };
    if (d > 9.7) d = 9.7 + (d - 9.7) * recip64(1.0 + (d - 9.7) * 1.5);   // clamp_rho
    const double A = P.A, T = P.T, bd = P.B * d, om = 1.0 - bd;
    double mu;
    if (P.mu_form == 1 || P.eos == EOS_PRW || P.eos == EOS_PRM) {
        const double q = 1.0 + 2.0 * bd - bd * bd, u = kSqrt2 - 1.0 + bd, r = recip64(om * q), rom = r * q, rq = r * om;
        mu = T * ln(d * rom) - P.AoPr * ln(u * u * rq) + T * rom - A * d * rq;
    } else if (P.eos == EOS_RKE || P.eos == EOS_RKS) {
        const double op = 1.0 + bd, r = recip64(om * op), rom = r * op;
        mu = T * ln(d * rom) + T * rom - P.AoB * ln(op) - A * d * (r * om);
    } else {
        const double rom = recip64(om);
        mu = P.eos == EOS_VDW ? T * ln(d * rom) + T * rom - 2.0 * A * d
                              : T * (ln(d) + (8.0 * bd - 9.0 * bd * bd + 3.0 * bd * bd * bd) * (rom * rom * rom)) - 2.0 * A * d;
    }
    return om == 0.0 ? T * __builtin_inf() : mu;   // at the densest packing, where recip64 has no value
}

// FP32 mu of an interface node from its FP32 Laplacian term Ka * lap: the EOS part
// in FP64, rounded once
__device__ __forceinline__ float mu_band(const DevParams &P, float d, float kal) {
    return (float)(P.K2s * mu_eos_fast<false>(P, (double)d) - (double)kal);
}
__device__ __forceinline__ bool in_band(const DevParams &P, float d) { return d > P.band_lo && d < P.band_hi; }

// mu at one fluid node; get(dx, dy, dz) returns rho at the offset node (along one axis).
// FP32: interface nodes (in_band) get the EOS part in FP64.
template <class TS, class Get>
__device__ __forceinline__ TS mu_node(const DevParams &P, Get get) {
    if constexpr (sizeof(TS) == 8) {
        const double d = get(0, 0, 0);
        double kal;
        if (P.lap_points == 7) {   // GradD7, Common.h:243-246
            auto ax = [&](int ux, int uy, int uz) {
                return 2 * get(-3 * ux, -3 * uy, -3 * uz) - 27 * get(-2 * ux, -2 * uy, -2 * uz)
                       + 270 * get(-ux, -uy, -uz) + 270 * get(ux, uy, uz) - 27 * get(2 * ux, 2 * uy, 2 * uz)
                       + 2 * get(3 * ux, 3 * uy, 3 * uz);
            };
            kal = P.Ka * (-d * 490 * 3 + ax(1, 0, 0) + ax(0, 1, 0) + ax(0, 0, 1)) / 180;
        } else {                   // GradD5, Common.h:189-192
            auto ax = [&](int ux, int uy, int uz) {
                return -get(-2 * ux, -2 * uy, -2 * uz) + get(-ux, -uy, -uz) * 16 + get(ux, uy, uz) * 16
                       - get(2 * ux, 2 * uy, 2 * uz);
            };
            kal = P.Ka * ((-d * 90 + ax(1, 0, 0) + ax(0, 1, 0) + ax(0, 0, 1)) / 12);
        }
        return P.K2s * mu_eos_fast<true>(P, d) - kal;
    } else {
        const float d = get(0, 0, 0);
        auto df = [&](int dx, int dy, int dz) { return (float)get(dx, dy, dz) - d; };
        float lap;
        if (P.lap_points == 7) {
            auto ax = [&](int ux, int uy, int uz) {
                return 2.0f * (df(-3 * ux, -3 * uy, -3 * uz) + df(3 * ux, 3 * uy, 3 * uz))
                       - 27.0f * (df(-2 * ux, -2 * uy, -2 * uz) + df(2 * ux, 2 * uy, 2 * uz))
                       + 270.0f * (df(-ux, -uy, -uz) + df(ux, uy, uz));
            };
            lap = (ax(1, 0, 0) + ax(0, 1, 0) + ax(0, 0, 1)) * (1.0f / 180.0f);
        } else {
            auto ax = [&](int ux, int uy, int uz) {
                return 16.0f * (df(-ux, -uy, -uz) + df(ux, uy, uz)) - (df(-2 * ux, -2 * uy, -2 * uz) + df(2 * ux, 2 * uy, 2 * uz));
            };
            lap = (ax(1, 0, 0) + ax(0, 1, 0) + ax(0, 0, 1)) * (1.0f / 12.0f);
        }
        const float kal = (float)P.Ka * lap;
        if (in_band(P, d)) return mu_band(P, d, kal);
        const float dc = d > 9.7f ? 9.7f + (d - 9.7f) * rcp_hw(1.0f + (d - 9.7f) * 1.5f) : d;   // clamp_rho
        const float m = mu_eos_fast(P.eos, P.mu_form, (float)P.A, (float)P.B, (float)P.T, dc);
        return (float)P.K2s * m - kal;
    }
}

// One thread per column (y, z) of the plane, marching along x over xc planes: the 2H + 1
// values along x stay in registers, the in-plane neighbours are read through the L1 (their
// lines are the ones neighbouring lanes and waves read), each one plane ahead.  Columns
// are numbered y * nz + z, so every lattice, one row in y included, fills its waves.
// Bound: latency and VALU (256^3 FP64 129 us against 56 us of traffic; FP32 75 us, 43 us of it
// VALU).  The LDS march below took 112 us in FP64 with a list of interface nodes apart (152 with
// the library's logarithm), 36 us against 14 on 3001 x 1 x 501 and 17 against 15 on
// 150 x 117 x 83; two nodes per thread, read as pairs, made the FP32 step 1 % slower.
// H: radius of the Laplacian, 2 (5 points) or 3 (7 points).  rho_solid (if given) receives
// the wall density of solid nodes, rho_copy (if given) the density of every node.
template <class TS, int H>
__global__ void __launch_bounds__(TPB) k_mu_columns(const DevParams P, const TS *__restrict__ rho, TS *__restrict__ mu,
                                                    TS *__restrict__ rho_solid, TS *__restrict__ rho_copy, int xc, int ncb) {
    const int pl = P.ny * P.nz;
    int t = blockIdx.x;
    {   // each XCD takes a contiguous range of workgroups, neighbours sharing an L2
        const int n = gridDim.x, k = t & 7;
        t = k * (n >> 3) + min(k, n & 7) + (t >> 3);
    }
    const int xa = t / ncb * xc, xb = min(xa + xc, P.nx);
    const int j = t % ncb * TPB + (int)threadIdx.x;
    if (j >= pl) return;
    const int y = j / P.nz, z = j - y * P.nz;
    const bool solid = is_solid(P, z);
    constexpr unsigned SZ = sizeof(TS);
    const unsigned jb = (unsigned)j * SZ;
    unsigned oy[2 * H], oz[2 * H];   // neighbours at distance -H..-1, 1..H
#pragma unroll
    for (int i = 0; i < 2 * H; ++i) {
        const int d = i < H ? i - H : i - H + 1;
        oy[i] = (unsigned)(wrap_off(y, d, P.ny) * P.nz + z) * SZ;
        oz[i] = (unsigned)(y * P.nz + wrap_off(z, d, P.nz)) * SZ;
    }
    auto plane = [&](int x) {
        x = P.nx >= 8 ? (x < 0 ? x + P.nx : (x >= P.nx ? x - P.nx : x)) : wrapc(x, P.nx);
        return rho + (size_t)x * pl;
    };
    TS xv[2 * H + 1], ya[2 * H], za[2 * H];
#pragma unroll
    for (int i = 0; i <= 2 * H; ++i) xv[i] = *lane_bytes(plane(xa - H + i), jb);
    {
        const TS *r = plane(xa);
#pragma unroll
        for (int i = 0; i < 2 * H; ++i) { ya[i] = *lane_bytes(r, oy[i]); za[i] = *lane_bytes(r, oz[i]); }
    }
    for (int x = xa; x < xb; ++x) {
        // the next plane's values; past the chunk the loads are not used
        const unsigned jo = in_loop(jb);
        const TS xn = *lane_bytes(plane(x + H + 1), jo);
        TS yn[2 * H], zn[2 * H];
        const TS *r = plane(x + 1);
#pragma unroll
        for (int i = 0; i < 2 * H; ++i) { yn[i] = *lane_bytes(r, in_loop(oy[i])); zn[i] = *lane_bytes(r, in_loop(oz[i])); }
        const size_t I = (size_t)x * pl;
        if (!solid)
            *lane_bytes(mu + I, jo) = mu_node<TS>(P, [&](int dx, int dy, int dz) {
                return dy ? ya[dy < 0 ? dy + H : dy + H - 1] : dz ? za[dz < 0 ? dz + H : dz + H - 1] : xv[dx + H];
            });
        else if (rho_solid) *lane_bytes(rho_solid + I, jo) = xv[H];
        if (rho_copy) *lane_bytes(rho_copy + I, jo) = xv[H];
#pragma unroll
        for (int i = 0; i < 2 * H; ++i) { xv[i] = xv[i + 1]; ya[i] = yn[i]; za[i] = zn[i]; }
        xv[2 * H] = xn;
    }
}

// The same as a march over 8 x 32 tiles: rho of planes x-H..x+H with an in-plane halo of H
// sits in an LDS ring of 2H + 2 planes (the extra slot receives the plane entering the ring
// while slower waves still read the one that left it, so one barrier a plane suffices), and
// each rho value is fetched from memory about once per tile.  Two planes are in flight.
// For large lattices of 4-byte densities, where the columns' reads past the L1 bound them
// (512x512x256: 265 us, 209 here: 2.5 TB/s of the 536 MB it cannot do without).
constexpr int kMuT = kTileY * kTileZ;
template <class TS, int H>
__global__ void __launch_bounds__(kMuT) k_mu_march(const DevParams P, const TS *__restrict__ rho, TS *__restrict__ mu,
                                                   TS *__restrict__ rho_solid, TS *__restrict__ rho_copy, int xc, int ntz,
                                                   int nty) {
    constexpr int R = 2 * H + 2, LZ = kTileZ + 2 * H, LP = (kTileY + 2 * H) * LZ;
    __shared__ TS s_rho[R][LP];
    int t = blockIdx.x;
    {   // each XCD takes a contiguous range of tiles, neighbours sharing an L2
        const int n = gridDim.x, k = t & 7;
        t = k * (n >> 3) + min(k, n & 7) + (t >> 3);
    }
    const int tzi = t % ntz;
    t /= ntz;
    const int y0 = t % nty * kTileY, z0 = tzi * kTileZ;
    const int xa = t / nty * xc, xb = min(xa + xc, P.nx);
    const int tid = threadIdx.x, ty = tid / kTileZ, tz = tid % kTileZ, y = y0 + ty, z = z0 + tz;
    const bool inr = y < P.ny && z < P.nz, solid = is_solid(P, z);
    const int pl = P.ny * P.nz;
    constexpr int HE = (LP + kMuT - 1) / kMuT;
    unsigned hoff[HE];
#pragma unroll
    for (int h = 0; h < HE; ++h) {
        const int e = min(tid + h * kMuT, LP - 1), ly = e / LZ, lz = e - ly * LZ;
        hoff[h] = (unsigned)(wrapc(y0 - H + ly, P.ny) * P.nz + wrapc(z0 - H + lz, P.nz)) * (unsigned)sizeof(TS);
    }
    auto fetch = [&](int x, TS (&v)[HE]) {   // past the chunk wrapped, and not used
        x = P.nx >= 8 ? (x < 0 ? x + P.nx : (x >= P.nx ? x - P.nx : x)) : wrapc(x, P.nx);
        const TS *r = rho + (size_t)x * pl;
#pragma unroll
        for (int h = 0; h < HE; ++h) v[h] = *lane_bytes(r, hoff[h]);
    };
    auto store = [&](int slot, const TS (&v)[HE]) {
#pragma unroll
        for (int h = 0; h < HE; ++h)
            if ((h + 1) * kMuT <= LP || tid + h * kMuT < LP) s_rho[slot][tid + h * kMuT] = v[h];
    };
    TS va[HE], vb[HE];
    {
        TS v[2 * H][HE];
#pragma unroll
        for (int k = 0; k < 2 * H; ++k) fetch(xa - H + k, v[k]);
#pragma unroll
        for (int k = 0; k < 2 * H; ++k) store(k, v[k]);
    }
    fetch(xa + H, va);
    fetch(xa + H + 1, vb);
    const int base = (ty + H) * LZ + tz + H;
    const unsigned jb = (unsigned)(inr ? y * P.nz + z : 0) * (unsigned)sizeof(TS);
    int s0 = 0;   // ring slot of plane x - H
    auto step = [&](int x, TS (&v)[HE]) {
        int slot[2 * H + 1];
#pragma unroll
        for (int d = 0; d <= 2 * H; ++d) slot[d] = s0 + d >= R ? s0 + d - R : s0 + d;
        store(slot[2 * H], v);   // plane x + H
        __syncthreads();
        fetch(x + H + 2, v);
        if (inr) {
            const size_t I = (size_t)x * pl;
            const TS d = s_rho[slot[H]][base];
            if (!solid)
                *lane_bytes(mu + I, jb) = mu_node<TS>(P, [&](int dx, int dy, int dz) { return s_rho[slot[dx + H]][base + dy * LZ + dz]; });
            else if (rho_solid) *lane_bytes(rho_solid + I, jb) = d;
            if (rho_copy) *lane_bytes(rho_copy + I, jb) = d;
        }
        s0 = s0 + 1 == R ? 0 : s0 + 1;
    };
    int x = xa;
    for (; x + 1 < xb; x += 2) {
        step(x, va);
        step(x + 1, vb);
    }
    if (x < xb) step(x, va);
}

}  // namespace

// x planes per workgroup of k_mu_march, 0: k_mu_columns.  The march from 6 million nodes of
// 4-byte densities on, where the tiles fill: us per launch, columns against march, FP32:
// 128^3 17.7 / 18.0, 1024x64x64 23 / 24, 192^3 42 / 38, 256^3 75 / 66, 384x384x256 150 / 127,
// 512x512x256 265 / 209 (FP16 265 / 216); tiles of one row (3001x1x501) 14 / 36.  Chunks of 32,
// 16 or 8 planes: 256^3 73 / 66 / 70, 512x512x256 209 / 222 / 250, 384x384x256 135 / 127 / 142,
// 192^3 45 / 42 / 38.  CPMP_MU=columns or =march (chunks of CPMP_XC, else 8) overrides.
int mu_march_chunk(int nx, int ny, int nz, int form) {
    if (fp64_storage(form)) return 0;
    const long long tiles = (long long)((ny + kTileY - 1) / kTileY) * ((nz + kTileZ - 1) / kTileZ);
    if (const char *e = std::getenv("CPMP_MU")) {
        const char *x = std::getenv("CPMP_XC");
        if (std::strcmp(e, "columns") == 0) return 0;
        if (std::strcmp(e, "march") == 0) return x ? std::min(std::max(std::atoi(x), 1), 1024) : 8;
    }
    if ((long long)nx * ny * nz < 6000000 || 10ll * ny * nz < 7 * tiles * kTileY * kTileZ) return 0;
    return (nx + 31) / 32 * tiles >= 8192 ? 32 : (nx + 15) / 16 * tiles >= 4096 ? 16 : 8;
}

// x planes per workgroup of k_mu_columns: enough workgroups for 8 waves per SIMD, at most 16
// (256^3 FP32 step 525 us, with 32 planes 530)
template <class TS>
static hipError_t launch(cpmp_ctx *c, void *rho_copy) {
    if constexpr (sizeof(TS) == 4) {
        if (c->mu_chunk > 0) {
            const int xc = c->mu_chunk, ntz = (c->p.nz + kTileZ - 1) / kTileZ, nty = (c->p.ny + kTileY - 1) / kTileY;
            const dim3 grid((unsigned)(ntz * nty * ((c->p.nx + xc - 1) / xc)));
            auto go = [&](auto h) {
                hipLaunchKernelGGL((k_mu_march<TS, decltype(h)::value>), grid, dim3(kMuT), 0, c->stream, c->dp, (const TS *)c->rho,
                                   (TS *)c->mu, (TS *)c->rho_next, (TS *)rho_copy, xc, ntz, nty);
            };
            if (c->dp.lap_points == 7) go(std::integral_constant<int, 3>{});
            else go(std::integral_constant<int, 2>{});
            return hipGetLastError();
        }
    }
    const int ncb = (int)blocks_for((long long)c->p.ny * c->p.nz);
    const int xc = std::max(1, std::min(16, c->p.nx * ncb / 2048));
    const dim3 grid((unsigned)(ncb * ((c->p.nx + xc - 1) / xc)));
    // double-buffered density: the solid values follow the step
    if (c->dp.lap_points == 7)
        hipLaunchKernelGGL((k_mu_columns<TS, 3>), grid, dim3(TPB), 0, c->stream, c->dp, (const TS *)c->rho, (TS *)c->mu,
                           (TS *)c->rho_next, (TS *)rho_copy, xc, ncb);
    else
        hipLaunchKernelGGL((k_mu_columns<TS, 2>), grid, dim3(TPB), 0, c->stream, c->dp, (const TS *)c->rho, (TS *)c->mu,
                           (TS *)c->rho_next, (TS *)rho_copy, xc, ncb);
    return hipGetLastError();
}

hipError_t launch_mu(cpmp_ctx *c, void *rho_copy) {
    return fp64_storage(c->form) ? launch<double>(c, rho_copy) : launch<float>(c, rho_copy);
}

}  // namespace cpmp
