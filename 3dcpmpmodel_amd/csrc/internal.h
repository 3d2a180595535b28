// internal.h -- context and launcher declarations shared by the library's
// translation units.  Not part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <string>

#include "../../include/cpmp.h"

namespace cpmp {

// Parameters as the kernels see them (one kernel argument; replaces the
// __constant__ symbols of FluidCuda.cu:67 and Common.h:96-153).
struct DevParams {
    int nx, ny, nz;
    int lo, hi;                 // solid layers at the z ends
    long long N;
    int eos, mu_form, lap_points, wall_scheme;
    int qp_on;                  // K1 or K2 non-zero
    double A, B, T, K2s, Ka;    // K2s = K*K
    double AoB, AoPr;           // A / B, A / (2 sqrt(2) B)
    double K1, K2;
    double ts[19];
    float tsf[19];              // ts in FP32 for the FP32 arithmetic forms
    double rho0;                // FP16 shift density
    int tiled, nty, ntz;        // tile-contiguous population sites (pop_site), tile counts in y, z
    int xc;                     // x planes per workgroup of the march kernels
    int unit_rates;             // the rates of rows 0, 1, 3, 5, 7, 10, 12, 16-18 are all 1 (reference set)
    int forcing;                // 0 exact-difference force term, 1 Guo
    // FP32 storage forms: fluid nodes with a density strictly inside (band_lo, band_hi)
    // -- the interface: between the Maxwell gas and liquid densities, less 2 % of their
    // gap at each end -- get the EOS chemical potential in FP64; empty (lo > hi) without
    // a two-phase region
    float band_lo, band_hi;
};

enum Kern { KW = CPMP_K_WALL, KM = CPMP_K_MU, KC = CPMP_K_COLLIDE, KR = CPMP_K_MACRO };

struct Timers {
    bool on = false;
    hipEvent_t ev[2 * CPMP_K_COUNT * 8] = {};
    double ms[CPMP_K_COUNT] = {};
    long long count[CPMP_K_COUNT] = {};
};

}  // namespace cpmp

struct cpmp_ctx {
    cpmp_params p;
    cpmp::DevParams dp;
    int64_t N = 0, NXY = 0;
    int form = 0;
    size_t pop_bytes = 0;       // bytes of one population value
    size_t scal_bytes = 0;      // bytes of one rho/mu value
    hipStream_t stream = nullptr;
    char *block = nullptr;      // the allocation that holds every buffer below
    bool open = false;          // counted among the device's contexts
    void *f[2] = {nullptr, nullptr};
    int cur = 0;
    void *rho = nullptr, *mu = nullptr;
    // rho_next: the density after the step, on lattices on moments and where the march sums
    // it; the FP16 form's previous density.  rbuf, cbuf: tile rings and chunk partial planes
    // of the march on exactly tiled lattices
    void *rho_next = nullptr, *rbuf = nullptr, *cbuf = nullptr;
    bool collide_v1 = false;    // one-thread-per-node collide (node_collide)
    bool moments = false;       // runs of steps carry 13 moments per node (moment_path)
    int step_chunk = 0;         // x planes per workgroup of the moment step
    int mu_chunk = 0;           // x planes per workgroup of the chemical-potential march (0: by columns)
    // a moment set; the population set that is not current holds the other.  mom_at: which
    // one holds the moments of the current populations (0 none, 1 mom, 2 the population set)
    void *mom = nullptr;
    int mom_at = 0;
    size_t fuse_bytes = 0;
    void *mv = nullptr;         // 3*N values of the scalar type, MV of the last step
    double *mu_w = nullptr;     // 2*NXY: bottom then top
    double *red = nullptr;      // reduction partials
    double *staging = nullptr;  // N doubles
    int64_t step = 0;
    bool mv_valid = false;
    cpmp::Timers *timers = nullptr;
};

namespace cpmp {

int set_error(int code, const char *fmt, ...);

// launchers (kernels.hip); all enqueue on ctx->stream
hipError_t launch_wall(cpmp_ctx *c);
// rho_copy (optional): receives a copy of rho as the kernel reads it (the adjoint's tape)
hipError_t launch_mu(cpmp_ctx *c, void *rho_copy = nullptr);
bool density_fused(const cpmp_ctx *c);
bool fuse_geometry(int nx, int ny, int nz, int xc, size_t *ring_elems, size_t *chunk_elems);
// forms whose populations, rho and mu are stored in FP64 (FP64, FP32A)
inline bool fp64_storage(int form) { return form == CPMP_FORM_FP64 || form == CPMP_FORM_FP32A; }
int mu_march_chunk(int nx, int ny, int nz, int form);
// x planes per march workgroup for a lattice and storage form (CPMP_XC overrides)
int march_chunk(int nx, int ny, int nz, int form);
// the one-thread-per-node collide instead of the x march (CPMP_COLLIDE=v1 / march
// override): FP64 lattices too small for 2048 march workgroups of 2 planes
bool node_collide(int nx, int ny, int nz, int form);
// runs of steps hand 12 moments per node and the density from one step to the next
// (the reference's unit rates; not the FP16 form, whose state is defined by its stored
// populations).  Lattices below 80 000 nodes keep the population kernels: there a step is
// a few launches' latency, and the march takes longer from end to end than a launch of one
// thread per node (us per step, population kernels against moments: 32^3 FP64 15.8 / 19.3,
// 48x40x36 FP32 23.8 / 26.0, FP64 26.8 / 29.2; 44x45x46 FP32 22.3 / 20.7, FP64 26.3 / 23.5).
// One-row FP32 lattices take the moments at any size: the population march of this form
// fills 1 of 8 lanes there (300x1x100 27.5 / 17.5).  Some lattices of 1 plane or 2 to 4 rows
// keep the populations at any size (thin_lattice).  CPMP_COLLIDE=moments takes the moments
// on a lattice of any size; CPMP_COLLIDE=v1 or march and, on lattices the march tiles cover,
// CPMP_FUSE=0 keep the populations.  The moment sets alternate with the population sets, so
// a lattice whose moment set is larger (edge columns of tiles a few nodes wide) keeps the
// populations whatever is asked for.
bool moment_path(const cpmp_params &p, const DevParams &d, bool fuse_off, bool covered);
constexpr int kMomentFields = 12;
int moment_chunk(int nx, int ny, int nz, int form);
// bytes of a moment set (which has to fit a population set)
size_t moment_bytes(int nx, int ny, int nz, int form);
// one collide and stream step, from the moments if they are current (c->mom_at), else from
// the populations, to moments and (out_pops) populations; rho_next receives the new
// density of the fluid nodes
hipError_t launch_moment_step(cpmp_ctx *c, bool out_pops, bool want_mv, void *uout);
// Adjoint workspaces up to this size are kept for the next call: allocating and freeing them
// took 3 to 50 ms a call, more than the sweep of a small lattice (128x128x64 FP32, 40 taped
// steps: 54 ms a call, 13.7 ms of it work); larger ones are returned after the call.  Each
// device keeps at most one idle block, which any of its contexts' calls takes for itself
// while it runs; it is returned when the device's last context closes, when an allocation of
// the library finds too little memory, and by cpmp_release_workspace.
constexpr size_t kAdjKeep = (size_t)8 << 30;
// the device's idle block, from now on the caller's (null: none)
char *workspace_take(int device, size_t *bytes);
// gives a block back that no work uses any more; the larger of it and an idle one is kept
void workspace_give(int device, char *block, size_t bytes);
size_t workspace_idle(int device);
// frees the idle block; its bytes
size_t workspace_release(int device);
// hipMalloc on the current device, which `device` names; once more without the idle block if
// memory is short.  A failure leaves no error behind for a later hipGetLastError.
hipError_t device_malloc(int device, void **p, size_t n);
constexpr int kTileY = 8, kTileZ = 32;   // in-plane tile of the march kernels and of tiled population storage
constexpr int kWallTile = 16;             // columns per edge of the wall-fill tiles (16 x 16 workgroups)
// copy one population set between the device layout and the reference node order
hipError_t launch_pop_relayout(cpmp_ctx *c, const void *src, void *dst, bool to_device_layout);
// uout (when given): u, grad mu, grad rho of every node, 9 N values of the
// storage scalar type (adjoint tape)
// last: the step ends a run (outside a run the populations are the state)
hipError_t launch_collide(cpmp_ctx *c, bool want_mv, void *uout = nullptr, bool last = true);
hipError_t launch_macro(cpmp_ctx *c);
// nsteps whole steps (MV on the last if wanted)
hipError_t launch_steps(cpmp_ctx *c, int nsteps, bool want_mv = true);
hipError_t launch_init_reference(cpmp_ctx *c, double radius, double width, double rg, double rl, double solid);
hipError_t launch_init_splash(cpmp_ctx *c, double radius, double width, double film, double rg, double rl);
hipError_t launch_init_spheres(cpmp_ctx *c, const cpmp_init_desc *d);
hipError_t launch_feq_from_rho(cpmp_ctx *c);
hipError_t launch_pop_from_double(cpmp_ctx *c, int q, const double *src, void *dst_pop);
hipError_t launch_pop_to_double(cpmp_ctx *c, int q, const void *src_pop, double *dst);
hipError_t launch_scalar_from_double(cpmp_ctx *c, const double *src, void *dst);
hipError_t launch_scalar_to_double(cpmp_ctx *c, const void *src, double *dst);
hipError_t launch_velocity(cpmp_ctx *c, double *out3);
// XZ plane y = tier of rho into out (nx*nz doubles, out[i*nz + k])
hipError_t launch_plane_y(cpmp_ctx *c, int tier, double *out);
// per-block (area, max height) partials of the cap fit into part (2 per block)
hipError_t launch_cap_columns(cpmp_ctx *c, double mid, double *part, unsigned *nblocks);
// liquid fraction of the fluid nodes of plane x, block partials (nblocks values)
hipError_t launch_plane_fraction(cpmp_ctx *c, int x, double rg, double rl, double *part, unsigned *nblocks);
hipError_t launch_force(cpmp_ctx *c, double *out3);
hipError_t launch_reduce(cpmp_ctx *c, double *host_out /* 12 */);
// the same reduction with its partials (reduce_scratch_doubles() values) in `part`
hipError_t launch_reduce_into(cpmp_ctx *c, double *part, double *host_out /* 12 */);
// cpmp_stats from the 12 reduction values; CPMP_ENAN (naming the first bad node) when
// a density is NaN or negative
int stats_from_reduction(cpmp_ctx *c, const double *v, cpmp_stats *out);
hipError_t launch_type(cpmp_ctx *c, double *out);
size_t reduce_scratch_doubles();

// host-side CPU evaluation of the per-node collision (self-test hook)
void host_collide_fp64(const double f[19], double rho, const double F[3], const double ts[19],
                       const double *qp, double out[19], double u[3], int forcing);

}  // namespace cpmp
