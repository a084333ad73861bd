/*
 * sf_internal.h -- interface between the C host layer (csrc/host/ C files,
 * compiled by gcc) and the HIP device layer (csrc/device/ HIP files, compiled by
 * hipcc for gfx950).  Not installed; callers use include/starflood*.h.
 *
 * Device launchers take device pointers and a stream, enqueue work and
 * return 0 or -1; they never synchronise unless their comment says so.
 */
#ifndef SF_INTERNAL_H
#define SF_INTERNAL_H

#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include "../../include/starflood_ext.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ---------- error reporting (host/params.c) ---------- */
/* Record and print "<func>() error: <msg>" in the reference's style. */
void sf_error(const char* func, const char* fmt, ...);
/* Check a HIP call; on failure record the error and return -1. */
int sf_hip_check(hipError_t e, const char* func, const char* what);
#define SF_HIP(call, func) do { if (sf_hip_check((call), (func), #call)) return STARFLOOD_FAILURE; } while (0)

/* Current process-wide parameters (host/params.c). */
const sf_params_t* sf_params(void);

/* ---------- per-simulation device context (host/context.c) ---------- */
typedef struct sf_tree_dev sf_tree_dev;   /* host/tree.c */

typedef struct sf_ctx {
	void* host_mem;          /* key: sim_t.mem */
	void* host_pinned_base;  /* the page-locked allocation holding sim_t.mem, or NULL (ordinary memory) */
	float* host_dev;         /* sim_t.mem as the device sees it, or NULL (ordinary memory) */
	unsigned int N;
	unsigned int dof;        /* reals per particle in sim.mem */
	unsigned int n_pad;      /* N rounded up to the PP j tile */
	float* d_mem;            /* device copy of sim.mem, same layout */
	float* d_body;           /* n_pad x 4: x, y, z, m (pad: m = 0) */
	double* d_x64;           /* 3N FP64 positions for the FAST drift */
	float* d_part;           /* partial sums of the PP and the SPH all-pairs passes */
	size_t part_bytes;
	double* d_red;           /* reduction scratch (blocks * SF_RED_VALUES), then the exact energy sums' */
	double* h_red;           /* pinned host mirror of the reduction result */
	double* h_red_dev;       /* the same as the device sees it */
	float* d_u;              /* SPH specific internal energy (N) */
	float* d_dudt;           /* its derivative (N) */
	float* d_sph_tmp;        /* SPH scratch (packed records, 12 n_pad floats) */
	void* d_sph_grid;        /* cell-grid pair search scratch (cubic model) */
	hipStream_t stream;
	sf_stats_t stats;        /* statistics of the last sim_step, */
	int have_stats;          /* where it left them on the host */
	int have_u;
} sf_ctx;

sf_ctx* sf_ctx_lookup(const void* host_mem, const char* func);
sf_ctx* sf_ctx_create(void* host_mem, unsigned int N, unsigned int dof);
void sf_ctx_destroy(sf_ctx* c);
/* Ensure the partial-sum scratch holds `bytes` bytes. */
int sf_ctx_reserve_part(sf_ctx* c, size_t bytes);
/* allocates (zeroed) d_u and d_dudt on first use */
int sf_ctx_ensure_u(sf_ctx* c);
/* The library's stream for work not tied to a simulation (lazy). */
hipStream_t sf_default_stream(void);

/* block offsets into d_mem / host mem (reference src/simulation.c:33-53) */
static inline float* sf_blk(float* base, unsigned int N, unsigned int e) { return base + (size_t)N * (size_t)e; }

#define SF_E_POS 0u
#define SF_E_VEL 3u
#define SF_E_ACC 6u
#define SF_E_MAS 9u
#define SF_E_POT 10u
#define SF_E_KEN 11u
#define SF_E_PEN 12u
#define SF_E_RAD 13u
#define SF_E_RHO 14u
#define SF_E_PRS 15u

/* mirror-mode transfers of blocks [e0, e0+count) (no-ops in RESIDENT mode), three
   of them at most; red (may be NULL, any mode): the
   SF_RED_VALUES results of a reduction, to h_red */
typedef struct sf_blocks {
	unsigned int e0, count;
} sf_blocks;
/* the two middle arguments, from a list of {e0, count} */
#define SF_SPANS(...) \
	(const sf_blocks[]){__VA_ARGS__}, (unsigned int)(sizeof((const sf_blocks[]){__VA_ARGS__}) / sizeof(sf_blocks))
int sf_upload_blocks(sf_ctx* c, const sf_blocks* span, unsigned int spans);
int sf_download_blocks(sf_ctx* c, const sf_blocks* span, unsigned int spans, const double* red);
int sf_finish(sf_ctx* c, const char* func);   /* synchronise the stream, report errors */

/* ---------- kernel timing (host/prof.c) ---------- */
/* Bracket a launch: sf_prof_begin returns a token passed to sf_prof_end. */
int sf_prof_begin(const char* name, hipStream_t s);
void sf_prof_end(int token, hipStream_t s);

/* ---------- device launchers (csrc/device) ---------- */
#define SF_RED_VALUES 16u    /* doubles per reduction partial */

/* `words` 32-bit words between device memory and page-locked host memory; dst
   and src are word aligned, at the same offset from a 16-byte boundary */
typedef struct sf_copy_range {
	void* dst;
	const void* src;
	size_t words;
} sf_copy_range;
#define SF_COPY_RANGES 4u
/* up to SF_COPY_RANGES of them by one kernel (host_copy.hip) */
int sfd_copy_ranges(const sf_copy_range* range, unsigned int count, hipStream_t s);
/* body[i] = (pos_i, m_i) for i < N, zero for N <= i < n_pad */
int sfd_pack_bodies(const float* pos, const float* mas, unsigned int N, unsigned int n_pad,
                    float* body, hipStream_t s);
/* sfd_kick_drift_fast, then sfd_pack_bodies, in one pass */
int sfd_kick_drift_pack(float* vel, const float* acc, double* x64, float* pos, const float* mas, unsigned int N,
                        unsigned int n_pad, float half_dt, double dt, float* body, hipStream_t s);

/* Reference-order PP gravity (src/gravity.c:693-812). */
int sfd_pp_exact(const float* pos, const float* mas, unsigned int N, float eps2, float negG,
                 int acc_phys, int kahan_acc, int kahan_pot, float* acc, float* pot, hipStream_t s);
/* its parameters, for a launch that makes it beside other sums */
typedef struct sf_exact_pp {
	float eps2, neg_g;
	int acc_phys, kahan_acc, kahan_pot;   /* kahan_acc: that of the other sums too */
	float* pot;
} sf_exact_pp;

/* What the fast force's combine does with each acceleration
   (device/force_epi.h): SF_EPI_STORE writes acc and (unless NULL) pot;
   SF_EPI_KICK also v += h a, ken and pen; SF_EPI_KDK takes the adjoint's
   integration from one force to the next (no acc, no pot). */
enum { SF_EPI_STORE = 0, SF_EPI_KICK, SF_EPI_KDK };
typedef struct {
	int kind;
	float *acc, *pot;
	float h;                       /* half a time step */
	float *v, *ken, *pen;
	double dt;                     /* SF_EPI_KDK from here */
	double* x64;
	float* x;                      /* copy of the opened step's positions, or NULL */
	int close, open;
	double* ck_x64;                /* checkpoint before the opening kick, or NULL */
	float *ck_v, *ck_a;
	float *xN, *vN;                /* the final state, or NULL */
} sf_force_epi;

/* What the force VJP's combine does with g (device/adjoint.hip): store it, or
   (step) lx += g, then either write lx and lv to gx0 and gv0 (where set) or
   lv += dt lx and the next VJP's inputs: nu = coef lv (coef m lv unless
   acc_phys) and, unless NULL, the bodies at x. */
typedef struct {
	int step;
	float* g;
	float *lx, *lv;   /* step from here */
	float dt, coef;
	int acc_phys;
	float *nu, *body;
	const float* x;
	float *gx0, *gv0;
} sf_vjp_epi;

/* Fast PP gravity of pos and mas (SF_EPI_STORE; body is then scratch) or of the
   n_pad packed bodies (a multiple of 1024; pos NULL, the other epilogues): partial
   sums into part (sfd_pp_part_bytes), then a fixed-order FP64 combine that ends
   with *epi (only SF_EPI_KDK writes body).  From kSymMin bodies each pair is
   evaluated once (device/pp_sym.hip); below, every i against every j. */
int sfd_pp_fast(const float* pos, const float* mas, float* body, unsigned int N, unsigned int n_pad, float eps2,
                double G, int acc_phys, float* part, const sf_force_epi* epi, hipStream_t s);
size_t sfd_pp_part_bytes(unsigned int n_pad);

/* FP64 direct sum for the listed particles (device idx list). */
int sfd_pp_f64(const float* pos, const float* mas, unsigned int N, double eps2, double G, int acc_phys,
               const unsigned int* idx, unsigned int n_idx, double* acc, double* pot, hipStream_t s);

/* Reference KDK pieces (src/simulation.c:381-451), FP32, no contraction. */
int sfd_kick_exact(float* vel, const float* acc, unsigned int n3, float half_dt, hipStream_t s);
int sfd_drift_exact(float* pos, const float* vel, unsigned int n3, float dt, hipStream_t s);
int sfd_kick_drift_exact(float* vel, const float* acc, float* pos, unsigned int n3, float half_dt, float dt,
                         hipStream_t s);
/* ken_i = (0.5 m_i) |v_i|^2, pen_i = m_i pot_i */
int sfd_energy_terms(const float* vel, const float* mas, const float* pot, unsigned int N,
                     float* ken, float* pen, hipStream_t s);
/* v += half_dt a (the fast policy's rounding) first, in the same pass */
int sfd_kick_energy_fast(float* vel, const float* acc, const float* mas, const float* pot, unsigned int N,
                         float half_dt, float* ken, float* pen, hipStream_t s);
/* exact_sum.hip: the sequential FP64 Kahan sums of ken and pen in index order
   (src/simulation.c:455-497), bit for bit, into out[0] and out[1]; part is
   scratch of sfd_energy_scratch_bytes(N).  pen NULL: the first sum alone.  red
   (may be NULL, with pen only): partials that sfd_kick_reduce_exact left, folded
   in the same launch. */
size_t sfd_energy_scratch_bytes(unsigned int N);
int sfd_energy_sums_exact(const float* ken, const float* pen, unsigned int N, void* part, double* out, double* red,
                          hipStream_t s);

/* FAST KDK: kick + FP64 drift fused; x64 refreshed from pos where they
   disagree (sfd_x64_refresh, or inside the drift). */
int sfd_x64_refresh(const float* pos, double* x64, unsigned int n3, hipStream_t s);
int sfd_kick_drift_fast(float* vel, const float* acc, double* x64, float* pos, unsigned int n3,
                        float half_dt, double dt, hipStream_t s);
/* sph.hip: u += half_dt du/dt (cubic SPH model) */
int sfd_sph_u_kick(float* u, const float* dudt, unsigned int N, float half_dt, hipStream_t s);

/* Deterministic FP64 reductions over the state: fills out[0..SF_RED_VALUES)
   with T, V, W, U, Px, Py, Pz, Lx, Ly, Lz.  x64 may be NULL (use pos).
   u may be NULL. red is scratch of sfd_reduce_scratch_doubles(N) doubles. */
unsigned int sfd_reduce_scratch_doubles(unsigned int N);
int sfd_reduce_state(const float* pos, const double* x64, const float* vel, const float* mas,
                     const float* pot, const float* ken, const float* pen, const float* u,
                     unsigned int N, double G, double eps, double* red, hipStream_t s);
/* v += half_dt a and sfd_energy_terms first, in the same pass */
int sfd_kick_reduce_state(const float* pos, const double* x64, float* vel, const float* acc, const float* mas,
                          const float* pot, float half_dt, float* ken, float* pen, const float* u, unsigned int N,
                          double G, double eps, double* red, hipStream_t s);
/* the same with the exact policy's roundings; the blocks' partials alone, for
   sfd_energy_sums_exact */
int sfd_kick_reduce_exact(const float* pos, float* vel, const float* acc, const float* mas, const float* pot,
                          float half_dt, float* ken, float* pen, const float* u, unsigned int N, double G,
                          double eps, double* red, hipStream_t s);

#ifdef __cplusplus
}
#endif

#endif /* SF_INTERNAL_H */
