/*
 * gravity.c -- solve_gravity_part_part with the reference's signature
 * (src/gravity.h:22, src/gravity.c:666-819), the FP64 direct-sum precision
 * reference, and the device-array force entry used by the adjoint.
 */
#include <stdio.h>
#include <stdlib.h>

#include "sf_host.h"

/* j slices of the cubic SPH all-pairs passes: enough blocks to give every CU
   several waves */
static unsigned int pp_slices(unsigned int n_pad) {
	/* one j range per wavefront of 64 i; about 128k wavefronts, while each
	   range keeps at least 256 j */
	const unsigned int iblocks = n_pad / 256u;
	unsigned int s = iblocks ? (32768u + iblocks - 1u) / iblocks : 1u;
	const unsigned int smax = n_pad / 256u;
	if (s > smax) s = smax;
	if (s > 64u) s = 64u;
	if (s < 1u) s = 1u;
	return s;
}

/* reference: (real)(EPSILON*EPSILON) is squared in double, then rounded */
static float eps2_f32(double eps) { return (float)(eps * eps); }

unsigned int sf_pp_slice_count(unsigned int n_pad) { return pp_slices(n_pad); }

size_t sf_pp_part_bytes(unsigned int n_pad) { return sfd_pp_part_bytes(n_pad); }

static int force(const sf_params_t* p, unsigned int N, unsigned int n_pad, const float* pos, const float* mas,
                 float* body, float* part, size_t part_bytes, const sf_force_epi* epi, hipStream_t s) {
	if (part_bytes < sf_pp_part_bytes(n_pad)) {
		sf_error("sfd_pp_fast", "%zu bytes of partial sums, %zu needed", part_bytes, sf_pp_part_bytes(n_pad));
		return -1;
	}
	return sfd_pp_fast(pos, mas, body, N, n_pad, eps2_f32(p->epsilon), p->G, p->acc_mode == SF_ACC_PHYSICAL, part, epi,
	                   s);
}

int sf_pp_force_packed(const sf_params_t* p, unsigned int N, unsigned int n_pad, float* body, float* part,
                       size_t part_bytes, const sf_force_epi* epi, hipStream_t s) {
	return force(p, N, n_pad, NULL, NULL, body, part, part_bytes, epi, s);
}

int sf_pp_force_arrays(const sf_params_t* p, unsigned int N, unsigned int n_pad, const float* pos, const float* mas,
                       float* body, float* part, size_t part_bytes, float* acc, float* pot, hipStream_t s) {
	const sf_force_epi epi = {.kind = SF_EPI_STORE, .acc = acc, .pot = pot};
	return force(p, N, n_pad, pos, mas, body, part, part_bytes, &epi, s);
}

sf_exact_pp sf_exact_pp_params(sf_ctx* c) {
	const sf_params_t* p = sf_params();
	return (sf_exact_pp){.eps2 = eps2_f32(p->epsilon), .neg_g = (float)(-p->G),
	                     .acc_phys = p->acc_mode == SF_ACC_PHYSICAL, .kahan_acc = p->kahan_solver,
	                     .kahan_pot = p->kahan_energy, .pot = sf_blk(c->d_mem, c->N, SF_E_POT)};
}

int sf_solve_gravity_pp(sf_ctx* c) {
	const sf_params_t* p = sf_params();
	const unsigned int N = c->N;
	const float *pos = sf_blk(c->d_mem, N, SF_E_POS), *mas = sf_blk(c->d_mem, N, SF_E_MAS);
	float *acc = sf_blk(c->d_mem, N, SF_E_ACC), *pot = sf_blk(c->d_mem, N, SF_E_POT);
	if (p->precision == SF_PRECISION_EXACT) {
		const sf_exact_pp e = sf_exact_pp_params(c);
		return sfd_pp_exact(pos, mas, N, e.eps2, e.neg_g, e.acc_phys, e.kahan_acc, e.kahan_pot, acc, pot, c->stream);
	}
	if (sf_ctx_reserve_part(c, sf_pp_part_bytes(c->n_pad))) return -1;
	return sf_pp_force_arrays(p, N, c->n_pad, pos, mas, c->d_body, c->d_part, c->part_bytes, acc, pot, c->stream);
}

int sf_step_gravity_pp(sf_ctx* c) {
	const sf_params_t* p = sf_params();
	const unsigned int N = c->N;
	const float h = 0.5f * (float)p->dt;
	float *vel = sf_blk(c->d_mem, N, SF_E_VEL), *acc = sf_blk(c->d_mem, N, SF_E_ACC);
	const sf_force_epi epi = {.kind = SF_EPI_KICK, .acc = acc, .pot = sf_blk(c->d_mem, N, SF_E_POT), .h = h, .v = vel,
	                          .ken = sf_blk(c->d_mem, N, SF_E_KEN), .pen = sf_blk(c->d_mem, N, SF_E_PEN)};
	if (sf_ctx_reserve_part(c, sf_pp_part_bytes(c->n_pad))) return -1;
	if (sfd_kick_drift_pack(vel, acc, c->d_x64, sf_blk(c->d_mem, N, SF_E_POS), sf_blk(c->d_mem, N, SF_E_MAS), N,
	                        c->n_pad, h, p->dt, c->d_body, c->stream))
		return -1;
	return sf_pp_force_packed(p, N, c->n_pad, c->d_body, c->d_part, c->part_bytes, &epi, c->stream);
}

/* reference src/gravity.c:667-819: reads pos, mas; writes acc (assigned, not
   accumulated) and pot. */
int solve_gravity_part_part(const sim_t* SF_RESTRICT sim_ptr) {
	if (!sim_ptr) return STARFLOOD_FAILURE;
	sf_ctx* c = sf_ctx_lookup(sim_ptr->mem, "solve_gravity_part_part");
	if (!c) return STARFLOOD_FAILURE;
	if (sf_upload_blocks(c, SF_SPANS({SF_E_POS, 3u}, {SF_E_MAS, 1u}))) return STARFLOOD_FAILURE;
	int rc = sf_solve_gravity_pp(c);
	if (sf_download_blocks(c, SF_SPANS({SF_E_ACC, 3u}, {SF_E_POT, 1u}), NULL)) rc = -1;
	if (sf_finish(c, "solve_gravity_part_part")) rc = -1;
	return rc ? STARFLOOD_FAILURE : STARFLOOD_SUCCESS;
}

int sf_pp_direct_f64(const sim_t* sim_ptr, const unsigned int* idx, unsigned int n_idx, double* acc_out,
                     double* pot_out) {
	if (!sim_ptr || (!idx && n_idx) || (n_idx && (!acc_out || !pot_out))) return STARFLOOD_FAILURE;
	sf_ctx* c = sf_ctx_lookup(sim_ptr->mem, "sf_pp_direct_f64");
	if (!c) return STARFLOOD_FAILURE;
	if (n_idx == 0) return STARFLOOD_SUCCESS;
	for (unsigned int k = 0; k < n_idx; ++k) {
		if (idx[k] >= c->N) {
			sf_error("sf_pp_direct_f64", "index %u out of range (N = %u)", idx[k], c->N);
			return STARFLOOD_FAILURE;
		}
	}
	const sf_params_t* p = sf_params();
	if (sf_upload_blocks(c, SF_SPANS({SF_E_POS, 3u}, {SF_E_MAS, 1u}))) return STARFLOOD_FAILURE;
	unsigned int* d_idx = NULL;
	double* d_out = NULL;
	int rc = 0;
	if (hipMalloc((void**)&d_idx, (size_t)n_idx * sizeof(unsigned int)) != hipSuccess ||
	    hipMalloc((void**)&d_out, (size_t)n_idx * 4u * sizeof(double)) != hipSuccess) {
		sf_error("sf_pp_direct_f64", "device allocation failed");
		rc = -1;
		goto done;
	}
	if (sf_hip_check(hipMemcpyAsync(d_idx, idx, (size_t)n_idx * sizeof(unsigned int), hipMemcpyHostToDevice,
	                                c->stream),
	                 "sf_pp_direct_f64", "index upload")) {
		rc = -1;
		goto done;
	}
	if (sfd_pp_f64(sf_blk(c->d_mem, c->N, SF_E_POS), sf_blk(c->d_mem, c->N, SF_E_MAS), c->N, p->epsilon * p->epsilon,
	               p->G, p->acc_mode == SF_ACC_PHYSICAL, d_idx, n_idx, d_out, d_out + 3u * (size_t)n_idx,
	               c->stream)) {
		rc = -1;
		goto done;
	}
	if (sf_hip_check(hipMemcpyAsync(acc_out, d_out, (size_t)n_idx * 3u * sizeof(double), hipMemcpyDeviceToHost,
	                                c->stream),
	                 "sf_pp_direct_f64", "download") ||
	    sf_hip_check(hipMemcpyAsync(pot_out, d_out + 3u * (size_t)n_idx, (size_t)n_idx * sizeof(double),
	                                hipMemcpyDeviceToHost, c->stream),
	                 "sf_pp_direct_f64", "download"))
		rc = -1;
	if (sf_finish(c, "sf_pp_direct_f64")) rc = -1;
done:
	if (d_idx) {
		hipStreamSynchronize(c->stream);
		hipFree(d_idx);
	}
	if (d_out) hipFree(d_out);
	return rc ? STARFLOOD_FAILURE : STARFLOOD_SUCCESS;
}
