// Launchers of the kernels in kernels.hip, called by the context code.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"

namespace cpi {

size_t elem_block_smem(int npe, int rule, int prec, int ml, int max_el, int kmax);
int elem_block_threads(int npe, int rule, int prec, int phys, int nblocks, int cus);
int elem_block_default_elements(int npe);
int elem_direct_threads(int npe);

// part: 0 = the whole element pass; with the surrogate (PHYS_EP_MLP) 1
// launches only the elastic pass, 2 only the network on the queue and 3
// only the walk over the deferred blocks, so each can be timed on its own
hipError_t launch_elem_block(const Params &p, int rule, int prec, int phys, bool aux,
                             int nblocks, size_t smem, hipStream_t s, int part = 0);
hipError_t prepare_elem_block(int npe, int rule, int prec, int phys, size_t smem);
// Events the following kernel launches of this host thread record at the
// kernel's own start and end (hipExtLaunchKernel); (null, null) restores
// plain launches.  For per-kernel timing outside graph capture.
void set_launch_events(hipEvent_t start, hipEvent_t stop);
// atomic: on n elements, those of list (device ids) if it is given; else n all
// of them
hipError_t launch_elem_direct(const Params &p, int rule, int prec, int phys, bool atomic,
                              const int32_t *list, int n, hipStream_t s);
// workgroups of the resident kernel the device can hold at once (0: there is
// none for this combination)
int resident_capacity(int npe, int rule, int prec, int phys, size_t smem, int cus);
hipError_t launch_resident(const Params &p, int rule, int prec, int phys, const Resident &rs,
                           int nblocks, size_t smem, hipStream_t s);
// its nodes of no element, after it
hipError_t launch_resident_loose(const Params &p, const Resident &rs, hipStream_t s);
hipError_t launch_mail_clear(const Resident &rs, int prec, hipStream_t s);
// LDS of a resident workgroup and bytes of the mail records
size_t resident_smem(size_t block_smem, int prec, int most);
size_t mail_bytes(int prec, size_t messages);
// prec: the element kernel's precision (its partials are stored in it)
hipError_t launch_node_bnd(const Params &p, int prec, bool aux, hipStream_t s);
// prec: the corner-force slots' precision (colour scatter)
hipError_t launch_node_all(const Params &p, int prec, bool aux, hipStream_t s);
hipError_t launch_node_init(const Params &p, hipStream_t s);
hipError_t launch_energy_reduce(const Params &p, hipStream_t s);
int energy_reduce_blocks();  // rows of p.ered (EP_N doubles each)
// lumped mass into p.m (scatter: 0 block, 1 colour, 2 atomic; list, n as
// launch_elem_direct)
hipError_t launch_mass(const Params &p, int rule, int scatter, int kind, double rho,
                       int nblocks, const int32_t *list, int n, hipStream_t s);
hipError_t launch_elem_dt(const Params &p, double *out, hipStream_t s);
// user-order host layouts (ninv: user node -> device id; spos: see
// k_export_elems).
// Parts: n nodes (elements), ninv, spos and last from the first of them on.
// Import: [n][3] into Vec3 and / or Node4 records (w = 0), null skipped.
hipError_t launch_import_nodes(const double *src, const int32_t *ninv, int n, Vec3 *d3, Node4 *d4,
                               hipStream_t s);
// Export: the arrays that are not null, vi = v - half_dt a
struct NodeExport {
  double *x, *v, *a, *vi;  // [n][3]
  double *m;               // [n]
  double *m3;              // [n][3], the mass in each component
  Ctl *ctl;                // a copy of the control block
  double half_dt;
};
hipError_t launch_export_nodes(const Params &p, const int32_t *ninv, int n, const NodeExport &o,
                               hipStream_t s);
// sig [n][nq][6], ep [n][nq] as doubles (null skipped)
hipError_t launch_export_elems(const Params &p, int prec, const uint32_t *spos, int n, double *sig,
                               double *ep, hipStream_t s);
// positions X0, velocities v0 (device order), forces, a and du zeroed
hipError_t launch_reset_nodes(const Params &p, const Vec3 *v0, hipStream_t s);
// smallest positive mass, one minimum per workgroup into out[blocks]
hipError_t launch_mass_min(const Params &p, double *out, int blocks, hipStream_t s);
// strain and stress [n][6] in user node order; last: per user node, the
// device id of the highest-numbered element holding it (-1: none, not written)
hipError_t launch_stress_node(const Params &p, const int32_t *last, int n, double *strain,
                              double *stress, hipStream_t s);
hipError_t launch_debug_strain(const Params &p, int rule, double alpha, int dcase, double nu,
                               double *out, hipStream_t s);
// the surrogate network on queue rows [0, n) (rows hold ceil(n/16)*16 rows
// of 32 bytes; see mlp_infer.h)
hipError_t launch_mlp_rows(const MlpParams *P, uint16_t *rows, int n, hipStream_t s);
// copies n4 32-byte records
hipError_t launch_stream_copy(const void *src, void *dst, long n4, hipStream_t s);

}  // namespace cpi
