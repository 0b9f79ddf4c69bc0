// Host-side launchers of the HIP kernels (implemented in the .hip files).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mhd_device.hpp"
#include "sources.hpp"

namespace pmf {

// Size of the per-block partial-result workspace (doubles) that the reductions use.
constexpr int kRedBlocks = 2048;
constexpr int kRedSlots = 24;  // doubles per block slot

// S: drag / radiation source terms (nullptr for the plain step).
template <class T>
void launch_step_ref(Fields<const T> U, Fields<T> O, T* ctp, const Grid& G, const StepParams<T>& P, bool ct,
                     hipStream_t st, const SrcParams<T>* S = nullptr);

// Fused tiled step (periodic GLM). Writes per-block CFL maxima of the new state into
// red (one double per block), unless that is null, and, unless dsmax is null, the final max into *dsmax and, if
// given, *hsmax (pinned host memory). Returns false when the grid shape is not supported by
// the fused kernel.
// zc: planes per z chunk (0 = the built-in choice); src: drag / radiation source terms
// (nullptr for the plain step).
// Pd: device-resident step scalars that replace P's (dt, ch, decay) in the kernel (P still
// selects the reconstruction and Riemann solver); nullptr = P as passed.
template <class T>
bool launch_step_fused(Fields<const T> U, Fields<T> O, const Grid& G, const StepParams<T>& P, double* red,
                       double* dsmax, hipStream_t st, int zc = 0, const SrcParams<T>* src = nullptr,
                       const StepParams<T>* Pd = nullptr, double* hsmax = nullptr);
// The maximum of red[0 .. nb) into *dsmax and, if given, *hsmax (pinned host memory).
void launch_fold_max(const double* red, int64_t nb, double* dsmax, double* hsmax, hipStream_t st);
// The device-side CFL stage of pmf_advance (evolve!'s rule, driver.jl:48-71, evaluated as
// the host does it): from the speed in dsmax[0], or for nb > 0 from the maximum of the
// previous step's partials red[0 .. nb), writes the step scalars to Pd and adds the step to
// clock[0] (reset: sets it), clock[1] = the step's dt.
template <class T>
void launch_step_params(const double* dsmax, const double* red, int64_t nb, const StepParams<T>& base,
                        StepParams<T>* Pd, double* clock, double cfl, double glm_ch_fac, double glm_cr, double dx,
                        int reset, hipStream_t st);
bool fused_supported(const Grid& G, int precision, int recon, int rsolve);
// Whether a :ref GLM step (src: with drag / radiation sources) is faster on the fused kernel with
// z chunks of zc planes than on the per-cell kernel.
bool ref_step_fused(const Grid& G, bool f64, int recon, bool src, int zc);
bool all_periodic(const Grid& G);
bool surrogate_grid(const Grid& G);
// The fused CT step (constrained-transport states, the :ref algorithm with each face
// solved once): the cell update into O and workspace slots 3-14 of ctp; ct_update! then
// finishes the step. src: the drag / radiation sources (no fallback masks: those belong
// to the :cube integrator). Unless workspace is CT_FILL, a variant that supports it forms the
// edge EMFs (slots 15-17) in the step, and writes slots 3-14 only with PPM under CT_DEFAULT;
// *edges tells whether it did (then ct_update! skips its edge pass). Returns false when the grid
// shape is not supported.
enum { CT_DEFAULT = -1, CT_LEAVE = 0, CT_FILL = 1 };  // workspace slots 3-14: not said, not needed, needed
template <class T>
bool launch_step_fused_ct(Fields<const T> U, Fields<T> O, T* ctp, const Grid& G, const StepParams<T>& P,
                          hipStream_t st, int zc = 0, const SrcParams<T>* src = nullptr, int workspace = CT_FILL,
                          bool* edges = nullptr);
// The surrogate-assisted fused step (float32, HLLD): simg is the network's LDS image,
// nsmooth accumulates the number of faces solved by the network.
bool launch_step_fused_surr(Fields<const float> U, Fields<float> O, const Grid& G, const StepParams<float>& P,
                            double* red, double* dsmax, const unsigned char* simg, float thr,
                            unsigned long long* nsmooth, hipStream_t st, double* hsmax);
// Number of workgroups (one partial maximum each) the fused kernel launches for G in the
// given precision with z chunks of zc planes (0 = the built-in choice).
int64_t fused_blocks(const Grid& G, bool f64, int zc = 0);
int fused_chunk(const Grid& G, bool f64);  // the built-in z chunk
// Relative time of `groups` workgroups of zc planes each on this device, `slots` of them per CU.
double fused_cost(int64_t groups, int zc, int slots);
int fused_slots();  // float workgroups the device holds at once, a multiple of eight
constexpr int kMinChunk = 4;  // smallest z chunk a caller may set (the built-in choice may be shorter)

// Geometry of the fused kernel's work decomposition: 16x12 column tiles (x fastest,
// then y; the last tile row may be ragged) marched through z chunks of zc planes.
struct FusedGeom {
  int32_t nx, ny, nz, ntx, nty, nchunks, zc;
  int32_t bc[3];  // per-axis boundary codes (BC_PERIODIC, BC_OUTFLOW, BC_REFLECT)
  int64_t plane, nc;
};
constexpr int kFusedTX = 16, kFusedTY = 12;

// One cube of an ensemble: both field sets (the step reads A and writes B on even
// steps, the reverse on odd ones), its geometry and its slice of the work-item list.
struct EnsCube {
  Fields<float> A, B;
  FusedGeom g;
  double dx;
  int32_t item0, nitems;
};
// Eight work queues (one per XCD): contiguous slices [base, base + len) of the items. Workgroup
// b takes item b / 8 of queue b % 8 first; the counters, one to a cache line, hand out the
// rest.
struct EnsQueues {
  int32_t base[8], len[8];
};
constexpr int kEnsCtrStride = 32;  // unsigneds from one queue's counter to the next
FusedGeom ens_geom(int n, int zc);
// Initial CFL maxima, one per work item (items are (cube, tile) pairs).
void launch_ens_wavespeed(const EnsCube* cubes, const int2* items, int nitems, const StepParams<float>& P,
                          double* red, int parity, hipStream_t st);
// Per-cube dt / ch / decay from the item maxima in red; clock holds (t, dt, smax) per cube.
void launch_ens_params(const EnsCube* cubes, int ncubes, const double* red, const StepParams<float>& base,
                       StepParams<float>* params, double* clock, unsigned* ctr, int nwg, float cfl, float fac, float cr,
                       hipStream_t st);
// The persistent step over all items (nwg workgroups, the same as launch_ens_params got; ctr =
// eight queue counters).
void launch_ens_step(const EnsCube* cubes, const int2* items, const EnsQueues& q, const StepParams<float>* params,
                     double* red, unsigned* ctr, int nwg, int parity, int recon, int rsolve, hipStream_t st);

// Passive species (passive_transport.jl): fractions from conserved densities in place
// (s2 may be null), and the backtrace into o1 (o2) of fractions (mode 0 / 1) or of an
// unconstrained scalar (mode 2) with the post-step velocity of U on an n^3 periodic grid.
template <class T> void launch_species_to_fractions(T* s1, T* s2, const T* rho, int64_t nc, T maxt, hipStream_t st);
template <class T>
void launch_backtrace(T* o1, T* o2, const T* a1, const T* a2, Fields<const T> U, int n, T dtdx, T maxt, int mode,
                      hipStream_t st);

template <class T>
void launch_wavespeed(Fields<const T> U, const Grid& G, const StepParams<T>& P, double* red, double* out,
                      hipStream_t st, double* hout = nullptr);
template <class T>
void launch_divb(Fields<const T> U, const Grid& G, T inv2dx, double* red, double* out3, hipStream_t st);
template <class T> void launch_totals(Fields<const T> U, const Grid& G, double* red, double* out8, hipStream_t st);
// ct_update! (ct.jl:158-173) on U. With P, red and dsmax: the cell-field pass also folds
// the CFL speed of the finished state into *dsmax (device) and, if given, *hsmax (pinned host
// memory), as the fused GLM step does.
// have_edges: slots 15-17 already hold this step's edge EMFs (formed by the step kernel).
template <class T>
void launch_ct_update(Fields<T> U, T* ctp, const Grid& G, T dtdx, bool compensate, hipStream_t st,
                      const StepParams<T>* P = nullptr, double* red = nullptr, double* dsmax = nullptr,
                      bool have_edges = false, double* hsmax = nullptr);
template <class T> void launch_divb_face(const T* ctp, const Grid& G, T invdx, double* red, double* out, hipStream_t st);
template <class T>
void launch_ct_install(Fields<T> U, T* ctp, const Grid& G, hipStream_t st);
template <class T>
void launch_ct_curl(const T* Ax, const T* Ay, const T* Az, T* bx, T* by, T* bz, const Grid& G, T invdx,
                    hipStream_t st);
template <class T>
void launch_riemann_batch(const T* L, const T* R, T* F, int64_t n, int dir, bool ct, const StepParams<T>& P,
                          hipStream_t st);

}  // namespace pmf
