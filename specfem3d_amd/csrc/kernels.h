// kernels.h -- launchers of the device kernels (all asynchronous on the given stream).
#pragma once

#include "mesh.h"

namespace sf {

// GLL constants passed to the element kernels by value (kernel-argument segment, read through
// the scalar cache): hp[i*5+l] = l'_l(x_i), hpw[i*5+l] = hp[i*5+l] w_i, wxy[a*5+b] = w_a w_b.
// Attenuation state of the elastic elements, in per-element blocks: the 18 memory-variable planes
// (component-major, SLS second) and the 6 strain planes of one element are contiguous, 125 points
// per plane. A stiffness launch in element order then reads and writes the state as a few
// sequential streams, and each plane of an element is one coalesced 500-byte run.
__host__ __device__ __forceinline__ int64_t r_idx(int64_t e, int plane, int p) { return (e * 18 + plane) * 125 + p; }
__host__ __device__ __forceinline__ int64_t eps_idx(int64_t e, int c, int p) { return (e * 6 + c) * 125 + p; }

struct GLLk {
  realw hp[25];
  realw hpw[25];
  realw wxy[25];
  // FMA builds, regular elements: hp * xix_regular and hpw * (jacobian_regular * xix_regular), which
  // fold the regular mapping and the jacobian weight into the contractions (fold_gll)
  realw hpr[25];
  realw hpwr[25];
};
inline void fold_gll(GLLk& G, realw xix_regular, realw jacobian_regular) {
  const realw jx = jacobian_regular * xix_regular;
  for (int q = 0; q < 25; q++) {
    G.hpr[q] = G.hp[q] * xix_regular;
    G.hpwr[q] = G.hpw[q] * jx;
  }
}
// the tables of a launch over regular elements alone: the folded ones in the place of the others
inline void regular_gll(GLLk& G, realw xix_regular, realw jacobian_regular) {
  fold_gll(G, xix_regular, jacobian_regular);
  for (int q = 0; q < 25; q++) {
    G.hp[q] = G.hpr[q];
    G.hpw[q] = G.hpwr[q];
  }
}
extern GLLk g_gll_host;
void set_gll_constants(const realw* hprime, const realw* hprimewgll, const realw* wgllwgll);

// Newmark pieces (k_update.hip)
void launch_predictor(hipStream_t s, int64_t n, realw* u, realw* v, realw* a, realw dt, realw dt2, realw dtsq2);
void launch_corrector(hipStream_t s, int64_t n, realw* v, realw* a, const realw* rmass, realw dt2);
// with `old`, also PML_displ_old = u + t1 v + t2 a of the corrected field (before the predictor)
void launch_corrector_predictor(hipStream_t s, int64_t n, realw* u, realw* v, realw* a, const realw* rmass,
                                realw dt2_prev, realw dt, realw dt2, realw dtsq2, realw* old = nullptr,
                                realw t1 = 0.f, realw t2 = 0.f);

// Gather assembly: the stiffness launches store local forces, 3 floats per slot in the solid and 1 in
// the fluid, and the pass that needs the acceleration (chi'' in the fluid) sums them, a point's slots in
// list order: a -= local[slot].
// The slot of point p = 5 row + i of the element at launch position pos: blocks of `eb` elements hold
// row by row the elements' five points, so that a row of points that runs through the elements of a
// block is contiguous (eb = 1: one element after the other).
__host__ __device__ __forceinline__ int gather_slot(int pos, int row, int i, int eb) {
  const int b = pos / eb;
  return b * eb * 125 + (row * eb + (pos - b * eb)) * 5 + i;
}
enum : uint16_t {
  AF_TERM = 1,   // boundary, coupling or source terms may have written the point's accel
  AF_EDGE = 2,   // point on the outer faces of the C-PML layers, or on the free surface of the fluid
  AF_MASS3 = 4,  // the point's three inverse masses differ (implicit Stacey term)
  AF_COUNT = 3   // shift of the number of slots
};
struct GatherArgs {
  int64_t g0, n;               // global points [g0, g0 + n)
  const uint16_t* info;        // AF_* and the number of slots << AF_COUNT, per global point
  const int* base;             // first slot entry of each 64 points from g0 on
  const int* idx;              // slots of every point, one point after the other
  const realw* local;
  int skip;                    // points with one of these flags end with zero: no contributions, no terms
  int clean;                   // accel is zero at every point without AF_TERM (it need not be read)
  realw *u, *v, *a;
  const realw* rm;             // inverse mass, 3 per point (read at AF_MASS3 points)
  const realw* rm1;            // ... and 1 per point (the others; every point of the fluid)
  realw dt2p;                  // corrector: dt/2
  realw dt, dt2, dtsq2;        // predictor
  realw* old;                  // PML_displ_old = u + t1 v + t2 a of the corrected field, or null
  realw t1, t2;
};
// what follows the sum: nothing (accel is left assembled), the corrector, or the corrector and the
// predictor of the next step (accel left zero)
enum { GATHER_ONLY = 0, GATHER_CORRECT = 1, GATHER_STEP = 2 };
// the acceleration or velocity that sum and corrector will give one point, from its slots at idx[first]
// on: for the receivers, which record a few points while the whole field waits for the next update. The
// operations are those of k_gather_update.
enum { WAIT_NONE = 0, WAIT_ACCEL = 1, WAIT_VELOC = 2 };
template <int NC>
__device__ __forceinline__ void waiting_value(const GatherArgs& A, int what, int64_t g, int first, realw out[NC]) {
  const int fl = A.info[g], cnt = fl >> AF_COUNT;
  const bool zero = fl & A.skip, full = !A.clean || (fl & AF_TERM);
  realw a[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) a[c] = full && !zero ? A.a[NC * g + c] : 0.f;
  for (int s = 0; s < (zero ? 0 : cnt); s++) {
    const realw* l = A.local + NC * (int64_t)A.idx[first + s];
#pragma unroll
    for (int c = 0; c < NC; c++) a[c] = a[c] + (-l[c]);
  }
#pragma unroll
  for (int c = 0; c < NC; c++) {
    a[c] = a[c] * (NC == 3 && (fl & AF_MASS3) ? A.rm[NC * g + c] : A.rm1[g]);
    out[c] = what == WAIT_ACCEL ? a[c] : A.v[NC * g + c] + A.dt2p * a[c];
  }
}
void launch_gather_update(hipStream_t s, const GatherArgs& a, int ncomp, int kind);
// slot lists (k_assembly.hip): the elements of `order` give the order of the sums, those of `launch`
// (nelem_launch of them) the slots, `pos0` launch positions on for the elements behind; allocates ptr
// (nglob + 1) and idx (125 nelem). lines: cache lines that the waves of a pass over all points touch
// with eb = 1 and with `eb`; idx holds slots for the returned one of the two.
int build_slot_lists(hipStream_t s, int nglob, int nspec, int nelem, const int* order, const int* launch, int nlaunch,
                     int pos0, int ncomp, int eb, const int* ibool, int*& ptr, int*& idx);
void launch_mark_points(hipStream_t s, int n, const int* ig, uint16_t bit, uint16_t* info);
// info (flags to be marked afterwards), base and rm1 of GatherArgs from the slot lists and the masses;
// rm null: one mass per point, rm1 is not written
// out[t] = ptr[ig[t]] (first slot entry of the receivers' points)
void launch_pick(hipStream_t s, int64_t n, const int* ig, const int* ptr, int* out);
void launch_gather_info(hipStream_t s, int64_t g0, int64_t n, const int* ptr, const realw* rm, uint16_t* info,
                        int* base, realw* rm1);

// element stiffness (k_elastic.hip / k_acoustic.hip)
// kinds of elements in a launch: regular ones, irregular ones, or the one before the other
enum { LINE_REG = 0, LINE_IRR = 1, LINE_BOTH = 2 };
struct ElasticArgs {
  int nelem;
  const int* elems;
  const int* ibool;
  const int* irregular;
  realw xix_regular, jacobian_regular;
  const realw* jac;        // 10 planes
  int64_t jac_plane;       // nspec_irr*125
  const float2* kappamu;
  const realw* displ;
  const realw* veloc;
  realw deltat;
  realw* R;                // 18 planes of nloc
  realw* eps;              // 6 planes of nloc
  const realw* fc;         // 3 planes
  const realw* fck;        // 3 planes
  const realw* fc_table;   // or: 6 planes of fc_rows distinct factor rows (fc 0..2, fck 3..5) ...
  const uint16_t* fc_index;  // ... and a row index per local point (null: use the planes)
  int fc_rows;
  realw* eps_tr3;          // nloc or null
  int64_t nloc;            // nspec*125
  realw alpha[3], beta[3], gamma[3];
  realw* local_out;        // local forces, 3 per slot (gather_slot)
  int eb;
  int nreg;                // listed regular elements, before the irregular ones
};
// att_variant: scheduling of the attenuation state in the point kernel (k_elastic_pt's AV)
void launch_elastic(hipStream_t s, const ElasticArgs& a, bool strain, bool att, bool exact,
                    int att_variant);
// deviatoric strain planes 0..4 and trace/3 of A.displ; with_trace also writes plane 5 = 3 * trace/3
void launch_element_strain(hipStream_t s, const ElasticArgs& a, realw* eps, realw* eps_tr3, bool with_trace,
                           bool exact);

// elastic kernel sums with the strain of the reconstructed displacement ElasticArgs::displ formed on the way
struct KernelSums {
  const realw *accel, *eps, *eps_tr3;  // adjoint field
  realw deltat;
  realw *rho_kl, *mu_kl, *kappa_kl;
};
void launch_kernels_line(hipStream_t s, const ElasticArgs& a, const KernelSums& k, bool exact);

// C-PML elements (k_pml.hip): stiffness with the convolution memory variables of
// compute_forces_viscoelastic_PML; per C-PML element blocks of 125-point planes
constexpr int SF_PML_NSTATE = 48;
constexpr int SF_PML_NCOEF = 42;
struct PmlArgs {
  int nelem;
  const int* elems;        // element ids ...
  const int* cpml;         // ... and their 0-based C-PML index
  const int* ibool;
  const int* irregular;
  realw xix_regular, jacobian_regular;
  const realw* jac;        // 10 planes
  int64_t jac_plane;
  const float2* kappamu;
  const realw* displ;
  const realw* veloc;
  const realw* pml_old;    // 3*nglob
  // per C-PML element: [2 ic] bit m set if coefficient plane m is one value over the element,
  // [2 ic + 1] bit m set if state plane m is live (its multiplier plane is not all zero; dead planes
  // are not stored and enter as zero)
  const uint64_t* masks;
  const int64_t* off;      // [2 ic]: offset of the element's packed coefficient planes, [2 ic + 1]: of its state
  realw* state;            // live state planes, 125 values each, packed per element in plane order
  const realw* coef;       // coefficient planes packed per element in plane order: 1 value if uniform, else 125
  realw t1, t2;            // deltatover2 (1 - 2 theta), deltatsqover2 (1 - theta)
  realw* local_out;        // local forces, 3 per slot (gather_slot)
  int eb, pos0;            // ... pos0: launch position of the first listed element
};
void launch_elastic_pml(hipStream_t s, const PmlArgs& a, bool exact);
// PML_displ_old at the listed points: u + t1 v + t2 a
void launch_pml_store_old(hipStream_t s, int n, const int* pts, const realw* u, const realw* v, const realw* a,
                          realw t1, realw t2, realw* old);
// zero u, v, a at the listed points (Dirichlet condition of the C-PML outer faces)
void launch_zero_points(hipStream_t s, int n, const int* pts, realw* u, realw* v, realw* a);

// Batched wavefields (k_batch.hip, batch.hip): groups of eight shots, each group a field of its own
// with rows of eight values: value (row r, shot s) of nrow rows at batch_idx, the next row of the same
// shot 8 further on. Rows are 3 g + c for the solid and g - g0 for the potentials.
__host__ __device__ __forceinline__ int64_t batch_idx(int64_t nrow, int64_t r, int s) {
  return (((int64_t)(s >> 3) * nrow + r) << 3) + (s & 7);
}
struct BatchArgs {
  int nelem;
  const int* elems;
  int ngroups;             // shot groups of the launch: of 4 or 8 shots (launch_*_batch)
  int s_first;             // first shot of the launch, a multiple of 8
  int S;                   // padded shot count
  int64_t nrow;            // rows of a group: 3 nglob
  const int* ibool;
  const int* irregular;
  realw xix_regular, jacobian_regular;
  const realw* jac;
  int64_t jac_plane;
  const float2* kappamu;
  const realw* u;
  const realw* v;          // viscoelastic: strain at u + dt v
  realw dt;
  // local forces: slot 125 ie + p of the launch, three rows of eight shots each; a block of loc_group
  // floats per group of eight
  realw* local;
  int64_t loc_group;
  int nreg;                // listed regular elements, before the irregular ones
  const int* nstep;        // per shot slot, decreasing (padding slots 0)
  const int* it;           // device step counter, 1-based current step
  // 3-SLS attenuation (k_visco_batch): per-shot memory variables and strain, one block per
  // (element, shot): value (e, shot, plane, p) at ((e * S + shot) * 18 + plane) * 125 + p
  // (strain: 6 planes)
  realw* R;
  realw* eps;
  const uint16_t* fc_index;    // SLS factor row per local point (or null: fc / fck planes)
  const realw* fc_table;       // 6 planes of fc_rows
  int fc_rows;
  const realw* fc;
  const realw* fck;
  int64_t nloc;
  realw alpha[3], beta[3], gamma[3];
};
// per-local-point flags of sf_batch_point_flags (for its callers: the engine has no use for them)
enum : unsigned char { BF_FIRST = 1, BF_LAST = 2, BF_ZERO = 4 };
// sc = shots per workgroup (4, 8)
void launch_elastic_batch(hipStream_t s, const BatchArgs& a, int sc, bool exact);
// viscoelastic (3 SLS) batched stiffness
void launch_visco_batch(hipStream_t s, const BatchArgs& a, int sc, bool exact);

// batched acoustic stiffness (k_batch.hip): potentials over the acoustic range of global points
struct BatchAcArgs {
  int nelem;
  const int* elems;
  int ngroups;             // shot groups of the launch, of 4 or 8 shots
  int s_first;             // first shot of the launch, a multiple of 8
  int64_t nrow;            // rows of a group: points of the acoustic range
  int64_t g0;              // first global point of the acoustic range
  const int* ibool;
  const int* irregular;
  realw xix_regular, jacobian_regular;
  const realw* jac;
  int64_t jac_plane;
  const realw* rho;        // rhostore, nspec*125
  const realw* pot;
  realw* local;            // slot 125 ie + p: a row of eight shots; loc_group floats per group of eight
  int64_t loc_group;
  const int* nstep;        // per shot slot, decreasing (padding slots 0)
  const int* it;           // device step counter, 1-based current step
};
// sc = shots per workgroup (4, 8)
void launch_acoustic_batch(hipStream_t s, const BatchAcArgs& a, int sc, bool exact);

struct AcousticArgs {
  int nelem;
  const int* elems;
  const int* ibool;
  const int* irregular;
  realw xix_regular, jacobian_regular;
  const realw* jac;
  int64_t jac_plane;
  const realw* rho;
  const realw* pot;
  realw* local_out;        // local forces, 1 per slot (gather_slot)
  int eb;
};
void launch_acoustic(hipStream_t s, const AcousticArgs& a, bool exact);


// boundary terms (k_boundary.hip)
// values of the sources in one step: as a launch argument where they fit (a copy from pinned memory to
// the device before the launch took 4 us of a 38 us step on 20x20x20 elements), else in device memory
constexpr int SF_SRC_VALS = 256;
struct SrcVals {
  realw v[SF_SRC_VALS];
  const realw* p;
};
enum { TERM_STACEY = 1, TERM_COUPLING = 2, TERM_SOURCE = 4, TERM_ADJOINT = 8 };
struct TermArgs {
  int n;                       // points that any term may touch
  const int* iglob;
  const int* head;             // 4 per point: its first face point, coupling point, source and adjoint pair, or -1
  int terms, flip;             // TERM_*; sign of the coupling
  FacePoints stacey, coupling, source, adjoint;  // of sources, ispec holds the owner
  const realw* in;             // veloc or chi'
  const realw* other;          // chi'' or displ of the coupling
  realw* out;                  // accel or chi''
  const realw *src_array, *src_kappa, *adj_h;
  SrcVals src, adj;
};
void launch_terms(hipStream_t s, const TermArgs& a, bool fluid);
// Stacey alone, also writing the boundary record
void launch_stacey_elastic(hipStream_t s, const FacePoints& f, const realw* veloc, realw* accel, realw* b_absorb);
void launch_stacey_elastic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_accel);
void launch_stacey_acoustic(hipStream_t s, const FacePoints& f, const realw* potd, realw* potdd, realw* b_absorb);
void launch_stacey_acoustic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_potdd);
void launch_free_surface(hipStream_t s, const FacePoints& f, realw* pot, realw* potd, realw* potdd);

// receivers (k_sources.hip)
void launch_seismo_el(hipStream_t s, int n, const int* list, const int* iglob, const double* h, const double* nu,
                      const realw* field, realw* out);
// ... of a field that waits to be summed (`what`: WAIT_*; first: slot entry of every receiver point)
void launch_seismo_el_waiting(hipStream_t s, int n, const int* list, const int* iglob, const double* h,
                              const double* nu, const GatherArgs& a, const int* first, int what, realw* out);
// receivers in acoustic elements: pressure = 1 records -sum h field into out[3 r] (out[3 r + 1..2] = 0),
// pressure = 0 the vector (1/rho) grad(field) interpolated and rotated by nu
struct AcReceiverArgs {
  int n;
  const int* list;
  const int* rec_ispec;
  const int* iglob;        // nrec*125 global points of the receiver elements
  const double* h;         // nrec*125 interpolation weights
  const double* nu;        // nrec*9
  const int* irregular;
  realw xix_regular;
  const realw* jac;
  int64_t jac_plane;
  const realw* rho;        // rhostore, nloc
  GatherArgs wait;         // ... of a field that waits to be summed
  const int* first;        // slot entry of every receiver point
};
void launch_seismo_ac(hipStream_t s, const AcReceiverArgs& a, const realw* field, int what, int pressure, realw* out);

// kernels / norms (k_kernels.hip)
void launch_compute_kernels_el(hipStream_t s, int nelem, const int* elems, const int* ibool, const realw* accel,
                               const realw* b_displ, const realw* eps, const realw* eps_tr3, const realw* b_eps,
                               const realw* b_eps_tr3, int64_t nloc, realw deltat, realw* rho_kl, realw* mu_kl,
                               realw* kappa_kl);
void launch_compute_kernels_ac(hipStream_t s, int nelem, const int* elems, const int* ibool, const int* irregular,
                               realw xix_regular, const realw* jac, int64_t jac_plane, const realw* rhostore,
                               const realw* pot, const realw* b_pot, const realw* b_potdd, realw deltat,
                               realw* rho_ac_kl, realw* kappa_ac_kl);
void launch_max_norm(hipStream_t s, int64_t npts, int ncomp, const realw* f, realw* out);

}  // namespace sf
