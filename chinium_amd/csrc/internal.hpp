// Internal host-side structures of the MI355X XC library (not part of the ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

#include "chinium_xc.h"

namespace chx {

// Batch and tile geometry shared by host planning and the kernels.
constexpr int kBatch = 64;     // quadrature points per batch (MFMA K for Vxc, M for density)
constexpr int kTile = 32;      // AOs per screening tile
constexpr int kGroup = 4;      // AO tiles per density work group (128 output columns)
constexpr int kSuper = 2;      // AO tiles per Vxc super-tile (64 x 64 output block)
constexpr int kPadAO = 128;    // nbasis is padded to a multiple of this (4 tiles)
constexpr int kMxTiles = 4;    // tiles per Vxc group of the cached tables (128 AOs)
constexpr int kMxWideTiles = 5;  // ... of the mixed form's wide shape (160 AOs)
constexpr int kChunkMax = 32;  // most consecutive batches that share one AO list
constexpr int kChunkLong = 512;  // ... where memory is short
constexpr int kCoef = 5;       // Vxc integrand coefficients per point: a, c_x, c_y, c_z, t
constexpr double kCoreRadius = 0.3;  // bohr: points this close to a nucleus with Z > 2 are batched apart

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void hip_check(hipError_t e, const char* what);
#define CHX_HIP(x) ::chx::hip_check((x), #x)

struct ShellH {
  int type;    // 0 s, 1 Cartesian p, -1 pure p, -2 pure d, -3 pure f
  int center;
  int nprim;
  int prim_off;
  int ao_off;  // offset in the reference AO order
};

int shell_size(int type);

// A component polynomial of a shell as monomials c x^i y^j z^k, in the
// reference's component order (molecule.cpp).
struct MonoTerm {
  double c;
  int i, j, k;
};
std::vector<std::vector<MonoTerm>> component_monomials(int type);
// A shell of an auxiliary (fitting) basis: angular momentum l (pure), centre,
// exponents, normalised contraction coefficients.
struct AuxShell {
  int l, center;
  std::vector<double> e, c;
};

// A device buffer owned by a handle.
template <class T> struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void alloc(size_t count) {
    if (count == n && p) return;
    release();
    if (count == 0) return;
    CHX_HIP(hipMalloc(&p, count * sizeof(T)));
    n = count;
  }
  T* alloc_get(size_t count) {
    alloc(count);
    return p;
  }
  void upload(const std::vector<T>& h, hipStream_t s) {
    alloc(h.size());
    if (!h.empty()) CHX_HIP(hipMemcpyAsync(p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s));
  }
  void copy_from(const DevBuf& o, hipStream_t s) {
    alloc(o.n);
    if (o.n) CHX_HIP(hipMemcpyAsync(p, o.p, o.n * sizeof(T), hipMemcpyDeviceToDevice, s));
  }
};

// One shell segment of a tile with everything its evaluation reads (mixed-precision
// form): the scalar unit fetches the first 80 bytes, which hold up to kSegInline
// primitives, and the rest only where a shell has more. A primitive is (-a log2 e,
// c, a c), so that exp(-a r^2) is one product and the hardware's exp2.
constexpr int kSegPrim = 12;  // primitives per record
constexpr int kSegInline = 4;
constexpr int kSegSame = 1 << 15;  // meta: the same centre as the record before (in the tile)
struct SegRec {
  double ax, ay, az;  // shell centre
  int meta;           // type & 0xff | nprim << 8 | first component << 16 | count << 24
  int col;            // AO offset in the tile
  float p[kSegPrim][3];
  float pad[4];
};
static_assert(sizeof(SegRec) == 192, "records start on 64-byte lines");

// Kernel-side view of the basis. Tiles are the chunks' own: every chunk of
// batches (see ChunkDev) holds the AOs alive in it, packed in 32-AO tiles, and
// tile_seg_off / seg / segrec list each tile's shell segments.
struct BasisView {
  const double* sh_xyz;   // 3 per shell
  const int* sh_type;
  const int* sh_nprim;
  const int* sh_poff;
  const double* p_exp;
  const double* p_coef;
  const int* tile_seg_off;  // tiles of all chunks + 1
  const int4* seg;          // (shell, first component, count, local AO offset in tile)
  const SegRec* segrec;     // per segment, same index as seg (mixed-precision form)
  const int* sh_atom;       // atom of each shell (XC gradient)
};

// A chunk: up to kChunkMax (short of memory: kChunkLong) consecutive batches (the batch order is spatial) and
// the list of the AOs above the screening threshold in any of them, packed in
// ntl tiles of 32 AOs (tiles tile0 .. tile0 + ntl - 1 of the grid's list). Every
// batch of the chunk carries all ntl tiles, so slot (batch, tile q) is
// bt_off[batch] + q, and the chunk's part of D is a dense (32 ntl)^2 matrix at
// doff in the gathered copy (elements; the split form holds hi, then lo).
struct ChunkDev {
  long doff;
  int tile0, ntl;
  int b0, nb;  // its batches b0 .. b0 + nb - 1
};
// A Vxc work item: the block (I, J) of super-tiles of one chunk over nbat of
// its batches; slot0 is the first batch's first slot.
struct VxcItem {
  int I, J, slot0, nbat, ntl, tile0, batch0, pad_;
};

// Cached tables: tiles I0 .. I0 + nI - 1 against J0 .. J0 + nJ - 1 (I0 <= J0) of a
// run (nbat batches of a chunk); the block's place u in U and its row length.
struct MxItem {
  long u;
  int I0, nI, J0, nJ, slot0, nbat, ntl, ldu, tile0, batch0;
};
// Row of one AO in a run's blocks: element k (k < len) is V at (that AO, ao_of[a0 + k]).
struct RowRef {
  long u;
  int a0, len;
};

// Grid set-up (kernels_grid.hip). rab: (R, 1 / R) of every pair of atoms, rows of
// becke_ld(natoms), the rest of a row (1, 1).
int becke_ld(int natoms);
void launch_becke(hipStream_t s, long npts, const double* px, const double* py, const double* pz, double* w,
                  const int* owner, int natoms, const double* atom_xyz, const double2* rab, int ld);
struct BisSeg { int lo, n, left; };  // points [lo, lo + n), the first `left` to go to the left half (0: a batch)
// Bisects the n points of the indexes idx level by level (segments levels[l] ..
// levels[l + 1] of segs); points and indexes end in pts / ids[levels.size() - 1
// odd or even] (without levels: pts[0] and idx).
void launch_bisect(hipStream_t s, long n, const int* idx, const double* px, const double* py, const double* pz,
                   const std::vector<int>& levels, const BisSeg* segs, double* pts[2], int* ids[2]);
void launch_batch_slots(hipStream_t s, int nbatches, const int2* batch, const double* pts, const int* idx, long stride,
                        const double* w, double* bx, double* by, double* bz, double* bw);
// Launchers (kernels.hip).
// alive: per batch nwords 64-bit words, bit k of word w set when shell 64 w + k
// comes closer than its reach (reach2: squared) to one of the batch's points
void launch_screen(hipStream_t s, int nbatches, int nshells, int nwords, const double* bx, const double* by,
                   const double* bz, const int* bn, const double* sh_xyz, const double* reach2,
                   unsigned long long* alive);
// The chunks' dense blocks of D (FP64): block r of the launch gathers the 32
// rows of tile r from D (reference order, column-major n x n), zero for padding.
// asym (may be null): *asym = gen when D is not symmetric to within rounding.
// tile0, d0: first tile, and place in the whole list of blocks of Dt's first element.
void launch_gather_d(hipStream_t s, int ntiles, int n, const double* D, const int* tile_chunk, const ChunkDev* chunks,
                     const int* ao_of, double* Dt, int* asym, int gen, int nmat = 1, size_t sO = 0, int tile0 = 0,
                     long d0 = 0);
void launch_pad_d(hipStream_t s, int n, int npad, const double* D, double* Dpad);
// mode 0: rho, grad rho / 2 into part ([group][4][64]); mode r = 1..3: the tau
// partial of direction r (part = component r - 1 of [group][3][64]). d0 as above.
void launch_density_f64(hipStream_t s, int mode, int ngroups, const int* grp_batch, const int* grp_tile,
                        const int* grp_ntiles, const int* b_chunk, const ChunkDev* chunks, const double* bx,
                        const double* by, const double* bz, BasisView bv, const double* Dt, long d0, double* part);
// One molecule of a multi-molecule functional launch: byte offsets of its
// buffers from the launch's base pointer, its slot count, its first block
// (entry nmol is a sentinel whose blk0 is the total block count) and its E/N slot.
struct FnMolecule {
  long grp_off, part, part_tau, w, rho, coef, en_part, cpart;
  int nslots, blk0, slot_en, ncpart;
};
void launch_functional_multi(hipStream_t s, const char* base, const FnMolecule* fm, int nmol, int nblocks,
                             const int* codes, int ncodes, int family, double* en);
void launch_functional(hipStream_t s, int nbatches, const int* grp_off, const double* part, const double* part_tau,
                       const double* bw, const int* codes, int ncodes, int family, int want_e, int want_v,
                       double* rho_out, double* coef, double* en_part, int en_blocks);
void launch_eval_functional(hipStream_t s, long n, const int* codes, int ncodes, const double* rho, const double* sigma,
                            const double* tau, double* exc, double* vrho, double* vsigma, double* vtau);
void launch_reduce_en(hipStream_t s, int nparts, const double* en_part, double* en);
void launch_fill(hipStream_t s, double* p, size_t n, double v);
// ncomp 1: a phi + c . grad phi; ncomp 4 adds the tau term (t = coef[4]).
void launch_vxc_f64(hipStream_t s, int ncomp, int nwork, const VxcItem* work, const int* ao_of, const double* bx,
                    const double* by, const double* bz, const double* coef, BasisView bv, double* Mint, int npad);
void launch_vrho_coef(hipStream_t s, long nslots, const double* vrho_w, double* coef);
// Cached-AO FP64 path (kernels_cached.hip).
void launch_ao_cache(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile,
                     const double* bx, const double* by, const double* bz, BasisView bv, double* cache);
// response path (closed shell, LDA/GGA)
constexpr int kFx = 8;  // per slot: v2rho2, v2rhosigma, v2sigma2, v_sigma, grad rho (3), -
// polarised (nspin = 2): vsigma (3), v2rho2 (3), v2rhosigma (6), v2sigma2 (6), grad rho_a (3), grad rho_b (3)
constexpr int kFxPol = 24;
void launch_functional_fpol(hipStream_t s, int nbatches, const int* grp_off, const double* part, const double* part_b,
                            const int* codes, int ncodes, int family, double* fx);
// outputs m0 .. m0 + nmat - 1 of [spin][perturbation] (nper perturbations)
void launch_response_coef_pol(hipStream_t s, int nbatches, const double* rhou, const double* fx, const double* bw,
                              int family, int m0, int nmat, int nper, double* coef);
void launch_eval_functional_fpol(hipStream_t s, long n, const int* codes, int ncodes, const double* rho,
                                 const double* sigma, double* v2rho2, double* v2rhosigma, double* v2sigma2);
void launch_functional_f(hipStream_t s, int nbatches, const int* grp_off, const double* part, const int* codes,
                         int ncodes, int family, double* fx);
void launch_point_rho(hipStream_t s, int nbatches, const int* grp_off, const double* part, double* rhou, int nmat,
                      size_t sP);
void launch_response_coef(hipStream_t s, int nbatches, const double* rhou, const double* fx, const double* bw,
                          int family, int nmat, double* coef);
void launch_eval_functional_f(hipStream_t s, long n, const int* codes, int ncodes, const double* rho,
                              const double* sigma, double* v2rho2, double* v2rhosigma, double* v2sigma2);
// spin-polarised (nspin = 2) functional, LDA/GGA and r2SCAN (part_tau / part_tau_b: meta-GGA)
void launch_functional_pol(hipStream_t s, int nbatches, const int* grp_off, const double* part, const double* part_b,
                           const double* part_tau, const double* part_tau_b, const double* bw, const int* codes,
                           int ncodes, int family, int want_e, int want_v, double* rho_out, double* coef,
                           double* coef_b, double* en_part, int en_blocks);
// at points, libxc's polarised layout; tau / vtau (meta-GGA) may be null
void launch_eval_functional_pol(hipStream_t s, long n, const int* codes, int ncodes, const double* rho,
                                const double* sigma, const double* tau, double* exc, double* vrho, double* vsigma,
                                double* vtau);
// Surrogate network (kernels_mlp.hip): 3 -> 64 -> 64 -> 64 -> 1, tanh. Offsets
// of the parameter block (floats); matrices are [out][in] (y = W x + b). The
// run copies the kernels read hold W2 transposed ([in][out]) at the same offset.
constexpr int kMlpH = 64;
constexpr int kMlpW1 = 0, kMlpB1 = 192, kMlpW2 = 256, kMlpB2 = 4352, kMlpW3 = 4416, kMlpB3 = 8512, kMlpW4 = 8576,
              kMlpB4 = 8640, kMlpParams = 8641;
// Descriptor box of the training data: t = (ln rho, s/(1+s), alpha/(1+alpha));
// the network input is u = (t - c) / h with c, h the box centre and half width.
struct MlpBox {
  float lo[3], hi[3];
  double rho_min;  // below: analytic functional (low-density tail)
  int nbase;       // the network predicts F - F_base of these analytic codes (0: the whole F)
  int base[2];
};
void launch_mlp_pack(hipStream_t s, const float* P, float* Prun, float* Pinf);
void launch_mlp_forward(hipStream_t s, long n, const float* U, const float* R, const unsigned* Wpk, float* F,
                        float* dF);
constexpr int kMlpPacked = 4 * 4 * 2 * 2 * 64 * 4;  // u32 words of the packed split-BF16 (hi, lo) MFMA weight fragments
void launch_mlp_pack_mx(hipStream_t s, const float* P, unsigned* Wpk);
// Gradient and loss as per-block sums (at most kMlpGradBlocks blocks; returns
// their number): Gpart[block][kMlpParams], losspart[block].
constexpr int kMlpGradBlocks = 256;
int launch_mlp_grad(hipStream_t s, long n, const float* U, const float* T, const float* C, float cs, const float* P,
                    float* Gpart, float* losspart);
// their sums: one Adam step on P, or the gradient to G; the loss is added to *loss
void launch_mlp_adam(hipStream_t s, int nparts, const float* Gpart, const float* losspart, float* P, float* M,
                     float* V, float* loss, float lr, int step);
void launch_mlp_reduce(hipStream_t s, int nparts, const float* Gpart, const float* losspart, float* G, float* loss);
void launch_mlp_features(hipStream_t s, long n, const double* rho, const double* sigma, const double* tau,
                         const int* codes, int ncodes, float* t, float* F);
void launch_mlp_eval(hipStream_t s, long n, const float* R, const unsigned* Wpk, const MlpBox& box, const int* codes,
                     int ncodes,
                     const double* rho, const double* sigma, const double* tau, double* exc, double* vrho,
                     double* vsigma, double* vtau, int* nfall);
void launch_functional_mlp(hipStream_t s, int nbatches, const int* grp_off, const double* part,
                           const double* part_tau, const double* bw, const float* R, const unsigned* Wpk,
                           const MlpBox& box, const int* codes, int ncodes, int want_e, int want_v, double* rho_out,
                           double* coef, double* en_part, int* nfall);
void launch_point_density(hipStream_t s, int nbatches, const int* grp_off, const double* part,
                          const double* part_tau, int has_tau, const double* bw, double* rho, double* sigma,
                          double* tau, double* w);
// (the launches below: nmat matrices of one launch, s*: doubles from one matrix's
// operand or result to the next one's; part1, coef1: the second one's (not null), of
// two; tau and ncomp 4 take one)
// rho, grad rho / 2 into part; part_tau (not null: meta-GGA): tau (asym / gen as launch_gather_d's)
void launch_density_c64(hipStream_t s, int ngroups, const int* grp_batch, const int* grp_tile, const int* grp_ntiles,
                        const int* bt_off, const int* b_chunk, const ChunkDev* chunks, const double* cache,
                        const double* Dt, const int* asym, int gen, double* part, double* part_tau, int nmat = 1,
                        size_t sD = 0, size_t sP = 0, double* part1 = nullptr);
// B = a phi + c . grad phi per slot (one component for every family)
void launch_make_b(hipStream_t s, int nbatches, const int* bt_off, const double* coef, const double* cache,
                   double* bmat, int nmat = 1, size_t sC = 0, size_t sB = 0, const double* coef1 = nullptr);
// upper blocks of V per run into U; ncomp 4 adds the tau term, its operand t d_r
// phi formed from the cache and coef[4] as it is loaded
void launch_vxc_c64(hipStream_t s, int ncomp, int nwork, const MxItem* work, const double* cache, const double* bmat,
                    const double* coef, double* U, int nmat = 1, size_t sB = 0, size_t sU = 0);
// M += A^T B over every pair of groups (items with I0, J0 in any order), A component 0 at `cache`.
// nmat products: A = cache + (m / nb) sA, B = bmat + (m % nb) sB, M + m sO.
struct ProdBatch {
  int nb = 1;
  size_t sA = 0, sB = 0, sO = 0;
};
void launch_prod_c64(hipStream_t s, int nwork, const MxItem* work, const int* ao_of, const double* cache,
                     const double* bmat, double* M, int npad, int nmat, const ProdBatch& pb);
void launch_finalize_sym(hipStream_t s, int n, int npad, const double* Mint, double* V);
// Device descriptor of one grid for the mixed-precision kernels. A kernel
// launch covers a list of (grid, item) pairs, so one launch can serve many
// molecules (a pack) as well as a single grid.
struct MolDev {
  const int *grp_batch, *grp_tile, *grp_ntiles, *bt_off;  // density work groups: batch, first tile, tiles
  const int* b_chunk;       // chunk of each batch
  const ChunkDev* chunks;
  const int* ao_of;         // AO of each column of the chunks' tiles (-1: padding)
  const double *bx, *by, *bz;                                          // points
  BasisView bv;
  const unsigned short* cache;  // split operand cache
  int sstride, toff;            // slot stride; offset of the transposed layout
  const unsigned short* Ds;     // the chunks' dense blocks of D, split: [hi, lo][nu][mu] per chunk
  int npad, ntiles, nslots, pad_;
  double *part, *part_tau;      // density partials
  const int *slot_batch, *slot_tile;
  const double* coef;           // Vxc integrand coefficients per point
  unsigned short* bt;           // B^T per slot
  const MxItem* cwork;          // Vxc work items
  float* U;                     // the runs' blocks of V (upper): Phi_I^T B_J, and uplane on, B_I^T Phi_J
  long uplane;
  // core batches (points within the core radius of a nucleus with Z > 2): their
  // density runs with the AO operands split in three bf16 terms; cache3 holds
  // the third term of their slots' AOg blocks [core slot][c][g][mu],
  // core_off the first core slot of each batch (-1: not a core batch),
  // core_grps the density groups of the core batches, main_grps those of the
  // other batches (the (rho, grad rho) launch's groups; null: every group)
  const unsigned short* cache3;
  const int *core_off, *core_grps, *main_grps;
  const int* asym;  // == gen: this build's D is not symmetric (meta-GGA)
  int gen, pad2_;
};
constexpr int kMxMaxTiles = 512;  // basis size the mixed form takes (npad <= 16384): no kernel's limit, nothing larger was run
constexpr int kMxMaxChunk = 128;  // longest run a caller may ask for, batches per Vxc work item

// XC nuclear gradient (kernels_grad.hip), FP64 cached form. gpart: kGradCopies
// partial gradients of 3 natoms.
constexpr int kGradCopies = 64;
void launch_xgrad_xz(hipStream_t s, int ngroups, const int* grp_batch, const int* grp_tile, const int* grp_ntiles,
                     const int* bt_off, const int* b_chunk, const ChunkDev* chunks, const double* cache,
                     const double* bmat, const double* Dt, int c1, int c2, double* xz);
void launch_xgrad_epi(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile, const int* slot_grp,
                      const int* slot_q, const double* bx, const double* by, const double* bz, BasisView bv,
                      const double* coef, const double* xz, int natoms, double* gpart, double* grad);
// skeleton density derivatives (rho, grad rho per nuclear coordinate) into
// rhos[3 atom + t][npt points][4], accumulated (clear it first)
// Skeleton Fock derivative: E^t = a d_t phi + (c . grad) d_t phi per slot into
// etab[t][slot][g][column] (zero it first), then F[3 A + t] in the reference's
// order from Q^t = (d_t Phi)^T B (qp[t]) and P^t = Phi^T E^t (qp[3 + t]).
void launch_skel_etab(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile, const double* bx,
                      const double* by, const double* bz, BasisView bv, const double* coef, double* etab);
void launch_fock_skel_fin(hipStream_t s, int n, int npad, int natoms, const double* qp,
                          const int* ao_atom, double* F);
// XC energy Hessian terms into H (np x np, np = 3 natoms):
// the per-slot diagonal-atom term (AO third derivatives, X and Y^r from xz1 /
// xz2), the f_xc term of the first-order skeleton densities rhos, and the D
// term from rr[3 t + s] = (d_t Phi)^T E^s (npad^2 each, internal order).
void launch_hess_terms(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile, const int* slot_grp,
                       const int* slot_q, const double* bx, const double* by, const double* bz, BasisView bv,
                       const double* coef, const double* xz1, const double* xz2, long npt, const double* rhos,
                       const double* fx, const double* bw, int family, int npad, const double* Dint,
                       const double* rr, const int* atom, int np, double* hpart, double* H);
size_t hess_part_elems(long npt, int np);  // doubles of hpart (partial sums)
void launch_skel_rho(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile, const int* slot_grp,
                     const int* slot_q, const double* bx, const double* by, const double* bz, BasisView bv,
                     const double* xz1, const double* xz2, long npt, double* rhos);

// Mixed-precision form (kernels_mixed.hip): MFMA operands cached as bf16
// hi/lo pairs, split-BF16 MFMA contractions with FP32 accumulation, FP32
// recomputation of the AO values outside the MFMA operands.
constexpr int kMxComp = 2 * kTile * kBatch;  // elements per component and layout of a slot
// slot_core / cache3 (may be null): the third bf16 term of the AOg block of each
// slot with slot_core >= 0, at cache3 + slot_core * nT * kBatch * kTile
void launch_ao_cache_mx(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile,
                        const double* bx, const double* by, const double* bz, BasisView bv, int nT, int sstride,
                        unsigned short* cache, const int* slot_core, unsigned short* cache3);
// The chunks' dense blocks of D in split form (as launch_gather_d), and (all n^2
// elements) R: what the two terms leave of D, D - hi - lo, in FP32 and in D's
// own (reference, column-major) order; asym (may be null): *asym = gen when D is
// not symmetric to within rounding
void launch_split_d(hipStream_t s, int ntiles, int n, const double* D, const int* tile_chunk, const ChunkDev* chunks,
                    const int* ao_of, unsigned short* Ds, float* R, int* asym, int gen);
// V (reference order) from the runs' blocks U (float: the two products, sU elements
// apart; double: their sum, nmat matrices sU elements apart) and, with R, the first-order energy
// correction for the split of D: partial sums of V . R into cpart
// (assemble_blocks(n) of them); launch_reduce_corr sums nparts partials into *out.
int assemble_blocks(int n);
template <class T>  // float (mixed form) or double
void launch_assemble(hipStream_t s, int n, const int* rowptr, const RowRef* rows, const int* ao_of, const T* U,
                     double* V, const float* R, double* cpart, int nmat, size_t sU);
void launch_reduce_corr(hipStream_t s, int nparts, const double* cpart, double* out);
// the packed form: per molecule of the table, en[2 slot_en] += its ncpart partials
void launch_corr_multi(hipStream_t s, const char* base, const FnMolecule* fm, int nmol, double* en);
void launch_bf16_check(hipStream_t s, unsigned n, unsigned* bad);
void launch_fill_u32(hipStream_t s, unsigned* p, size_t n, unsigned v);
// One launch over the grid `one` (descriptor by value): density work groups,
// B^T slot blocks, Vxc work items. Density: rho, grad rho; with_tau: tau too.
// ncore_groups: the core groups' rho, grad rho with three-term operands too (GGA: in the same launch)
void launch_density_mx(hipStream_t s, int with_tau, int nitems, int ncore_groups, const MolDev& one);
// B^T of every slot for ncomp components
void launch_make_b_mx(hipStream_t s, int ncomp, const MolDev& one);
// wide: groups of up to kMxWideTiles tiles instead of kMxTiles
void launch_vxc_mx(hipStream_t s, int ncomp, int wide, int nitems, const MolDev& one);
// Persistent stage launches over many molecules (packs, LDA/GGA): tab holds one
// descriptor per molecule with byte offsets from base in place of pointers;
// starts (nmol + 1) the first item of each molecule in the stage's flat list.
enum { kStageDensity = 0, kStageCore = 1, kStageMakeB = 2, kStageVxc = 3, kStageVxcWide = 4 };
void launch_stage_multi(hipStream_t s, int stage, int ncomp, const char* base, const MolDev* tab, const int* starts,
                        int nmol, int total);

}  // namespace chx

// Opaque handle definitions.
namespace chx {
std::vector<AuxShell> aux_basis_shells(const chx_mol* m, const std::string& data_root, const std::string& basis);
}

struct chx_mol {
  int natoms = 0;
  std::vector<int> Z;
  std::vector<double> xyz;
  std::vector<chx::ShellH> shells;
  std::vector<double> exps, coefs;
  int nbasis = 0;
};

struct chx_mlp {
  hipStream_t stream = nullptr;
  chx::DevBuf<float> P, Prun, Pinf, M, V, loss;  // canonical, run (FP32), run (BF16-rounded); Adam state
  chx::DevBuf<float> Gpart;                      // per-block gradients and losses (kMlpGradBlocks of each)
  chx::DevBuf<unsigned> Wpk;                         // packed BF16 MFMA fragments of the inference weights
  chx::DevBuf<float> U, T, C;                        // training set: inputs, targets, sample weights
  std::vector<double> cprefix;                       // prefix sums of C (minibatch normalisation)
  long ndata = 0;
  int step = 0;
  bool have_box = false;
  chx::MlpBox box{};
  ~chx_mlp() {
    if (stream) (void)hipStreamDestroy(stream);
  }
};

struct chx_xc {
  std::vector<int> codes;
  int family = 0;
  double exx = 0;
  int spin = 1;
  const chx_mlp* surrogate = nullptr;  // when set, Evaluate runs the network (meta-GGA grids)
};

struct chx_grid {
  int device = 0;
  hipStream_t stream = nullptr;
  int nthreads = 1;
  int type = 0;
  int precision = CHX_PREC_FP64;
  double screen_thr = 1e-14;
  chx_mol mol;

  // AOs in the reference's order; matrices of the build (M) have npad rows.
  int nbasis = 0, npad = 0, ntiles = 0;
  std::vector<double> sh_xyz;
  std::vector<int> sh_type, sh_nprim, sh_poff, sh_atom, sh_ao;  // sh_ao: first AO of the shell
  std::vector<double> p_exp, p_coef;
  std::vector<int> tile_seg_off;
  std::vector<int4> seg;

  // Points: nbatches x kBatch slots (padding slots carry w = 0).
  long npoints = 0;
  int nbatches = 0;
  std::vector<int> batch_n;        // real points per batch
  std::vector<double> hx, hy, hz, hw;  // slot arrays (host copy)

  // Screening products (built by get_ao).
  bool ao_ready = false;
  // Bumped whenever the plan, the work lists or a buffer a captured pack graph
  // addresses may change (grid_plan, set_vxc_chunk, reallocations).
  unsigned long plan_gen = 0;
  std::vector<chx::ChunkDev> chunks;   // consecutive batches that share an AO list
  std::vector<int> chunk_b0;           // first batch of each chunk (and the end)
  std::vector<int> b_chunk, tile_chunk, ao_of;
  size_t dt_elems = 0;                 // elements of the chunks' dense blocks of D
  std::vector<int> seg_chunk;          // AO values recomputed: first chunk of each segment (and the end)
  size_t seg_elems = 0;                // ... elements of the largest segment's blocks of D
  std::vector<int> bt_off;             // first slot of each batch
  std::vector<int> grp_batch, grp_tile, grp_ntiles, grp_off;  // density work groups
  std::vector<chx::VxcItem> vwork;     // Vxc work items (64-AO super-tiles I <= J), AO values recomputed
  // Cached-AO path: phi and grad phi per alive (batch, tile) slot kept in HBM.
  bool cached = false;
  int cache_mode = -1;               // -1 automatic, 0 never, 1 always
  std::vector<int> slot_batch, slot_tile;
  int vxc_chunk = 0;                 // batches per Vxc work item; 0 = by the item count
  int min_run = 1;                   // ... and at least this many, where shorter runs' blocks have no room
  int vxc_shape = -1;                // mixed form's Vxc groups: -1 by basis size, 0 up to 4 tiles, 1 up to 5
  int mx_wide = 0;                   // mixed form: Vxc over groups of up to 5 tiles (large bases)
  std::vector<chx::MxItem> mwork;       // Vxc work items of the cached tables
  std::vector<chx::MxItem> pwork;       // FP64 form: items of the plain products (skeleton derivatives)
  size_t u_elems = 0;                   // elements of the runs' blocks of V (mixed form: of either product's)
  // mixed form: core batches (density with three-term operands)
  double core_radius = chx::kCoreRadius;  // bohr; 0 turns the core treatment off
  int ncore_batches = 0;
  std::vector<int> core_grps, main_grps;
  chx::DevBuf<unsigned short> d_cmx3;
  chx::DevBuf<int> d_core_off, d_core_grps, d_main_grps, d_slot_core;
  chx::DevBuf<double> d_cache, d_bmat, d_Mint;
  chx::DevBuf<int> d_slot_batch, d_slot_tile;
  chx::DevBuf<chx::MxItem> d_mwork, d_pwork;
  chx::DevBuf<chx::RowRef> d_rows;
  chx::DevBuf<int> d_rowptr;
  chx::DevBuf<float> d_U;
  chx::DevBuf<double> d_U64;
  chx::DevBuf<int> d_asym;              // number of the last build whose D was not symmetric
  int d_gen = 0;                        // builds counted
  chx::DevBuf<double> d_ws;             // derivative calls' workspace (Workspace in api.cpp)
  bool ws_live = false;
  chx::DevBuf<int> d_ao_atom;           // atom of each AO (-1: padding), with the slot tables below
  bool slot_tables = false;             // ... of this plan are on the device
  double flops_build = 0, mean_tiles = 0;
  std::vector<double> batch_work;  // g_b n_b^2 per batch (points x kept AOs squared)
  double core_flops = 0;           // the core batches' three-term (rho, grad rho) launch: 2 sum g_b n_b^2

  // Device mirrors.
  chx::DevBuf<double> d_sh_xyz, d_p_exp, d_p_coef;
  chx::DevBuf<chx::SegRec> d_segrec;
  int max_nprim = 0;
  // Mixed form: split AO cache (AOg + nT transposed components per slot), B^T, split D.
  chx::DevBuf<unsigned short> d_cmx, d_bmx, d_Dsplit;
  chx::MolDev hmol{};                 // descriptor of this grid (mixed form), passed to kernels by value
  int mx_sstride = 0, mx_nT = 0, bmx_comps = 0;
  chx::DevBuf<int> d_sh_type, d_sh_nprim, d_sh_poff, d_tile_seg_off, d_sh_atom;
  chx::DevBuf<int4> d_seg;
  chx::DevBuf<double> d_x, d_y, d_z, d_w;
  chx::DevBuf<int> d_bn;
  chx::DevBuf<chx::ChunkDev> d_chunks;
  chx::DevBuf<int> d_b_chunk, d_tile_chunk, d_ao_of;
  chx::DevBuf<int> d_bt_off, d_grp_batch, d_grp_tile, d_grp_ntiles, d_grp_off;
  chx::DevBuf<chx::VxcItem> d_vwork;
  chx::DevBuf<int> d_codes;

  // Per-iteration state.
  // d_en: E, N and (mixed form) the first-order correction for the split of D
  chx::DevBuf<double> d_Din, d_Dt, d_part, d_part_tau, d_rho, d_coef, d_en_part, d_en, d_Vout;
  // mixed form: D - hi - lo per spin (FP32, reference order) and the partial sums of V . (D - hi - lo)
  chx::DevBuf<float> d_Dres;
  chx::DevBuf<double> d_cpart;
  // corr_pending: the last Evaluate computed E and v in the mixed form, so the potential's build
  // adds the correction to E; corr_done: a build since then has; vout_ready: d_Vout holds that
  // potential (vout_nspin matrices)
  bool corr_pending = false, corr_done = false, vout_ready = false;
  int vout_nspin = 0;
  int v_family = 0;    // family of the potential on the grid (set by Evaluate / set_vrho)
  int en_blocks = 0;
  // XC gradient (Grid::getDensitySkeleton / getEnergyGrad)
  chx::DevBuf<double> d_Dskel, d_Dskel_t;  // D of the skeleton calls: npad^2, and its chunk blocks
  std::vector<int> slot_grp, slot_q;
  chx::DevBuf<int> d_slot_grp, d_slot_q;
  bool have_skeleton = false;
  bool have_density = false, have_eval = false, have_v = false;
  // response path: f_xc at the ground-state density, perturbed densities
  chx::DevBuf<double> d_fx, d_rhou;
  int fx_family = -1;  // family of the f_xc on the grid (-1: none)
  int fx_nspin = 1;    // spin count of that f_xc (2: kFxPol values per slot)
  int nmats_u = 0;     // perturbed densities held in d_rhou (per spin)
  int nspin_u = 1;     // spin count of those densities ([spin][mat] in d_rhou)
  // spin-polarised densities (nspin = 2): beta partials and coefficients; alpha in d_part / d_coef
  int nspin = 1;    // spin count of the density on the grid
  int v_nspin = 1;  // spin count of the potential on the grid
  chx::DevBuf<double> d_part_b, d_part_tau_b, d_coef_b, d_coef_save;
  // surrogate functional: points that fell back to the analytic functional in the last Evaluate
  chx::DevBuf<int> d_nfall;
  bool surrogate_used = false;

  // Optional per-kernel HIP-event timing (stage ids in chx_grid_kernel_times).
  bool profile = false;
  struct Pending { int stage; hipEvent_t a, b; };
  std::vector<Pending> pending;
  double stage_ms[8] = {0};
  long stage_n[8] = {0};
  void mark_begin(int stage, hipEvent_t* a);
  void mark_end(int stage, hipEvent_t a);
  void collect_times();
  int eval_family = -1;
  double last_E = 0, last_N = 0;

  chx::BasisView view() const;
};
