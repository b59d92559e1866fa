// Host-only checks of the library's planning and call code (gridgen.cpp, api.cpp): the HIP runtime and
// the kernel launches are replaced by the ones below, so that a plan, a call's arguments and what happens
// when memory runs out can be looked at without a GPU. Device memory is host memory under a byte budget;
// a launch checks that the tables it would read are there and returns.
//   host_plan <check> <data root>; exit status 0 when it holds.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <string>
#include <vector>

#include "internal.hpp"

// ---- the runtime ---------------------------------------------------------------------------------
namespace fake {
size_t budget = (size_t)64 << 30, used = 0;
std::map<char*, size_t> live;  // base -> bytes
hipError_t last = hipSuccess;
hipError_t done(hipError_t e) { return e == hipSuccess ? e : last = e; }
// p lies in a live allocation with at least n bytes behind it
bool at(const void* p, size_t n = 1) {
  auto it = live.upper_bound((char*)p);
  if (p == nullptr || it == live.begin()) return false;
  --it;
  return (char*)p + n <= it->first + it->second;
}
int failed = 0;
void check(bool ok, const char* what) {
  if (ok) return;
  ++failed;
  std::printf("FAILED: %s\n", what);
}
}  // namespace fake
#define CHECK(x) fake::check((x), #x)

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (fake::used + n > fake::budget) return fake::done(hipErrorOutOfMemory);
  *p = std::calloc(n ? n : 1, 1);
  fake::live[(char*)*p] = n;
  fake::used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = fake::live.find((char*)p);
  if (it == fake::live.end()) return hipSuccess;
  fake::used -= it->second;
  fake::live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = fake::budget > fake::used ? fake::budget - fake::used : 0;
  *t = fake::budget;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = fake::last;
  fake::last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}

// ---- the launches ----------------------------------------------------------------------------------
namespace chx {
using fake::at;
static void launched() { CHX_HIP(hipGetLastError()); }
std::vector<std::pair<std::string, const void*>> nulls;
int becke_ld(int natoms) { return natoms; }
void launch_becke(hipStream_t, long, const double*, const double*, const double*, double*, const int*, int,
                  const double*, const double2*, int) {}
void launch_bisect(hipStream_t, long n, const int* idx, const double* px, const double* py, const double* pz,
                   const std::vector<int>& levels, const BisSeg*, double* pts[2], int* ids[2]) {
  for (int k = 0; k < 2; ++k)  // in the points' own order
    for (long i = 0; i < n; ++i) {
      pts[k][i] = px[idx[i]];
      pts[k][n + i] = py[idx[i]];
      pts[k][2 * n + i] = pz[idx[i]];
      ids[k][i] = idx[i];
    }
}
void launch_batch_slots(hipStream_t, int nb, const int2* batch, const double* pts, const int* idx, long stride,
                        const double* w, double* bx, double* by, double* bz, double* bw) {
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < kBatch; ++k) {
      const int p = batch[b].x + (k < batch[b].y ? k : 0), s = b * kBatch + k;
      bx[s] = pts[p];
      by[s] = pts[stride + p];
      bz[s] = pts[2 * stride + p];
      bw[s] = k < batch[b].y ? w[idx[p]] : 0.0;
    }
}
void launch_screen(hipStream_t, int nb, int nsh, int nwords, const double* bx, const double* by, const double* bz,
                   const int* bn, const double* sh, const double* reach2, unsigned long long* alive) {
  for (int b = 0; b < nb; ++b)
    for (int s = 0; s < nsh; ++s)
      for (int k = 0; k < bn[b]; ++k) {
        const double x = bx[b * kBatch + k] - sh[3 * s], y = by[b * kBatch + k] - sh[3 * s + 1],
                     z = bz[b * kBatch + k] - sh[3 * s + 2];
        if (x * x + y * y + z * z < reach2[s]) alive[(size_t)b * nwords + (s >> 6)] |= 1ull << (s & 63);
      }
}
void launch_fill(hipStream_t, double* p, size_t n, double) { CHECK(n == 0 || at(p, n * sizeof(double))); launched(); }
void launch_fill_u32(hipStream_t, unsigned* p, size_t n, unsigned) { CHECK(n == 0 || at(p, n * 4)); launched(); }
void launch_ao_cache(hipStream_t, int, const int*, const int*, const double*, const double*, const double*, BasisView,
                     double*) { launched(); }
void launch_ao_cache_mx(hipStream_t, int, const int*, const int*, const double*, const double*, const double*,
                        BasisView, int, int, unsigned short*, const int*, unsigned short*) { launched(); }
std::vector<char> gathered;  // chunks whose blocks of D are in place
size_t density_groups = 0;   // density groups run since it was cleared
void launch_gather_d(hipStream_t, int ntiles, int, const double*, const int* tile_chunk, const ChunkDev* chunks,
                     const int*, double* Dt, int*, int, int nmat, size_t sO, int tile0, long d0) {
  gathered.assign(1 << 16, 0);
  for (int t = tile0; t < tile0 + ntiles; ++t) {
    const ChunkDev& c = chunks[tile_chunk[t]];
    CHECK(c.tile0 >= tile0 && c.tile0 + c.ntl <= tile0 + ntiles);  // whole chunks
    CHECK(at(Dt + (c.doff - d0)) && at(Dt + (nmat - 1) * sO + (c.doff - d0), 8192 * (size_t)c.ntl * c.ntl));
    gathered[tile_chunk[t]] = 1;
  }
  launched();
}
void launch_density_f64(hipStream_t, int mode, int ng, const int* batch, const int* tile, const int*,
                        const int* b_chunk, const ChunkDev* chunks, const double*, const double*, const double*,
                        BasisView, const double* Dt, long d0, double* part) {
  for (int k = 0; k < ng; ++k) {
    const ChunkDev& c = chunks[b_chunk[batch[k]]];
    CHECK(gathered[b_chunk[batch[k]]] && tile[k] >= c.tile0 && tile[k] < c.tile0 + c.ntl);
    CHECK(at(Dt + (c.doff - d0)) && at(Dt + (c.doff - d0), 8192 * (size_t)c.ntl * c.ntl));
  }
  CHECK(ng == 0 || at(part, ((size_t)(ng - 1) * (mode ? 3 : 4) + 1) * 512));
  density_groups += ng;
  launched();
}
void launch_point_rho(hipStream_t, int, const int*, const double* part, double* rhou, int, size_t) {
  CHECK(at(part) && at(rhou));
  launched();
}
void launch_vxc_f64(hipStream_t, int, int, const VxcItem*, const int*, const double*, const double*, const double*,
                    const double*, BasisView, double* M, int npad) { CHECK(at(M, 8 * npad * npad)); launched(); }
void launch_finalize_sym(hipStream_t, int, int, const double*, double* V) { CHECK(at(V)); launched(); }
void launch_pad_d(hipStream_t, int, int npad, const double*, double* D) {
  CHECK(at(D, sizeof(double) * npad * npad));
  launched();
}
void launch_density_c64(hipStream_t, int, const int*, const int*, const int*, const int*, const int*, const ChunkDev*,
                        const double*, const double*, const int*, int, double* part, double*, int, size_t, size_t,
                        double*) { CHECK(at(part)); launched(); }
void launch_functional(hipStream_t, int, const int* off, const double*, const double*, const double*, const int*, int,
                       int, int, int, double*, double*, double*, int) { CHECK(at(off)); launched(); }
void launch_functional_f(hipStream_t, int, const int*, const double*, const int*, int, int, double*) { launched(); }
void launch_reduce_en(hipStream_t, int, const double*, double* en) { CHECK(at(en)); launched(); }
void launch_split_d(hipStream_t, int, int, const double*, const int*, const ChunkDev*, const int*, unsigned short* Ds,
                    float* R, int*, int) { CHECK(at(Ds) && at(R)); launched(); }
void launch_density_mx(hipStream_t, int, int, int, const MolDev& m) { CHECK(at(m.part)); launched(); }
void launch_make_b_mx(hipStream_t, int, const MolDev& m) { CHECK(at(m.bt)); launched(); }
void launch_vxc_mx(hipStream_t, int, int, int nitems, const MolDev& m) {
  for (int k = 0; k < nitems; ++k) CHECK(at(m.cwork + k, sizeof(MxItem)) && at(m.U + m.cwork[k].u) && at(m.U + m.uplane + m.cwork[k].u));
  launched();
}
void launch_reduce_corr(hipStream_t, int, const double*, double* out) { CHECK(at(out)); launched(); }
void launch_make_b(hipStream_t, int, const int*, const double*, const double*, double* b, int, size_t, size_t,
                   const double*) { CHECK(at(b)); launched(); }
void launch_vxc_c64(hipStream_t, int, int nwork, const MxItem*, const double*, const double*, const double*, double* U,
                    int, size_t, size_t) { CHECK(nwork == 0 || at(U)); launched(); }
int assemble_blocks(int n) { return n; }
template <class T>
void launch_assemble(hipStream_t, int n, const int* rowptr, const RowRef* rows, const int*, const T* U, double* V,
                     const float*, double*, int nmat, size_t sU) {
  const size_t last = sizeof(T) == 4 ? sU : (nmat - 1) * sU;
  CHECK(at(rowptr, 4 * (n + 1)) && at(V, sizeof(double) * n * n));
  for (int e = 0; e < rowptr[n]; ++e) CHECK(at(U + rows[e].u, sizeof(T) * rows[e].len) && at(U + last + rows[e].u, sizeof(T) * rows[e].len));
  launched();
}
template void launch_assemble<float>(hipStream_t, int, const int*, const RowRef*, const int*, const float*, double*,
                                     const float*, double*, int, size_t);
template void launch_assemble<double>(hipStream_t, int, const int*, const RowRef*, const int*, const double*, double*,
                                      const float*, double*, int, size_t);
void launch_xgrad_xz(hipStream_t, int, const int*, const int*, const int*, const int*, const int*, const ChunkDev*,
                     const double*, const double*, const double*, int, int, double*) { launched(); }
void launch_skel_rho(hipStream_t, int, const int*, const int*, const int*, const int*, const double*, const double*,
                     const double*, BasisView, const double*, const double*, long, double*) { launched(); }
void launch_skel_etab(hipStream_t, int, const int*, const int*, const double*, const double*, const double*, BasisView,
                      const double*, double*) { launched(); }
void launch_prod_c64(hipStream_t, int, const MxItem*, const int*, const double*, const double*, double*, int, int,
                     const ProdBatch&) { launched(); }
void launch_fock_skel_fin(hipStream_t, int n, int, int, const double*, const int* ao_atom, double*) {
  CHECK(at(ao_atom, sizeof(int) * n));  // read for every AO
  launched();
}
size_t hess_part_elems(long, int np) { return (size_t)np * np; }
void launch_hess_terms(hipStream_t, int, const int*, const int*, const int*, const int*, const double*, const double*,
                       const double*, BasisView, const double*, const double*, const double*, long, const double*,
                       const double*, const double*, int, int npad, const double*, const double*, const int* atom, int,
                       double*, double*) {
  CHECK(at(atom, sizeof(int) * npad));  // read for every AO and padding column
  launched();
}
}  // namespace chx

// ---- the checks --------------------------------------------------------------------------------------
namespace {
std::string root;

// nat hydrogens 2 bohr apart with nsh s shells each (exponents 0.1 .. 1: everything overlaps everything), SG-1
chx_grid* grid(int nat, int nsh, double expo = 0.1) {
  std::vector<int> Z(nat, 1);
  std::vector<double> xyz(3 * nat, 0.0);
  for (int a = 0; a < nat; ++a) xyz[3 * a] = 2.0 * a;
  chx_mol* m;
  chx_grid* g;
  CHECK(chx_mol_create(nat, Z.data(), xyz.data(), &m) == CHX_OK);
  for (int a = 0; a < nat; ++a)
    for (int k = 0; k < nsh; ++k) {
      const double e = expo * (1 + 9.0 * k / nsh), c = 1;
      CHECK(chx_mol_add_shell(m, a, 0, 1, &e, &c) == CHX_OK);
    }
  if (chx_grid_create(m, "SG-1", root.c_str(), 1, 0, &g) != CHX_OK) {
    std::printf("%s\n", chx_last_error());
    std::exit(2);
  }
  chx_mol_destroy(m);
  return g;
}
chx_xc* functional(int code) {
  chx_xc* xc;
  CHECK(chx_xc_create(1, &code, 1, &xc) == CHX_OK);
  return xc;
}

// Skeleton calls on a plan whose threshold leaves no shell alive.
void empty_lists() {
  chx_grid* g = grid(2, 3);
  const int n = 6;
  chx_xc* xc = functional(1);
  std::vector<double> D(n * n, 0.1), F(6 * n * n), H(36);
  for (double thr : {1e6, 1e-14}) {  // the second plan has slots
    CHECK(chx_grid_set_screening(g, thr) == CHX_OK);
    CHECK(chx_grid_get_ao(g, 0, 0) == CHX_OK);
    CHECK((g->slot_tile.size() == 0) == (thr > 1));
    CHECK(chx_grid_get_density(g, D.data(), 1, n) == CHX_OK);
    CHECK(chx_xc_evaluate(xc, g, "ev") == CHX_OK);
    CHECK(chx_grid_fock(g, F.data(), 1, n) == CHX_OK);
    CHECK(chx_xc_evaluate(xc, g, "f") == CHX_OK);
    CHECK(chx_grid_get_density_skeleton(g, D.data(), 1, n) == CHX_OK);
    CHECK(chx_grid_fock_skeleton(g, F.data(), 1, n) == CHX_OK);
    CHECK(chx_grid_energy_hess(g, H.data()) == CHX_OK);
  }
  chx_xc_destroy(xc);
  chx_grid_destroy(g);
}

int build(chx_grid* g, const chx_xc* xc, const std::vector<double>& D, std::vector<double>& F) {
  int rc = chx_grid_get_density(g, D.data(), 1, g->nbasis);
  if (rc == CHX_OK) rc = chx_xc_evaluate(xc, g, "ev");
  if (rc == CHX_OK) rc = chx_grid_fock(g, F.data(), 1, g->nbasis);
  return rc;
}

// Run lengths and plans that do not fit: the call fails, and what was there before stays usable or is
// known to be gone (no call reaches a freed table).
void failed_plans() {
  const size_t all = fake::budget;
  for (int form : {CHX_PREC_FP64, CHX_PREC_MIXED}) {
    chx_grid* g = grid(1, 300);
    chx_xc* xc = functional(1);
    const int n = g->nbasis;
    std::vector<double> D((size_t)n * n, 0.1), F((size_t)n * n);
    CHECK(chx_grid_set_precision(g, form) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK && g->cached);
    CHECK(chx_grid_set_vxc_chunk(g, 4) == CHX_OK);
    CHECK(build(g, xc, D, F) == CHX_OK);
    const size_t u = g->u_elems, per = 8;  // (mixed form: two FP32 products)
    // shorter runs: more blocks than there is room for
    fake::budget = fake::used + u * per;
    const unsigned long gen = g->plan_gen;
    CHECK(chx_grid_set_vxc_chunk(g, 1) == CHX_ERR_DEVICE);
    CHECK(g->ao_ready && g->plan_gen != gen && g->vxc_chunk == 4 && g->u_elems == u);
    CHECK(fake::at(form == CHX_PREC_FP64 ? (void*)g->d_U64.p : (void*)g->d_U.p, u * per));
    if (form == CHX_PREC_MIXED) CHECK(g->hmol.U == g->d_U.p && g->hmol.cwork == g->d_mwork.p);
    CHECK(chx_grid_fock(g, F.data(), 1, n) == CHX_OK && build(g, xc, D, F) == CHX_OK);
    // no room for any: the plan is gone, and getAO makes another of it
    fake::budget = 0;
    CHECK(chx_grid_set_vxc_chunk(g, 1) == CHX_ERR_DEVICE);
    CHECK(!g->ao_ready && g->vxc_chunk == 4);
    CHECK(chx_grid_fock(g, F.data(), 1, n) == CHX_ERR_STATE && build(g, xc, D, F) == CHX_ERR_STATE);
    fake::budget = all;
    CHECK(chx_grid_get_ao(g, 0, 0) == CHX_OK && build(g, xc, D, F) == CHX_OK && g->u_elems == u);
    // a plan that fails half way
    CHECK(chx_grid_set_type(g, 2) == CHX_OK);
    fake::budget = fake::used;
    CHECK(chx_grid_get_ao(g, 0, 0) != CHX_OK);
    CHECK(chx_grid_fock(g, F.data(), 1, n) == CHX_ERR_STATE && build(g, xc, D, F) == CHX_ERR_STATE);
    fake::budget = all;
    CHECK(chx_grid_get_ao(g, 0, 0) == CHX_OK && build(g, xc, D, F) == CHX_OK);
    if (form == CHX_PREC_MIXED) {  // the other group size
      CHECK(chx_grid_set_vxc_shape(g, 0) == CHX_OK && chx_grid_set_vxc_chunk(g, 1) == CHX_OK);
      fake::budget = 0;
      CHECK(chx_grid_set_vxc_shape(g, 1) == CHX_ERR_DEVICE || g->d_U.p);
      CHECK(chx_grid_fock(g, F.data(), 1, n) == (g->ao_ready ? CHX_OK : CHX_ERR_STATE));
      fake::budget = all;
    }
    chx_xc_destroy(xc);
    chx_grid_destroy(g);
  }
}

// Plans under a byte budget: longer runs, longer chunks, the form without tables and its segments, in
// this order, and every build within the budget.
void budgets() {
  const size_t all = fake::budget;
  for (int form : {CHX_PREC_FP64, CHX_PREC_MIXED}) {
    chx_grid* g = grid(4, 160);  // 640 AOs, all alive in most batches
    chx_xc* xc = functional(1);
    const int n = g->nbasis;
    std::vector<double> D((size_t)n * n, 0.1), F((size_t)n * n);
    CHECK(chx_grid_set_precision(g, form) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK && g->cached);
    size_t slots = 0;
    for (const chx::ChunkDev& c : g->chunks) slots += (size_t)c.nb * c.ntl;
    const double table = slots * (form == CHX_PREC_MIXED ? 3.0 * chx::kMxComp * 2 : 5.0 * 2048 * 8);
    const double blocks = form == CHX_PREC_MIXED ? 4.0 * g->dt_elems + 8.0 * g->u_elems
                                                 : 8.0 * g->dt_elems + 8.0 * g->u_elems;
    const size_t u0 = g->u_elems, d0 = g->dt_elems, chunks0 = g->chunks.size();
    chx_grid_destroy(g);
    const double share = form == CHX_PREC_MIXED ? 0.9 : 0.8;
    int longer_runs = 0, longer_chunks = 0, recomputed = 0, refused = 0;
    for (double f = 1.2; f > 0.02; f *= 0.93) {  // room for the tables and f of their blocks, down to a part of the tables
      g = grid(4, 160);
      CHECK(chx_grid_set_precision(g, form) == CHX_OK);
      const double room = f > 0.1 ? table + f * blocks : table * f / 0.1;
      fake::budget = fake::used + (size_t)(room / share);
      const int rc = chx_grid_get_ao(g, 0, 0);
      if (rc != CHX_OK) {
        CHECK(form == CHX_PREC_MIXED && room < table + blocks);
        ++refused;
      } else {
        CHECK(g->cached || form == CHX_PREC_FP64);
        chx::density_groups = 0;
        CHECK(build(g, xc, D, F) == CHX_OK);
        if (!g->cached) {
          CHECK(chx::density_groups == g->grp_batch.size());
          CHECK(chx_grid_get_density_u(g, D.data(), 1, 1, n) == CHX_OK);
          CHECK(chx::density_groups == 2 * g->grp_batch.size());
          ++recomputed;
        } else if (g->dt_elems < d0) {
          ++longer_chunks;
        } else if (g->u_elems < u0) {
          ++longer_runs;
        }
        for (const chx::ChunkDev& c : g->chunks) CHECK(c.nb <= chx::kChunkLong);
      }
      fake::budget = all;
      chx_grid_destroy(g);
    }
    std::printf("form %d: %zu chunks; plans with longer runs %d, longer chunks %d, without tables %d, refused %d\n", form,
                chunks0, longer_runs, longer_chunks, recomputed, refused);
    CHECK(longer_runs > 0 && longer_chunks > 0);
    CHECK(form == CHX_PREC_MIXED ? refused > 0 : recomputed > 0);
    chx_xc_destroy(xc);
  }
}

// A grid planned again has the room of its former plan: the same tables, also where both would not fit,
// and the other form's tables in the place of its own.
void planned_again() {
  const size_t all = fake::budget;
  for (int form : {CHX_PREC_FP64, CHX_PREC_MIXED}) {
    chx_grid* g = grid(2, 160);
    chx_xc* xc = functional(1);
    const int n = g->nbasis;
    std::vector<double> D((size_t)n * n, 0.1), F((size_t)n * n);
    const size_t before = fake::used;
    CHECK(chx_grid_set_precision(g, form) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK && g->cached);
    const size_t u = g->u_elems, d = g->dt_elems;
    fake::budget = before + (fake::used - before) * 3 / 2;
    for (double thr : {1e-13, 1e-14}) {
      CHECK(chx_grid_set_screening(g, thr) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK && g->cached);
      CHECK(build(g, xc, D, F) == CHX_OK);
    }
    CHECK(g->u_elems == u && g->dt_elems == d && g->min_run == 1);
    CHECK(chx_grid_set_precision(g, form == CHX_PREC_FP64 ? CHX_PREC_MIXED : CHX_PREC_FP64) == CHX_OK);
    CHECK(chx_grid_get_ao(g, 0, 0) == CHX_OK && build(g, xc, D, F) == CHX_OK);
    CHECK(chx_grid_set_precision(g, form) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK && g->cached);
    CHECK(build(g, xc, D, F) == CHX_OK && g->u_elems == u);
    fake::budget = all;
    chx_xc_destroy(xc);
    chx_grid_destroy(g);
  }
}

// A shell is in the list of every batch in which one of its components or their derivatives exceeds the
// threshold: contractions of steep and diffuse primitives of either sign, coarse thresholds, exponents of 0.
void reaches() {
  std::mt19937 rng(3);
  auto uni = [&](double a, double b) { return a + (b - a) * (rng() / 4294967296.0); };
  for (int trial = 0; trial < 60; ++trial) {
    chx_mol* m;
    chx_grid* g;
    const int Z = 1;
    const double at[3] = {0, 0, 0};
    CHECK(chx_mol_create(1, &Z, at, &m) == CHX_OK);
    static const int types[] = {0, 1, -2, -3};
    std::vector<std::vector<double>> e, c;
    for (int k = 0; k < 12; ++k) {
      const int np = 1 + rng() % 4;
      std::vector<double> ee, cc;
      for (int p = 0; p < np; ++p) {
        ee.push_back(trial % 6 == 5 && p == 0 ? (k % 2 ? 0.0 : -1e-4) : std::pow(10.0, uni(-2, 6)));
        cc.push_back(uni(-1, 1) * std::pow(10.0, uni(-2, 2)));
      }
      CHECK(chx_mol_add_shell(m, 0, types[k % 4], np, ee.data(), cc.data()) == CHX_OK);
      e.push_back(ee);
      c.push_back(cc);
    }
    CHECK(chx_grid_create(m, "SG-1", root.c_str(), 1, 0, &g) == CHX_OK);
    for (double thr : {0.0, 1e-14, 1e-6, 1e-3, 0.1, 1.0, 30.0}) {
      CHECK(chx_grid_set_screening(g, thr) == CHX_OK && chx_grid_get_ao(g, 0, 0) == CHX_OK);
      int missing = 0;
      for (int k = 0; k < 12; ++k)
        for (int b = 0; b < g->nbatches; ++b) {
          const chx::ChunkDev& ch = g->chunks[g->b_chunk[b]];
          bool listed = false;
          for (int i = 0; i < ch.ntl * chx::kTile; ++i) listed |= g->ao_of[ch.tile0 * chx::kTile + i] == g->sh_ao[k];
          if (listed) continue;
          for (int i = 0; i < g->batch_n[b]; ++i) {
            const double x = g->hx[b * chx::kBatch + i], y = g->hy[b * chx::kBatch + i], z = g->hz[b * chx::kBatch + i];
            double A = 0, A1 = 0;
            for (size_t p = 0; p < e[k].size(); ++p) {
              const double t = c[k][p] * std::exp(-e[k][p] * (x * x + y * y + z * z));
              A += t;
              A1 -= 2 * e[k][p] * t;
            }
            // one component of the type and its gradient
            const double q[4] = {1, x, std::sqrt(3.0) * x * y, z * (z * z - 1.5 * (x * x + y * y))};
            const double dx[4] = {0, 1, std::sqrt(3.0) * y, -3 * x * z}, dz[4] = {0, 0, 0, 3 * z * z - 1.5 * (x * x + y * y)};
            const int t = k % 4;
            const double v = std::max({std::fabs(A * q[t]), std::fabs(A1 * x * q[t] + A * dx[t]),
                                       std::fabs(A1 * z * q[t] + A * dz[t])});
            missing += v > thr * (1 + 1e-12);
          }
        }
      if (missing) std::printf("trial %d threshold %g: %d values above it left out\n", trial, thr, missing);
      CHECK(missing == 0);
    }
    chx_grid_destroy(g);
    chx_mol_destroy(m);
  }
}
}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> checks = {
      {"empty_lists", empty_lists}, {"failed_plans", failed_plans}, {"budgets", budgets}, {"planned_again", planned_again}, {"reaches", reaches}};
  if (argc != 3 || !checks.count(argv[1])) return 2;
  root = argv[2];
  checks.at(argv[1])();
  std::printf("%s: %s\n", argv[1], fake::failed ? "failed" : "ok");
  return fake::failed != 0;
}
