// Grid construction and batch planning (host side).
//
// Restates Grid::Grid (src/Grid/GridGeneration.cpp:27-162,232-310) for the
// GPU: atom-centred Lebedev x radial points, Becke partition weights (FP64,
// on the device), then this build's own batching: spatially compact batches
// of 64 points (recursive bisection along the longest box edge) instead of
// the reference's 128-point halves of the generation order. Batch membership
// changes only the order of summation.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <fstream>
#include <numeric>
#include <sstream>

#include "internal.hpp"

namespace chx {
namespace {

struct LebOrbit { int type; double a, b, v; };
struct LebRule { int n, first, count; };
#include "lebedev_table.inc"

const char* kElemNames[] = {"", "H", "He", "Li", "Be", "B", "C", "N", "O", "F", "Ne", "Na", "Mg", "Al", "Si",
                            "P", "S", "Cl", "Ar", "K", "Ca", "Sc", "Ti", "V", "Cr", "Mn", "Fe", "Co", "Ni",
                            "Cu", "Zn", "Ga", "Ge", "As", "Se", "Br", "Kr"};

// Octahedral orbit of a generator (Lebedev-Laikov types 1-6).
void expand_orbit(const LebOrbit& o, std::vector<std::array<double, 4>>& out) {
  double g[3];
  switch (o.type) {
    case 1: g[0] = 1; g[1] = 0; g[2] = 0; break;
    case 2: g[0] = 0; g[1] = g[2] = std::sqrt(0.5); break;
    case 3: g[0] = g[1] = g[2] = std::sqrt(1.0 / 3.0); break;
    case 4: g[0] = g[1] = o.a; g[2] = std::sqrt(1.0 - 2.0 * o.a * o.a); break;
    case 5: g[0] = o.a; g[1] = std::sqrt(1.0 - o.a * o.a); g[2] = 0; break;
    case 6: g[0] = o.a; g[1] = o.b; g[2] = std::sqrt(1.0 - o.a * o.a - o.b * o.b); break;
    default: throw Error(CHX_ERR_ARG, "bad Lebedev orbit");
  }
  static const int perm[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
  std::vector<std::array<double, 3>> base;
  for (const auto& p : perm) {
    std::array<double, 3> c = {g[p[0]], g[p[1]], g[p[2]]};
    if (std::find(base.begin(), base.end(), c) == base.end()) base.push_back(c);
  }
  for (const auto& c : base)
    for (int s = 0; s < 8; ++s) {
      const double sx = (s & 1) ? -1.0 : 1.0, sy = (s & 2) ? -1.0 : 1.0, sz = (s & 4) ? -1.0 : 1.0;
      if ((c[0] == 0 && sx < 0) || (c[1] == 0 && sy < 0) || (c[2] == 0 && sz < 0)) continue;
      out.push_back({sx * c[0], sy * c[1], sz * c[2], o.v});
    }
}

const std::vector<std::array<double, 4>>& lebedev(int n) {
  static std::vector<std::vector<std::array<double, 4>>> cache(6000);
  if (n <= 0 || n >= (int)cache.size()) throw Error(CHX_ERR_FILE, "Lebedev rule not available");
  auto& r = cache[n];
  if (!r.empty()) return r;
  for (const LebRule& lr : kLebRules) {
    if (lr.n != n) continue;
    for (int k = 0; k < lr.count; ++k) expand_orbit(kLebOrbits[lr.first + k], r);
    if ((int)r.size() != n) throw Error(CHX_ERR_FILE, "Lebedev expansion size mismatch");
    return r;
  }
  throw Error(CHX_ERR_FILE, "Lebedev rule not available");
}

struct Radial { std::vector<double> r, w; std::vector<int> nang; };

// .grid file (Grids/README.md:1-11): "ngroups nshells", radial line ("em R" or
// "de2 alpha xmin xmax"), then "npoints nshells" per group from the nucleus out.
Radial read_grid_file(const std::string& path) {
  std::ifstream f(path);
  if (!f.good()) throw Error(CHX_ERR_FILE, "Missing element grid file in folder!");
  std::string line;
  int ngroups = 0, ntot = 0;
  if (!std::getline(f, line)) throw Error(CHX_ERR_FILE, "Corrupted grid file");
  { std::stringstream ss(line); ss >> ngroups >> ntot; }
  if (ngroups <= 0 || ntot <= 1) throw Error(CHX_ERR_FILE, "Corrupted grid file");
  if (!std::getline(f, line)) throw Error(CHX_ERR_FILE, "Corrupted grid file");
  std::stringstream ss(line);
  std::string formula;
  ss >> formula;
  Radial R;
  R.r.resize(ntot);
  R.w.resize(ntot);
  if (formula == "de2") {  // GridGeneration.cpp:90-100
    double alpha, x0, x1;
    ss >> alpha >> x0 >> x1;
    const double h = (x1 - x0) / (double)(ntot - 1);
    for (int i = 0; i < ntot; ++i) {
      const double xi = h * i + x0;
      R.r[i] = std::exp(alpha * xi - std::exp(-xi));
      R.w[i] = std::exp(3 * alpha * xi - 3 * std::exp(-xi)) * (alpha + std::exp(-xi)) * h;
    }
  } else if (formula == "em") {  // GridGeneration.cpp:103-113
    double Rm;
    ss >> Rm;
    for (int i = 0; i < ntot; ++i) {
      const double ii = i + 1;
      R.r[i] = Rm * std::pow(ii / (ntot + 1 - ii), 2);
      R.w[i] = 2 * std::pow(Rm, 3) * (ntot + 1) * std::pow(ii, 5) / std::pow(ntot + 1 - ii, 7);
    }
  } else {
    throw Error(CHX_ERR_FILE, "Unrecognized radial formula!");
  }
  for (int k = 0; k < ngroups; ++k) {
    if (!std::getline(f, line)) throw Error(CHX_ERR_FILE, "Corrupted grid file");
    std::stringstream gs(line);
    int npts = 0, nsh = 0;
    gs >> npts >> nsh;
    for (int s = 0; s < nsh; ++s) R.nang.push_back(npts);
  }
  if ((int)R.nang.size() != ntot) throw Error(CHX_ERR_FILE, "Corrupted grid file");
  return R;
}

// Nuclei with Z > 2 by cells of at least 1 bohr over their bounding box, to find
// the nucleus (if any) within r <= 1 bohr of a point. A cell lists the nuclei of
// the 27 cells around it, so that a point reads one cell (mostly an empty one): a
// hash table asked for 27 keys per point took half of a geometry step's host time.
struct HeavyCells {
  const std::vector<double>& xyz;
  double lo[3] = {0, 0, 0}, h = 1 + 1e-6;  // the edge: 1 bohr and a margin for rounding
  long n[3] = {0, 0, 0};
  std::vector<int> start, atoms;  // cell c: atoms[start[c]] .. atoms[start[c + 1]]
  HeavyCells(const chx_mol& m) : xyz(m.xyz) {
    std::vector<int> heavy;
    double hi[3] = {0, 0, 0};
    for (int a = 0; a < m.natoms; ++a) {
      const double* c = &xyz[3 * a];
      if (m.Z[a] <= 2 || !(std::fabs(c[0]) + std::fabs(c[1]) + std::fabs(c[2]) < 1e100)) continue;
      for (int d = 0; d < 3; ++d) {
        lo[d] = heavy.empty() ? c[d] : std::min(lo[d], c[d]);
        hi[d] = heavy.empty() ? c[d] : std::max(hi[d], c[d]);
      }
      heavy.push_back(a);
    }
    if (heavy.empty()) return;
    auto cells = [&] {
      double c = 1;
      for (int d = 0; d < 3; ++d) c *= std::floor((hi[d] - lo[d]) / h) + 4;
      return c;
    };
    while (cells() > 1 << 21) h *= 2;
    for (int d = 0; d < 3; ++d) {
      lo[d] -= 2 * h;  // so that no nucleus is in an outermost cell
      n[d] = (long)std::floor((hi[d] - lo[d]) / h) + 2;
    }
    std::vector<int> count((size_t)(n[0] * n[1] * n[2]) + 1, 0);
    auto each = [&](auto&& f) {  // the cells around each nucleus
      for (int d = 0; d < 27; ++d)
        for (int a : heavy) {
          long c[3];
          for (int k = 0; k < 3; ++k) c[k] = (long)std::floor((xyz[3 * a + k] - lo[k]) / h);
          f(((c[0] + d / 9 - 1) * n[1] + c[1] + d / 3 % 3 - 1) * n[2] + c[2] + d % 3 - 1, a);
        }
    };
    each([&](long c, int) { ++count[c + 1]; });
    for (size_t c = 1; c < count.size(); ++c) count[c] += count[c - 1];
    start = count;
    atoms.resize(start.back());
    each([&](long c, int a) { atoms[count[c]++] = a; });
  }
  long cell(double x, double y, double z) const {  // -1: outside
    const double c[3] = {std::floor((x - lo[0]) / h), std::floor((y - lo[1]) / h), std::floor((z - lo[2]) / h)};
    for (int d = 0; d < 3; ++d)
      if (!(c[d] >= 0 && c[d] < (double)n[d])) return -1;
    return ((long)c[0] * n[1] + (long)c[1]) * n[2] + (long)c[2];
  }
  // a heavy atom within sqrt(r2) of (x, y, z), sqrt(r2) <= 1; -1 if none
  int near(double x, double y, double z, double r2) const {
    if (atoms.empty()) return -1;
    const long c = cell(x, y, z);
    if (c < 0) return -1;
    for (int k = start[c]; k < start[c + 1]; ++k) {
      const int a = atoms[k];
      const double ex = x - xyz[3 * a], ey = y - xyz[3 * a + 1], ez = z - xyz[3 * a + 2];
      if (ex * ex + ey * ey + ez * ez < r2) return a;
    }
    return -1;
  }
};

// Recursive bisection into batches of exactly kBatch points (one remainder): what
// goes to the left depends on the numbers of points only, so all levels' segments
// are known before any point has moved. levels: first segment of each level, and the end.
void bisect_plan(const std::vector<long>& sets, std::vector<BisSeg>& segs, std::vector<int>& levels,
                 std::vector<int2>& batches) {
  std::vector<BisSeg> cur;
  auto add = [&](std::vector<BisSeg>& v, long lo, long n) {
    if (n > 0) v.push_back(BisSeg{(int)lo, (int)n, n <= kBatch ? 0 : kBatch * (int)((n + kBatch - 1) / kBatch / 2)});
  };
  for (size_t k = 0; k + 1 < sets.size(); ++k) add(cur, sets[k], sets[k + 1] - sets[k]);
  levels.assign(1, 0);
  while (std::any_of(cur.begin(), cur.end(), [](const BisSeg& s) { return s.left > 0; })) {
    segs.insert(segs.end(), cur.begin(), cur.end());
    levels.push_back((int)segs.size());
    std::vector<BisSeg> next;
    for (const BisSeg& s : cur) {
      add(next, s.lo, s.left ? s.left : s.n);
      if (s.left) add(next, s.lo + s.left, s.n - s.left);
    }
    cur.swap(next);
  }
  for (const BisSeg& s : cur) batches.push_back(make_int2(s.lo, s.n));
}

}  // namespace

const std::vector<std::array<double, 4>>& lebedev_rule(int n) { return lebedev(n); }

void ensure_stream(chx_grid* g) {
  if (g->stream) return;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) throw Error(CHX_ERR_DEVICE, "no HIP device available");
  CHX_HIP(hipGetDevice(&g->device));
  CHX_HIP(hipStreamCreate(&g->stream));
}

// Build points, weights, batches and the internal AO layout.
void grid_build(chx_grid* g, const std::string& grid_name, const std::string& data_root) {
  const chx_mol& m = g->mol;
  const int nat = m.natoms;
  if (nat <= 0) throw Error(CHX_ERR_ARG, "molecule has no atoms");
  if (m.nbasis <= 0) throw Error(CHX_ERR_ARG, "molecule has no basis");
  // ---- atom-centred points in generation order (atom -> shell -> angular point)
  std::vector<double> px, py, pz, pw;
  std::vector<int> owner;
  std::vector<Radial> radial(37);  // one file per element
  for (int a = 0; a < nat; ++a) {
    const int Z = m.Z[a];
    if (Z < 1 || Z > 36) throw Error(CHX_ERR_ARG, "unsupported element");
    Radial& R = radial[Z];
    if (R.r.empty()) R = read_grid_file(data_root + "/Grids/" + grid_name + "/" + kElemNames[Z] + ".grid");
    const double* c = &m.xyz[3 * a];
    for (size_t s = 0; s < R.r.size(); ++s) {
      const auto& L = lebedev(R.nang[s]);
      for (const auto& l : L) {
        px.push_back(l[0] * R.r[s] + c[0]);
        py.push_back(l[1] * R.r[s] + c[1]);
        pz.push_back(l[2] * R.r[s] + c[2]);
        pw.push_back(R.w[s] * 4 * M_PI * l[3]);
        owner.push_back(a);
      }
    }
  }
  const long G = (long)px.size();
  if (G > (1l << 30)) throw Error(CHX_ERR_UNSUPPORTED, "more than 2^30 grid points");
  // ---- Becke weights on the device (FP64); the data files are all read by now
  ensure_stream(g);
  DevBuf<double> dx, dy, dz, dw;
  {
    const int ld = becke_ld(nat);
    std::vector<double2> rab((size_t)nat * ld, make_double2(1.0, 1.0));
    for (int b = 0; b < nat; ++b)
      for (int c = 0; c < nat; ++c) {
        if (b == c) continue;
        const double dx = m.xyz[3 * b] - m.xyz[3 * c], dy = m.xyz[3 * b + 1] - m.xyz[3 * c + 1],
                     dz = m.xyz[3 * b + 2] - m.xyz[3 * c + 2];
        const double R = std::sqrt(dx * dx + dy * dy + dz * dz);
        rab[(size_t)b * ld + c] = make_double2(R, 1.0 / R);
      }
    DevBuf<double> dxyz;
    DevBuf<double2> drab;
    DevBuf<int> down;
    dx.upload(px, g->stream); dy.upload(py, g->stream); dz.upload(pz, g->stream); dw.upload(pw, g->stream);
    down.upload(owner, g->stream);
    dxyz.upload(m.xyz, g->stream);
    drab.upload(rab, g->stream);
    launch_becke(g->stream, G, dx.p, dy.p, dz.p, dw.p, down.p, nat, dxyz.p, drab.p, ld);
    CHX_HIP(hipMemcpyAsync(pw.data(), dw.p, sizeof(double) * G, hipMemcpyDeviceToHost, g->stream));
    CHX_HIP(hipStreamSynchronize(g->stream));
  }
  // ---- drop exactly-zero weights, batch the rest spatially
  // The points within kCoreRadius of a nucleus with Z > 2 (atomic cores, where
  // the density is largest) are batched apart, per atom, so that the mixed
  // form's three-term core treatment covers few batches; the rest is bisected
  // as one set. Only the batch membership depends on this.
  std::vector<int> keep;
  std::vector<long> sets = {0};
  {
    const double rc2 = kCoreRadius * kCoreRadius;
    const HeavyCells hc(m);
    std::vector<std::vector<int>> core(nat);
    std::vector<int> rest;
    rest.reserve(G);
    for (long i = 0; i < G; ++i) {  // any nucleus with Z > 2, not only the point's own atom's
      if (pw[i] == 0.0) continue;
      const int a = hc.near(px[i], py[i], pz[i], rc2);
      (a >= 0 ? core[a] : rest).push_back((int)i);
    }
    keep.reserve(G);
    for (int a = 0; a < nat; ++a) {
      keep.insert(keep.end(), core[a].begin(), core[a].end());
      sets.push_back((long)keep.size());
    }
    keep.insert(keep.end(), rest.begin(), rest.end());
    sets.push_back((long)keep.size());
  }
  std::vector<BisSeg> segs;
  std::vector<int> levels;
  std::vector<int2> batches;
  bisect_plan(sets, segs, levels, batches);
  g->npoints = (long)keep.size();
  g->nbatches = (int)batches.size();
  const size_t nslots = (size_t)g->nbatches * kBatch;
  g->hx.assign(nslots, 0); g->hy.assign(nslots, 0); g->hz.assign(nslots, 0); g->hw.assign(nslots, 0);
  g->batch_n.assign(g->nbatches, 0);
  for (int b = 0; b < g->nbatches; ++b) g->batch_n[b] = batches[b].y;
  g->d_x.alloc(nslots); g->d_y.alloc(nslots); g->d_z.alloc(nslots); g->d_w.alloc(nslots);
  if (nslots) {
    const long n = g->npoints;
    DevBuf<double> pts[2];
    DevBuf<int> ids[2], didx;
    DevBuf<BisSeg> dsegs;
    DevBuf<int2> dbat;
    for (int k = 0; k < 2; ++k) {
      pts[k].alloc(3 * (size_t)n);
      ids[k].alloc(n);
    }
    didx.upload(keep, g->stream);
    dsegs.upload(segs, g->stream);
    dbat.upload(batches, g->stream);
    double* pp[2] = {pts[0].p, pts[1].p};
    int* ip[2] = {ids[0].p, ids[1].p};
    launch_bisect(g->stream, n, didx.p, dx.p, dy.p, dz.p, levels, dsegs.p, pp, ip);
    const size_t nl = levels.size() - 1;
    launch_batch_slots(g->stream, g->nbatches, dbat.p, pp[nl & 1], nl ? ip[nl & 1] : didx.p, n, dw.p, g->d_x.p,
                       g->d_y.p, g->d_z.p, g->d_w.p);
    const size_t bytes = sizeof(double) * nslots;
    CHX_HIP(hipMemcpyAsync(g->hx.data(), g->d_x.p, bytes, hipMemcpyDeviceToHost, g->stream));
    CHX_HIP(hipMemcpyAsync(g->hy.data(), g->d_y.p, bytes, hipMemcpyDeviceToHost, g->stream));
    CHX_HIP(hipMemcpyAsync(g->hz.data(), g->d_z.p, bytes, hipMemcpyDeviceToHost, g->stream));
    CHX_HIP(hipMemcpyAsync(g->hw.data(), g->d_w.p, bytes, hipMemcpyDeviceToHost, g->stream));
    CHX_HIP(hipStreamSynchronize(g->stream));
  }
  // ---- shells in the reference's AO order
  g->nbasis = m.nbasis;
  g->npad = ((m.nbasis + kPadAO - 1) / kPadAO) * kPadAO;
  g->ntiles = g->npad / kTile;
  g->sh_xyz.clear(); g->sh_type.clear(); g->sh_nprim.clear(); g->sh_poff.clear(); g->sh_atom.clear();
  g->sh_ao.clear(); g->p_exp.clear(); g->p_coef.clear();
  g->max_nprim = 0;
  for (const ShellH& s : m.shells) {
    const int a = s.center;
    g->sh_xyz.push_back(m.xyz[3 * a]); g->sh_xyz.push_back(m.xyz[3 * a + 1]); g->sh_xyz.push_back(m.xyz[3 * a + 2]);
    g->sh_type.push_back(s.type);
    g->sh_atom.push_back(a);
    g->sh_nprim.push_back(s.nprim);
    g->sh_ao.push_back(s.ao_off);
    g->sh_poff.push_back((int)g->p_exp.size());
    g->max_nprim = std::max(g->max_nprim, s.nprim);
    for (int p = 0; p < s.nprim; ++p) {
      g->p_exp.push_back(m.exps[s.prim_off + p]);
      g->p_coef.push_back(m.coefs[s.prim_off + p]);
    }
  }
  // ---- device copies
  hipStream_t st = g->stream;
  g->d_sh_xyz.upload(g->sh_xyz, st); g->d_sh_type.upload(g->sh_type, st); g->d_sh_nprim.upload(g->sh_nprim, st);
  g->d_sh_atom.upload(g->sh_atom, st);
  g->d_sh_poff.upload(g->sh_poff, st); g->d_p_exp.upload(g->p_exp, st); g->d_p_coef.upload(g->p_coef, st);
  g->d_bn.upload(g->batch_n, st);
  CHX_HIP(hipStreamSynchronize(st));
  g->ao_ready = false;
}

// The distance from a shell's centre beyond which neither |phi| nor any
// |d phi / d x_k| of its components exceeds thr, from the bounds
//   |phi| <= r^l F(r),  |d phi| <= r^l G(r) + l r^(l-1) F(r),
//   F = sum_p |c_p| exp(-a_p r^2),  G = sum_p 2 a_p r |c_p| exp(-a_p r^2)
// (the components' angular parts are at most 1 and their derivatives at most l
// on the unit sphere). Every term falls beyond sqrt((l + 1) / (2 a_min)), so
// the last crossing is bisected there, or searched below when the threshold is
// that coarse. A zero threshold keeps a shell until its exponentials underflow; a
// shell with an exponent that does not decay is kept everywhere.
static double shell_reach(int type, int np, const double* e, const double* c, double thr) {
  const int l = std::abs(type);
  auto bound = [&](double r) {
    double F = 0, G = 0;
    for (int p = 0; p < np; ++p) {
      const double t = std::fabs(c[p]) * std::exp(-e[p] * r * r);
      F += t;
      G += 2 * e[p] * r * t;
    }
    const double rl = std::pow(r, l);
    return std::max(rl * F, rl * G + (l ? l * std::pow(r, l - 1) * F : 0.0));
  };
  double amin = e[0];
  for (int p = 1; p < np; ++p) amin = std::min(amin, e[p]);
  if (!(amin > 0)) return HUGE_VAL;
  double lo = std::sqrt((l + 1) / (2 * amin)), hi = lo + std::sqrt(800 / amin);
  if (bound(lo) > thr) {
    for (int k = 0; k < 100; ++k) {
      const double mid = 0.5 * (lo + hi);
      if (bound(mid) > thr) lo = mid; else hi = mid;
    }
    return hi * (1 + 1e-9);
  }
  const int steps = 4096;
  for (int k = steps; k >= 0; --k)
    if (bound(lo * k / steps) > thr) return lo * (k + 1) / steps;
  return 0.0;
}

// Cuts the batches into chunks with one AO list each. A batch's own list is
// short (a few hundred of a large molecule's thousands of AOs), which is what
// makes the contractions cheap, but a chunk's block of D is gathered once per
// chunk and its blocks of V are stored and read back once per run, so neighbours
// are merged while the merged list's cost stays below that of the two: cost =
// n^2 (points + kChunkCost), n the list's length in whole tiles, the second term
// those blocks in units of one point's contraction. kChunkCost = 256 gives 7 to
// 23 batches per chunk at 1.2 to 1.7 times the work of single batches' lists over
// (H2O)1 .. (H2O)128, C18 and alkanes. Builds in us at 64 / 128 / 256 / 512 /
// 1024: mixed (H2O)16 730 / 721 / 705 / 726 / 757, (H2O)48 r2SCAN 7940 / 7990 /
// 8010 / 8410 / 8790, (H2O)128 13650 / 12390 / 11900 / 12300 / 12770, alkane C24
// 618 / 594 / 582 / 588 / 633; FP64, whose contractions cost more beside the same
// blocks, (H2O)16 2090 / 2150 / 2220 / 2290 / 2430, C18 8810 / 9390 / 9670 / 9860 /
// 10010 (one value for both forms is kept here). At most `longest` batches make a chunk.
static void build_chunks(chx_grid* g, int nwords, const std::vector<unsigned long long>& alive, int longest) {
  constexpr double kChunkCost = 256.0;
  const int nb = g->nbatches, nsh = (int)g->sh_type.size();
  std::vector<int> sizes;  // shell sizes present, with the mask of the shells of that size
  std::vector<std::vector<unsigned long long>> mask;
  for (int s = 0; s < nsh; ++s) {
    const int n = shell_size(g->sh_type[s]);
    size_t k = std::find(sizes.begin(), sizes.end(), n) - sizes.begin();
    if (k == sizes.size()) {
      sizes.push_back(n);
      mask.emplace_back(nwords, 0ull);
    }
    mask[k][s >> 6] |= 1ull << (s & 63);
  }
  auto cost = [&](const unsigned long long* w, const unsigned long long* v, int batches) {
    int n = 0;
    for (size_t k = 0; k < sizes.size(); ++k)
      for (int i = 0; i < nwords; ++i) n += sizes[k] * __builtin_popcountll((w[i] | (v ? v[i] : 0ull)) & mask[k][i]);
    const double t = (n + kTile - 1) / kTile * kTile;
    return t * t * (double(kBatch) * batches + kChunkCost);
  };
  g->chunks.clear(); g->chunk_b0.clear(); g->tile_chunk.clear(); g->ao_of.clear();
  g->tile_seg_off.clear(); g->seg.clear();
  g->b_chunk.assign(nb, 0);
  g->dt_elems = 0;
  std::vector<unsigned long long> cur(nwords);
  for (int b0 = 0; b0 < nb;) {
    std::copy_n(&alive[(size_t)b0 * nwords], nwords, cur.begin());
    int b1 = b0 + 1;
    double c = cost(cur.data(), nullptr, 1);
    while (b1 < nb && b1 - b0 < longest) {
      const unsigned long long* v = &alive[(size_t)b1 * nwords];
      const double cm = cost(cur.data(), v, b1 - b0 + 1);
      if (cm > c + cost(v, nullptr, 1)) break;
      for (int i = 0; i < nwords; ++i) cur[i] |= v[i];
      c = cm;
      ++b1;
    }
    // the list, packed: shells in AO order, one that does not fit a tile continues in the next
    ChunkDev ch{(long)g->dt_elems, (int)g->tile_chunk.size(), 0, b0, b1 - b0};
    int col = kTile;
    for (int s = 0; s < nsh; ++s) {
      if (!(cur[s >> 6] >> (s & 63) & 1ull)) continue;
      for (int k = 0, n = shell_size(g->sh_type[s]); k < n;) {
        if (col == kTile) {  // next tile
          g->tile_seg_off.push_back((int)g->seg.size());
          g->tile_chunk.push_back((int)g->chunks.size());
          g->ao_of.resize(g->ao_of.size() + kTile, -1);
          ++ch.ntl;
          col = 0;
        }
        const int cnt = std::min(n - k, kTile - col);
        g->seg.push_back(make_int4(s, k, cnt, col));
        for (int i = 0; i < cnt; ++i) g->ao_of[g->ao_of.size() - kTile + col + i] = g->sh_ao[s] + k + i;
        k += cnt;
        col += cnt;
      }
    }
    g->dt_elems += (size_t)ch.ntl * kTile * ch.ntl * kTile;
    for (int b = b0; b < b1; ++b) g->b_chunk[b] = (int)g->chunks.size();
    g->chunks.push_back(ch);
    g->chunk_b0.push_back(b0);
    b0 = b1;
  }
  g->chunk_b0.push_back(nb);
  g->tile_seg_off.push_back((int)g->seg.size());
}

// The form that recomputes AO values: segments of chunks whose blocks of D are gathered
// together, into at most an eighth of the room (or one chunk's, the matrix at most).
static void build_segments(chx_grid* g, double room) {
  const size_t cap = (size_t)(room / 8 / sizeof(double));
  g->seg_chunk.assign(1, 0);
  g->seg_elems = 0;
  size_t cur = 0;
  for (size_t c = 0; c < g->chunks.size(); ++c) {
    const size_t n = (size_t)g->chunks[c].ntl * kTile * g->chunks[c].ntl * kTile;
    if (cur > 0 && cur + n > cap) {
      g->seg_chunk.push_back((int)c);
      cur = 0;
    }
    cur += n;
    g->seg_elems = std::max(g->seg_elems, cur);
  }
  g->seg_chunk.push_back((int)g->chunks.size());
}

// Vxc work items: per chunk every block (I, J) of super-tiles of `sup` tiles
// (upper: only I <= J), cut into runs of at most `len` of its batches.
// Chunk-major, so that the items that run together on one XCD share the
// chunk's operand slots in its L2.
static void build_items(const chx_grid* g, int sup, bool upper, int len, std::vector<VxcItem>& out) {
  out.clear();
  for (size_t c = 0; c < g->chunks.size(); ++c) {
    const ChunkDev& ch = g->chunks[c];
    const int ns = (ch.ntl + sup - 1) / sup;
    for (int b = g->chunk_b0[c]; b < g->chunk_b0[c + 1]; b += len) {
      const int nbat = std::min(len, g->chunk_b0[c + 1] - b);
      for (int I = 0; I < ns; ++I)
        for (int J = upper ? I : 0; J < ns; ++J)
          out.push_back(VxcItem{I, J, g->bt_off[b], nbat, ch.ntl, ch.tile0, b, 0});
    }
  }
}

// The longest run (a power of two up to the chunk length) that still leaves
// enough items. A run's blocks are written once, so long runs write less; but an
// item is a serial chain of its run's K steps, which shows unless several times
// more items than the chip holds are there. An FP64 step is some ten times as
// long, so runs past 4 batches do not pay there. Times by run length, in us, Vxc
// launch and V's assembly, mixed form, GGA, def2-SVP: (H2O)16 / SG-2 197 + 101 (4),
// 189 + 57 (8), 210 + 38 (16), 261 + 29 (32); (H2O)4 / SG-1 15 + 15 (2), 17 + 12 (4),
// 71 + 9 (32); (H2O)128 / SG-2 3578 + 1549 (8), 3508 + 1012 (16), 3548 + 774 (32).
// A meta-GGA step is four times as long and would take shorter runs in the largest
// systems: (H2O)48 / SG-2 r2SCAN 2951 + 587 (4), 3214 + 330 (8), 3689 + 201 (the rule).
// Builds in FP64: (H2O)16 1140 (1), 977 (4),
// 1141 (16); C18 / def2-TZVP r2SCAN 2317 (1), 2298 (4), 2665 (16); H2O 97 (1), 105 (4).
static int default_len(const chx_grid* g, int sup, bool upper) {
  const bool mixed = g->precision == CHX_PREC_MIXED;
  for (int len = kChunkMax; len > 1; len /= 2) {
    if (!mixed && len > 4) continue;
    const long want = len > 8 ? 4096 : 160;
    long n = 0;
    for (size_t c = 0; c < g->chunks.size(); ++c) {
      const long ns = (g->chunks[c].ntl + sup - 1) / sup, nb = g->chunk_b0[c + 1] - g->chunk_b0[c];
      n += (upper ? ns * (ns + 1) / 2 : ns * ns) * ((nb + len - 1) / len);
    }
    if (n >= want) return len;
  }
  return 1;
}

// Cached tables: runs of at most len batches of a chunk; per run the groups of its
// tiles (at most sup, equal to within one) and an item per pair I <= J. U holds
// per run and group I the row panel of I's rows, columns from I0 to the list's
// end; rows/rowptr list for every AO its row in every run that holds it, from
// the AO's own column on (the upper triangle).
static void build_mwork(chx_grid* g, int sup, int len, std::vector<RowRef>& rows, std::vector<int>& rowptr) {
  g->mwork.clear();
  g->u_elems = 0;
  rowptr.assign(g->nbasis + 1, 0);
  const size_t nch = g->chunks.size();
  for (size_t c = 0; c < nch; ++c) {
    const int runs = (g->chunk_b0[c + 1] - g->chunk_b0[c] + len - 1) / len, a0 = g->chunks[c].tile0 * kTile;
    for (int i = 0; i < g->chunks[c].ntl * kTile; ++i)
      if (g->ao_of[a0 + i] >= 0) rowptr[g->ao_of[a0 + i] + 1] += runs;
  }
  for (int i = 0; i < g->nbasis; ++i) rowptr[i + 1] += rowptr[i];
  rows.resize(rowptr[g->nbasis]);
  std::vector<int> at(rowptr.begin(), rowptr.end() - 1);
  for (size_t c = 0; c < nch; ++c) {
    const ChunkDev& ch = g->chunks[c];
    if (ch.ntl == 0) continue;
    const int ng = (ch.ntl + sup - 1) / sup, a0 = ch.tile0 * kTile;
    int nreal = ch.ntl * kTile;  // the list's AOs: only its last tile is padded
    while (g->ao_of[a0 + nreal - 1] < 0) --nreal;
    for (int b = g->chunk_b0[c]; b < g->chunk_b0[c + 1]; b += len) {
      const int nbat = std::min(len, g->chunk_b0[c + 1] - b);
      for (int I = 0; I < ng; ++I) {
        const int I0 = ch.ntl * I / ng, I1 = ch.ntl * (I + 1) / ng, ldu = (ch.ntl - I0) * kTile;
        for (int J = I; J < ng; ++J) {
          const int J0 = ch.ntl * J / ng, J1 = ch.ntl * (J + 1) / ng;
          g->mwork.push_back(MxItem{(long)g->u_elems + (J0 - I0) * kTile, I0, I1 - I0, J0, J1 - J0, g->bt_off[b], nbat,
                                    ch.ntl, ldu, ch.tile0, b});
        }
        for (int r = I0 * kTile; r < std::min(I1 * kTile, nreal); ++r)
          rows[at[g->ao_of[a0 + r]]++] = RowRef{(long)g->u_elems + (long)(r - I0 * kTile) * (ldu + 1), a0 + r, nreal - r};
        g->u_elems += (size_t)(I1 - I0) * kTile * ldu;
      }
    }
  }
}

// u_elems of build_mwork for these groups and runs.
static size_t run_elems(const chx_grid* g, int sup, int len) {
  size_t n = 0;
  for (const ChunkDev& ch : g->chunks) {
    if (ch.ntl == 0) continue;
    const int ng = (ch.ntl + sup - 1) / sup;
    size_t run = 0;
    for (int I = 0; I < ng; ++I) {
      const int I0 = ch.ntl * I / ng, I1 = ch.ntl * (I + 1) / ng;
      run += (size_t)(I1 - I0) * kTile * (ch.ntl - I0) * kTile;
    }
    n += run * ((ch.nb + len - 1) / len);
  }
  return n;
}

// Tiles per Vxc group of the cached tables.
static int group_tiles(const chx_grid* g) {
  return g->precision == CHX_PREC_MIXED && g->mx_wide ? kMxWideTiles : kMxTiles;
}

// Run length of the cached tables' Vxc work items by the rule, not below what the plan found
// room for; the caller's where it set one.
int auto_run(const chx_grid* g) { return std::max(default_len(g, group_tiles(g), true), g->min_run); }
static int run_length(const chx_grid* g) { return g->vxc_chunk > 0 ? g->vxc_chunk : auto_run(g); }

static double slot_bytes(const chx_grid* g, int nT) {
  double slots = 0;
  for (const ChunkDev& ch : g->chunks) slots += (double)ch.nb * ch.ntl;
  return slots * (g->precision == CHX_PREC_MIXED ? 3.0 * nT * kMxComp * sizeof(unsigned short)
                                                 : 5.0 * kBatch * kTile * sizeof(double));
}

// What the tables of the cached forms take (bytes) at a run length. FP64: phi, grad phi
// and B per slot, the chunks' blocks of D, the runs' blocks of V. Mixed: the split operand
// cache (nT components in two layouts, 2 bytes an element) and B^T per slot, the core
// slots' third terms, D's blocks in two terms, either product of the runs.
static double table_bytes(const chx_grid* g, int nT, const std::vector<char>& core, int len) {
  const double runs = (double)run_elems(g, group_tiles(g), len);
  if (g->precision != CHX_PREC_MIXED) return slot_bytes(g, nT) + (g->dt_elems + runs) * sizeof(double);
  double core_slots = 0;
  for (size_t b = 0; b < core.size(); ++b) core_slots += core[b] * g->chunks[g->b_chunk[b]].ntl;
  return slot_bytes(g, nT) + (core_slots * nT * kBatch * kTile + 2.0 * g->dt_elems) * sizeof(unsigned short) +
         2 * runs * sizeof(float);
}

// Vxc work items of the cached tables over groups of up to kMxTiles tiles or
// (mixed form, wide) kMxWideTiles; FP64 form: also every pair of groups for the
// plain products. Uploads them; the host vectors outlive the copies (synchronises).
void build_cwork(chx_grid* g) {
  hipStream_t st = g->stream;
  const bool mixed = g->precision == CHX_PREC_MIXED;
  const int sup = group_tiles(g);
  std::vector<RowRef> rows;
  std::vector<int> rowptr;
  build_mwork(g, sup, run_length(g), rows, rowptr);
  if (mixed) {
    g->d_U64.release();
    g->d_U.alloc(std::max<size_t>(1, 2 * g->u_elems));
  } else {
    g->d_U.release();
    g->d_U64.alloc(std::max<size_t>(1, g->u_elems));
  }
  g->d_mwork.upload(g->mwork, st);
  g->d_rows.upload(rows, st);
  g->d_rowptr.upload(rowptr, st);
  g->pwork.clear();
  if (mixed) {
    g->hmol.cwork = g->d_mwork.p;
    g->hmol.U = g->d_U.p;
    g->hmol.uplane = (long)g->u_elems;
  } else {
    for (const MxItem& m : g->mwork) {
      g->pwork.push_back(m);
      if (m.I0 != m.J0) {
        MxItem t = m;
        std::swap(t.I0, t.J0);
        std::swap(t.nI, t.nJ);
        g->pwork.push_back(t);
      }
    }
  }
  g->d_pwork.upload(g->pwork, st);
  CHX_HIP(hipStreamSynchronize(st));
}

// After a failure half way: no plan and nothing that was made with it, for this
// grid's calls and for a pack that holds it.
static void drop_plan(chx_grid* g) {
  ++g->plan_gen;
  g->ao_ready = g->have_density = g->have_eval = g->have_v = g->have_skeleton = g->slot_tables = false;
  g->corr_pending = g->corr_done = g->vout_ready = false;
  g->fx_family = -1;
  g->nmats_u = 0;
}

// Mixed form: Vxc over groups of up to kMxWideTiles tiles. -1: from npad 1024 on.
static int wide_groups(const chx_grid* g) {
  return g->precision == CHX_PREC_MIXED && (g->vxc_shape == 1 || (g->vxc_shape < 0 && g->npad >= 1024)) ? 1 : 0;
}

// Rebuilds the Vxc work items for another run length or group size without touching
// the AO tables. Where the new runs' blocks cannot be allocated the call fails and the
// former ones, which fitted, are made again; should that fail too, the plan is dropped.
static void rebuild_runs(chx_grid* g, int chunk, int shape) {
  const int was_chunk = g->vxc_chunk, was_shape = g->vxc_shape;
  g->vxc_chunk = chunk;
  g->vxc_shape = shape;
  if (!g->ao_ready || !g->cached) return;
  ++g->plan_gen;
  auto rebuild = [&] {
    g->mx_wide = wide_groups(g);
    build_cwork(g);
  };
  try {
    rebuild();
  } catch (...) {
    g->vxc_chunk = was_chunk;
    g->vxc_shape = was_shape;
    try {
      rebuild();
    } catch (...) {
      drop_plan(g);
    }
    throw;
  }
}

void set_vxc_chunk(chx_grid* g, int chunk) { rebuild_runs(g, chunk, g->vxc_shape); }

// Vxc block shape of the mixed form (-1: groups of up to 5 tiles from npad 1024
// on, of up to 4 below; 0, 1: either), rebuilding the work items.
void set_vxc_shape(chx_grid* g, int shape) {
  if (g->precision != CHX_PREC_MIXED) g->vxc_shape = shape;
  else rebuild_runs(g, g->vxc_chunk, shape);
}

// Bytes of the tables that the grid's former plan holds; with release, they are freed.
static size_t former_tables(chx_grid* g, bool release) {
  size_t n = 0;
  auto add = [&](auto& b) {
    n += b.n * sizeof(*b.p);
    if (release) b.release();
  };
  add(g->d_cache); add(g->d_bmat); add(g->d_U64); add(g->d_Dt);
  add(g->d_cmx); add(g->d_bmx); add(g->d_U); add(g->d_Dsplit); add(g->d_cmx3);
  return n;
}

// Screening and work plans (Grid::getAO counterpart).
static void make_plan(chx_grid* g) {
  hipStream_t st = g->stream;
  g->d_ws.release();
  const int nb = g->nbatches, nsh = (int)g->sh_type.size(), nwords = (nsh + 63) / 64;
  std::vector<double> reach2(nsh);
  std::vector<int> kinds;  // one shell of each kind (atoms of an element repeat theirs)
  for (int s = 0; s < nsh; ++s) {
    const int np = g->sh_nprim[s];
    const double *e = &g->p_exp[g->sh_poff[s]], *c = &g->p_coef[g->sh_poff[s]];
    auto same = [&](int k) {
      return g->sh_type[k] == g->sh_type[s] && g->sh_nprim[k] == np && std::equal(e, e + np, &g->p_exp[g->sh_poff[k]]) &&
             std::equal(c, c + np, &g->p_coef[g->sh_poff[k]]);
    };
    const auto it = std::find_if(kinds.begin(), kinds.end(), same);
    if (it != kinds.end()) {
      reach2[s] = reach2[*it];
      continue;
    }
    kinds.push_back(s);
    const double r = shell_reach(g->sh_type[s], np, e, c, g->screen_thr);
    reach2[s] = r * r;
  }
  std::vector<unsigned long long> alive((size_t)nb * nwords, 0ull);
  {
    DevBuf<double> d_reach;
    DevBuf<unsigned long long> d_alive;
    d_reach.upload(reach2, st);
    d_alive.alloc(std::max<size_t>(1, alive.size()));
    launch_screen(st, nb, nsh, nwords, g->d_x.p, g->d_y.p, g->d_z.p, g->d_bn.p, g->d_sh_xyz.p, d_reach.p,
                  d_alive.p);
    if (nb)
      CHX_HIP(hipMemcpyAsync(alive.data(), d_alive.p, sizeof(alive[0]) * alive.size(), hipMemcpyDeviceToHost, st));
    CHX_HIP(hipStreamSynchronize(st));
  }
  const bool mixed = g->precision == CHX_PREC_MIXED;
  const int nT = g->type >= 2 ? 4 : 1;
  if (mixed && g->ntiles > kMxMaxTiles)
    throw Error(CHX_ERR_UNSUPPORTED, "the mixed-precision form takes at most " + std::to_string(kMxMaxTiles * kTile) +
                                         " basis functions");
  if (mixed && g->max_nprim > kSegPrim)
    throw Error(CHX_ERR_UNSUPPORTED, "the mixed-precision form takes at most " + std::to_string(kSegPrim) +
                                         " primitives per shell");
  // core batches of the mixed form: any real point within core_radius of a nucleus with Z > 2
  std::vector<char> core;
  if (mixed && g->core_radius > 0) {
    core.assign(nb, 0);
    const double r2c = g->core_radius * g->core_radius;  // <= 1 bohr: the cells' reach
    const HeavyCells hc(g->mol);
    for (int b = 0; b < nb; ++b)
      for (int q = 0; q < g->batch_n[b] && !core[b]; ++q) {
        const size_t p = (size_t)b * kBatch + q;
        core[b] = hc.near(g->hx[p], g->hy[p], g->hz[p], r2c) >= 0;
      }
  }
  // The chunks, and whether their tables have room. D's and V's blocks grow with a list's
  // square once per chunk and run, the tables only with its length per batch: where the
  // whole does not fit, runs are made longer (up to the chunk), then chunks (up to
  // kChunkLong batches, which costs nothing where the lists are alike; where they differ
  // the chunks stay short and the blocks small).
  size_t free_b = 0, total_b = 0;
  CHX_HIP(hipMemGetInfo(&free_b, &total_b));
  const double share = mixed ? 0.9 : 0.8, room = share * (double)(free_b + former_tables(g, false));
  g->mx_wide = wide_groups(g);
  bool fits = false;
  for (int longest = kChunkMax; !fits; longest *= 2) {
    build_chunks(g, nwords, alive, longest);
    g->min_run = 1;
    fits = table_bytes(g, nT, core, run_length(g)) <= room;
    while (!fits && g->vxc_chunk == 0 && g->min_run < longest) {
      g->min_run *= 2;
      fits = table_bytes(g, nT, core, run_length(g)) <= room;
    }
    if (longest >= kChunkLong || (!mixed && g->cache_mode == 0) || slot_bytes(g, nT) > room) break;
  }
  if (mixed && !fits)
    throw Error(CHX_ERR_DEVICE, "the mixed-precision form needs " +
                                    std::to_string(table_bytes(g, nT, core, run_length(g)) / 1e9) +
                                    " GB of device memory for its AO cache");
  g->cached = mixed || g->cache_mode == 1 || (g->cache_mode == -1 && fits);
  if (!g->cached || table_bytes(g, nT, core, run_length(g)) > share * (double)free_b) former_tables(g, true);
  if (!g->cached) build_segments(g, room);
  g->bt_off.assign(nb + 1, 0);
  g->batch_work.assign(nb, 0.0);
  g->slot_batch.clear(); g->slot_tile.clear();
  g->grp_batch.clear(); g->grp_tile.clear(); g->grp_ntiles.clear();
  g->grp_off.assign(nb + 1, 0);
  std::vector<int> chunk_nao(g->chunks.size(), 0);
  for (size_t i = 0; i < g->ao_of.size(); ++i)
    if (g->ao_of[i] >= 0) ++chunk_nao[g->tile_chunk[i / kTile]];
  double flops = 0, tiles = 0;
  for (int b = 0; b < nb; ++b) {
    const ChunkDev& ch = g->chunks[g->b_chunk[b]];
    g->bt_off[b] = (int)g->slot_tile.size();
    g->grp_off[b] = (int)g->grp_batch.size();
    for (int q = 0; q < ch.ntl; ++q) {
      g->slot_batch.push_back(b);
      g->slot_tile.push_back(ch.tile0 + q);
    }
    for (int q = 0; q < ch.ntl; q += kGroup) {
      g->grp_batch.push_back(b);
      g->grp_tile.push_back(ch.tile0 + q);
      g->grp_ntiles.push_back(std::min(kGroup, ch.ntl - q));
    }
    tiles += ch.ntl;
    const double n = chunk_nao[g->b_chunk[b]];
    g->batch_work[b] = (double)g->batch_n[b] * n * n;
    flops += g->batch_work[b];
  }
  g->bt_off[nb] = (int)g->slot_tile.size();
  g->grp_off[nb] = (int)g->grp_batch.size();
  g->mean_tiles = nb ? tiles / nb : 0;
  // k contractions per build (GGA: Phi D and Phi^T B; meta-GGA adds three of
  // each for tau), 2 flops per multiply-add
  g->flops_build = (g->type >= 2 ? 8.0 : 2.0) * 2.0 * flops;
  const size_t nslot = g->slot_tile.size();
  // the tiles' segment records, and the plan's tables on the device
  std::vector<SegRec> rec(g->seg.size());  // lives until the synchronisation at the end
  for (size_t k = 0; k < g->seg.size(); ++k) {
    const int4 sg = g->seg[k];
    const int sh = sg.x, np = g->sh_nprim[sh], po = g->sh_poff[sh];
    SegRec& r = rec[k];
    std::memset(&r, 0, sizeof(r));
    r.ax = g->sh_xyz[3 * sh]; r.ay = g->sh_xyz[3 * sh + 1]; r.az = g->sh_xyz[3 * sh + 2];
    r.meta = (g->sh_type[sh] & 0xff) | (std::min(np, kSegPrim) << 8) | (sg.y << 16) | (sg.z << 24);
    r.col = sg.w;
    if (k > 0 && sg.w > 0 && g->sh_atom[g->seg[k - 1].x] == g->sh_atom[sh]) r.meta |= kSegSame;
    for (int p = 0; p < np && p < kSegPrim; ++p) {
      r.p[p][0] = (float)(-1.4426950408889634 * g->p_exp[po + p]);
      r.p[p][1] = (float)g->p_coef[po + p];
      r.p[p][2] = (float)(g->p_exp[po + p] * g->p_coef[po + p]);
    }
  }
  g->d_segrec.upload(rec, st);
  g->d_tile_seg_off.upload(g->tile_seg_off, st); g->d_seg.upload(g->seg, st);
  g->d_chunks.upload(g->chunks, st); g->d_b_chunk.upload(g->b_chunk, st);
  g->d_tile_chunk.upload(g->tile_chunk, st); g->d_ao_of.upload(g->ao_of, st);
  g->d_slot_batch.upload(g->slot_batch, st); g->d_slot_tile.upload(g->slot_tile, st);
  g->vwork.clear();
  g->mwork.clear();
  if (g->cached) g->d_Mint.release();
  else g->d_Mint.alloc((size_t)g->npad * g->npad);
  if (g->cached) {
    if (mixed) {
      g->d_cache.release();
      g->d_bmat.release();
      g->mx_nT = nT;
      g->mx_sstride = 2 * nT * kMxComp;  // AOg then AOt, nT components each
      g->d_cmx.alloc(std::max<size_t>(1, nslot * (size_t)g->mx_sstride));
      g->bmx_comps = nT;
      g->d_bmx.alloc(std::max<size_t>(1, nslot * (size_t)nT * kMxComp));
      g->d_Dsplit.alloc(std::max<size_t>(1, 2 * g->dt_elems));
      std::vector<int> core_off(nb, -1), slot_core(std::max<size_t>(1, nslot), -1);
      g->core_grps.clear();
      g->main_grps.clear();
      g->ncore_batches = 0;
      g->core_flops = 0.0;
      int ncore_slots = 0;
      if (!core.empty()) {
        for (int b = 0; b < nb; ++b) {
          if (!core[b]) {
            for (int k = g->grp_off[b]; k < g->grp_off[b + 1]; ++k) g->main_grps.push_back(k);
            continue;
          }
          ++g->ncore_batches;
          g->core_flops += 2.0 * g->batch_work[b];
          core_off[b] = ncore_slots;
          for (int it = g->bt_off[b]; it < g->bt_off[b + 1]; ++it) slot_core[it] = ncore_slots++;
          for (int k = g->grp_off[b]; k < g->grp_off[b + 1]; ++k) g->core_grps.push_back(k);
        }
      }
      static const std::vector<int> neg1{-1}, zero1{0};  // placeholders outlive the asynchronous copies
      g->d_core_off.upload(core_off.empty() ? neg1 : core_off, st);
      g->d_slot_core.upload(slot_core.empty() ? neg1 : slot_core, st);
      g->d_core_grps.upload(g->core_grps.empty() ? zero1 : g->core_grps, st);
      if (g->core_grps.empty()) g->main_grps.clear();  // no core batches: the launch takes every group
      g->d_main_grps.upload(g->main_grps.empty() ? zero1 : g->main_grps, st);
      g->d_cmx3.alloc(std::max<size_t>(1, (size_t)ncore_slots * nT * kBatch * kTile));
      launch_ao_cache_mx(st, (int)nslot, g->d_slot_batch.p, g->d_slot_tile.p, g->d_x.p, g->d_y.p, g->d_z.p,
                         g->view(), nT, g->mx_sstride, g->d_cmx.p, ncore_slots ? g->d_slot_core.p : nullptr,
                         g->d_cmx3.p);
      CHX_HIP(hipStreamSynchronize(st));  // the host vectors above go out of scope
    } else {
      g->d_cmx.release();
      g->d_bmx.release();
      g->d_Dsplit.release();
      g->d_Dres.release();
      g->d_cpart.release();
      g->mx_nT = g->mx_sstride = g->bmx_comps = 0;
      g->d_cache.alloc(std::max<size_t>(1, nslot * (size_t)4 * kBatch * kTile));
      g->d_bmat.alloc(std::max<size_t>(1, nslot * (size_t)kBatch * kTile));
      launch_ao_cache(st, (int)nslot, g->d_slot_batch.p, g->d_slot_tile.p, g->d_x.p, g->d_y.p, g->d_z.p, g->view(),
                      g->d_cache.p);
    }
  } else {
    g->d_cache.release();
    g->d_bmat.release();
    build_items(g, kSuper, true, default_len(g, kSuper, true), g->vwork);
    g->d_vwork.upload(g->vwork, st);
    g->d_cmx.release();
    g->d_bmx.release();
    g->d_Dsplit.release();
    g->d_Dres.release();
    g->d_cpart.release();
  }
  g->d_bt_off.upload(g->bt_off, st);
  g->d_grp_batch.upload(g->grp_batch, st); g->d_grp_tile.upload(g->grp_tile, st);
  g->d_grp_ntiles.upload(g->grp_ntiles, st); g->d_grp_off.upload(g->grp_off, st);
  // per-iteration buffers
  const size_t nslots = (size_t)nb * kBatch;
  if (mixed) g->d_Dt.release();
  else g->d_Dt.alloc(std::max<size_t>(1, g->cached ? g->dt_elems : g->seg_elems));
  g->d_Din.alloc((size_t)g->nbasis * g->nbasis);
  g->d_Vout.alloc((size_t)g->nbasis * g->nbasis);
  g->d_part.alloc(std::max<size_t>(1, g->grp_batch.size() * 4 * kBatch));
  g->d_rho.alloc(std::max<size_t>(1, nslots));
  g->d_coef.alloc(std::max<size_t>(kCoef, kCoef * nslots));
  g->d_part_tau.alloc(g->type >= 2 ? std::max<size_t>(1, g->grp_batch.size() * 3 * kBatch) : 1);
  g->en_blocks = (int)std::max<size_t>(1, (nslots + 255) / 256);
  g->d_en_part.alloc(2 * (size_t)g->en_blocks);
  g->d_en.alloc(3);
  launch_fill(st, g->d_en.p, 3, 0.0);
  if (g->type >= 2) {
    g->d_asym.alloc(1);
    launch_fill_u32(st, (unsigned*)g->d_asym.p, 1, 0u);
  } else {
    g->d_asym.release();
  }
  g->d_gen = 0;
  if (mixed) {  // split remainder of D per spin, and the partial sums of V . remainder
    g->d_Dres.alloc(2 * (size_t)g->nbasis * g->nbasis);
    g->d_cpart.alloc(2 * (size_t)assemble_blocks(g->nbasis));
  }
  g->hmol = MolDev{};
  if (g->cached) build_cwork(g);
  if (mixed) {  // descriptor of this grid for the mixed kernels
    MolDev& m = g->hmol;
    m.grp_batch = g->d_grp_batch.p; m.grp_tile = g->d_grp_tile.p; m.grp_ntiles = g->d_grp_ntiles.p;
    m.bt_off = g->d_bt_off.p; m.b_chunk = g->d_b_chunk.p; m.chunks = g->d_chunks.p; m.ao_of = g->d_ao_of.p;
    m.bx = g->d_x.p; m.by = g->d_y.p; m.bz = g->d_z.p;
    m.bv = g->view();
    m.cache = g->d_cmx.p; m.sstride = g->mx_sstride; m.toff = g->mx_nT * kMxComp;
    m.Ds = g->d_Dsplit.p; m.npad = g->npad; m.ntiles = g->ntiles; m.nslots = (int)nslot;
    m.part = g->d_part.p; m.part_tau = g->d_part_tau.p;
    m.slot_batch = g->d_slot_batch.p; m.slot_tile = g->d_slot_tile.p;
    m.coef = g->d_coef.p; m.bt = g->d_bmx.p;
    m.cache3 = g->d_cmx3.p;
    m.asym = g->d_asym.p;
    m.core_off = g->d_core_off.p;
    m.core_grps = g->d_core_grps.p;
    m.main_grps = g->core_grps.empty() ? nullptr : g->d_main_grps.p;
  }
  CHX_HIP(hipStreamSynchronize(st));
  g->ao_ready = true;
  ++g->plan_gen;
  g->have_density = g->have_eval = g->have_v = g->have_skeleton = false;
  g->corr_pending = g->corr_done = g->vout_ready = false;
  g->slot_tables = false;
}

void grid_plan(chx_grid* g) {
  try {
    make_plan(g);
  } catch (...) {
    drop_plan(g);
    throw;
  }
}

}  // namespace chx

int chx_lebedev_rule_impl(int n, double* xyzw) {
  const auto& r = chx::lebedev_rule(n);
  for (size_t i = 0; i < r.size(); ++i)
    for (int k = 0; k < 4; ++k) xyzw[4 * i + k] = r[i][k];
  return (int)r.size();
}

chx::BasisView chx_grid::view() const {
  chx::BasisView v;
  v.sh_xyz = d_sh_xyz.p;
  v.sh_atom = d_sh_atom.p;
  v.sh_type = d_sh_type.p;
  v.sh_nprim = d_sh_nprim.p;
  v.sh_poff = d_sh_poff.p;
  v.p_exp = d_p_exp.p;
  v.p_coef = d_p_coef.p;
  v.tile_seg_off = d_tile_seg_off.p;
  v.seg = d_seg.p;
  v.segrec = d_segrec.p;
  return v;
}
