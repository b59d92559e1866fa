// FP64 plain form with the AO tables cached in HBM.
//
// phi and grad phi do not change between SCF iterations, so they are computed
// once per grid (at Grid::getAO, as the reference caches its AO tables,
// src/Grid/Grid.cpp:22-33) for every (batch, 32-AO tile of its list) slot and kept in
// HBM (~80 KB per slot). Each iteration then streams them through two MFMA
// contractions:
//   density: X = Phi_b D_b, then rho = sum X phi and grad rho / 2 = sum X grad phi
//            from the cache;
//   Vxc:     V_IJ = Phi_I^T B_J + B_I^T Phi_J over groups of up to 128 of the
//            list's AOs, B = a phi + c . grad phi built once per iteration by
//            k_make_b, summed over the runs by k_assemble.
// Meta-GGA adds tau = 1/2 sum_r (d_r Phi D) . d_r phi (three more density
// products) and sum_r (d_r Phi)^T T_r to V.
// Layouts: cache[slot][c][g][32] (c = phi, d/dx, d/dy, d/dz), bmat[slot][g][32].
//
// A v_mfma_f64_16x16x4 holds its SIMD for 64 cycles and takes 512 bytes per
// operand, so a wave that owns 64 x 64 (or 64 x 32) results needs 8 to 12 bytes
// per cycle: the waves read their operands straight from the caches in operand
// order (rows of 128 bytes), with no LDS stage and no barrier, the next loads in
// flight while the products of the current ones run.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace chx {

constexpr int kSlotAO = 4 * kBatch * kTile;  // doubles per cached slot
constexpr int kSlotB = kBatch * kTile;

// ---------------------------------------------------------------------------
// AO cache: one block per slot.
__global__ __launch_bounds__(256) void k_ao_cache(const int* __restrict__ slot_batch, const int* __restrict__ slot_tile,
                                                  const double* __restrict__ bx, const double* __restrict__ by,
                                                  const double* __restrict__ bz, BasisView bv,
                                                  double* __restrict__ cache) {
  __shared__ double px[kBatch], py[kBatch], pz[kBatch];
  const int s = blockIdx.x, tid = threadIdx.x;
  const int b = slot_batch[s], t = slot_tile[s];
  double* out = cache + (size_t)s * kSlotAO;
  if (tid < kBatch) {
    px[tid] = bx[b * kBatch + tid];
    py[tid] = by[b * kBatch + tid];
    pz[tid] = bz[b * kBatch + tid];
  }
  // padding AOs of a chunk's last tile are zero
  const int4 last = bv.seg[bv.tile_seg_off[t + 1] - 1];
  const int nao = last.w + last.z;
  for (int e = tid; e < 4 * kBatch * (kTile - nao); e += 256) {
    const int w = kTile - nao;
    const int c = e / (kBatch * w), r = e % (kBatch * w);
    out[((size_t)c * kBatch + r / w) * kTile + nao + r % w] = 0.0;
  }
  __syncthreads();
  const int s0 = bv.tile_seg_off[t], s1 = bv.tile_seg_off[t + 1];
  for (int item = tid; item < (s1 - s0) * kBatch; item += 256) {
    const int g = item % kBatch;
    const int4 sg = bv.seg[s0 + item / kBatch];
    double v[7], gx[7], gy[7], gz[7];
    shell_eval<true>(bv, sg.x, px[g], py[g], pz[g], v, gx, gy, gz);
#pragma unroll
    for (int m = 0; m < 7; ++m)
      if (m < sg.z) {
        const int col = sg.w + m;
        out[(0 * kBatch + g) * kTile + col] = v[sg.y + m];
        out[(1 * kBatch + g) * kTile + col] = gx[sg.y + m];
        out[(2 * kBatch + g) * kTile + col] = gy[sg.y + m];
        out[(3 * kBatch + g) * kTile + col] = gz[sg.y + m];
      }
  }
}

void launch_ao_cache(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile,
                     const double* bx, const double* by, const double* bz, BasisView bv, double* cache) {
  if (nslots == 0) return;
  hipLaunchKernelGGL(k_ao_cache, dim3(nslots), dim3(256), 0, s, slot_batch, slot_tile, bx, by, bz, bv, cache);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Density from the cache. Block = (batch, group of <= 4 tiles of its list as
// output columns). A wave owns one tile's 32 columns of X = Phi D: all 64 points
// (4 waves), or with TAU 32 points of all four products Phi D, (d_r Phi) D (8
// waves). K runs over the list's tiles in 8-AO pieces: lane (lk, lrow) holds AOs
// 2 lk, 2 lk + 1 of point lrow (one 16-byte load, 64 contiguous bytes per
// point), and rows 2 lk, 2 lk + 1 of D, so both see the same order of K.
// tau = sum_r x_r^T D x_r (x_r = d_r phi) is a quadratic form: for a symmetric D
// (asym != gen) the wave's tau products run over the tiles up to its own, those
// before it counted twice (accumulators doubled when it is reached).
// C18 / def2-TZVP / SG-3: 4.6 ms (7.6 in four launches with LDS stages).
// NM = 2: two matrices (spins, perturbations) against the same phi, which is then
// read once for both, the epilogue's grad phi too. Radical C7 / UKS, def2-SVP /
// SG-1: 0.25 ms for both spins, 0.28 in two launches.
template <bool TAU, int NM>
__global__ __launch_bounds__(TAU ? 512 : 256, 2) void k_density_c64(
    const int* __restrict__ grp_batch, const int* __restrict__ grp_tile, const int* __restrict__ grp_ntiles,
    const int* __restrict__ bt_off, const int* __restrict__ b_chunk, const ChunkDev* __restrict__ chunks,
    const double* __restrict__ cache, const double* __restrict__ Dt, size_t sD, const int* __restrict__ asym, int gen,
    double* __restrict__ part, size_t sP, double* __restrict__ part1, double* __restrict__ part_tau) {
  static_assert(!TAU || NM == 1, "tau takes one matrix");
  constexpr int NC = TAU ? 4 : 1, NR = TAU ? 2 : 4, NOUT = TAU ? 5 : 4;
  __shared__ double red[kGroup][NM * NOUT][kBatch];
  Dt += blockIdx.y * NM * sD;
  part += blockIdx.y * NM * sP;
  if (!part1) part1 = part + sP;
  const int grp = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;
  const int q = TAU ? wave >> 1 : wave, row0 = TAU ? 32 * (wave & 1) : 0;  // the wave's tile of the group, first point
  const int b = grp_batch[grp], nt = grp_ntiles[grp];
  const ChunkDev ch = chunks[b_chunk[b]];
  const int nk = ch.ntl, ld = nk * kTile, it0 = bt_off[b], tq = grp_tile[grp] - ch.tile0 + q;  // the tile in the list
  if (q < nt) {
    const bool sym = TAU && *asym != gen;
    const double* __restrict__ A0 = cache + (size_t)it0 * kSlotAO + (row0 + lrow) * kTile + 2 * lk;
    const double* __restrict__ D0 = Dt + ch.doff + (size_t)(2 * lk) * ld + tq * kTile + lrow;
    dbl4 acc[NC * NM][NR][2];
#pragma unroll
    for (int d = 0; d < NC * NM; ++d)
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[d][r][h] = dbl4{0, 0, 0, 0};
    // pieces [p0, p1) of K: AOs 8 (p % 4).. of tile p / 4; every load is unconditional (a branch around
    // one makes the compiler wait for all that are in flight)
    auto run = [&](auto with_tau, int p0, int p1) {
      constexpr int ND = decltype(with_tau)::value ? NC : 1;
      if (p0 >= p1) return;
      double2 a[2][ND][NR];
      double bb[2][NM][2][2];  // [buffer][matrix][row of the pair][half]
      auto load = [&](int p, int buf) {
        const int k = p >> 2, o = 8 * (p & 3);
        const double* __restrict__ pa = A0 + (size_t)k * kSlotAO + o;
        const double* __restrict__ pd = D0 + (size_t)(k * kTile + o) * ld;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int r = 0; r < NR; ++r)
            a[buf][d][r] = *reinterpret_cast<const double2*>(pa + d * kSlotB + 16 * r * kTile);
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) bb[buf][m][e][h] = pd[m * sD + (size_t)e * ld + 16 * h];
      };
      auto step = [&](int buf) {
#pragma unroll
        for (int d = 0; d < ND * NM; ++d)  // component d, or (one component) matrix d
#pragma unroll
          for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const double2 x = a[buf][NM == 1 ? d : 0][r];
              acc[d][r][h] = mfma_f64(x.x, bb[buf][NM == 1 ? 0 : d][0][h], acc[d][r][h]);
              acc[d][r][h] = mfma_f64(x.y, bb[buf][NM == 1 ? 0 : d][1][h], acc[d][r][h]);
            }
      };
      load(p0, 0);
      for (int p = p0; p < p1; p += 2) {  // whole tiles: an even number of pieces
        load(p + 1, 1);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products that they run beside
        step(0);
        load(min(p + 2, p1 - 1), 0);
        __builtin_amdgcn_sched_barrier(0);
        step(1);
      }
    };
    if (sym) {
      run(std::true_type{}, 0, 4 * tq);
#pragma unroll
      for (int d = 1; d < NC; ++d)
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int h = 0; h < 2; ++h) acc[d][r][h] *= 2.0;
      run(std::true_type{}, 4 * tq, 4 * tq + 4);
      run(std::false_type{}, 4 * tq + 4, 4 * nk);
    } else {
      run(std::true_type{}, 0, 4 * nk);
    }
    // X[g = row0 + 16 r + 4 i + lk][nu = 16 h + lrow] of the wave's tile, against phi and grad phi;
    // sums over the tile's columns (the 16 lanes of a row)
    const double* __restrict__ src = cache + (size_t)(it0 + tq) * kSlotAO + (row0 + lk) * kTile + lrow;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      double f[2][4][4];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int d = 0; d < 4; ++d) f[h][i][d] = src[d * kSlotB + (16 * r + 4 * i) * kTile + 16 * h];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < NM * NOUT; ++c) {
          const int m = NM == 1 ? 0 : c / NOUT, o = c % NOUT;
          double v = 0.0;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (o < 4) v += acc[m][r][h][i] * f[h][i][o & 3];
            if (o == 4) {
#pragma unroll
              for (int d = 1; d < NC; ++d) v += acc[d][r][h][i] * f[h][i][d];
            }
          }
          v += __shfl_xor(v, 1, 64);
          v += __shfl_xor(v, 2, 64);
          v += __shfl_xor(v, 4, 64);
          v += __shfl_xor(v, 8, 64);
          if (lrow == 4 * i + (o & 3)) red[q][c][row0 + 16 * r + 4 * i + lk] = v;
        }
    }
  }
  // the sums over the group's tiles
  __syncthreads();
  for (int e = tid; e < (TAU ? 7 : 4 * NM) * kBatch; e += TAU ? 512 : 256) {
    const int c = e / kBatch, g = e % kBatch;
    double v = 0.0;
    if (c < NM * NOUT)
      for (int t = 0; t < nt; ++t) v += red[t][c][g];
    if (c < 4)
      part[(size_t)grp * 4 * kBatch + c * kBatch + g] = v;
    else if (NM == 2)
      part1[(size_t)grp * 4 * kBatch + (c - 4) * kBatch + g] = v;
    else  // part_tau: [group][3][64], summed over the directions in the first
      part_tau[(size_t)grp * 3 * kBatch + (c - 4) * kBatch + g] = v;
  }
}

void launch_density_c64(hipStream_t s, int ngroups, const int* grp_batch, const int* grp_tile, const int* grp_ntiles,
                        const int* bt_off, const int* b_chunk, const ChunkDev* chunks, const double* cache,
                        const double* Dt, const int* asym, int gen, double* part, double* part_tau, int nmat,
                        size_t sD, size_t sP, double* part1) {
  if (ngroups == 0) return;
  const int pairs = part_tau ? 0 : nmat / 2, done = 2 * pairs;
  if (pairs)
    hipLaunchKernelGGL((k_density_c64<false, 2>), dim3(ngroups, pairs), dim3(256), 0, s, grp_batch, grp_tile,
                       grp_ntiles, bt_off, b_chunk, chunks, cache, Dt, sD, asym, gen, part, sP, part1, nullptr);
  if (part_tau)
    hipLaunchKernelGGL((k_density_c64<true, 1>), dim3(ngroups), dim3(512), 0, s, grp_batch, grp_tile, grp_ntiles,
                       bt_off, b_chunk, chunks, cache, Dt, sD, asym, gen, part, sP, nullptr, part_tau);
  else if (done < nmat)
    hipLaunchKernelGGL((k_density_c64<false, 1>), dim3(ngroups), dim3(256), 0, s, grp_batch, grp_tile, grp_ntiles,
                       bt_off, b_chunk, chunks, cache, Dt + done * sD, sD, asym, gen, part + done * sP, sP, nullptr,
                       nullptr);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// B = a phi + c . grad phi for every slot of a batch (one block per batch),
// one component per slot for every family: the meta-GGA operand
// T_r = t d_r phi (t = w v_tau / 4, so that V = M + M^T carries
// (1/2) w v_tau grad phi_mu . grad phi_nu) is formed from the cached d_r phi
// while the Vxc kernel loads it, instead of being stored.
// kMakeBMat matrices at a time read phi and grad phi once for all of them.
constexpr int kMakeBMat = 4;
__global__ __launch_bounds__(256) void k_make_b(const int* __restrict__ bt_off, const double* __restrict__ coef,
                                                size_t sC, const double* __restrict__ coef1,
                                                const double* __restrict__ cache, double* __restrict__ bmat,
                                                size_t sB, int nmat) {
  __shared__ double cf[kMakeBMat][4][kBatch];
  const int b = blockIdx.x, tid = threadIdx.x, m0 = blockIdx.y * kMakeBMat, nm = min(kMakeBMat, nmat - m0);
  for (int e = tid; e < nm * 4 * kBatch; e += 256) {
    const int m = e / (4 * kBatch), c = (e / kBatch) % 4, g = e % kBatch;
    const double* __restrict__ src = coef1 && m0 + m == 1 ? coef1 : coef + (m0 + m) * sC;
    cf[m][c][g] = src[kCoef * ((size_t)b * kBatch + g) + c];
  }
  __syncthreads();
  bmat += m0 * sB;
  for (int it = bt_off[b]; it < bt_off[b + 1]; ++it) {
    const double* src = cache + (size_t)it * kSlotAO;
    double* dst = bmat + (size_t)it * kSlotB;
    for (int e = tid; e < kSlotB; e += 256) {
      const int g = e / kTile;
      const double v = src[e], dx = src[kSlotB + e], dy = src[2 * kSlotB + e], dz = src[3 * kSlotB + e];
#pragma unroll
      for (int m = 0; m < kMakeBMat; ++m)
        if (m < nm) dst[m * sB + e] = cf[m][0][g] * v + cf[m][1][g] * dx + cf[m][2][g] * dy + cf[m][3][g] * dz;
    }
  }
}

void launch_make_b(hipStream_t s, int nbatches, const int* bt_off, const double* coef, const double* cache,
                   double* bmat, int nmat, size_t sC, size_t sB, const double* coef1) {
  if (nbatches == 0) return;
  hipLaunchKernelGGL(k_make_b, dim3(nbatches, (nmat + kMakeBMat - 1) / kMakeBMat), dim3(256), 0, s, bt_off, coef, sC,
                     coef1, cache, bmat, sB, nmat);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Contractions over the points, C_IJ = sum_g A_I[g]^T B_J[g], for groups I and J
// of up to 4 of a chunk's tiles over a run of its batches. 4 waves in a 2 x 2
// grid, each owning half of the row and of the column blocks (up to 64 x 64).
// Passes over the batch's 64 points, 4 points per product, lane (lk, lrow) point
// lk and AO lrow of either operand:
//   KIND 0: V of one run, upper blocks I0 <= J0: phi^T B, and for I < J B^T phi
//           into the same accumulators; I = J is symmetrised through LDS;
//   KIND 1: the same with the meta-GGA passes (d_r phi)^T (t d_r phi) first (t =
//           coef[4] of the point; twice t for I < J, the term is symmetric);
//   KIND 2: A^T B alone for any (I, J), added to M by FP64 atomics.
// KIND 0 and 1 store the block once into U (see k_assemble). C18 / def2-TZVP
// r2SCAN: 4.3 ms (9.6 with both triangles, LDS stages and atomics into M).
constexpr int kSymStrip = 32;  // columns of the diagonal block transposed at a time
template <int KIND>
__global__ __launch_bounds__(256, 2) void k_vxc_c64(const MxItem* __restrict__ work, const double* __restrict__ cache,
                                                    const double* __restrict__ bmat, const double* __restrict__ coef,
                                                    const int* __restrict__ ao_of, double* __restrict__ out,
                                                    int npad, ProdBatch pb) {
  int item = blockIdx.x;
  if (gridDim.y > 1) {  // an item's matrices side by side on one XCD: they share the operand A
    const int nm = gridDim.y, full = gridDim.x / 8 * 8, lin = blockIdx.y * gridDim.x + blockIdx.x;
    const int r = lin - full * nm, rest = gridDim.x - full;
    const int mat = r < 0 ? lin / 8 % nm : r / rest;
    item = r < 0 ? lin / (8 * nm) * 8 + lin % 8 : full + r % rest;
    cache += (mat / pb.nb) * pb.sA;
    bmat += (mat % pb.nb) * pb.sB;
    out += mat * pb.sO;
  }
  const MxItem wk = work[item];
  const bool diag = wk.I0 == wk.J0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;
  const int nr = wk.nI, nc = wk.nJ, r0 = nr * (wave & 1), c0 = nc * (wave >> 1);  // the wave's row and column blocks
  const int ntau = KIND == 1 ? 3 : 0, npass = ntau + (KIND == 2 || diag ? 1 : 2);
  dbl4 acc[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = dbl4{0, 0, 0, 0};
  double a[2][2][4], bb[2][2][4], tt[2][2];  // [buffer][4-point step of the pair][block]
  const int lo = lk * kTile + lrow;
  auto load = [&](int k, int buf) {  // piece k: 8 points of one pass of one batch
    const int p8 = k & 7, pass = (k >> 3) % npass, it = (k >> 3) / npass;
    const size_t s0 = (size_t)wk.slot0 + (size_t)it * wk.ntl;
    const bool tau = pass < ntau, swap = pass > ntau;
    const double* __restrict__ pa = (swap ? bmat + (s0 + wk.I0) * kSlotB
                                          : cache + (s0 + wk.I0) * kSlotAO + (tau ? pass + 1 : 0) * kSlotB) +
                                    8 * p8 * kTile + lo;
    const double* __restrict__ pB = (tau    ? cache + (s0 + wk.J0) * kSlotAO + (pass + 1) * kSlotB
                                     : swap ? cache + (s0 + wk.J0) * kSlotAO
                                            : bmat + (s0 + wk.J0) * kSlotB) +
                                    8 * p8 * kTile + lo;
    const int sa = swap ? kSlotB : kSlotAO, sb = tau || swap ? kSlotAO : kSlotB;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      double t = 1.0;  // (non-tau passes load one too)
      if (KIND == 1) t = coef[kCoef * ((size_t)(wk.batch0 + it) * kBatch + 8 * p8 + 4 * e + lk) + 4];
      if (KIND == 1) tt[buf][e] = t;
#pragma unroll
      for (int r = 0; r < 4; ++r) {  // past the group: its last block again (a branch would wait for all loads)
        const int q = r0 + min(r, nr - 1);
        a[buf][e][r] = pa[(size_t)(q >> 1) * sa + (q & 1) * 16 + 4 * e * kTile];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int q = c0 + min(c, nc - 1);
        bb[buf][e][c] = pB[(size_t)(q >> 1) * sb + (q & 1) * 16 + 4 * e * kTile];
      }
    }
  };
  auto step = [&](int k, int buf) {
    double scale = 1.0;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (KIND == 1) scale = (k >> 3) % npass < ntau ? (diag ? 1.0 : 2.0) * tt[buf][e] : 1.0;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < nc) {
          const double v = KIND == 1 ? scale * bb[buf][e][c] : bb[buf][e][c];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (r < nr) acc[r][c] = mfma_f64(a[buf][e][r], v, acc[r][c]);
        }
    }
  };
  const int n8 = wk.nbat * npass * 8;  // even
  load(0, 0);
  for (int k = 0; k < n8; k += 2) {
    load(k + 1, 1);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products that they run beside
    step(k, 0);
    load(min(k + 2, n8 - 1), 0);
    __builtin_amdgcn_sched_barrier(0);
    step(k + 1, 1);
  }
  // C layout: acc[r][c][i] = C[row 16 (r0 + r) + 4 i + lk][column 16 (c0 + c) + lrow]
  if (KIND == 2) {
    const int* __restrict__ ao = ao_of + (size_t)wk.tile0 * kTile;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mu = ao[wk.I0 * kTile + 16 * (r0 + r) + 4 * i + lk];
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c < nc) {
              const int nu = ao[wk.J0 * kTile + 16 * (c0 + c) + lrow];
              if (mu >= 0 && nu >= 0) unsafeAtomicAdd(&out[(size_t)mu * npad + nu], acc[r][c][i]);
            }
        }
      }
    return;
  }
  double* __restrict__ U = out + wk.u;
  const int ld = wk.ldu;
  if (!diag) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nr) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < nc) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              U[(size_t)(16 * (r0 + r) + 4 * i + lk) * ld + 16 * (c0 + c) + lrow] = acc[r][c][i];
          }
      }
    return;
  }
  __shared__ double T[kSymStrip][4 * kTile + 4];
  for (int s = 0; s < 2 * nc; s += kSymStrip / 16) {  // U = M + M^T, 32 rows at a time
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c < nc && c0 + c >= s && c0 + c < s + kSymStrip / 16) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r < nr) {
#pragma unroll
            for (int i = 0; i < 4; ++i) T[16 * (c0 + c - s) + lrow][16 * (r0 + r) + 4 * i + lk] = acc[r][c][i];
          }
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nr && r0 + r >= s && r0 + r < s + kSymStrip / 16) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c < nc) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int row = 16 * (r0 + r) + 4 * i + lk, col = 16 * (c0 + c) + lrow;
              U[(size_t)row * ld + col] = acc[r][c][i] + T[row - 16 * s][col];
            }
          }
      }
  }
}

void launch_vxc_c64(hipStream_t s, int ncomp, int nwork, const MxItem* work, const double* cache, const double* bmat,
                    const double* coef, double* U, int nmat, size_t sB, size_t sU) {
  if (nwork == 0) return;
  const ProdBatch pb{nmat, 0, sB, sU};
  if (ncomp == 4)
    hipLaunchKernelGGL(k_vxc_c64<1>, dim3(nwork), dim3(256), 0, s, work, cache, bmat, coef, nullptr, U, 0, pb);
  else
    hipLaunchKernelGGL(k_vxc_c64<0>, dim3(nwork, nmat), dim3(256), 0, s, work, cache, bmat, coef, nullptr, U, 0, pb);
  CHX_HIP(hipGetLastError());
}

void launch_prod_c64(hipStream_t s, int nwork, const MxItem* work, const int* ao_of, const double* cache,
                     const double* bmat, double* M, int npad, int nmat, const ProdBatch& pb) {
  if (nwork == 0) return;
  hipLaunchKernelGGL(k_vxc_c64<2>, dim3(nwork, nmat), dim3(256), 0, s, work, cache, bmat, nullptr, ao_of, M, npad, pb);
  CHX_HIP(hipGetLastError());
}

// V (reference order, column-major) = M + M^T.
__global__ void k_finalize_sym(int n, int npad, const double* __restrict__ Mint, double* __restrict__ V) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)n * n) return;
  const int col = (int)(idx / n), row = (int)(idx % n);
  V[idx] = Mint[(size_t)row * npad + col] + Mint[(size_t)col * npad + row];
}

void launch_finalize_sym(hipStream_t s, int n, int npad, const double* Mint, double* V) {
  const long tot = (long)n * n;
  hipLaunchKernelGGL(k_finalize_sym, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, n, npad, Mint, V);
  CHX_HIP(hipGetLastError());
}

}  // namespace chx
