// Grid set-up on the device: Becke weights and the bisection of the points into
// batches (GridGeneration.cpp:75-153 and the sub-grid split after it).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"

namespace chx {

// ---------------------------------------------------------------------------
// Becke partition (GridGeneration.cpp:136-153): w *= P_owner / sum_B P_B,
// P_B = prod_{C != B} s(mu_BC), s = (1 - p(p(p(mu))))/2, p(m) = 1.5m - 0.5m^3.
// All pairs of atoms per point (lane = point): bound by the FP64 rate. Eight
// atoms B go through the C's together: the distance to C is formed once for the
// eight and their products are independent chains (distances kept in LDS instead
// left one wave per SIMD and were slower). The division by R_BC is a product with
// its reciprocal and two corrections by the remainder (P. Markstein, IBM J. Res.
// Dev. 34, 1990: correctly rounded from a quotient within one ulp), so that
// weights, and which of them are zero, are those of the division. (H2O)24 / SG-1:
// 1.65 ms (3.4 with a division and two square roots in every pair).
constexpr int kBeckeB = 8;
__device__ __forceinline__ double becke_factor(double num, double2 r) {  // r = (R, 1 / R)
  double q = num * r.y;
  q = __builtin_fma(__builtin_fma(-q, r.x, num), r.y, q);
  double m = __builtin_fma(__builtin_fma(-q, r.x, num), r.y, q);
  m = 1.5 * m - 0.5 * m * m * m;
  m = 1.5 * m - 0.5 * m * m * m;
  m = 1.5 * m - 0.5 * m * m * m;
  return 0.5 * (1.0 - m);
}

__global__ __launch_bounds__(64) void k_becke(long npts, const double* __restrict__ px, const double* __restrict__ py,
                                              const double* __restrict__ pz, double* __restrict__ w,
                                              const int* __restrict__ owner, int natoms,
                                              const double* __restrict__ axyz, const double2* __restrict__ rab, int ld) {
  const long i0 = (long)blockIdx.x * 64 + threadIdx.x, i = i0 < npts ? i0 : npts - 1;
  const double x = px[i], y = py[i], z = pz[i];
  auto distance = [&](int a) {
    const double dx = x - axyz[3 * a], dy = y - axyz[3 * a + 1], dz = z - axyz[3 * a + 2];
    return ::sqrt(dx * dx + dy * dy + dz * dz);
  };
  const int me = owner[i];
  double total = 0, mine = 0;
  for (int b = 0; b < natoms; b += kBeckeB) {
    double d[kBeckeB], p[kBeckeB];
#pragma unroll
    for (int q = 0; q < kBeckeB; ++q) {
      d[q] = distance(min(b + q, natoms - 1));
      p[q] = 1.0;
    }
    for (int c = 0; c < natoms; ++c) {
      const double rc = distance(c);
      const double2* __restrict__ r = rab + (size_t)c * ld + b;  // (R_CB = R_BC)
      bool alive = false;
#pragma unroll
      for (int q = 0; q < kBeckeB; ++q) {
        const double f = becke_factor(d[q] - rc, r[q]);
        p[q] = c != b + q && p[q] != 0.0 ? p[q] * f : p[q];  // a product that has reached zero stays there
        alive |= p[q] != 0.0;
      }
      if ((c & 7) == 7 && !__any(alive)) break;
    }
#pragma unroll
    for (int q = 0; q < kBeckeB; ++q)
      if (b + q < natoms) {
        total += p[q];
        if (b + q == me) mine = p[q];
      }
  }
  if (i0 < npts) w[i] *= mine / total;
}

void launch_becke(hipStream_t s, long npts, const double* px, const double* py, const double* pz, double* w,
                  const int* owner, int natoms, const double* atom_xyz, const double2* rab, int ld) {
  if (npts == 0) return;
  hipLaunchKernelGGL(k_becke, dim3((unsigned)((npts + 63) / 64)), dim3(64), 0, s, npts, px, py, pz, w, owner, natoms,
                     atom_xyz, rab, ld);
  CHX_HIP(hipGetLastError());
}

int becke_ld(int natoms) { return (natoms + kBeckeB - 1) / kBeckeB * kBeckeB; }

// ---------------------------------------------------------------------------
// One level of the bisection: a block takes a segment [lo, lo + n) and moves its
// points so that the `left` first ones along the longest axis of its bounding box
// (by coordinate, then by index) come first, both halves keeping their order; a
// segment that is a batch already (left = 0) is copied. Selection: 1024 equal
// bins over the range of the candidates, the bin that holds the wanted rank gives
// the next candidates, and the last kBisCand or fewer are ranked against each
// other; where the coordinates are all equal the index takes their place. Bins
// are monotone in the coordinate, so the result is exact. Bound by the passes
// over the segment (7 of its axis), for the first levels by the one block that
// makes them. (H2O)24 / SG-1, 264 000 points, all levels: 2.4 ms (22 on the host).
constexpr int kBisThreads = 1024, kBisWaves = kBisThreads / 64, kBisBins = 1024, kBisCand = 1024;
constexpr int kBisUnroll = 8;

__device__ __forceinline__ double bis_key(double v) { return fmin(fmax(v, -1e300), 1e300); }  // a total order

// min and max over the block, to all threads; ends with the scratch free again
__device__ __forceinline__ void block_min_max(double& mn, double& mx, double (*red)[2]) {
  for (int o = 32; o > 0; o >>= 1) {
    mn = fmin(mn, __shfl_xor(mn, o, 64));
    mx = fmax(mx, __shfl_xor(mx, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6][0] = mn;
    red[threadIdx.x >> 6][1] = mx;
  }
  __syncthreads();
  for (int w = 0; w < kBisWaves; ++w) {
    mn = fmin(mn, red[w][0]);
    mx = fmax(mx, red[w][1]);
  }
  __syncthreads();
}

__global__ __launch_bounds__(kBisThreads) void k_bisect(const BisSeg* __restrict__ segs,
                                                        const double* __restrict__ src, const int* __restrict__ sidx,
                                                        double* __restrict__ dst, int* __restrict__ didx, long stride) {
  __shared__ double red[kBisWaves][2], ckey[kBisCand], tkey;
  __shared__ int hist[kBisBins], cidx[kBisCand], scan[kBisWaves], ncand, bin_k, bin_m, bin_before, tidx;
  const BisSeg sg = segs[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = sg.n;
  src += sg.lo;
  sidx += sg.lo;
  dst += sg.lo;
  didx += sg.lo;
  if (sg.left == 0) {
    for (int i = tid; i < n; i += kBisThreads) {
      for (int d = 0; d < 3; ++d) dst[d * stride + i] = src[d * stride + i];
      didx[i] = sidx[i];
    }
    return;
  }
  // f(key, index) over the segment; kBisUnroll loads in flight (one block walks up to the whole grid)
  auto each = [&](const double* __restrict__ kp, bool with_idx, auto&& f) {
    for (int i0 = tid; i0 < n; i0 += kBisUnroll * kBisThreads) {
      double v[kBisUnroll];
      int id[kBisUnroll];
#pragma unroll
      for (int q = 0; q < kBisUnroll; ++q) v[q] = kp[min(i0 + q * kBisThreads, n - 1)];
      if (with_idx) {
#pragma unroll
        for (int q = 0; q < kBisUnroll; ++q) id[q] = sidx[min(i0 + q * kBisThreads, n - 1)];
      }
#pragma unroll
      for (int q = 0; q < kBisUnroll; ++q)
        if (i0 + q * kBisThreads < n) f(bis_key(v[q]), with_idx ? id[q] : 0);
    }
  };
  // the longest axis
  double a = 0, b = 0;
  int axis = 0;
  for (int d = 0; d < 3; ++d) {
    double mn = 1e300, mx = -1e300;
    each(src + d * stride, false, [&](double v, int) {
      mn = fmin(mn, v);
      mx = fmax(mx, v);
    });
    block_min_max(mn, mx, red);
    if (d == 0 || mx - mn > b - a) {
      a = mn;
      b = mx;
      axis = d;
    }
  }
  const double* __restrict__ key = src + axis * stride;
  // candidates: keys in [a, b], or with by_idx the points at val with an index in [a, b]
  int k = sg.left - 1, m = n;
  bool by_idx = false;
  double val = 0;
  auto cand = [&](double v, int id, double& kv) {
    kv = by_idx ? (double)id : v;
    return kv >= a && kv <= b && (!by_idx || v == val);
  };
  auto to_index = [&] {  // the candidates' keys are all equal: on to their indexes
    double mn = 1e300, mx = -1e300;
    each(key, true, [&](double v, int id) {
      if (v == a) {
        mn = fmin(mn, (double)id);
        mx = fmax(mx, (double)id);
      }
    });
    block_min_max(mn, mx, red);
    by_idx = true;
    val = a;
    a = mn;
    b = mx;
  };
  while (m > kBisCand) {  // the same in every thread; the first and the last candidate part company each time
    if (a == b) {
      if (by_idx) break;  // (indexes differ: not reached)
      to_index();
    }
    const double scale = kBisBins / (b - a);
    auto bin = [&](double v) {
      if (!(scale < 1e300)) return v > a ? kBisBins - 1 : 0;
      return min(kBisBins - 1, (int)((v - a) * scale));
    };
    for (int i = tid; i < kBisBins; i += kBisThreads) hist[i] = 0;
    __syncthreads();
    each(key, by_idx, [&](double v, int id) {
      double kv;
      if (cand(v, id, kv)) atomicAdd(&hist[bin(kv)], 1);
    });
    __syncthreads();
    // the bin of rank k (kBisBins == kBisThreads)
    const int h = hist[tid];
    int c = h;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(c, o, 64);
      if (lane >= o) c += t;
    }
    if (lane == 63) scan[wave] = c;
    __syncthreads();
    for (int w = 0; w < wave; ++w) c += scan[w];
    if (k < c && k >= c - h) {
      bin_k = tid;
      bin_m = h;
      bin_before = c - h;
    }
    __syncthreads();
    const int bk = bin_k;
    m = bin_m;
    k -= bin_before;
    double mn = 1e300, mx = -1e300;
    each(key, by_idx, [&](double v, int id) {
      double kv;
      if (cand(v, id, kv) && bin(kv) == bk) {
        mn = fmin(mn, kv);
        mx = fmax(mx, kv);
      }
    });
    block_min_max(mn, mx, red);
    a = mn;
    b = mx;
  }
  // rank the last ones against each other
  if (tid == 0) ncand = 0;
  __syncthreads();
  each(key, true, [&](double v, int id) {
    double kv;
    if (cand(v, id, kv)) {
      const int q = atomicAdd(&ncand, 1);
      if (q < kBisCand) {
        ckey[q] = kv;
        cidx[q] = id;
      }
    }
  });
  __syncthreads();
  const int nc = min(ncand, kBisCand);
  if (tid < nc) {
    const double mk = ckey[tid];
    const int mi = cidx[tid];
    int rank = 0;
    for (int q = 0; q < nc; ++q) rank += ckey[q] < mk || (ckey[q] == mk && cidx[q] < mi);
    if (rank == k) {
      tkey = by_idx ? val : mk;
      tidx = mi;
    }
  }
  __syncthreads();
  const double tk = tkey;
  const int ti = tidx;
  // split, in order: rows of kBisThreads points, four at a time; hist holds the waves' counts (two sets)
  int nl = 0, done = 0;
  for (int c0 = 0, set = 0; c0 < n; c0 += 4 * kBisThreads, set ^= 1) {
    int* __restrict__ cnt = hist + set * 4 * kBisWaves;
    bool in[4], go[4];
    unsigned long long bl[4], bi[4];
    double pt[4][3];
    int id[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = min(c0 + r * kBisThreads + tid, n - 1);
#pragma unroll
      for (int d = 0; d < 3; ++d) pt[r][d] = src[d * stride + i];
      id[r] = sidx[i];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      in[r] = c0 + r * kBisThreads + tid < n;
      const double v = bis_key(axis == 0 ? pt[r][0] : axis == 1 ? pt[r][1] : pt[r][2]);
      go[r] = in[r] && (v < tk || (v == tk && id[r] <= ti));
      bl[r] = __ballot(go[r]);
      bi[r] = __ballot(in[r]);
      if (lane == 0) cnt[r * kBisWaves + wave] = __popcll(bl[r]);
    }
    __syncthreads();
    const int own = cnt[lane];  // 4 rows x 16 waves = 64 counts
    int c = own;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(c, o, 64);
      if (lane >= o) c += t;
    }
    const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = r * kBisWaves + wave, before = __shfl(c - own, e, 64);
      const int pl = nl + before + __popcll(bl[r] & below);
      const int pr = sg.left + done - nl + (64 * e - before) + __popcll(bi[r] & ~bl[r] & below);
      const int q = go[r] ? pl : pr;
      if (in[r] && q < n) {
#pragma unroll
        for (int d = 0; d < 3; ++d) dst[d * stride + q] = pt[r][d];
        didx[q] = id[r];
      }
    }
    nl += __shfl(c, 63, 64);
    done += min(4 * kBisThreads, n - c0);
  }
}

// Points of the kept indexes, in their order.
__global__ __launch_bounds__(256) void k_take_points(long n, const int* __restrict__ idx, const double* __restrict__ px,
                                                     const double* __restrict__ py, const double* __restrict__ pz,
                                                     double* __restrict__ out, long stride) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int j = idx[i];
  out[i] = px[j];
  out[stride + i] = py[j];
  out[2 * stride + i] = pz[j];
}

// The batches' slots: points and weights, padding slots repeat the first point with w = 0.
__global__ __launch_bounds__(64) void k_batch_slots(const int2* __restrict__ batch, const double* __restrict__ pts,
                                                    const int* __restrict__ idx, long stride,
                                                    const double* __restrict__ w, double* __restrict__ bx,
                                                    double* __restrict__ by, double* __restrict__ bz,
                                                    double* __restrict__ bw) {
  const int2 bt = batch[blockIdx.x];  // first point, number of points
  const int k = threadIdx.x, p = bt.x + (k < bt.y ? k : 0);
  const size_t s = (size_t)blockIdx.x * kBatch + k;
  bx[s] = pts[p];
  by[s] = pts[stride + p];
  bz[s] = pts[2 * stride + p];
  bw[s] = k < bt.y ? w[idx[p]] : 0.0;
}

void launch_bisect(hipStream_t s, long n, const int* idx, const double* px, const double* py, const double* pz,
                   const std::vector<int>& levels, const BisSeg* segs, double* pts[2], int* ids[2]) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_take_points, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, idx, px, py, pz, pts[0], n);
  const int* from = idx;
  for (size_t l = 0; l + 1 < levels.size(); ++l) {  // from pts[l % 2], idx or ids[l % 2] to the other
    hipLaunchKernelGGL(k_bisect, dim3(levels[l + 1] - levels[l]), dim3(kBisThreads), 0, s, segs + levels[l],
                       pts[l & 1], from, pts[~l & 1], ids[~l & 1], n);
    from = ids[~l & 1];
  }
  CHX_HIP(hipGetLastError());
}

void launch_batch_slots(hipStream_t s, int nbatches, const int2* batch, const double* pts, const int* idx, long stride,
                        const double* w, double* bx, double* by, double* bz, double* bw) {
  if (nbatches == 0) return;
  hipLaunchKernelGGL(k_batch_slots, dim3(nbatches), dim3(kBatch), 0, s, batch, pts, idx, stride, w, bx, by, bz, bw);
  CHX_HIP(hipGetLastError());
}

}  // namespace chx
