// Mixed-precision form: the two dense contractions on split-BF16 MFMA.
//
// Every FP32 operand x is held as a pair of bf16 numbers, hi = bf16(x) and
// lo = bf16(x - hi), so that hi + lo carries 16 significant bits. A product
// x*y is formed as hi*hi' + hi*lo' + lo*hi' on v_mfma_f32_16x16x32_bf16 with
// FP32 accumulation (the dropped lo*lo' term is below 2^-16 |x y|). The
// functional, the E_xc / N_e sums and the final V accumulation stay FP64.
//
// The MFMA operands are cached at Grid::getAO in this split form (as the
// reference caches its AO tables once, src/Grid/Grid.cpp:22-33), nT = 1
// component (phi), or 4 (phi, d/dx, d/dy, d/dz) for meta-GGA, in two layouts:
//   AOg [c][g=0..63][hl][mu=0..31]  (K = mu contiguous: A of the density X = Phi D)
//   AOt [c][hl][mu=0..31][g=0..63]  (K = g contiguous: A of Vxc M = Phi^T B)
// 8 KB per component and layout per slot. Values needed outside the MFMA
// operands (the density epilogue, the Vxc integrand B) are recomputed in FP32
// from the basis: the hardware exp makes that cheaper than reading them back.
// The MFMA operand layouts used below: lane l, element e of the 8-vector holds
//   A[i = l % 16][k = 8 (l / 16) + e],  B[k = 8 (l / 16) + e][j = l % 16],
// and result register r of lane l is C[4 (l / 16) + r][l % 16].
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "internal.hpp"

namespace chx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;
// 16 bytes of operand data; a native vector (HIP's u32x4 is a struct whose
// copies the compiler may keep in private memory)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMxRow = 2 * kTile;             // one AOg row: 32 hi then 32 lo
constexpr int kMxT = 2 * kTile * kBatch;      // elements per component of AOg, AOt and Bt

// float -> bf16, round to nearest even: the hardware conversion
// (v_cvt_pk_bf16_f32). k_bf16_check compares it with the bit-level rule
// f2bf_rne on the device.
__device__ __forceinline__ u16 f2bf(float f) { return __builtin_bit_cast(u16, (__bf16)f); }
__device__ __forceinline__ u16 f2bf_rne(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ __forceinline__ float bf2f(u16 h) { return __uint_as_float((unsigned)h << 16); }
__device__ __forceinline__ void split_bf(float x, u16& hi, u16& lo) {
  hi = f2bf(x);
  lo = f2bf(x - bf2f(hi));
}

// Device check of the conversion: n pseudo-random finite floats spread over
// many binades; counts values where the hardware result differs from f2bf_rne.
__global__ void k_bf16_check(unsigned n, unsigned* __restrict__ bad) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsigned h = i * 2654435761u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  const unsigned e = 64u + (h >> 25);  // biased exponent 64..191
  const float f = __uint_as_float((h & 0x807fffffu) | (e << 23));
  if (f2bf(f) != f2bf_rne(f)) atomicAdd(bad, 1u);
}

__global__ void k_fill_u32(unsigned* p, size_t n, unsigned v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_u32(hipStream_t s, unsigned* p, size_t n, unsigned v) {
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  CHX_HIP(hipGetLastError());
}

void launch_bf16_check(hipStream_t s, unsigned n, unsigned* bad) {
  hipLaunchKernelGGL(k_bf16_check, dim3((n + 255) / 256), dim3(256), 0, s, n, bad);
  CHX_HIP(hipGetLastError());
}
__device__ __forceinline__ bf16x8 as_bf(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ f32x4 mfma3(u32x4 ah, u32x4 al, u32x4 bh, u32x4 bl, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(al), as_bf(bh), c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(ah), as_bf(bl), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(ah), as_bf(bh), c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// AO cache in split form: one block per slot. Values are evaluated in FP64,
// rounded to FP32 and split.
__global__ __launch_bounds__(256) void k_ao_cache_mx(const int* __restrict__ slot_batch, const int* __restrict__ slot_tile,
                                                     const double* __restrict__ bx, const double* __restrict__ by,
                                                     const double* __restrict__ bz, BasisView bv, int nT, int sstride,
                                                     u16* __restrict__ cache,
                                                     const int* __restrict__ slot_core, u16* __restrict__ cache3) {
  __shared__ float E[4][kBatch][kTile + 1];
  __shared__ double px[kBatch], py[kBatch], pz[kBatch];
  const int s = blockIdx.x, tid = threadIdx.x;
  const int b = slot_batch[s], t = slot_tile[s];
  for (int e = tid; e < 4 * kBatch * (kTile + 1); e += 256) (&E[0][0][0])[e] = 0.0f;  // padding AOs stay zero
  if (tid < kBatch) {
    px[tid] = bx[b * kBatch + tid];
    py[tid] = by[b * kBatch + tid];
    pz[tid] = bz[b * kBatch + tid];
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
        E[0][g][col] = (float)v[sg.y + m];
        E[1][g][col] = (float)gx[sg.y + m];
        E[2][g][col] = (float)gy[sg.y + m];
        E[3][g][col] = (float)gz[sg.y + m];
      }
  }
  __syncthreads();
  u16* out = cache + (size_t)s * sstride;
  for (int e = tid; e < nT * kBatch * kTile; e += 256) {
    const int c = e / (kBatch * kTile), g = (e / kTile) % kBatch, mu = e % kTile;
    u16 hi, lo;
    split_bf(E[c][g][mu], hi, lo);
    out[(c * kBatch + g) * kMxRow + mu] = hi;
    out[(c * kBatch + g) * kMxRow + kTile + mu] = lo;
  }
  u16* outt = out + nT * kMxT;
  for (int e = tid; e < nT * kTile * kBatch; e += 256) {
    const int c = e / (kTile * kBatch), mu = (e / kBatch) % kTile, g = e % kBatch;
    u16 hi, lo;
    split_bf(E[c][g][mu], hi, lo);
    outt[c * kMxT + mu * kBatch + g] = hi;
    outt[c * kMxT + kTile * kBatch + mu * kBatch + g] = lo;
  }
  const int cs = slot_core ? slot_core[s] : -1;
  if (cs >= 0) {  // core slot: the third term x - hi - lo, AOg order without the hl plane
    u16* o3 = cache3 + (size_t)cs * nT * kBatch * kTile;
    for (int e = tid; e < nT * kBatch * kTile; e += 256) {
      const int c = e / (kBatch * kTile), g = (e / kTile) % kBatch, mu = e % kTile;
      const float x = E[c][g][mu];
      u16 hi, lo;
      split_bf(x, hi, lo);
      o3[e] = f2bf((x - bf2f(hi)) - bf2f(lo));
    }
  }
}

void launch_ao_cache_mx(hipStream_t s, int nslots, const int* slot_batch, const int* slot_tile,
                        const double* bx, const double* by, const double* bz, BasisView bv, int nT, int sstride,
                        unsigned short* cache, const int* slot_core, unsigned short* cache3) {
  if (nslots == 0) return;
  hipLaunchKernelGGL(k_ao_cache_mx, dim3(nslots), dim3(256), 0, s, slot_batch, slot_tile, bx, by, bz, bv, nT,
                     sstride, cache, slot_core, cache3);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// The chunks' dense blocks of D in split form: per chunk [hl][nu][mu], ld = 32
// ntl. One block per tile of the chunks (its 32 rows nu against the chunk's
// columns mu), as k_gather_d; the blocks past the tiles form R (kRestBlock
// elements each), what the split leaves of D, D - hi - lo (its FP32 rounding
// included), at D's own position. The products see hi + lo; sum V . R, with V
// the potential of this density, is the first-order energy of the remainder
// (dE/dD = V), which the energy takes back when the potential is built
// (k_assemble). With asym (meta-GGA) the last blocks compare D with D^T: an
// element more than 1e-12 sqrt(D_ii D_jj) off (products of FP64 rounding stay far
// below, as this does below the split) sets *asym = gen, this build's number.
// One launch: small molecules (and packs of them) are bound by the launches.
constexpr int kRestBlock = 4096;
__global__ __launch_bounds__(256) void k_split_gather(int n, const double* __restrict__ D,
                                                      const int* __restrict__ tile_chunk,
                                                      const ChunkDev* __restrict__ chunks,
                                                      const int* __restrict__ ao_of, u16* __restrict__ Ds,
                                                      int ntiles, long n2, float* __restrict__ R, int nrest,
                                                      int* __restrict__ asym, int gen) {
  const int t = blockIdx.x;
  if (t >= ntiles + nrest) {  // 32 x 32 tile pair (i <= j) of the symmetry check
    check_symmetry(t - ntiles - nrest, n, D, 1e-12, asym, gen);
    return;
  }
  if (t >= ntiles) {
    const long e0 = (long)(t - ntiles) * kRestBlock, e1 = e0 + kRestBlock < n2 ? e0 + kRestBlock : n2;
    for (long i = e0 + threadIdx.x; i < e1; i += 256) {
      const double v = D[i];
      u16 hi, lo;
      split_bf((float)v, hi, lo);
      R[i] = (float)(v - (double)bf2f(hi) - (double)bf2f(lo));
    }
    return;
  }
  const ChunkDev c = chunks[tile_chunk[t]];
  const int ld = c.ntl * kTile;
  const size_t plane = (size_t)ld * ld;
  u16* __restrict__ out = Ds + 2 * c.doff + (size_t)(t - c.tile0) * kTile * ld;
  const int* __restrict__ cols = ao_of + (size_t)c.tile0 * kTile;
  __shared__ int rows[kTile];
  __shared__ float T[kTile][kTile + 1];
  if (threadIdx.x < kTile) rows[threadIdx.x] = ao_of[(size_t)t * kTile + threadIdx.x];
  for (int q = 0; q < c.ntl; ++q) {  // 32 x 32 sub-blocks, transposed through LDS so that both sides run along AOs
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * kTile; e += 256) {
      const int r = e & (kTile - 1), k = e >> 5, rr = rows[r], cc = cols[q * kTile + k];
      T[r][k] = rr >= 0 && cc >= 0 ? (float)D[(size_t)cc * n + rr] : 0.f;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kTile * kTile / 2; e += 256) {  // two columns per thread
      const int r = e >> 4, k = 2 * (e & 15);
      u16 h0, l0, h1, l1;
      split_bf(T[r][k], h0, l0);
      split_bf(T[r][k + 1], h1, l1);
      const size_t o = (size_t)r * ld + q * kTile + k;
      *reinterpret_cast<unsigned*>(out + o) = (unsigned)h0 | ((unsigned)h1 << 16);
      *reinterpret_cast<unsigned*>(out + plane + o) = (unsigned)l0 | ((unsigned)l1 << 16);
    }
  }
}

void launch_split_d(hipStream_t s, int ntiles, int n, const double* D, const int* tile_chunk, const ChunkDev* chunks,
                    const int* ao_of, unsigned short* Ds, float* R, int* asym, int gen) {
  const long n2 = (long)n * n;
  const int nrest = (int)((n2 + kRestBlock - 1) / kRestBlock);
  const unsigned nb = (unsigned)(ntiles + nrest + (asym ? symmetry_blocks(n) : 0));
  hipLaunchKernelGGL(k_split_gather, dim3(nb), dim3(256), 0, s, n, D, tile_chunk, chunks, ao_of, Ds, ntiles, n2, R, nrest,
                     asym, gen);
  CHX_HIP(hipGetLastError());
}

__device__ __forceinline__ double block_sum_d(double v) {
  __shared__ double red[16];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
  return t;
}

// V from the runs' blocks U (see k_vxc_mx): block mu sums row mu, columns nu >=
// mu, of every run whose list holds AO mu into FP64 sums in LDS, writes V[mu][nu]
// and V[nu][mu] (reference order), and with R the partial sum of V . R over them.
// 16 waves; a run's row is contiguous in U, kAsmUnroll rows are in flight per
// wave. Up to kAsmLds / 16 = 512 AOs each wave has a copy of the sums (COPIES =
// 16), so that a plain LDS read-add-write does, its rows ordered by wave-scope
// fences (which cost no instruction); larger rows share one (COPIES = 1)
// through ds_add_f64, which is the bound there, some 130 cycles per wave: fewer
// waves with copies are slower still. With one FP32 block per run: (H2O)16 48 us
// against 86 shared; (H2O)48 250 us shared against 363 with 4 waves; (H2O)128 700 us
// against 1430 with 2. With both products of a run, added here in FP64 (def2-SVP /
// SG-2): (H2O)16 57 us (48 with one FP32 sum), (H2O)48 157 to 201 (157 to 163),
// (H2O)128 0.78 ms (0.62).
// The FP64 atomics to HBM that all this replaces, one per element of M and run
// at about 40 G/s, took most of the Vxc launch. kAsmLds sums per block: larger
// bases take several column ranges (grid y).
constexpr int kAsmLds = 8192;
constexpr int kAsmUnroll = 8;
constexpr int kAsmThreads = 1024;
static int asm_copies(int n) { return n <= kAsmLds / 16 ? 16 : 1; }
static int asm_ranges(int n) { return (n + kAsmLds / asm_copies(n) - 1) / (kAsmLds / asm_copies(n)); }
int assemble_blocks(int n) { return n * asm_ranges(n); }

template <int COPIES, class T>
__global__ __launch_bounds__(kAsmThreads) void k_assemble(int n, const int* __restrict__ rowptr,
                                                             const RowRef* __restrict__ rows,
                                                             const int* __restrict__ ao_of,
                                                             const T* __restrict__ U, double* __restrict__ V,
                                                             const float* __restrict__ R,
                                                             double* __restrict__ cpart, size_t sU) {
  extern __shared__ double asum[];
  constexpr bool kTwo = sizeof(T) == 4;  // both products in FP32, the second sU elements on
  if (!kTwo) U += blockIdx.z * sU;       // the matrix of the launch
  V += (size_t)blockIdx.z * n * n;
  constexpr int kCols = kAsmLds / COPIES, kWaves = kAsmThreads / 64;
  const int mu = blockIdx.x, c0 = blockIdx.y * kCols, w = min(kCols, n - c0), tid = threadIdx.x;
  if (c0 + w <= mu) {  // below the diagonal: the block of row nu writes it
    if (R && tid == 0) cpart[(size_t)blockIdx.y * n + mu] = 0.0;
    return;
  }
  for (int i = tid; i < w * COPIES; i += kAsmThreads) asum[i] = 0.0;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  double* sum = COPIES == 1 ? asum : asum + (size_t)wave * w;
  const int e1 = rowptr[mu + 1];
  for (int e = rowptr[mu] + wave * kAsmUnroll; e < e1; e += kWaves * kAsmUnroll) {
    RowRef r[kAsmUnroll];
    int len = 0;
#pragma unroll
    for (int q = 0; q < kAsmUnroll; ++q) {
      r[q] = rows[min(e + q, e1 - 1)];
      if (e + q >= e1) r[q].len = 0;
      len = max(len, r[q].len);
    }
    for (int k0 = 0; k0 < len; k0 += 64) {  // every lane to the end: the fences below are for the whole wave
      const int k = k0 + lane;
      int nu[kAsmUnroll];
      T v[kAsmUnroll], v2[kAsmUnroll];
#pragma unroll
      for (int q = 0; q < kAsmUnroll; ++q) {  // clamped, not skipped: the loads go out together
        const int kk = min(k, max(r[q].len - 1, 0));
        nu[q] = ao_of[r[q].a0 + kk] - c0;
        v[q] = U[r[q].u + kk];
        if (kTwo) v2[q] = U[sU + r[q].u + kk];
        if (k >= r[q].len) nu[q] = -1;
      }
#pragma unroll
      for (int q = 0; q < kAsmUnroll; ++q) {
        const double x = kTwo ? (double)v[q] + (double)v2[q] : (double)v[q];
        if (nu[q] >= 0 && nu[q] < w) {
          if (COPIES == 1)
            __hip_atomic_fetch_add(&sum[nu[q]], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          else
            sum[nu[q]] += x;
        }
        if (COPIES > 1) {  // a row's columns differ, two rows' may not: one row's sums before the next one's
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
          __builtin_amdgcn_wave_barrier();
        }
      }
    }
  }
  __syncthreads();
  double acc = 0.0;
  for (int i = max(0, mu - c0) + tid; i < w; i += kAsmThreads) {
    double v = asum[i];
#pragma unroll
    for (int c = 1; c < COPIES; ++c) v += asum[(size_t)c * w + i];
    const size_t up = (size_t)mu * n + c0 + i, lo = (size_t)(c0 + i) * n + mu;
    V[up] = v;
    V[lo] = v;
    if (R) acc += v * (up == lo ? (double)R[up] : (double)R[up] + (double)R[lo]);
  }
  if (R) {
    acc = block_sum_d(acc);
    if (tid == 0) cpart[(size_t)blockIdx.y * n + mu] = acc;
  }
}

template <class T>
void launch_assemble(hipStream_t s, int n, const int* rowptr, const RowRef* rows, const int* ao_of, const T* U,
                     double* V, const float* R, double* cpart, int nmat, size_t sU) {
  if (n == 0) return;
  const int copies = asm_copies(n);
  const dim3 grid(n, asm_ranges(n), nmat);
  const size_t lds = (size_t)std::min(n, kAsmLds / copies) * copies * sizeof(double);
  if (copies == 16)
    hipLaunchKernelGGL((k_assemble<16, T>), grid, dim3(kAsmThreads), lds, s, n, rowptr, rows, ao_of, U, V, R, cpart, sU);
  else
    hipLaunchKernelGGL((k_assemble<1, T>), grid, dim3(kAsmThreads), lds, s, n, rowptr, rows, ao_of, U, V, R, cpart, sU);
  CHX_HIP(hipGetLastError());
}
template void launch_assemble<float>(hipStream_t, int, const int*, const RowRef*, const int*, const float*, double*,
                                     const float*, double*, int, size_t);
template void launch_assemble<double>(hipStream_t, int, const int*, const RowRef*, const int*, const double*, double*,
                                      const float*, double*, int, size_t);

__global__ __launch_bounds__(256) void k_reduce_corr(int nparts, const double* __restrict__ cpart,
                                                     double* __restrict__ out) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < nparts; i += 256) acc += cpart[i];
  acc = block_sum_d(acc);
  if (threadIdx.x == 0) *out = acc;
}

void launch_reduce_corr(hipStream_t s, int nparts, const double* cpart, double* out) {
  hipLaunchKernelGGL(k_reduce_corr, dim3(1), dim3(256), 0, s, nparts, cpart, out);
  CHX_HIP(hipGetLastError());
}

// One block per molecule of a pack lane: its partials (at base + cpart) added
// to its energy, after the functional's sums have written it.
__global__ __launch_bounds__(256) void k_corr_multi(const char* __restrict__ base, const FnMolecule* __restrict__ fm,
                                                    double* __restrict__ en) {
  const FnMolecule m = fm[blockIdx.x];
  const double* cpart = reinterpret_cast<const double*>(base + m.cpart);
  double acc = 0.0;
  for (int i = threadIdx.x; i < m.ncpart; i += 256) acc += cpart[i];
  acc = block_sum_d(acc);
  if (threadIdx.x == 0) en[2 * m.slot_en] += acc;
}

void launch_corr_multi(hipStream_t s, const char* base, const FnMolecule* fm, int nmol, double* en) {
  if (nmol <= 0) return;
  hipLaunchKernelGGL(k_corr_multi, dim3((unsigned)nmol), dim3(256), 0, s, base, fm, en);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Angular parts of one shell in FP32 (same conventions as shell_eval:
// src/Grid/AO/{S,CartP,PureP,PureD,PureF}.hpp). phi_m = R Q_m and
// grad phi_m = grad R Q_m + R grad Q_m with R = sum_p c_p exp(-a_p r^2), so an
// operation sees the radial part once per shell (op.begin / op.end) and, per
// component, op.comp(column, Q, dQ/dx, dQ/dy, dQ/dz). The shell type is a
// template argument: each type's polynomials are straight-line code, the
// constant derivatives fold away, and components first..first+cnt-1 are
// emitted with compile-time indices.
template <int TYPE, class Op>
__device__ __forceinline__ void emit_shell_f32(float x, float y, float z, int first, int cnt, int col, Op& op) {
  constexpr int n = TYPE == 0 ? 1 : TYPE == -2 ? 5 : TYPE == -3 ? 7 : 3;
  float q[n], qx[n], qy[n], qz[n];
  const float r3 = 1.7320508075688772f, r6 = 2.449489742783178f, r10 = 3.1622776601683795f, r15 = 3.872983346207417f;
  if (TYPE == 0) {
    q[0] = 1.f; qx[0] = qy[0] = qz[0] = 0.f;
  } else if (TYPE == 1) {  // Cartesian p: x, y, z
    q[0] = x; qx[0] = 1.f; qy[0] = 0.f; qz[0] = 0.f;
    q[1] = y; qx[1] = 0.f; qy[1] = 1.f; qz[1] = 0.f;
    q[2] = z; qx[2] = 0.f; qy[2] = 0.f; qz[2] = 1.f;
  } else if (TYPE == -1) {  // pure p: y, z, x
    q[0] = y; qx[0] = 0.f; qy[0] = 1.f; qz[0] = 0.f;
    q[1] = z; qx[1] = 0.f; qy[1] = 0.f; qz[1] = 1.f;
    q[2] = x; qx[2] = 1.f; qy[2] = 0.f; qz[2] = 0.f;
  } else if (TYPE == -2) {
    q[0] = r3 * x * y;                     qx[0] = r3 * y; qy[0] = r3 * x;  qz[0] = 0.f;
    q[1] = r3 * y * z;                     qx[1] = 0.f;    qy[1] = r3 * z;  qz[1] = r3 * y;
    q[2] = z * z - 0.5f * (x * x + y * y); qx[2] = -x;     qy[2] = -y;      qz[2] = 2.f * z;
    q[3] = r3 * x * z;                     qx[3] = r3 * z; qy[3] = 0.f;     qz[3] = r3 * x;
    q[4] = 0.5f * r3 * (x * x - y * y);    qx[4] = r3 * x; qy[4] = -r3 * y; qz[4] = 0.f;
  } else {
    const float xx = x * x, yy = y * y, zz = z * z;
    const float c10 = 0.25f * r10, c6 = 0.25f * r6;
    q[0] = c10 * y * (3.f * xx - yy);     qx[0] = c10 * 6.f * x * y;  qy[0] = c10 * 3.f * (xx - yy);             qz[0] = 0.f;
    q[1] = r15 * x * y * z;               qx[1] = r15 * y * z;        qy[1] = r15 * x * z;                       qz[1] = r15 * x * y;
    q[2] = c6 * y * (4.f * zz - xx - yy); qx[2] = -c6 * 2.f * x * y;  qy[2] = c6 * (4.f * zz - xx - 3.f * yy);  qz[2] = c6 * 8.f * y * z;
    q[3] = z * (zz - 1.5f * (xx + yy));   qx[3] = -3.f * x * z;       qy[3] = -3.f * y * z;                      qz[3] = 3.f * zz - 1.5f * (xx + yy);
    q[4] = c6 * x * (4.f * zz - xx - yy); qx[4] = c6 * (4.f * zz - 3.f * xx - yy); qy[4] = -c6 * 2.f * x * y;   qz[4] = c6 * 8.f * x * z;
    q[5] = 0.5f * r15 * (xx - yy) * z;    qx[5] = r15 * x * z;        qy[5] = -r15 * y * z;                      qz[5] = 0.5f * r15 * (xx - yy);
    q[6] = c10 * x * (xx - 3.f * yy);     qx[6] = c10 * 3.f * (xx - yy); qy[6] = -c10 * 6.f * x * y;             qz[6] = 0.f;
  }
  if (first == 0 && cnt == n) {  // the usual case: the whole shell lies in this tile
#pragma unroll
    for (int m = 0; m < n; ++m) op.comp(col + m, q[m], qx[m], qy[m], qz[m]);
  } else {
#pragma unroll
    for (int m = 0; m < n; ++m) {
      const int k = m - first;  // component m of the shell is AO col + k of the tile
      if (k >= 0 && k < cnt) op.comp(col + k, q[m], qx[m], qy[m], qz[m]);
    }
  }
}

// One wave walks one tile at 64 points, lane = point. Every segment record
// comes in through scalar loads and the shell loop is uniform across the
// wave: no divergence, no LDS, no block barrier. The offset from the centre
// is taken in FP64 (points and centres are tens of bohr apart, the offsets
// that matter are small), everything after it in FP32 with the hardware exp2.
// The basis tables are read through the constant address space: they never
// change while a kernel runs, and so are always read with scalar loads (a
// kernel that also issues LDS DMA loads would otherwise get vector loads).
using cvec4 = const __attribute__((address_space(4))) u32x4;
struct SegHead {  // the first 80 bytes of a record
  double ax, ay, az;
  int meta, col;
  float p[kSegInline][3];
};
__device__ __forceinline__ SegHead load_seghead(const SegRec* recs, int k) {
  static_assert(sizeof(SegHead) == 5 * sizeof(u32x4) && offsetof(SegRec, p) == offsetof(SegHead, p), "record layout");
  u32x4 w[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) w[i] = ((cvec4*)(recs + k))[i];
  SegHead r;
  __builtin_memcpy(&r, w, sizeof(SegHead));
  return r;
}

// R = sum_p c_p exp(-a_p r^2) and sum_p a_p c_p exp(-a_p r^2) over NP primitives
template <int NP>
__device__ __forceinline__ void radial_f32(const SegHead& h, const SegRec* rec, float r2, float& A0, float& A1) {
  A0 = A1 = 0.f;
  auto add = [&](float e, float c, float ec) {
    const float v = __builtin_amdgcn_exp2f(e * r2);
    A0 += c * v;
    A1 += ec * v;
  };
#pragma unroll
  for (int i = 0; i < (NP < kSegInline ? NP : kSegInline); ++i) add(h.p[i][0], h.p[i][1], h.p[i][2]);
  if (NP > kSegInline) {
    constexpr int kMore = NP > kSegInline ? (3 * (NP - kSegInline) + 3) / 4 : 1;
    u32x4 w[kMore];
#pragma unroll
    for (int i = 0; i < kMore; ++i) w[i] = ((cvec4*)rec)[5 + i];
#pragma unroll
    for (int i = kSegInline; i < NP; ++i) {
      const int o = 3 * (i - kSegInline);
      add(__uint_as_float(w[o / 4][o % 4]), __uint_as_float(w[(o + 1) / 4][(o + 1) % 4]),
          __uint_as_float(w[(o + 2) / 4][(o + 2) % 4]));
    }
  }
}

// PREFETCH: the next record is loaded while the current one is evaluated
// (for an Op that reads no LDS, whose waits would take the record load along).
template <bool PREFETCH = false, class Op>
__device__ __forceinline__ void walk_tile_f32(const BasisView& bv, int t, double px, double py, double pz, Op& op) {
  using cint = const __attribute__((address_space(4))) int;
  const int s0 = ((cint*)bv.tile_seg_off)[t], s1 = ((cint*)bv.tile_seg_off)[t + 1];
  float x = 0.f, y = 0.f, z = 0.f, r2 = 0.f;
  SegHead nxt;
  if (PREFETCH && s0 < s1) nxt = load_seghead(bv.segrec, s0);
  for (int k = s0; k < s1; ++k) {
    SegHead rec;
    if (PREFETCH) {
      rec = nxt;
      nxt = load_seghead(bv.segrec, k + 1 < s1 ? k + 1 : k);
    } else {
      rec = load_seghead(bv.segrec, k);
    }
    if (!(rec.meta & kSegSame)) {  // a new centre (the shells of an atom follow each other)
      x = (float)(px - rec.ax);
      y = (float)(py - rec.ay);
      z = (float)(pz - rec.az);
      r2 = x * x + y * y + z * z;
    }
    float A0, A1;
    const SegRec* rp = bv.segrec + k;
    const int np = (rec.meta >> 8) & 0x7f;
    if (np == 1) {  // primitive count: straight-line code per count
      radial_f32<1>(rec, rp, r2, A0, A1);
    } else {
      switch (np) {
        case 2: radial_f32<2>(rec, rp, r2, A0, A1); break;
        case 3: radial_f32<3>(rec, rp, r2, A0, A1); break;
        case 4: radial_f32<4>(rec, rp, r2, A0, A1); break;
        case 5: radial_f32<5>(rec, rp, r2, A0, A1); break;
        case 6: radial_f32<6>(rec, rp, r2, A0, A1); break;
        case 7: radial_f32<7>(rec, rp, r2, A0, A1); break;
        case 8: radial_f32<8>(rec, rp, r2, A0, A1); break;
        default: radial_f32<kSegPrim>(rec, rp, r2, A0, A1); break;  // unused slots hold c = 0
      }
    }
    // R = A0, grad R = -2 r A1
    op.begin(A0, -2.f * x * A1, -2.f * y * A1, -2.f * z * A1);
    const int first = (rec.meta >> 16) & 0xff, cnt = rec.meta >> 24;
    switch ((int)(signed char)(rec.meta & 0xff)) {
      case 0: emit_shell_f32<0>(x, y, z, first, cnt, rec.col, op); break;
      case 1: emit_shell_f32<1>(x, y, z, first, cnt, rec.col, op); break;
      case -1: emit_shell_f32<-1>(x, y, z, first, cnt, rec.col, op); break;
      case -2: emit_shell_f32<-2>(x, y, z, first, cnt, rec.col, op); break;
      default: emit_shell_f32<-3>(x, y, z, first, cnt, rec.col, op); break;
    }
    op.end();
  }
}

// Density epilogue on one tile at this lane's point, as sums per shell of X Q
// and X grad Q times R and grad R: with X = Phi D, o[0] = sum_nu X_nu phi_nu and
// o[1..3] = sum_nu X_nu grad phi_nu; TAU: with X_r = (d_r Phi) D also
// o[4 + r] = sum_nu X_r,nu d_r phi_nu, from the same walk over the shells (the
// walk, not the MFMAs, is most of a GGA density on lists of a few hundred AOs). The
// three directions stay apart: they are added in FP64, where the functional sums tau.
// X is held in registers (uniform column index: no memory access).
typedef float f32x32 __attribute__((ext_vector_type(32)));
constexpr int kXPitch = kBatch + 4;  // of X^T in LDS: 16-byte rows that 16 lanes write without bank conflicts
template <bool TAU>
struct DensEpi {
  f32x32 xv[TAU ? 4 : 1];
  float o[TAU ? 7 : 4] = {};
  float R, Rx, Ry, Rz, S0, Sx, Sy, Sz, Tx, Ty, Tz, Ux, Uy, Uz;
  // xq: X^T of this tile at this lane's point, xq[col * kXPitch]
  __device__ void load(int d, const float* xq) {
#pragma unroll
    for (int c = 0; c < kTile; ++c) xv[d][c] = xq[c * kXPitch];
  }
  __device__ void begin(float a, float ax, float ay, float az) {
    R = a; Rx = ax; Ry = ay; Rz = az;
    S0 = Sx = Sy = Sz = 0.f;
    if (TAU) Tx = Ty = Tz = Ux = Uy = Uz = 0.f;
  }
  __device__ void comp(int col, float q, float qx, float qy, float qz) {
    const float v = xv[0][col];
    S0 += v * q;
    Sx += v * qx;
    Sy += v * qy;
    Sz += v * qz;
    if (TAU) {
      const float vx = xv[TAU ? 1 : 0][col], vy = xv[TAU ? 2 : 0][col], vz = xv[TAU ? 3 : 0][col];
      Tx += vx * q;
      Ty += vy * q;
      Tz += vz * q;
      Ux += vx * qx;
      Uy += vy * qy;
      Uz += vz * qz;
    }
  }
  __device__ void end() {
    o[0] += R * S0;
    o[1] += Rx * S0 + R * Sx;
    o[2] += Ry * S0 + R * Sy;
    o[3] += Rz * S0 + R * Sz;
    if (TAU) {
      o[TAU ? 4 : 0] += R * Ux + Rx * Tx;
      o[TAU ? 5 : 0] += R * Uy + Ry * Ty;
      o[TAU ? 6 : 0] += R * Uz + Rz * Tz;
    }
  }
};

// ---------------------------------------------------------------------------
// Density. Block = (batch, group of <= 4 tiles of its list as output columns), 4
// waves in a 2 x 2 grid: wave (wr, wc) owns rows g = 32 wr..+31 and columns
// 64 wc..+63 of X = Phi_b D_b (64 x 128). K loop over the list's tiles
// (32 AOs = one MFMA K step). A K step's operands (A: 64 points x 32 AOs, D:
// 128 columns x 32 AOs, hi and lo) are 24 fragments of 1 KB that the waves'
// DMA loads (global_load_lds_dwordx4: lane i -> bytes 16 i of the fragment)
// bring from memory straight into LDS (no VGPR staging), coalesced, in a
// swizzled order from which the MFMA lanes read without bank conflicts.
// Per step: wait for the step's fragments, read the wave's 12 into registers,
// barrier, start the DMA of the next step into the same buffer, run the
// wave's 24 MFMAs while it lands (one buffer of 24 KB, 28 with the third terms,
// under X^T's 34: 39.5 KB in all, so four blocks share a CU and cover each
// other's barriers). Epilogue: X goes to LDS, wave q loads
// tile q's columns at its lane's point into registers and contracts them with
// phi / grad phi recomputed in FP32.
constexpr int kDxFrag = 64;  // u32x4 per fragment
constexpr int kDxA = 8;      // A fragments per step: [row block][hl]
constexpr int kDxB = 16;     // D fragments per step: [column block][hl]
constexpr int kDxA3 = 4;     // P3: third-term A fragments per step: [row block]
struct DensMxSmem {
  union {
    u32x4 F[(kDxA + kDxB + kDxA3) * kDxFrag];  // one K step's fragments
    float X[kGroup * kTile][kXPitch];          // epilogue: X^T [nu][g]
  };
  float red[kGroup][4][kBatch];
  double px[kBatch], py[kBatch], pz[kBatch];
};

// A = phi; epilogue rho and grad rho / 2 (4 components into part).
// P3 (core batches only): the AO operand carries a third bf16 term (x - hi -
// lo, 24 significant bits in all) from the core slots' side cache, and a
// product takes the five terms hi hi, lo hi, hi lo, lo2 hi and lo lo: the AO
// values at FP32 level where the density is largest, and D as hi + lo exactly
// (its remainder D - hi - lo, the same in every batch, is taken back in the
// energy to first order once the potential is built).
// Blocks walk the core group list; the others run the two-term kernel.
// The grid's descriptor comes by value (a kernel argument: every pointer in it
// is known to address global memory, and uniform table reads become scalar
// loads; a descriptor read from device memory would leave them flat).
// r: the block's item (after the XCD-aware remap) within the molecule's launch.
template <bool P3>
__device__ __forceinline__ void density_mx_body(const MolDev& m, int r, DensMxSmem& sm) {
  using lds_ptr = __attribute__((address_space(3))) void*;
  const int grp = P3 ? m.core_grps[r] : m.main_grps ? m.main_grps[r] : r;
  const u16* __restrict__ cache = m.cache;
  const size_t sstride = (size_t)m.sstride;
  double* __restrict__ part = m.part;
  const BasisView bv = m.bv;  // descriptor fields in registers, read once
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;
  const int wr = wave & 1, wc = wave >> 1;
  const int b = m.grp_batch[grp];
  const int nt = m.grp_ntiles[grp], j0 = m.grp_tile[grp];
  const ChunkDev ch = m.chunks[m.b_chunk[b]];
  const int it0 = m.bt_off[b], nk = ch.ntl, ld = nk * kTile;  // the batch's slots it0.. are its K steps
  if (tid < kBatch) {
    sm.px[tid] = m.bx[b * kBatch + tid];
    sm.py[tid] = m.by[b * kBatch + tid];
    sm.pz[tid] = m.bz[b * kBatch + tid];
  }
  // The wave's fragments are f = wave + 4 j. A (j = 0, 1): row block f >> 1,
  // hl f & 1. D (j = 2..5, f' = f - 8): column block c = f' >> 1 (tile c >> 1,
  // half c & 1), hl f' & 1; columns past the group's tiles read a present
  // tile's rows (their X columns are never used). A fragment is 16 rows of
  // 64 bytes; DMA lane i fetches row i >> 2, 16-byte chunk (i & 3) ^ sw(row)
  // (four neighbouring lanes read one contiguous 64-byte run: coalesced), and
  // the MFMA lane that needs (row, chunk) reads it back at frag_idx(row, chunk)
  // (the XOR keeps those LDS reads free of bank conflicts). P3 adds the AO
  // operand's third term: A3 row block = wave.
  const int drow = lane >> 2, dch = (lane & 3) ^ ((drow >> 2) & 3);
  const int fidx = 4 * lrow + (lk ^ ((lrow >> 2) & 3));  // this lane's MFMA operand in a fragment
  int offa[2], offb[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int f = wave + 4 * j;
    offa[j] = (16 * (f >> 1) + drow) * kMxRow + (f & 1) * kTile + 8 * dch;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int f = wave + 4 * j, c = f >> 1, q = c >> 1;
    offb[j] = (f & 1) * ld * ld + ((j0 - ch.tile0 + (q < nt ? q : 0)) * kTile + 16 * (c & 1) + drow) * ld + 8 * dch;
  }
  const u16* __restrict__ Ds = m.Ds + 2 * ch.doff;
  const u16* __restrict__ c3 = nullptr;
  if (P3) {
    // this batch's core slots in the side cache: [core slot][c][g][mu]
    c3 = m.cache3 + ((size_t)m.core_off[b] * (m.toff / 2)) +
         (16 * wave + drow) * kTile + 8 * dch;
  }
  __syncthreads();
  auto dma = [&](int k) {
    const u16* a = cache + (size_t)(it0 + k) * sstride;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_global_load_lds(a + offa[j], (lds_ptr)(sm.F + (wave + 4 * j) * kDxFrag), 16, 0, 0);
    const int ti = k * kTile;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_global_load_lds(Ds + offb[j] + ti, (lds_ptr)(sm.F + (kDxA + wave + 4 * j) * kDxFrag), 16, 0, 0);
    if (P3)
      __builtin_amdgcn_global_load_lds(c3 + (size_t)k * (m.toff / 2),
                                       (lds_ptr)(sm.F + (kDxA + kDxB + wave) * kDxFrag), 16, 0, 0);
  };

  f32x4 acc[2][4];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ncb = 2 * (nt - 2 * wc);  // the wave's column blocks that hold group tiles (may be <= 0)
  dma(0);
  for (int k = 0; k < nk; ++k) {
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's fragments of step k are in LDS
    __syncthreads();                     // ... and every other wave's
    u32x4 a[2][2], bq[4][2], a3[2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) a[r][h] = sm.F[((2 * wr + r) * 2 + h) * kDxFrag + fidx];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) bq[c][h] = sm.F[(kDxA + (4 * wc + c) * 2 + h) * kDxFrag + fidx];
    if (P3) {
#pragma unroll
      for (int r = 0; r < 2; ++r) a3[r] = sm.F[(kDxA + kDxB + 2 * wr + r) * kDxFrag + fidx];
    }
    __syncthreads();  // every wave holds its fragments: the buffer is free
    if (k + 1 < nk) dma(k + 1);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c < ncb) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          f32x4 v = acc[r][c];
          if (P3) {  // the small terms first
            v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(a[r][1]), as_bf(bq[c][1]), v, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf(a3[r]), as_bf(bq[c][0]), v, 0, 0, 0);
          }
          acc[r][c] = mfma3(a[r][0], a[r][1], bq[c][0], bq[c][1], v);
        }
      }
  }

  // Epilogue. X[g = 32 wr + 16 r + 4 lk + i][n = 64 wc + 16 c + lrow] -> LDS as X^T.
  __syncthreads();  // every wave is done with the fragments
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      *reinterpret_cast<f32x4*>(&sm.X[64 * wc + 16 * c + lrow][32 * wr + 16 * r + 4 * lk]) = acc[r][c];
  __syncthreads();
  DensEpi<false> epi;
  if (wave < nt) {  // wave q = tile q of the group; lane = point
    epi.load(0, &sm.X[kTile * wave][lane]);
    walk_tile_f32<true>(bv, j0 + wave, sm.px[lane], sm.py[lane], sm.pz[lane], epi);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) sm.red[wave][c][lane] = epi.o[c];
  __syncthreads();
  {
    const int c = tid / kBatch, g = tid % kBatch;
    double v = 0.0;
    for (int q = 0; q < nt; ++q) v += (double)sm.red[q][c][g];
    part[(size_t)grp * 4 * kBatch + c * kBatch + g] = v;
  }
}
// The first ncore blocks take the core groups (their products are longer), the
// others the rest: one launch, since the core batches alone leave the chip half empty.
__global__ __launch_bounds__(256, 4) void k_density_mx(MolDev m, int ncore) {
  __shared__ DensMxSmem sm;
  if ((int)blockIdx.x < ncore) density_mx_body<true>(m, xcd_remap(blockIdx.x, ncore), sm);
  else density_mx_body<false>(m, xcd_remap(blockIdx.x - ncore, gridDim.x - ncore), sm);
}

// Meta-GGA density in one launch: the products Phi D and (d_r Phi) D share one D
// block per K step (48 fragments: A_0..A_3, then D); one walk over the shells
// contracts all four (DensEpi<true>) into rho, grad rho / 2 and tau. Same
// indexing as k_density_mx. tau = sum_r x_r^T D x_r (x_r = d_r phi) is a
// quadratic form, so for a symmetric D its products stop at the group's own
// tiles: K steps before them count twice (the accumulators are doubled when the
// group's first tile is reached), steps after them carry rho alone. A D that
// the symmetry check (k_split_gather) flagged takes every step once.
// (H2O)48 / def2-SVP / SG-2: 2.6 ms, against 5.0 with every step and a walk per
// component.
struct DensMxMggaSmem {
  union {
    u32x4 F[(4 * kDxA + kDxB) * kDxFrag];  // one K step's fragments: A_0..A_3, D
    float X[kGroup * kTile][kXPitch];
  };
  float red[kGroup][7][kBatch];
  double px[kBatch], py[kBatch], pz[kBatch];
};

__global__ __launch_bounds__(256, 2) void k_density_mx_mgga(MolDev m) {
  using lds_ptr = __attribute__((address_space(3))) void*;
  __shared__ DensMxMggaSmem sm;
  const int grp = xcd_remap(blockIdx.x, gridDim.x);
  const u16* __restrict__ cache = m.cache;  // components 0 (phi), 1..3 (d_r phi)
  const size_t sstride = (size_t)m.sstride;
  const BasisView bv = m.bv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;
  const int wr = wave & 1, wc = wave >> 1;
  const int b = m.grp_batch[grp];
  const int nt = m.grp_ntiles[grp], j0 = m.grp_tile[grp];
  const ChunkDev ch = m.chunks[m.b_chunk[b]];
  const int it0 = m.bt_off[b], nk = ch.ntl, ld = nk * kTile;
  if (tid < kBatch) {
    sm.px[tid] = m.bx[b * kBatch + tid];
    sm.py[tid] = m.by[b * kBatch + tid];
    sm.pz[tid] = m.bz[b * kBatch + tid];
  }
  const int drow = lane >> 2, dch = (lane & 3) ^ ((drow >> 2) & 3);
  const int fidx = 4 * lrow + (lk ^ ((lrow >> 2) & 3));
  int offa[2], offb[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int f = wave + 4 * j;
    offa[j] = (16 * (f >> 1) + drow) * kMxRow + (f & 1) * kTile + 8 * dch;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int f = wave + 4 * j, c = f >> 1, q = c >> 1;
    offb[j] = (f & 1) * ld * ld + ((j0 - ch.tile0 + (q < nt ? q : 0)) * kTile + 16 * (c & 1) + drow) * ld + 8 * dch;
  }
  const u16* __restrict__ Ds = m.Ds + 2 * ch.doff;
  __syncthreads();
  const bool sym = *m.asym != m.gen;
  const int t0 = j0 - ch.tile0;                // the group's first tile
  const int ktau = sym ? t0 + nt : nk;         // steps that carry tau
  auto dma = [&](int k) {
    const u16* a = cache + (size_t)(it0 + k) * sstride;
    const int nd = k < ktau ? 4 : 1;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nd)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        __builtin_amdgcn_global_load_lds(a + (size_t)r * kMxT + offa[j],
                                         (lds_ptr)(sm.F + (r * kDxA + wave + 4 * j) * kDxFrag), 16, 0, 0);
    const int ti = k * kTile;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_global_load_lds(Ds + offb[j] + ti, (lds_ptr)(sm.F + (4 * kDxA + wave + 4 * j) * kDxFrag), 16,
                                       0, 0);
  };

  f32x4 acc[4][2][4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[d][r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ncb = 2 * (nt - 2 * wc);
  dma(0);
  for (int k = 0; k < nk; ++k) {
    const bool tau = k < ktau;
    if (sym && k == t0) {
#pragma unroll
      for (int d = 1; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[d][r][c] *= 2.f;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's fragments of step k are in LDS
    __syncthreads();                     // ... and every other wave's
    u32x4 a[4][2][2], bq[4][2];
#pragma unroll
    for (int d = 0; d < 4; ++d)
      if (d == 0 || tau)
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) a[d][r][h] = sm.F[(d * kDxA + (2 * wr + r) * 2 + h) * kDxFrag + fidx];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) bq[c][h] = sm.F[(4 * kDxA + (4 * wc + c) * 2 + h) * kDxFrag + fidx];
    __syncthreads();  // every wave holds its fragments: the buffer is free
    if (k + 1 < nk) dma(k + 1);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c < ncb) {
#pragma unroll
        for (int d = 0; d < 4; ++d)
          if (d == 0 || tau)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            acc[d][r][c] = mfma3(a[d][r][0], a[d][r][1], bq[c][0], bq[c][1], acc[d][r][c]);
      }
  }
  DensEpi<true> epi;
#pragma unroll
  for (int d = 0; d < 4; ++d) {  // X_d -> LDS as X_d^T -> registers of the lane that holds the point
    __syncthreads();  // the previous user of the X area is done
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<f32x4*>(&sm.X[64 * wc + 16 * c + lrow][32 * wr + 16 * r + 4 * lk]) = acc[d][r][c];
    __syncthreads();
    epi.load(d, &sm.X[kTile * wave][lane]);
  }
  if (wave < nt) walk_tile_f32<true>(bv, j0 + wave, sm.px[lane], sm.py[lane], sm.pz[lane], epi);
#pragma unroll
  for (int c = 0; c < 7; ++c) sm.red[wave][c][lane] = epi.o[c];
  __syncthreads();
  for (int e = tid; e < 7 * kBatch; e += 256) {
    const int c = e / kBatch, g = e % kBatch;
    double v = 0.0;
    for (int q = 0; q < nt; ++q) v += (double)sm.red[q][c][g];
    if (c < 4)
      m.part[(size_t)grp * 4 * kBatch + c * kBatch + g] = v;
    else  // part_tau: [group][3][64]
      m.part_tau[(size_t)grp * 3 * kBatch + (c - 4) * kBatch + g] = v;
  }
}

void launch_density_mx(hipStream_t s, int with_tau, int nitems, int ncore_groups, const MolDev& one) {
  if (with_tau && nitems > 0) {
    hipLaunchKernelGGL(k_density_mx_mgga, dim3(nitems), dim3(256), 0, s, one);
    nitems = 0;  // the core groups come after it
  }
  if (nitems + ncore_groups > 0)
    hipLaunchKernelGGL(k_density_mx, dim3(nitems + ncore_groups), dim3(256), 0, s, one, ncore_groups);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// B^T in split form, one wave per slot (lane = point), from phi and grad phi
// recomputed in FP32:
//   Bt[slot][0][hl][nu][g] = split(a phi + c . grad phi),
//   meta-GGA (NC = 4) adds Bt[slot][r][hl][nu][g] = split(t d_r phi), t = w v_tau / 4.
// Neighbouring lanes exchange halves, so that an AO's two rows of 128 bytes in
// the slot's [c][hl][nu][g] block go out in one store of the wave; columns past
// the tile's last AO are written as zeros. No LDS stage and no barrier, so
// occupancy is set by registers alone. Bound by the walk's instructions and the
// waits for its records ((H2O)128 / def2-SVP / SG-2: 1.8 ms for 4 GB; the stores
// alone take 0.8).
template <int NC>
struct MakeB {
  u16* sv;       // where this lane's pairs go in the [c][hl][nu][g] block
  unsigned sel;  // byte selection of its pairs
  float ca, cx, cy, cz, ct, R, Rx, Ry, Rz, s1;
  __device__ void begin(float a, float ax, float ay, float az) {
    R = a; Rx = ax; Ry = ay; Rz = az;
    s1 = ca * a + cx * ax + cy * ay + cz * az;  // (a + c . grad) R
  }
  __device__ void put(int c, int col, float v) {
    u16 hi, lo;
    split_bf(v, hi, lo);
    const int own = hi | (int)lo << 16, other = __builtin_amdgcn_mov_dpp(own, 0xb1, 0xf, 0xf, true);  // lane ^ 1
    *reinterpret_cast<unsigned*>(sv + c * kMxT + col * kBatch) = __builtin_amdgcn_perm(other, own, sel);
  }
  __device__ void comp(int col, float q, float qx, float qy, float qz) {
    put(0, col, q * s1 + R * (cx * qx + cy * qy + cz * qz));  // a phi + c . grad phi
    if (NC == 4) {
      put(1, col, ct * (Rx * q + R * qx));
      put(2, col, ct * (Ry * q + R * qy));
      put(3, col, ct * (Rz * q + R * qz));
    }
  }
  __device__ void end() {}
};

template <int NC>
__device__ __forceinline__ void make_b_slot(const MolDev& m, int item, int g) {
  if (item >= m.nslots) return;
  const BasisView bv = m.bv;  // descriptor fields in registers, read once
  int slot = item, b = m.slot_batch[item], t = m.slot_tile[item];
  if (NC == 1) {  // a chunk's items tile by tile, so that the waves that run together read the same records
    const ChunkDev ch = m.chunks[m.b_chunk[b]];
    const int local = (b - ch.b0) * ch.ntl + t - ch.tile0, q = local / ch.nb;
    b = ch.b0 + local - q * ch.nb;
    t = ch.tile0 + q;
    slot = item - local + (b - ch.b0) * ch.ntl + q;
  }
  const size_t p = (size_t)b * kBatch + g;
  const double* __restrict__ coef = m.coef + kCoef * p;
  MakeB<NC> op;
  // even lanes store the hi parts of points g, g + 1, odd lanes the lo parts of g - 1, g
  op.sv = m.bt + (size_t)slot * NC * kMxT + (g & 1) * (kTile * kBatch) + (g & ~1);
  op.sel = g & 1 ? 0x03020706u : 0x05040100u;
  op.ca = (float)coef[0];
  op.cx = (float)coef[1];
  op.cy = (float)coef[2];
  op.cz = (float)coef[3];
  op.ct = (float)coef[4];
  walk_tile_f32<true>(bv, t, m.bx[p], m.by[p], m.bz[p], op);
  // zeros past the tile's last AO (its segments are in column order)
  const int s1 = bv.tile_seg_off[t + 1];
  int nao = 0;
  if (s1 > bv.tile_seg_off[t]) {
    const int4 sg = bv.seg[s1 - 1];  // (shell, first component, count, local offset)
    nao = sg.w + sg.z;
  }
  for (int col = nao; col < kTile; ++col)
#pragma unroll
    for (int c = 0; c < NC; ++c) *reinterpret_cast<unsigned*>(op.sv + c * kMxT + col * kBatch) = 0u;
}
template <int NC>
__global__ __launch_bounds__(NC == 4 ? 64 : 256) void k_make_b_mx(MolDev m) {
  constexpr int W = NC == 4 ? 1 : 4;  // waves per block
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  make_b_slot<NC>(m, blockIdx.x * W + wave, threadIdx.x & 63);
}

void launch_make_b_mx(hipStream_t s, int ncomp, const MolDev& one) {
  const int waves = one.nslots;
  if (waves == 0) return;
  if (ncomp == 4)
    hipLaunchKernelGGL((k_make_b_mx<4>), dim3(waves), dim3(64), 0, s, one);
  else
    hipLaunchKernelGGL((k_make_b_mx<1>), dim3((waves + 3) / 4), dim3(256), 0, s, one);
  CHX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Vxc: one block of one run's V, U_IJ = sum_g Phi_I^T B_J + B_I^T Phi_J over
// the run's batches, for groups I <= J of at most MT of the chunk's tiles (the
// groups of a list are equal to within a tile, so no block is mostly padding).
// Only the upper blocks are formed. For I < J the two products follow each other
// (second pass: the operands swap roles); for I = J there is one product M, and M^T
// comes from it through LDS at the end. Both go to U as they are, in FP32 like the
// accumulators, and k_assemble adds them in FP64. The tau part (NC = 4) is symmetric,
// M_tau = sum_r (d_r Phi)^T (t d_r Phi): its steps run first and once, doubled for
// I < J.
// A K step is 32 points of one component: the row group's and the column
// group's operands, hi and lo, fragments of 1 KB (16 rows of 64 bytes) that the
// waves' DMA loads bring straight into LDS, coalesced and swizzled as in the
// density kernel. Two LDS buffers and one barrier per step: after it, step k's
// fragments are in LDS and every wave has read step k - 1's buffer, so the DMA
// of step k + 1 goes there before step k's fragment reads and products. 4 waves
// in a 2 x 2 grid, each owning half of the row and of the column blocks (up to
// MT x MT fragments of 16 x 16; MT = 5 is the largest whose two buffers leave
// room for two blocks per CU).
// Either product is stored once per run, row-major, the row panel of group I from
// column I0 on, the second one uplane elements after the first; of a block on the
// diagonal the upper half. (H2O)16 / def2-SVP / SG-2 186 us, (H2O)128 3.55 ms; one
// accumulator for both and one store, which adds them in FP32, took 175 us and 3.51
// ms: fewer bytes. A second set of accumulators, their FP64 sum stored at the end, is
// no faster than two stores (188 us with whole diagonal blocks, 190 so stored; with
// MT = 5 it does not fit the registers).
template <int MT>
struct VxcMxSmem {
  u32x4 F[2][8 * MT * kDxFrag];  // step k in buffer k & 1: row group's fragments, then the column group's
};

template <int NC, int MT>
__device__ __forceinline__ void vxc_mx_body(const MolDev& m, int item) {
  using lds_ptr = __attribute__((address_space(3))) void*;
  constexpr int PT = 32 * MT + 4;  // pitch of the transposed strip
  __shared__ VxcMxSmem<MT> sm;
  const MxItem wk = m.cwork[item];
  const int nI = wk.nI, RB = 2 * nI, CB = 2 * wk.nJ, nf = 2 * (RB + CB);
  const bool diag = wk.I0 == wk.J0;
  const u16* __restrict__ cache = m.cache + m.toff;
  const u16* __restrict__ bt = m.bt;
  const size_t sstride = (size_t)m.sstride;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lk = lane >> 4;
  const int wr = wave & 1, wc = wave >> 1;
  const int r0 = nI * wr, nc = wk.nJ, c0 = nc * wc;  // the wave's row blocks r0 .. r0 + nI - 1, columns c0 ..
  // The wave's fragments are f = wave + 4 j: hl f & 1, rows 16 ((f >> 1) & 1)..+15
  // of tile f >> 2 of the row group (f < 2 RB) or of the column group.
  const int drow = lane >> 2, dch = (lane & 3) ^ ((drow >> 2) & 3);
  const int fidx = 4 * lrow + (lk ^ ((lrow >> 2) & 3));
  const int off = (wave & 1) * (kTile * kBatch) + drow * kBatch + 8 * dch;
  const int nbat = wk.nbat;
  const int ntau = NC == 4 ? 6 * nbat : 0;  // tau steps, first
  const int kswap = ntau + 2 * nbat;        // first step of the second product
  const int nstage = kswap + (diag ? 0 : 2 * nbat);
  auto dma = [&](int k, int buf) {  // issue step k's loads: (batch, half of its points, component, product)
    const bool swap = k >= kswap;
    int it, h, c;
    if (k < ntau) {
      it = k / 6; h = (k / 3) % 2; c = 1 + k % 3;
    } else {
      const int q = k - (swap ? kswap : ntau);
      it = q >> 1; h = q & 1; c = 0;
    }
    const int s0 = wk.slot0 + it * wk.ntl;
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j) {
      const int f = wave + 4 * j;
      if (f < nf) {
        const bool row = f < 2 * RB;
        const int fr = row ? f : f - 2 * RB;
        const size_t slot = (size_t)(s0 + (row ? wk.I0 : wk.J0) + (fr >> 2));
        const u16* p = (row != swap ? cache + slot * sstride : bt + slot * (NC * kMxT)) + c * kMxT + h * 32 +
                       ((fr >> 1) & 1) * (16 * kBatch);
        __builtin_amdgcn_global_load_lds(p + off, (lds_ptr)(sm.F[buf] + f * kDxFrag), 16, 0, 0);
      }
    }
  };
  f32x4 acc[MT][MT];
  float* __restrict__ U = m.U + wk.u;
  const int ld = wk.ldu;
  dma(0, 0);
  for (int pass = 0, k = 0; k < nstage; ++pass) {  // the products of the run, one after the other
    const int kend = pass == 0 ? kswap : nstage;
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
      for (int c = 0; c < MT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (; k < kend; ++k) {
      if (NC == 4 && k == ntau && !diag) {  // 2 M_tau
#pragma unroll
        for (int r = 0; r < MT; ++r)
#pragma unroll
          for (int c = 0; c < MT; ++c) acc[r][c] *= 2.f;
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's fragments of step k are in LDS
      __syncthreads();                     // ... and every other wave's, and step k - 1's buffer is read
      if (k + 1 < nstage) dma(k + 1, (k + 1) & 1);
      const u32x4* F = sm.F[k & 1];
      u32x4 a[MT][2];
#pragma unroll
      for (int r = 0; r < MT; ++r)
        if (r < nI) {
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) a[r][hh] = F[((r0 + r) * 2 + hh) * kDxFrag + fidx];
        }
#pragma unroll
      for (int c = 0; c < MT; ++c)
        if (c < nc) {
          const u32x4* Fc = F + (2 * RB + (c0 + c) * 2) * kDxFrag + fidx;
          const u32x4 bh = Fc[0], bl = Fc[kDxFrag];
#pragma unroll
          for (int r = 0; r < MT; ++r)
            if (r < nI) acc[r][c] = mfma3(a[r][0], a[r][1], bh, bl, acc[r][c]);
        }
    }
    float* __restrict__ out = U + pass * m.uplane + (size_t)(16 * r0 + 4 * lk) * ld + 16 * c0 + lrow;
#pragma unroll
    for (int r = 0; r < MT; ++r)
      if (r < nI) {
#pragma unroll
        for (int c = 0; c < MT; ++c)
          if (c < nc && (!diag || c0 + c >= r0 + r)) {  // (below the diagonal nothing is read)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[(size_t)(16 * r + i) * ld + 16 * c] = acc[r][c][i];
          }
      }
  }
  if (!diag) return;
  // M^T, 64 rows at a time: the strip's 64 columns of M go to LDS transposed
  float* T = reinterpret_cast<float*>(&sm.F[0][0]);
  static_assert(sizeof(float) * 64 * PT <= sizeof(sm), "a strip fits the fragment buffers");
  const int n = 16 * CB;
  for (int s = 0; s < CB; s += 4) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < MT; ++c)
      if (c < nc && c0 + c >= s && c0 + c < s + 4) {
#pragma unroll
        for (int r = 0; r < MT; ++r)
          if (r < nI)
            *reinterpret_cast<f32x4*>(T + (16 * (c0 + c - s) + lrow) * PT + 16 * (r0 + r) + 4 * lk) = acc[r][c];
      }
    __syncthreads();
    float* __restrict__ out = U + m.uplane + (size_t)(16 * s) * ld;
    const int rows = min(64, n - 16 * s);
    for (int e = tid; e < rows * (n / 4); e += 256) {
      const int row = e / (n / 4), col = e % (n / 4) * 4;
      if (col + 3 >= 16 * s + row)
        *reinterpret_cast<f32x4*>(out + (size_t)row * ld + col) = *reinterpret_cast<const f32x4*>(T + row * PT + col);
    }
  }
}
template <int NC, int MT>
__global__ __launch_bounds__(256, 2) void k_vxc_mx(MolDev m) {
  vxc_mx_body<NC, MT>(m, xcd_remap(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------------------
// Persistent stage kernels over many molecules (packs). A table holds one
// descriptor per molecule whose pointer fields are byte offsets from a base
// kernel argument; rebase() adds the base, so every table address the kernels
// form derives from a kernel argument and stays a global-memory access (a
// descriptor read from device memory with its own pointers would leave them
// flat). starts[k] is the first item of molecule k in the stage's flat item
// list (starts[nmol] = total). A fixed grid of blocks walks the list: virtual
// block v = blockIdx.x + j gridDim.x takes item xcd_remap(v, total) (gridDim.x
// a multiple of 8, so each XCD keeps a contiguous range), finds its molecule by
// bisection, and runs the single-molecule body on it.
template <class T>
__device__ __forceinline__ T* rb(const char* base, T* off) {
  return reinterpret_cast<T*>(const_cast<char*>(base) + reinterpret_cast<long>(off));
}
__device__ __forceinline__ MolDev rebase(const char* base, const MolDev& o) {
  MolDev m = o;
  m.grp_batch = rb(base, o.grp_batch); m.grp_tile = rb(base, o.grp_tile); m.grp_ntiles = rb(base, o.grp_ntiles);
  m.bt_off = rb(base, o.bt_off);
  m.b_chunk = rb(base, o.b_chunk); m.chunks = rb(base, o.chunks); m.ao_of = rb(base, o.ao_of);
  m.bx = rb(base, o.bx); m.by = rb(base, o.by); m.bz = rb(base, o.bz);
  m.bv.sh_xyz = rb(base, o.bv.sh_xyz); m.bv.sh_type = rb(base, o.bv.sh_type);
  m.bv.sh_nprim = rb(base, o.bv.sh_nprim); m.bv.sh_poff = rb(base, o.bv.sh_poff);
  m.bv.p_exp = rb(base, o.bv.p_exp); m.bv.p_coef = rb(base, o.bv.p_coef);
  m.bv.tile_seg_off = rb(base, o.bv.tile_seg_off); m.bv.seg = rb(base, o.bv.seg);
  m.bv.segrec = rb(base, o.bv.segrec); m.bv.sh_atom = rb(base, o.bv.sh_atom);
  m.cache = rb(base, o.cache); m.Ds = rb(base, o.Ds);
  m.part = rb(base, o.part); m.part_tau = rb(base, o.part_tau);
  m.slot_batch = rb(base, o.slot_batch); m.slot_tile = rb(base, o.slot_tile);
  m.coef = rb(base, o.coef); m.bt = rb(base, o.bt);
  m.cwork = rb(base, o.cwork); m.U = rb(base, o.U);
  m.cache3 = rb(base, o.cache3);
  m.asym = rb(base, o.asym);
  m.core_off = rb(base, o.core_off); m.core_grps = rb(base, o.core_grps); m.main_grps = rb(base, o.main_grps);
  return m;
}
__device__ __forceinline__ int item_owner(const int* __restrict__ starts, int nmol, int item) {
  int lo = 0, hi = nmol;  // the last molecule whose first item is <= item
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (starts[mid] <= item) lo = mid; else hi = mid;
  }
  return lo;
}
// A block's items come in increasing order (xcd_remap keeps each block's XCD),
// so after the first bisection its molecule cursor only moves forward.
__device__ __forceinline__ int item_owner_from(const int* __restrict__ starts, int nmol, int item, int k) {
  if (k < 0) return item_owner(starts, nmol, item);
  while (k + 1 < nmol && starts[k + 1] <= item) ++k;
  return k;
}

template <bool P3>
__global__ __launch_bounds__(256, 4) void k_density_mx_multi(const char* base, const MolDev* __restrict__ tab,
                                                                      const int* __restrict__ starts, int nmol,
                                                                      int total) {
  __shared__ DensMxSmem sm;
  int k = -1;
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int item = xcd_remap(v, total);
    k = item_owner_from(starts, nmol, item, k);
    density_mx_body<P3>(rebase(base, tab[k]), item - starts[k], sm);
    __syncthreads();  // the next item reuses the block's LDS
  }
}

template <int NC>
__global__ __launch_bounds__(256) void k_make_b_mx_multi(const char* base, const MolDev* __restrict__ tab,
                                                         const int* __restrict__ starts, int nmol, int total) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int k = -1;
  for (int v = blockIdx.x * 4 + wave; v < total; v += gridDim.x * 4) {  // one wave per slot, no LDS
    k = item_owner_from(starts, nmol, v, k);
    make_b_slot<NC>(rebase(base, tab[k]), v - starts[k], threadIdx.x & 63);
  }
}

template <int NC, int MT>
__global__ __launch_bounds__(256, 2) void k_vxc_mx_multi(const char* base, const MolDev* __restrict__ tab,
                                                         const int* __restrict__ starts, int nmol, int total) {
  int k = -1;
  for (int v = blockIdx.x; v < total; v += gridDim.x) {
    const int item = xcd_remap(v, total);
    k = item_owner_from(starts, nmol, item, k);
    vxc_mx_body<NC, MT>(rebase(base, tab[k]), item - starts[k]);
    __syncthreads();
  }
}

// Blocks of a persistent launch: the kernel's resident blocks per CU times the
// CUs, a multiple of 8, at most the items (rounded up to 8).
template <class K>
static int persistent_blocks(K kernel, int threads, int total) {
  static int ncu = 0;
  if (!ncu) {
    int dev = 0;
    CHX_HIP(hipGetDevice(&dev));
    CHX_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  }
  int per_cu = 0;
  CHX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0));
  const long full = (long)std::max(1, per_cu) * ncu;
  const long want = std::min<long>(full, ((long)total + 7) / 8 * 8);
  return (int)std::max<long>(8, want / 8 * 8);
}

void launch_stage_multi(hipStream_t s, int stage, int ncomp, const char* base, const MolDev* tab, const int* starts,
                        int nmol, int total) {
  if (total <= 0) return;
  switch (stage) {
    case kStageDensity: {
      auto k = k_density_mx_multi<false>;
      hipLaunchKernelGGL(k, dim3(persistent_blocks(k, 256, total)), dim3(256), 0, s, base, tab, starts, nmol, total);
      break;
    }
    case kStageCore: {
      auto k = k_density_mx_multi<true>;
      hipLaunchKernelGGL(k, dim3(persistent_blocks(k, 256, total)), dim3(256), 0, s, base, tab, starts, nmol, total);
      break;
    }
    case kStageMakeB: {
      if (ncomp != 1) throw Error(CHX_ERR_UNSUPPORTED, "persistent packs are built for LDA and GGA");
      auto k = k_make_b_mx_multi<1>;
      const int blocks = persistent_blocks(k, 256, (total + 3) / 4);
      hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, s, base, tab, starts, nmol, total);
      break;
    }
    case kStageVxc: {
      if (ncomp != 1) throw Error(CHX_ERR_UNSUPPORTED, "persistent packs are built for LDA and GGA");
      auto k = k_vxc_mx_multi<1, 4>;
      hipLaunchKernelGGL(k, dim3(persistent_blocks(k, 256, total)), dim3(256), 0, s, base, tab, starts, nmol, total);
      break;
    }
    case kStageVxcWide: {
      if (ncomp != 1) throw Error(CHX_ERR_UNSUPPORTED, "persistent packs are built for LDA and GGA");
      auto k = k_vxc_mx_multi<1, 5>;
      hipLaunchKernelGGL(k, dim3(persistent_blocks(k, 256, total)), dim3(256), 0, s, base, tab, starts, nmol, total);
      break;
    }
    default:
      throw Error(CHX_ERR_ARG, "unknown pack stage");
  }
  CHX_HIP(hipGetLastError());
}

void launch_vxc_mx(hipStream_t s, int ncomp, int wide, int nitems, const MolDev& one) {
  if (nitems == 0) return;
  if (wide && ncomp == 4)
    hipLaunchKernelGGL((k_vxc_mx<4, 5>), dim3(nitems), dim3(256), 0, s, one);
  else if (wide)
    hipLaunchKernelGGL((k_vxc_mx<1, 5>), dim3(nitems), dim3(256), 0, s, one);
  else if (ncomp == 4)
    hipLaunchKernelGGL((k_vxc_mx<4, 4>), dim3(nitems), dim3(256), 0, s, one);
  else
    hipLaunchKernelGGL((k_vxc_mx<1, 4>), dim3(nitems), dim3(256), 0, s, one);
  CHX_HIP(hipGetLastError());
}

}  // namespace chx
