// pf_misc.hip — deterministic FP64 reductions, seeded-setup kernels and form conversion.
// All floating-point expressions keep the reference's evaluation order; the library is built
// with -ffp-contract=off so no multiply-add is fused, and HIP's division and square root are
// IEEE correctly rounded on gfx950.
#include "pf_kernels.h"

namespace pfamd {
// ----------------------------------------------------------------------------------------------
// Deterministic FP64 reductions.  Stage 1: each block reduces a contiguous cell range with a
// fixed tree; stage 2: one block reduces the partials in index order.
template <class F, int K, int P>
__global__ __launch_bounds__(256) void reduce_stage1(const uint16_t *__restrict__ id,
                                                     const typename F::T *__restrict__ phi,
                                                     const typename F::T *__restrict__ pfrac,
                                                     const typename F::C *__restrict__ c0,
                                                     const typename F::C *__restrict__ c1, int ns,
                                                     long ncell, long per_block,
                                                     RedPartial *__restrict__ out) {
  __shared__ RedPartial sh[256];
  RedPartial r;
  r.mass[0] = r.mass[1] = 0.0;
  r.pf[0] = r.pf[1] = r.pf[2] = 0.0;
  r.cmax[0] = r.cmax[1] = -1e300;
  r.cmin[0] = r.cmin[1] = 1e300;
  r.serr = 0.0;
  r.nif = r.nnf = 0;
  const long beg = long(blockIdx.x) * per_block;
  const long end = min(beg + per_block, ncell);
  for (long c = beg + threadIdx.x; c < end; c += 256) {
    bool bad = false;
    for (int s = 0; s < ns; ++s) {
      const double v = conc_effective<F>(s == 0 ? c0 : c1, c, ncell);
      r.mass[s] += v;
      r.cmax[s] = fmax(r.cmax[s], v);
      r.cmin[s] = fmin(r.cmin[s], v);
      bad = bad || !isfinite(v);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const double v = double(pfrac[c * P + p]);
      r.pf[p] += v;
      bad = bad || !isfinite(v);
    }
    double sp = 0.0;
#pragma unroll
    for (int s = 0; s < K; ++s) sp += double(phi[c * K + s]);
    bad = bad || !isfinite(sp);
    r.serr = fmax(r.serr, fabs(sp - 1.0));
    uint32_t g[K];
    load_ids<K>(id, c, g);
    r.nif += (K > 1 && g[1] != 0) ? 1 : 0;
    r.nnf += bad ? 1 : 0;
  }
  sh[threadIdx.x] = r;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      RedPartial &a = sh[threadIdx.x];
      const RedPartial &o = sh[threadIdx.x + w];
      for (int s = 0; s < 2; ++s) {
        a.mass[s] += o.mass[s];
        a.cmax[s] = fmax(a.cmax[s], o.cmax[s]);
        a.cmin[s] = fmin(a.cmin[s], o.cmin[s]);
      }
      for (int p = 0; p < 3; ++p) a.pf[p] += o.pf[p];
      a.serr = fmax(a.serr, o.serr);
      a.nif += o.nif;
      a.nnf += o.nnf;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = sh[0];
}

__global__ __launch_bounds__(256) void reduce_stage2(RedPartial *__restrict__ part, int nparts) {
  __shared__ RedPartial sh[256];
  RedPartial r;
  r.mass[0] = r.mass[1] = 0.0;
  r.pf[0] = r.pf[1] = r.pf[2] = 0.0;
  r.cmax[0] = r.cmax[1] = -1e300;
  r.cmin[0] = r.cmin[1] = 1e300;
  r.serr = 0.0;
  r.nif = r.nnf = 0;
  // thread t reduces partials t*chunk .. (t+1)*chunk-1 in order
  const int chunk = (nparts + 255) / 256;
  for (int i = threadIdx.x * chunk; i < min(nparts, (threadIdx.x + 1) * chunk); ++i) {
    const RedPartial &o = part[i];
    for (int s = 0; s < 2; ++s) {
      r.mass[s] += o.mass[s];
      r.cmax[s] = fmax(r.cmax[s], o.cmax[s]);
      r.cmin[s] = fmin(r.cmin[s], o.cmin[s]);
    }
    for (int p = 0; p < 3; ++p) r.pf[p] += o.pf[p];
    r.serr = fmax(r.serr, o.serr);
    r.nif += o.nif;
    r.nnf += o.nnf;
  }
  sh[threadIdx.x] = r;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      RedPartial &a = sh[threadIdx.x];
      const RedPartial &o = sh[threadIdx.x + w];
      for (int s = 0; s < 2; ++s) {
        a.mass[s] += o.mass[s];
        a.cmax[s] = fmax(a.cmax[s], o.cmax[s]);
        a.cmin[s] = fmin(a.cmin[s], o.cmin[s]);
      }
      for (int p = 0; p < 3; ++p) a.pf[p] += o.pf[p];
      a.serr = fmax(a.serr, o.serr);
      a.nif += o.nif;
      a.nnf += o.nnf;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) part[0] = sh[0];
}

// ----------------------------------------------------------------------------------------------
// Seeded setup kernels (FP64 domains).

// Tessellation (MicrostructureConstruction.cpp:68-109): nearest seed under the per-axis periodic
// distance with the reduction stretch; strict '>' keeps the lowest seed index on ties.  Writes
// slot 0 = grain code (phase 2), phi = 1, value_phase = (0,1[,0]).
//
// A workgroup owns blocks of 8 x 8 x 4 cells (16 x 16 of a plane) and first drops the seeds that cannot be nearest to any
// of them: along an axis the periodic distance changes by at most the offset, so over a block of
// half-width w around its centre it lies within w of the centre's, and a seed whose smallest possible
// distance exceeds another seed's largest possible one (with a margin for rounding) is out.  A block
// keeps a few seeds of hundreds; only theirs are evaluated per cell, in seed order.
// 256^3, 128 seeds: 2.67 -> 0.22 ms, 940 MB written at 4.2 TB/s.  512^3, 512 seeds: 74.7 -> 2.4 ms.
template <int K, int P>
__global__ __launch_bounds__(256) void voronoi_kernel(const double *__restrict__ seeds, int G,
                                                      double reduction, int nx, int ny, int nz,
                                                      long ncell, uint16_t *__restrict__ id,
                                                      double *__restrict__ phi,
                                                      double *__restrict__ pfrac) {
  __shared__ double sx[256], sy[256], sz[256];
  __shared__ int sq[256];
  __shared__ double best[4];
  __shared__ int kept[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int e = nz == 1 ? 4 : 3, w = 1 << e, wz = nz == 1 ? 1 : 4;  // block w x w x wz
  const long bx = (nx + w - 1) / w, by = (ny + w - 1) / w, bz = (nz + wz - 1) / wz;
  for (long blk = blockIdx.x; blk < bx * by * bz; blk += gridDim.x) {
    const int tx = int(blk % bx), ty = int((blk / bx) % by), tz = int(blk / (bx * by));
    const int x = tx * w + (t & (w - 1)), y = ty * w + ((t >> e) & (w - 1));
    const int z = tz * wz + (t >> (2 * e));
    const bool valid = x < nx && y < ny && z < nz;
    const int i = x + 1, j = y + 1, k = z + 1;  // 1-based cells, as the seeds
    auto axis = [](double s, double c, int n) {
      const double a = fabs(s - c);
      return a < 0.5 * n ? a : n - a;
    };
    // bounds of the squared distance of a seed over the block (1-based cells w tx + 1 .. w tx + w, ...)
    const double rw = 0.5 * (w - 1), rz = 0.5 * (wz - 1);
    const double mx = w * double(tx) + 1. + rw, my = w * double(ty) + 1. + rw;
    const double mz = wz * double(tz) + 1. + rz;
    auto bounds = [&](double px, double py, double pz, double &lo, double &hi) {
      const double dx = fabs(axis(px, mx, nx)), dy = fabs(axis(py, my, ny)), dz = fabs(axis(pz, mz, nz));
      const double ix = 1. / (1. - reduction), iy = 1. - reduction;
      const double lx = fmax(dx - rw, 0.) * ix, ly = fmax(dy - rw, 0.) * iy, lz = fmax(dz - rz, 0.);
      const double hx = (dx + rw) * ix, hy = (dy + rw) * iy, hz = dz + rz;
      lo = lx * lx + ly * ly + lz * lz;
      hi = hx * hx + hy * hy + hz * hz;
    };
    double least = 1e300;
    for (int q = t; q < G; q += 256) {
      double lo, hi;
      bounds(seeds[3 * q], seeds[3 * q + 1], seeds[3 * q + 2], lo, hi);
      least = fmin(least, hi);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) least = fmin(least, __shfl_xor(least, d));
    if (lane == 0) best[wave] = least;
    __syncthreads();
    least = fmin(fmin(best[0], best[1]), fmin(best[2], best[3])) * (1. + 1e-9);
    const double a0 = nx / (1. - reduction), a1 = ny / (1. - reduction), a2 = nz / (1. - reduction);
    double temp1 = a0 * a0 + a1 * a1 + a2 * a2;
    int index = 0;
    for (int base = 0; base < G; base += 256) {
      const int q = base + t;
      double px = 0., py = 0., pz = 0.;
      bool keep = false;
      if (q < G) {
        px = seeds[3 * q];
        py = seeds[3 * q + 1];
        pz = seeds[3 * q + 2];
        double lo, hi;
        bounds(px, py, pz, lo, hi);
        keep = !(lo > least);
      }
      const unsigned long long m = __ballot(keep);
      if (lane == 0) kept[wave] = __popcll(m);
      __syncthreads();  // (also: the previous chunk's seeds have been read)
      int at = __popcll(m & ((1ull << lane) - 1ull));
      for (int v = 0; v < wave; ++v) at += kept[v];
      const int count = kept[0] + kept[1] + kept[2] + kept[3];
      if (keep) {
        sx[at] = px;
        sy[at] = py;
        sz[at] = pz;
        sq[at] = q + 1;
      }
      __syncthreads();
      for (int s = 0; s < count; ++s) {
        const double ax = fabs(sx[s] - i), ay = fabs(sy[s] - j), az = fabs(sz[s] - k);
        const double dx = ax < 0.5 * nx ? ax : nx - ax;
        const double dy = ay < 0.5 * ny ? ay : ny - ay;
        const double dz = az < 0.5 * nz ? az : nz - az;
        const double ex = dx / (1. - reduction), ey = dy * (1. - reduction);
        const double temp2 = ex * ex + ey * ey + dz * dz;
        if (temp1 > temp2) {
          temp1 = temp2;
          index = sq[s];
        }
      }
    }
    __syncthreads();  // before the next block's seeds
    if (!valid) continue;
    const long cell = x + long(nx) * (y + long(ny) * z);
    uint32_t g[K];
#pragma unroll
    for (int s = 0; s < K; ++s) g[s] = 0;
    g[0] = (2u << 14) | uint32_t(index);
    store_ids<K>(id, cell, g);
#pragma unroll
    for (int s = 0; s < K; ++s) phi[cell * K + s] = s == 0 ? 1.0 : 0.0;
#pragma unroll
    for (int p = 0; p < P; ++p) pfrac[cell * P + p] = p == 1 ? 1.0 : 0.0;
  }
}

// total_conc = dot(value_phase, per-phase initial concentration) (MicrostructureConstruction.cpp:58)
template <int P>
__global__ __launch_bounds__(256) void construct_conc_kernel(const double *__restrict__ pfrac,
                                                             double c1, double c2, double c3,
                                                             long ncell, double *__restrict__ c) {
  const long cell = long(blockIdx.x) * 256 + threadIdx.x;
  if (cell >= ncell) return;
  const double ic[3] = {c1, c2, c3};
  double t = 0.0;
#pragma unroll
  for (int p = 0; p < P; ++p) t += pfrac[cell * P + p] * ic[p];
  c[cell] = t;
}

__device__ inline uint64_t splitmix64(uint64_t x) {
  uint64_t z = x + 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

// Nucleation flag (nucleation.cpp:12): slots in use minus the matrix-phase carbon of the cell
// times (1 - 0.001 u); u from the counter-based generator keyed by (seed, cell).
template <int K, int P>
__global__ __launch_bounds__(256) void nucleation_flag_kernel(
    const uint16_t *__restrict__ id, const double *__restrict__ pfrac,
    const double *__restrict__ c0, const DiffConsts<double> dc, uint64_t seed_key, long ncell,
    float *__restrict__ flag, uint8_t *__restrict__ mark) {
  const long cell = long(blockIdx.x) * 256 + threadIdx.x;
  if (cell >= ncell) return;
  uint32_t g[K];
  load_ids<K>(id, cell, g);
  int cnt = 0;
#pragma unroll
  for (int s = 0; s < K; ++s) cnt += g[s] > 0 ? 1 : 0;
  double ph[P];
#pragma unroll
  for (int p = 0; p < P; ++p) ph[p] = pfrac[cell * P + p];
  // value_conc1(2,cell): the full partition of phase 2
  double t1 = 0.0, t2 = 0.0;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    t1 += ph[j] * dc.pk[1][j];
    t2 += ph[j] * dc.pc[1][j];
  }
  const float c2 = float((c0[cell] - t2) / t1);
  const float u = float(double(splitmix64(seed_key + uint64_t(cell)) >> 40) * (1.0 / 16777216.0));
  flag[cell] = float(double(float(cnt)) - double(c2) * (1. - 0.001 * double(u)));
  mark[cell] = 0;
}

// The first maximum of the nucleation flag in storage order (larger value, then smaller index) is
// kept per chunk of kFlagChunk consecutive cells.  Painting a nucleus changes flags only inside its
// box: a workgroup owns one chunk that the box touches, paints the chunk's cells and takes the chunk's
// new maximum in the same pass; the last workgroup to end takes the maximum over the chunks, the next
// nucleus's centre.  One small launch per nucleus instead of three and a pass over the whole domain.
// 256^3: 32.7 (23.4 + 4.9 + 4.4) -> 10.3 us per nucleus, the latency of its chain (centre, flags,
// two reductions, the count, the maxima).  512^3: 271 -> 13.8 us.
//
// A flag and its cell as one number that grows with the flag and, for equal flags, falls with the
// cell; 0 is no cell, a NaN sorts below every number.
__device__ inline unsigned long long flag_key(float v, int cell) {
  uint32_t u = __float_as_uint(v + 0.f);  // (-0 as +0)
  u = (u & 0x80000000u) ? ~u : u | 0x80000000u;
  if (v != v) u = 0;
  return (static_cast<unsigned long long>(u) << 32) | uint32_t(~cell);
}
// the largest of a workgroup of 1024 threads, in every thread
__device__ inline unsigned long long block_best(unsigned long long m, unsigned long long (&part)[16]) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = max(m, __shfl_xor(m, d));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  m = part[threadIdx.x & 15];
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) m = max(m, __shfl_xor(m, d));
  return m;
}
__global__ __launch_bounds__(1024) void flag_chunks_kernel(const float *__restrict__ flag, int ncell,
                                                           unsigned long long *__restrict__ best) {
  __shared__ unsigned long long part[16];
  const int beg = int(blockIdx.x) * kFlagChunk, len = min(kFlagChunk, ncell - beg);
  unsigned long long m = 0;
#pragma unroll
  for (int o = 0; o < kFlagChunk; o += 1024) {
    const int q = o + int(threadIdx.x);
    if (q < len) m = max(m, flag_key(flag[beg + q], beg + q));
  }
  m = block_best(m, part);
  if (threadIdx.x == 0) best[blockIdx.x] = m;
}
// one workgroup: the cell of the maximum over the chunks; centre[1] is the paint's count of workgroups
__global__ __launch_bounds__(1024) void flag_centre_kernel(const unsigned long long *__restrict__ best,
                                                           int nchunk, int *__restrict__ centre) {
  __shared__ unsigned long long part[16];
  unsigned long long m = 0;
  for (int q = threadIdx.x; q < nchunk; q += 1024) m = max(m, best[q]);
  m = block_best(m, part);
  if (threadIdx.x == 0) {
    centre[0] = int(~uint32_t(m));
    centre[1] = 0;
  }
}

// Paint a nucleus around the centre (nucleation.cpp:15-37): cells closer than radius become it
// (slot 0 = code, phi = 1, value_phase = (1,0,0)); cells closer than 2*radius leave the flag at
// zero.  The box of half-width R = ceil(2 radius) around the centre holds every affected cell; along
// an axis shorter than 2R+1 it is the whole axis.  blockIdx.y is a plane of the box; its rows are at
// most two runs of cells (the y axis wraps once), and blockIdx.x counts the chunks that these touch.
// (More planes than a grid may have are taken in turns.)  Runs of several planes can share a chunk:
// the workgroups then write the same values, and no one uses a flag that another changes (a painted
// cell's is taken as zero).
// The chunk maxima cross workgroups inside the launch: they are stored and read at device scope, and
// the count that orders them is an acquire-release one, so the last workgroup sees all of them.
template <int K, int P>
__global__ __launch_bounds__(1024) void nucleus_paint_kernel(
    int *__restrict__ centre, int code, float radius, int R, int nx, int ny, int nz, int cy_n, int cz_n,
    uint16_t *__restrict__ id, double *__restrict__ phi, double *__restrict__ pfrac,
    float *__restrict__ flag, uint8_t *__restrict__ mark, int ncell,
    unsigned long long *__restrict__ best, int nchunk) {
  __shared__ unsigned long long part[16];
  __shared__ int last;
  const int mid = centre[0], plane = nx * ny;
  const int cx = mid % nx, cy = (mid / nx) % ny, cz = mid / plane;
  auto wrapped = [](int v, int n) { return ((v % n) + n) % n; };
  const int y0 = cy_n == ny ? 0 : wrapped(cy - R, ny);
  const int yn = min(cy_n, ny - y0), yw = cy_n - yn;  // rows before and after the wrap
  for (int iz = blockIdx.y; iz < cz_n; iz += gridDim.y) {
    const int z = cz_n == nz ? iz : wrapped(cz - R + iz, nz);
    const int run0 = plane * z + nx * y0, run1 = plane * z;
    const int c0 = run0 / kFlagChunk, n0 = (run0 + nx * yn - 1) / kFlagChunk - c0 + 1;
    const int c1 = run1 / kFlagChunk, n1 = yw ? (run1 + nx * yw - 1) / kFlagChunk - c1 + 1 : 0;
    const int b = blockIdx.x;
    if (b >= n0 + n1) continue;
    const int chunk = b < n0 ? c0 + b : c1 + (b - n0);
    const int beg = chunk * kFlagChunk, len = min(kFlagChunk, ncell - beg);
    float v[kFlagChunk / 1024];
#pragma unroll
    for (int o = 0; o < kFlagChunk / 1024; ++o) {
      const int q = o * 1024 + int(threadIdx.x);
      v[o] = q < len ? flag[beg + q] : 0.f;
    }
    unsigned long long m = 0;
#pragma unroll
    for (int o = 0; o < kFlagChunk / 1024; ++o) {
      const int q = o * 1024 + int(threadIdx.x);
      if (q >= len) continue;
      const int cell = beg + q;
      const int row = cell / nx, x = cell - row * nx, zz = row / ny, y = row - zz * ny;
      const int off[3] = {abs(cx - x), abs(cy - y), abs(cz - zz)}, ext[3] = {nx, ny, nz};
      float dist = 0.f;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const long ad = off[d], bd = ext[d] - off[d];
        const float s1 = float(ad * ad), s2 = float(bd * bd);
        dist += fminf(s1, s2);
      }
      const float Dist = sqrtf(dist);
      if (Dist < radius) {
        uint32_t g[K];
#pragma unroll
        for (int s = 0; s < K; ++s) g[s] = 0;
        g[0] = uint32_t(code) & 0xffffu;
        store_ids<K>(id, cell, g);
#pragma unroll
        for (int s = 0; s < K; ++s) phi[long(cell) * K + s] = s == 0 ? 1.0 : 0.0;
#pragma unroll
        for (int p = 0; p < P; ++p) pfrac[long(cell) * P + p] = p == 0 ? 1.0 : 0.0;
        mark[cell] = 1;
      }
      if (Dist < 2 * radius) flag[cell] = v[o] = 0.f;
      m = max(m, flag_key(v[o], cell));
    }
    m = block_best(m, part);
    if (threadIdx.x == 0)
      __hip_atomic_store(best + chunk, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();  // `part` has been read
  }
  // every thread has read the centre (one with nothing to paint passes no barrier above) before this
  // workgroup is counted: the last one changes it
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(centre + 1, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
           int(gridDim.x * gridDim.y) - 1;
  __syncthreads();
  if (!last) return;
  unsigned long long m = 0;
  for (int q = threadIdx.x; q < nchunk; q += 1024)
    m = max(m, __hip_atomic_load(best + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  m = block_best(m, part);
  if (threadIdx.x == 0) {  // every workgroup has read its centre
    centre[0] = int(~uint32_t(m));
    centre[1] = 0;
  }
}

__global__ __launch_bounds__(256) void nucleus_conc_kernel(const uint8_t *__restrict__ mark,
                                                           double value, long ncell,
                                                           double *__restrict__ c) {
  const long cell = long(blockIdx.x) * 256 + threadIdx.x;
  if (cell >= ncell) return;
  if (mark[cell]) c[cell] = value;
}

// mean + sd * (sum of 12 uniforms - 6): an Irwin-Hall approximation of a Gaussian whose value
// is reproduced exactly by any IEEE double evaluation in this order
__global__ __launch_bounds__(256) void solute_noise_kernel(double mean, double sd,
                                                           uint64_t seed_key, long ncell,
                                                           double *__restrict__ c) {
  const long cell = long(blockIdx.x) * 256 + threadIdx.x;
  if (cell >= ncell) return;
  double acc = 0.0;
  for (int q = 0; q < 12; ++q)
    acc += double(splitmix64(seed_key + uint64_t(cell) * 12 + q) >> 11) *
           (1.0 / 9007199254740992.0);
  c[cell] = mean + sd * (acc - 6.0);
}

// FP64 domain -> mixed domain (round each stored value; compensation starts at zero)
// grid-stride: n reaches N*K elements (2^32 at 1024^3, K = 4), beyond one launch's work-items
__global__ __launch_bounds__(256) void convert_f64_to_f32(const double *__restrict__ src,
                                                          float *__restrict__ dst, long n) {
  for (long i = long(blockIdx.x) * 256 + threadIdx.x; i < n; i += long(gridDim.x) * 256)
    dst[i] = float(src[i]);
}
__global__ __launch_bounds__(256) void convert_conc_f64_to_mixed(const double *__restrict__ src,
                                                                 float *__restrict__ dst, long n) {
  const long i = long(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) {
    dst[i] = float(src[i]);
    if (i < (n + 1) / 2) comp_bytes(dst, n)[i] = 0;  // the code bytes of cells 2i, 2i + 1
  }
}

// explicit instantiations used by the host dispatch (pf_api.hip)
#define PF_INST_RED(F, K, P)                                                                     \
  template __global__ void reduce_stage1<F, K, P>(const uint16_t *, const F::T *, const F::T *,  \
                                                  const F::C *, const F::C *, int, long, long,   \
                                                  RedPartial *);
PF_INST_RED(FormF64, 4, 2)
PF_INST_RED(FormF64, 4, 3)
PF_INST_RED(FormF64, 6, 2)
PF_INST_RED(FormF64, 6, 3)
PF_INST_RED(FormMixed, 4, 2)
PF_INST_RED(FormMixed, 4, 3)
PF_INST_RED(FormMixed, 6, 2)
PF_INST_RED(FormMixed, 6, 3)

// Fields of the VTI dump (write_data.cpp:42-82): korn = 0 where slot 2 holds a grain, else the
// phase of slot 1 (the grain code's top bits; 0 for an empty cell); conc = the total carbon
// concentration (mixed form: the stored value minus its compensation, as pf_download_state
// reports it), as float.
template <class F>
__global__ __launch_bounds__(256) void vti_fields_kernel(const uint16_t *__restrict__ id,
                                                         const int KI,
                                                         const typename F::C *__restrict__ c,
                                                         const long ncell,
                                                         int32_t *__restrict__ korn,
                                                         float *__restrict__ conc) {
  const long cell = long(blockIdx.x) * 256 + threadIdx.x;
  if (cell >= ncell) return;
  const int g1 = id[cell * KI], g2 = id[cell * KI + 1];
  korn[cell] = g2 != 0 ? 0 : (g1 >> 14);
  conc[cell] = float(conc_effective<F>(c, cell, ncell));
}
template __global__ void vti_fields_kernel<FormF64>(const uint16_t *, int, const double *, long,
                                                    int32_t *, float *);
template __global__ void vti_fields_kernel<FormMixed>(const uint16_t *, int, const float *, long,
                                                      int32_t *, float *);

#define PF_INST_SETUP(K, P)                                                                      \
  template __global__ void voronoi_kernel<K, P>(const double *, int, double, int, int, int,      \
                                                long, uint16_t *, double *, double *);           \
  template __global__ void nucleation_flag_kernel<K, P>(const uint16_t *, const double *,        \
                                                        const double *, const DiffConsts<double>, \
                                                        uint64_t, long, float *, uint8_t *);     \
  template __global__ void nucleus_paint_kernel<K, P>(                                           \
      int *, int, float, int, int, int, int, int, int, uint16_t *, double *, double *, float *,    \
      uint8_t *, int, unsigned long long *, int);
PF_INST_SETUP(4, 2)
PF_INST_SETUP(4, 3)
PF_INST_SETUP(6, 2)
PF_INST_SETUP(6, 3)
template __global__ void construct_conc_kernel<2>(const double *, double, double, double, long,
                                                  double *);
template __global__ void construct_conc_kernel<3>(const double *, double, double, double, long,
                                                  double *);

}  // namespace pfamd
