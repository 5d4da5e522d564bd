// pf_diffuse_direct.h — the one-launch diffusion sub-step of 3D domains (pf_diffuse_direct.hip).
#pragma once
#include <algorithm>

#include "pf_diffuse_common.h"

namespace pfamd {

// n / d and n % d for 0 <= n < 2^31 by one multiplication with the rounded-up reciprocal (Granlund and
// Montgomery's division by invariant integers): with s = ceil(log2 d) and
// m = ceil(2^(31+s) / d) < 2^32 the error m * d - 2^(31+s) is below 2^s, so n * error stays below
// 2^(31+s) and the quotient is exact.
struct FastDiv {
  uint32_t d = 1, mul = 0x80000000u, shift = 31;
  FastDiv() = default;
  explicit FastDiv(uint32_t div) : d(div) {
    uint32_t s = 0;
    while ((1ull << s) < div) ++s;
    shift = 31 + s;
    mul = uint32_t(((1ull << shift) + div - 1) / div);
  }
  __host__ __device__ uint32_t quot(uint32_t n) const { return uint32_t((uint64_t(n) * mul) >> shift); }
  __host__ __device__ uint32_t rem(uint32_t n) const { return n - d * quot(n); }
};

struct DirectGeom {
  int nlist;     // workgroups of the listed cells, ahead of the others
  int nbulk;     // workgroups of the bulk cells
  int nmore;     // workgroups of the listed cells behind the others
  int flip;      // walk the bulk cells from the last to the first
  int nx, ny, nz;
  FastDiv row;   // runs of V cells per row (mixed, V == 1: cells per row)
  FastDiv rows;  // rows per plane
};

// One sub-step: the bulk cells of every phase in runs of V cells times U planes per thread, the
// listed cells (flag 0; mixed: the byte pairs that hold one) by the first workgroups.  `packed`: the
// bulk flags, two bits per cell (general_count_kernel).  MORE: geo.nmore > 0 (a kernel of its own: the test
// for workgroups behind the bulk cells costs the allocation-free call at 128^3 1.5 %).
template <class F, int P, bool NOFLUX, int V, int U, bool MORE>
__global__ void diffuse_direct_kernel(const typename F::C *__restrict__ cin,
                                      typename F::C *__restrict__ cout,
                                      const typename F::T *__restrict__ pfrac,
                                      const uint32_t *__restrict__ packed,
                                      const int *__restrict__ list, const int *__restrict__ count,
                                      const DiffConsts<typename F::A> dc, const DirectGeom geo);

// the part of the geometry that does not depend on the run length
inline DirectGeom direct_geometry(int nx, int ny, int nz, bool flip) {
  const long n = long(nx) * ny * nz;
  DirectGeom g;
  g.nx = nx;
  g.ny = ny;
  g.nz = nz;
  g.flip = flip;
  // The listed part: one entry per thread up to a sixteenth of the cells (a round of entries is a
  // chain of three memory latencies and the full formula), at least 64 workgroups where the domain
  // has that many (40 x 24 x 16 with 4 workgroups: 11.0 us, with 60: 4.3).  Domains of up to 2^20 cells
  // have seven times as many again behind the bulk cells, which end at once where the list is
  // short: 64^3 FP64 with every cell listed 11.8 us, 37.1 without them (18.2 in a listed pass of its own),
  // with 3 % listed 4.9 either way.  (The bulk workgroups going on with the list instead: every cell
  // listed 16.4, and 1.5-3.5 % on short lists at 128^3.)  Never more than one entry per thread,
  // so there are at most (n + 255) / 256 of them.
  g.nlist = int(std::min<long>(1024, std::max<long>((n + 4095) / 4096, std::min<long>(64, (n + 255) / 256))));
  g.nmore = n <= (1L << 20) ? int(std::min<long>(7L * g.nlist, (n + 255) / 256 - g.nlist)) : 0;
  return g;
}
// runs of V cells times U planes; pairs: byte pairs in storage order instead
inline void set_runs(DirectGeom &g, bool pairs, int V, int U) {
  const long n = long(g.nx) * g.ny * g.nz;
  g.row = FastDiv(uint32_t(pairs ? g.nx : g.nx / V));
  g.rows = FastDiv(uint32_t(g.ny));
  const long items = pairs ? (n + 1) / 2 : long(g.nx / V) * g.ny * ((g.nz + U - 1) / U);
  g.nbulk = int((items + 255) / 256);
}

// Run length: 16 bytes where the rows hold a whole number of runs, so that every run is aligned and
// within one row; rows of odd length take single cells (FP64) or byte pairs in storage order (mixed).
// Two planes per thread: 128^3 10.5 us against 11.2 with one and 10.7 with four (FP64), 224^3 34.0
// against 38.8 and 35.5.
//
// `flip` alternates between the sub-steps: a pass that starts where the last one ended finds that end
// still cached where several domains share the memory-side cache.  Step, always forwards / alternating,
// three domains in turn: 176^3 FP64 4.64 / 4.36 ms, 192^3 6.35 / 6.24, 216^3 mixed 5.56 / 5.34; one domain
// alone 0.4-0.7 % longer (192^3 4.62 / 4.63).
template <class F, int P, bool NOF>
hipError_t launch_direct(hipStream_t stream, const typename F::C *cin, typename F::C *cout,
                         const typename F::T *pfrac, const uint32_t *packed, const int *list,
                         const int *count, const DiffConsts<typename F::A> &dc, int nx, int ny, int nz,
                         bool flip) {
  DirectGeom g = direct_geometry(nx, ny, nz, flip);
  auto go = [&](auto v, auto u) {
    constexpr int V = decltype(v)::value, U = decltype(u)::value;
    set_runs(g, F::kMixed && V == 1, V, U);
    auto kernel = g.nmore > 0 ? diffuse_direct_kernel<F, P, NOF, V, U, true>
                              : diffuse_direct_kernel<F, P, NOF, V, U, false>;
    hipLaunchKernelGGL(kernel, dim3(unsigned(g.nlist + g.nbulk + g.nmore)), dim3(256), 0, stream, cin,
                       cout, pfrac, packed, list, count, dc, g);
  };
  using std::integral_constant;
  if constexpr (F::kMixed) {
    if (nx % 4 == 0) go(integral_constant<int, 4>(), integral_constant<int, 2>());
    else if (nx % 2 == 0) go(integral_constant<int, 2>(), integral_constant<int, 2>());
    else go(integral_constant<int, 1>(), integral_constant<int, 1>());
  } else {
    // (a caller's own array, in the accelerator calls, may be aligned to one value only)
    const bool aligned =
        (reinterpret_cast<uintptr_t>(cin) | reinterpret_cast<uintptr_t>(cout)) % 16 == 0;
    if (nx % 2 == 0 && aligned) go(integral_constant<int, 2>(), integral_constant<int, 2>());
    else go(integral_constant<int, 1>(), integral_constant<int, 2>());
  }
  return hipGetLastError();
}

}  // namespace pfamd
