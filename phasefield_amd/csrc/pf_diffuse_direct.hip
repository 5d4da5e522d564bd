// pf_diffuse_direct.hip — one diffusion sub-step in one launch, for 3D domains whose concentration
// stays in the memory-side cache and for rows that hold no whole number of 16-byte runs (the formula
// and its bulk reduction: pf_diffuse.hip).
//
// Up to 128^3 a sub-step is bound by the launches and by one round of memory latency, not by bytes
// (an empty launch takes 1.6 us, a pass over 64^3 cells 2.8 us), so the bulk cells and the listed
// cells share one launch: the first (and, for long lists, the last) workgroups take the list, the
// others the bulk cells, and each cell is written by exactly one of them (a bulk thread skips what the
// flags list).  The bulk part keeps nothing in LDS and has no loop: every load of a thread is issued before the first is used,
// and each XCD takes a contiguous range of the domain, so the y and z neighbours come from its L2
// (128^3 FP64 pass alone: 6.6 us with contiguous ranges, 7.3 us in launch order, 4.1 us for a plain
// copy).  Flags are read as two bits per cell.
// Sub-step, before (plane-marching kernel, then the listed pass) and after, 3D seeded states:
//   40 x 24 x 16 FP64  12.5 -> 4.3 us     101 x 75 x 67 FP64   13.1 -> 5.9 us
//   64^3 mixed         13.3 -> 5.8 us     101 x 75 x 67 mixed  30.0 -> 6.3 us
//   128^3 FP64         17.9 -> 10.1 us    128^3 mixed          14.3 -> 8.5 us
//   192^3 FP64         43.3 -> 24.8 us    192^3 mixed          32.8 -> 18.2 us
// Up to 128^3 what is left is launch, two rounds of latency and the listed cells' arithmetic
// (divisions and square roots); above, the traffic of the caches.
#include "pf_diffuse_direct_impl.h"

namespace pfamd {

namespace {

// the stencil of cell i
template <class F, int P, bool NOFLUX>
__device__ inline void load_stencil(const typename F::C *__restrict__ cin,
                                    const typename F::T *__restrict__ pfrac, uint32_t i, int nx, int ny,
                                    int nz, StencilLoad<F, P, 6> &s) {
  int x, y, z;
  cell_coords(i, nx, ny, x, y, z);
  const uint32_t ux = uint32_t(nx), plane = ux * uint32_t(ny), vol = plane * uint32_t(nz);
  const long nb[6] = {long(x == 0 ? i + ux - 1u : i - 1u),
                      long(x == nx - 1 ? i + 1u - ux : i + 1u),
                      long(y == 0 ? i + plane - ux : i - ux),
                      long(y == ny - 1 ? i + ux - plane : i + ux),
                      long(z == 0 ? (NOFLUX ? i : i + vol - plane) : i - plane),
                      long(z == nz - 1 ? (NOFLUX ? i : i + plane - vol) : i + plane)};
  stencil_load<F, P, 6>(cin, pfrac, i, long(vol), nb, s);
}
// the increment of a bulk cell: the reduced form with the phase its value_phase names
template <int P>
__device__ inline float bulk_del(const StencilLoad<FormMixed, P, 6> &s, const DiffConsts<float> &dc) {
  float Dp = dc.D[0];
#pragma unroll
  for (int p = 1; p < P; ++p)
    if (s.me.ph[p] == 1.f) Dp = dc.D[p];
  BulkAcc<FormMixed> acc;
  acc.first(s.nb[0].c - s.me.c, Dp);
#pragma unroll
  for (int f = 1; f < 6; ++f) acc.add(s.nb[f].c - s.me.c, Dp);
  return acc.result(dc.r, Dp * dc.r);
}

}  // namespace

template <class F, int P, bool NOFLUX, int V, int U, bool MORE>
__global__ __launch_bounds__(256) void diffuse_direct_kernel(
    const typename F::C *__restrict__ cin, typename F::C *__restrict__ cout,
    const typename F::T *__restrict__ pfrac, const uint32_t *__restrict__ packed,
    const int *__restrict__ list, const int *__restrict__ count,
    const DiffConsts<typename F::A> dc, const DirectGeom geo) {
  constexpr int NF = 6;
  const int nx = geo.nx, ny = geo.ny, nz = geo.nz;
  const uint32_t plane = uint32_t(nx) * uint32_t(ny);
  const long n = long(plane) * nz;
  const int b = blockIdx.x;

  const int bulk = b - geo.nlist;
  if (MORE ? __builtin_expect(unsigned(bulk) >= unsigned(geo.nbulk), 0) : bulk < 0) {
    const int group = bulk < 0 ? b : b - geo.nbulk;
    // the first entry is read along with the list's length (the list has room for every cell)
    // (unsigned: an index below 2^31 and a round of threads)
    const uint32_t stride = uint32_t(geo.nlist + (MORE ? geo.nmore : 0)) * 256u;
    uint32_t k = uint32_t(group) * 256u + threadIdx.x;
    int e = list[min(long(k), n - 1)];
    const uint32_t m = uint32_t(*count);
    for (; k < m; k += stride, e = k < m ? list[k] : 0) {
      if constexpr (F::kMixed) {
        // a byte pair (ListOrder::pairs): both cells are computed and stored, with their code byte;
        // the one that is not listed takes its bulk form
        const uint32_t j = uint32_t(e) & 0x3fffffffu, mask = uint32_t(e) >> 30;
        const uint32_t i0 = 2 * j, i1 = min(i0 + 1u, uint32_t(n) - 1u);
        StencilLoad<F, P, NF> s0, s1;
        load_stencil<F, P, NOFLUX>(cin, pfrac, i0, nx, ny, nz, s0);
        load_stencil<F, P, NOFLUX>(cin, pfrac, i1, nx, ny, nz, s1);
        const float d0 = (mask & 1u) ? stencil_del<F, P, NF>(s0, dc) : bulk_del<P>(s0, dc);
        const float d1 = (mask & 2u) ? stencil_del<F, P, NF>(s1, dc) : bulk_del<P>(s1, dc);
        CompCode q0, q1;
        const float v0 = mixed_step(s0.me.c, d0, s0.q, comp_hash(i0, dc.key), q0);
        const float v1 = mixed_step(s1.me.c, d1, s1.q, comp_hash(i1, dc.key), q1);
        uint32_t byte = uint32_t(q0) & 15u;
        cout[i0] = v0;
        if (i1 != i0) {
          cout[i1] = v1;
          byte |= (uint32_t(q1) & 15u) << 4;
        }
        comp_bytes(cout, n)[j] = uint8_t(byte);
      } else {
        const uint32_t i = uint32_t(e);
        StencilLoad<F, P, NF> st;
        load_stencil<F, P, NOFLUX>(cin, pfrac, i, nx, ny, nz, st);
        stencil_update<F, P, NF>(cout, i, n, st, dc);
      }
    }
    return;
  }

  direct_bulk<F, P, NOFLUX, V, U>(cin, cout, packed, dc, geo, bulk);
}

#define PF_INST_DIRECT(F, P, NOF, V, U, MORE)                                                 \
  template __global__ void diffuse_direct_kernel<F, P, NOF, V, U, MORE>(                      \
      const F::C *, F::C *, const F::T *, const uint32_t *, const int *, const int *,          \
      const DiffConsts<F::A>, DirectGeom);
#define PF_INST_DIRECT_NOF(F, P, V, U)     \
  PF_INST_DIRECT(F, P, false, V, U, false) \
  PF_INST_DIRECT(F, P, false, V, U, true)  \
  PF_INST_DIRECT(F, P, true, V, U, false)  \
  PF_INST_DIRECT(F, P, true, V, U, true)
#define PF_INST_DIRECT_P(P)            \
  PF_INST_DIRECT_NOF(FormF64, P, 1, 2)   \
  PF_INST_DIRECT_NOF(FormF64, P, 2, 2)   \
  PF_INST_DIRECT_NOF(FormMixed, P, 1, 1) \
  PF_INST_DIRECT_NOF(FormMixed, P, 2, 2) \
  PF_INST_DIRECT_NOF(FormMixed, P, 4, 2)
PF_INST_DIRECT_P(2)
PF_INST_DIRECT_P(3)

}  // namespace pfamd
