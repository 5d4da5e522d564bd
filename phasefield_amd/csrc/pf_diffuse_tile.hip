// pf_diffuse_tile.hip — several diffusion sub-steps of one solute in one launch, for domains of
// independent planes (2D; the formula and its bulk reduction: pf_diffuse.hip).
//
// One sub-step of a 2D domain is a few microseconds of launch and memory latency around almost no
// work, so a workgroup takes its tile through `steps` sub-steps: it loads the tile with a halo of
// that many cells, keeps the values in LDS, and every sub-step the cells that are still exact shrink
// by one layer.  The halo is computed again by the neighbouring tiles, with the same operations in
// the same order, so the result is bitwise that of single sub-steps.
//
// A bulk cell (flag p) is owned by a thread and takes the reduced update.  The listed cells (flag 0)
// are compacted per tile; each is an entry of one thread, which keeps the cell's face weights and
// partition constants in registers for all sub-steps of the launch and publishes the cell's
// partition in LDS for the entries next to it.  A tile with more listed cells than threads gives every
// thread two.  Two of three phases would not fit the registers: where a tile that full has the third
// phase it takes the full formula from memory, every sub-step.  The two-phase FP64 kernel is held to 96
// registers (a few values of the second instance are spilled): at 116 every step took 3 % longer in turn
// with other domains' kernels.  Per sub-step, one domain, every cell listed, from memory (as it was) /
// with two entries / single sub-steps:
//   256^2 FP64             6.98 / 2.85 / 8.1 us   1000 x 600 FP64    27.8 / 14.9 / 20.4 us
//   256^2 mixed            4.45 / 3.12 / 8.7      1000 x 600 mixed   16.3 / 12.9 / 14.0
//   256^2, third absent    8.52 / 2.17 / 8.7      1200^2 FP64        54.2 / 29.0 / 35.6
// The third phase's terms are 0 * (0 - 0) where no entry of a wavefront and none of its neighbours has
// that phase, and are left out there (256^2 accelerator call 322 -> 307 us).
//
// A one-cell-thick domain whose stencil has six faces (the accelerator calls) runs here as well: its
// z faces join a cell to itself and carry no flux, only the NaN of a partition that is not finite
// (SELF_Z; an infinite bulk cell becomes NaN without them).
#include "pf_diffuse_tile.h"

#include <type_traits>

namespace pfamd {

template <class F, int P, bool SELF_Z>
__global__ __launch_bounds__(kTileNT, P == 2 ? (F::kMixed ? 8 : 5) : 4) void diffuse_tile_kernel(
    const typename F::C *__restrict__ cin, typename F::C *__restrict__ cout,
    const typename F::T *__restrict__ pfrac, const uint8_t *__restrict__ flag,
    const DiffConsts<typename F::A> dc, const TileGeom geo, const long ncell, const uint32_t k0,
    const int solute) {
  using A = typename F::A;
  constexpr int NF = 4, NT = kTileNT, V = kTileV, CELLS = NT * V;
  constexpr int NONE = CELLS + CELLS * P;  // the partition of an absent phase
  static_assert(NONE < 65535, "16-bit element indices");
  static_assert(V <= 8 && V * P <= 32, "packed codes and presence bits");
  __shared__ A L[NONE + 1];            // the cells' values; behind them the entries' partitions; 0
  __shared__ uint16_t slot_of[CELLS];  // a listed cell's entry, 0xffff for the others
  __shared__ uint16_t list[CELLS];     // the listed cells
  __shared__ uint8_t codes[F::kMixed ? CELLS : 1];
  __shared__ int counter;
  const int t = threadIdx.x;
  const int nx = geo.nx, ny = geo.ny, S = geo.steps;
  // Workgroup b runs on XCD b % 8: of every 256 tiles in a row (one per compute unit) each XCD takes a
  // contiguous eighth, so that neighbouring tiles share its L2 and tiles full of listed cells, which
  // lie side by side, spread over the XCDs (1000 x 600 FP64, 30 % of the plane listed: 14.5 us per
  // sub-step with eighths of all tiles, 7.7 with these).
  const int b = blockIdx.x, group = b & ~255;
  const int m = min(256, geo.nblocks - group), xcd = b & 7;
  const int logical = group + xcd * (m >> 3) + min(xcd, m & 7) + ((b & 255) >> 3);
  const int tx = logical % geo.nbx, tyz = logical / geo.nbx;
  const int ty = tyz % geo.nby;
  const uint32_t plane0 = uint32_t(nx) * uint32_t(ny) * uint32_t(tyz / geo.nby);
  const int ix0 = tx * geo.bx, iy0 = ty * geo.by;
  const int ibx = min(geo.bx, nx - ix0), iby = min(geo.by, ny - iy0);
  const int X = ibx + 2 * S, Y = iby + 2 * S, ncells = X * Y;
  const int ox = ix0 - S, oy = iy0 - S;

  if (t == 0) {
    counter = 0;
    L[NONE] = A(0);
  }
  __syncthreads();

  auto wrapn = [](int i, int e) {  // into [0, e), from any distance (a halo may span the domain)
    i %= e;
    return i < 0 ? i + e : i;
  };
  // The thread's cells t + k * NT: place in the domain, sub-steps a bulk cell stays exact for (0: not
  // updated here), phase - 1, whether it is of the tile itself.
  uint32_t gi[V];
  int depth[V];
  uint32_t phase = 0, inside = 0, general = 0, qs = 0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int idx = t + k * NT;
    gi[k] = 0;
    depth[k] = 0;
    bool gen = false;
    if (idx < ncells) {
      const int ly = int(unsigned(idx) / unsigned(X)), lx = idx - ly * X;
      gi[k] = plane0 + uint32_t(wrapn(ox + lx, nx)) + uint32_t(nx) * uint32_t(wrapn(oy + ly, ny));
      const int f = flag[gi[k]];
      L[idx] = A(cin[gi[k]]);
      if constexpr (F::kMixed) qs |= (uint32_t(comp_load(cin, ncell, gi[k])) & 15u) << (4 * k);
      gen = f == 0;
      if (!gen) {
        depth[k] = min(min(lx, X - 1 - lx), min(ly, Y - 1 - ly));
        phase |= uint32_t(f - 1) << (2 * k);
      } else {
        general |= 1u << k;
      }
      if (lx >= S && lx < X - S && ly >= S && ly < Y - S) inside |= 1u << k;
    }
    // the tile's listed cells, compacted (their order changes no result)
    const unsigned long long m = __ballot(gen);
    int base = 0;
    const int lane = t & 63;
    if (lane == 0 && m) base = atomicAdd(&counter, __popcll(m));
    base = __shfl(base, 0);
    const int slot = base + __popcll(m & ((1ull << lane) - 1ull));
    if (idx < ncells) slot_of[idx] = gen ? uint16_t(slot) : uint16_t(0xffff);
    if (gen) {
      list[slot] = uint16_t(idx);
      if constexpr (F::kMixed) codes[idx] = uint8_t((qs >> (4 * k)) & 15u);
    }
  }
  __syncthreads();
  const int ng = counter;

  auto key_of = [&](int s) -> uint32_t {
    return F::kMixed ? comp_step_key(k0 + uint32_t(s - 1), solute) : 0u;
  };
  // One sub-step of the thread's bulk cells, from L into nv.  No branch between the cells: an
  // inactive one reads the neighbourhood of cell (1, 1), so the loads and sums of the V cells overlap
  // (a sub-step is one chain of LDS and FP64 latencies; with a branch per cell it was V of them).
  A nv[V];
  auto bulk_step = [&](int s, uint32_t key) {
    bool any = false;
#pragma unroll
    for (int k = 0; k < V; ++k) any = any || depth[k] >= s;
    if (!__any(any)) return;
    A c[V], f[V][4];
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const int at = depth[k] >= s ? t + k * NT : X + 1;
      c[k] = L[at];
      f[k][0] = L[at - 1];
      f[k][1] = L[at + 1];
      f[k][2] = L[at - X];
      f[k][3] = L[at + X];
    }
#pragma unroll
    for (int k = 0; k < V; ++k) {
      A Dp = dc.D[0];
#pragma unroll
      for (int q = 1; q < P; ++q)
        if (((phase >> (2 * k)) & 3u) == uint32_t(q)) Dp = dc.D[q];
      BulkAcc<F> acc;
      acc.first(f[k][0] - c[k], Dp);
      acc.add(f[k][1] - c[k], Dp);
      acc.add(f[k][2] - c[k], Dp);
      acc.add(f[k][3] - c[k], Dp);
      const A del = acc.result(dc.r, Dp * dc.r);
      if constexpr (F::kMixed) {
        CompCode qo;
        nv[k] = mixed_step(c[k], del, comp_unpack(qs >> (4 * k)), comp_hash(gi[k], key), qo);
        if (depth[k] >= s) qs = (qs & ~(15u << (4 * k))) | ((uint32_t(qo) & 15u) << (4 * k));
      } else {
        nv[k] = c[k] + del;
      }
    }
  };
  auto bulk_write = [&](int s) {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (depth[k] >= s) L[t + k * NT] = nv[k];
  };
  // what faces that join a cell to itself add: 0, or NaN where a partition is not finite
  static_assert(!SELF_Z || !F::kMixed, "an FP64 sum starts from it");
  auto self_z = [](const auto &c) {
    A z = c[0] * A(0);
#pragma unroll
    for (size_t p = 1; p < sizeof(c) / sizeof(c[0]); ++p) z = __builtin_elementwise_fma(c[p], A(0), z);
    return z;
  };
  // a listed cell's place, its neighbours' in the domain and in L, and its depth
  struct Cell {
    uint32_t g, gn[4];
    int off[4], depth;
  };
  auto locate = [&](int idx, Cell &o) {
    const int ly = int(unsigned(idx) / unsigned(X)), lx = idx - ly * X;
    const int gx = wrapn(ox + lx, nx), gy = wrapn(oy + ly, ny);
    const uint32_t unx = uint32_t(nx), plane = unx * uint32_t(ny);
    const uint32_t g = plane0 + uint32_t(gx) + unx * uint32_t(gy);
    o.g = g;
    o.depth = min(min(lx, X - 1 - lx), min(ly, Y - 1 - ly));
    o.off[0] = -1;
    o.off[1] = 1;
    o.off[2] = -X;
    o.off[3] = X;
    o.gn[0] = gx == 0 ? g + unx - 1u : g - 1u;
    o.gn[1] = gx == nx - 1 ? g + 1u - unx : g + 1u;
    o.gn[2] = gy == 0 ? g + plane - unx : g - unx;
    o.gn[3] = gy == ny - 1 ? g + unx - plane : g + unx;
  };

  // whether a cell of the tile has the third phase (or one of its constants is not finite)
  auto third_phase = [&]() {
    bool has = !(dc.D[2] * A(0) == A(0));
#pragma unroll
    for (int i = 0; i < 3; ++i) has = has || !((dc.pk[i][2] + dc.pc[i][2]) * A(0) == A(0));
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (t + k * NT < ncells)
        has = has || ((general >> k) & 1u ? !(pfrac[long(gi[k]) * P + 2] == typename F::T(0))
                                          : ((phase >> (2 * k)) & 3u) == 2u);
    return __syncthreads_or(has) != 0;
  };
  // the sub-steps, with up to G listed cells per thread and PH phases (those behind are absent)
  auto run = [&](auto entries, auto phases) {
    constexpr int G = decltype(entries)::value, PH = decltype(phases)::value;
    A w[G][NF * PH], t1[G][PH], t2[G][PH], cp[G][PH], sc[G];
    int sdepth[G];
    // saddr: a neighbour's partition in L by face and phase, two places per word.  A bulk neighbour's
    // is its value for the phase it has and 0 for the others (0 * (value - c) would be NaN once the
    // value overflows).
    static_assert(PH * NF % 2 == 0, "two places per word");
    uint32_t saddr[G][NF * PH / 2], sgi[G], present = 0;
    CompCode sq[G];
    // partition_cell of an entry's value (the division by t1 = 1 of a unit cell changes nothing)
    // whether an entry of the wavefront or a neighbour has the third phase (or its D is not finite)
    bool third = true;
    auto partition = [&](int j) {
#pragma unroll
      for (int p = 0; p < PH; ++p) {
        if (p == 2 && !third) continue;
        const A v = (sc[j] - t2[j][p]) / t1[j][p];
        cp[j][p] = ((present >> (j * PH + p)) & 1u) ? v : A(0);
      }
    };
    bool has = false;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int slot = t + j * NT;
      sdepth[j] = -1;
      sq[j] = 0;
      sgi[j] = 0;
      sc[j] = A(0);
#pragma unroll
      for (int q = 0; q < NF * PH / 2; ++q) saddr[j][q] = 0;
#pragma unroll
      for (int p = 0; p < PH; ++p) {
        t1[j][p] = A(1);
        t2[j][p] = cp[j][p] = A(0);
      }
#pragma unroll
      for (int q = 0; q < NF * PH; ++q) w[j][q] = A(0);
      if (slot < ng) {
        const int idx = list[slot];
        Cell o;
        locate(idx, o);
        sdepth[j] = o.depth;
        sgi[j] = o.g;
        A ph[PH], phn[NF][PH];
#pragma unroll
        for (int p = 0; p < PH; ++p) ph[p] = A(pfrac[long(o.g) * P + p]);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int p = 0; p < PH; ++p) phn[f][p] = A(pfrac[long(o.gn[f]) * P + p]);
        if constexpr (PH == 3) {
          has = has || !(ph[2] == A(0));
#pragma unroll
          for (int f = 0; f < NF; ++f) has = has || !(phn[f][2] == A(0));
        }
        // (a cell of the outermost layer is never updated; only its partition is read)
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const int nidx = o.depth > 0 ? idx + o.off[f] : idx;
          const uint32_t s2 = slot_of[nidx];
#pragma unroll
          for (int p = 0; p < PH; ++p) {
            const uint32_t a = s2 != 0xffffu      ? uint32_t(CELLS) + s2 * uint32_t(PH) + uint32_t(p)
                               : phn[f][p] > A(0) ? uint32_t(nidx)
                                                  : uint32_t(NONE);
            const int q = f * PH + p;
            saddr[j][q >> 1] |= a << (16 * (q & 1));
          }
        }
#pragma unroll
        for (int i = 0; i < PH; ++i) {
          if (ph[i] > A(0)) present |= 1u << (j * PH + i);
          A a = ph[0] * dc.pk[i][0], c = ph[0] * dc.pc[i][0];
#pragma unroll
          for (int q = 1; q < PH; ++q) {
            a += ph[q] * dc.pk[i][q];
            c += ph[q] * dc.pc[i][q];
          }
          t1[j][i] = a;
          t2[j][i] = c;
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int p = 0; p < PH; ++p) w[j][f * PH + p] = face_weight<A>(phn[f][p] * ph[p]);
        if constexpr (F::kMixed) sq[j] = comp_unpack(codes[idx]);
        sc[j] = L[idx];
        partition(j);
#pragma unroll
        for (int p = 0; p < PH; ++p) L[CELLS + slot * PH + p] = cp[j][p];
      }
    }
    if constexpr (PH == 3) third = __any(has) || !(dc.D[2] * A(0) == A(0));
    __syncthreads();
    const int waves_first = t & ~63;  // entries of this wavefront: waves_first + j * NT and on
    for (int s = 1; s <= S; ++s) {
      const uint32_t key = key_of(s);
      bulk_step(s, key);
#pragma unroll
      for (int j = 0; j < G; ++j) {
        if (waves_first + j * NT >= ng) break;  // wave-uniform
        DelAcc<F, PH> acc;
        if constexpr (SELF_Z) acc.s[0] = self_z(cp[j]);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int p = 0; p < PH; ++p) {
            if (p == 2 && !third) continue;  // 0 * (0 - 0)
            const int q = f * PH + p;
            const uint32_t a = (saddr[j][q >> 1] >> (16 * (q & 1))) & 0xffffu;
            const A term = w[j][q] * (L[a] - cp[j][p]);
            if (f == 0) acc.first(p, term, dc);
            else acc.add(p, term, dc);
          }
        const A del = acc.result(dc);
        A v;
        CompCode qo = 0;
        if constexpr (F::kMixed) v = mixed_step(sc[j], del, sq[j], comp_hash(sgi[j], key), qo);
        else v = sc[j] + del;
        if (sdepth[j] >= s) {
          sc[j] = v;
          if constexpr (F::kMixed) sq[j] = qo;
        }
        partition(j);
      }
      __syncthreads();
      bulk_write(s);
#pragma unroll
      for (int j = 0; j < G; ++j)
        if (sdepth[j] >= s) {
          const int slot = t + j * NT;
          L[list[slot]] = sc[j];
#pragma unroll
          for (int p = 0; p < PH; ++p) L[CELLS + slot * PH + p] = cp[j][p];
        }
      __syncthreads();
    }
    if constexpr (F::kMixed) {
#pragma unroll
      for (int j = 0; j < G; ++j)
        if (sdepth[j] > 0) codes[list[t + j * NT]] = uint8_t(uint32_t(sq[j]) & 15u);
    }
  };
  using std::integral_constant;
  if (__builtin_expect(ng <= NT, 1)) {
    run(integral_constant<int, 1>(), integral_constant<int, P>());
  } else if (P == 2 || !third_phase()) {
    run(integral_constant<int, V>(), integral_constant<int, 2>());
  } else if constexpr (P == 3) {
    // two entries of three phases do not fit the registers: the full formula from memory, the new
    // values kept behind the cells until every thread has read
    for (int s = 1; s <= S; ++s) {
      const uint32_t key = key_of(s);
      bulk_step(s, key);
      for (int i = t; i < ng; i += NT) {
        const int idx = list[i];
        Cell o;
        locate(idx, o);
        A v = L[idx];
        if (o.depth >= s) {
          StencilLoad<F, P, NF> st;
          st.me.c = typename F::C(v);
#pragma unroll
          for (int p = 0; p < P; ++p) st.me.ph[p] = pfrac[long(o.g) * P + p];
          A z = A(0);
          if constexpr (SELF_Z) {  // (before the neighbours are loaded: registers)
            CellPF<A> me;
            partition_cell<F, P>(st.me, dc, me);
            z = self_z(me.c);
            asm volatile("" : "+v"(z));
          }
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            st.nb[f].c = typename F::C(L[idx + o.off[f]]);
#pragma unroll
            for (int p = 0; p < P; ++p) st.nb[f].ph[p] = pfrac[long(o.gn[f]) * P + p];
          }
          A del = stencil_del<F, P, NF>(st, dc);
          if constexpr (SELF_Z) del += z;
          if constexpr (F::kMixed) {
            CompCode qo;
            v = mixed_step(v, del, comp_unpack(codes[idx]), comp_hash(o.g, key), qo);
            codes[idx] = uint8_t(uint32_t(qo) & 15u);
          } else {
            v = v + del;
          }
        }
        L[CELLS + i] = v;
      }
      __syncthreads();
      bulk_write(s);
      for (int i = t; i < ng; i += NT) L[list[i]] = L[CELLS + i];
      __syncthreads();
    }
  }

#pragma unroll
  for (int k = 0; k < V; ++k)
    if ((inside >> k) & 1u) cout[gi[k]] = typename F::C(L[t + k * NT]);
  if constexpr (F::kMixed) {
    // the codes, two cells per byte: a byte whose two cells are this tile's is stored, a byte that it
    // shares with another tile takes its own half by an atomic
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (((inside & ~general) >> k) & 1u) codes[t + k * NT] = uint8_t((qs >> (4 * k)) & 15u);
    __syncthreads();
    const int half = ibx / 2 + 1, items = half * iby;
    uint8_t *cb = comp_bytes(cout, ncell);
    for (int i = t; i < items; i += NT) {
      const int r = i / half, m = i - r * half;
      const long g0 = long(plane0) + ix0 + long(nx) * (iy0 + r);
      const long c0 = (g0 & ~1L) + 2 * m;  // the byte's first cell
      const int l0 = S + int(c0 - g0) + X * (S + r);
      const bool lo = c0 >= g0 && c0 < g0 + ibx, hi = c0 + 1 >= g0 && c0 + 1 < g0 + ibx;
      if (lo && hi)
        cb[c0 >> 1] = uint8_t(codes[l0] | (codes[l0 + 1] << 4));
      else if (lo)
        comp_put_atomic(cout, ncell, c0, CompCode(codes[l0]));
      else if (hi)
        comp_put_atomic(cout, ncell, c0 + 1, CompCode(codes[l0 + 1]));
    }
  }
}

#define PF_INST_TILE(F, P, SELF_Z)                                                              \
  template __global__ void diffuse_tile_kernel<F, P, SELF_Z>(                                   \
      const F::C *, F::C *, const F::T *, const uint8_t *, const DiffConsts<F::A>, TileGeom,     \
      long, uint32_t, int);
PF_INST_TILE(FormF64, 2, false)
PF_INST_TILE(FormF64, 3, false)
PF_INST_TILE(FormF64, 3, true)
PF_INST_TILE(FormMixed, 2, false)
PF_INST_TILE(FormMixed, 3, false)

}  // namespace pfamd
