// pf_diffuse_direct_impl.h — the bulk part of the one-launch sub-step kernels (pf_diffuse_direct.hip, and
// the reverse sub-step of pf_adjoint.hip, which is the same update of the adjoint).
#pragma once
#include "pf_diffuse_direct.h"

namespace pfamd {

template <class A, int V> struct Run {  // V consecutive values at any alignment of A
  A v[V];
};
template <class A, int V> __device__ inline Run<A, V> load_run(const A *p) {
  Run<A, V> r;
  if constexpr (V == 1) {
    r.v[0] = p[0];
  } else {
    const VecA<A, V> x = *reinterpret_cast<const VecA<A, V> *>(p);
#pragma unroll
    for (int k = 0; k < V; ++k) r.v[k] = x.v[k];
  }
  return r;
}
// two bits per cell (general_count_kernel's `packed`): the V cells from cell i on, i % V == 0
template <int V> __device__ inline uint32_t load_flags(const uint32_t *packed, uint32_t i) {
  return (packed[i >> 4] >> (2 * (i & 15u))) & ((1u << (2 * V)) - 1u);
}
// the diffusivity of flag f (1-based phase)
template <class A, int P> __device__ inline A phase_d(const DiffConsts<A> &dc, uint32_t f) {
  A d = dc.D[0];
#pragma unroll
  for (int p = 1; p < P; ++p)
    if (f == uint32_t(p + 1)) d = dc.D[p];
  return d;
}

// The bulk cells of workgroup bb of geo.nbulk (256 threads).
template <class F, int P, bool NOFLUX, int V, int U>
__device__ inline void direct_bulk(const typename F::C *__restrict__ cin,
                                   typename F::C *__restrict__ cout,
                                   const uint32_t *__restrict__ packed,
                                   const DiffConsts<typename F::A> &dc, const DirectGeom &geo,
                                   const int bb) {
  using A = typename F::A;
  using C = typename F::C;
  const int nx = geo.nx, ny = geo.ny, nz = geo.nz;
  const uint32_t plane = uint32_t(nx) * uint32_t(ny);
  const long n = long(plane) * nz;
  // The bulk cells: workgroup b runs on XCD b % 8 (the grid's list part shifts that for all alike), and
  // each XCD takes a contiguous range of the runs (x fastest, then y, then chunks of U planes).
  const int nb = geo.nbulk;
  const int per = nb >> 3, rem = nb & 7, xcd = bb & 7;
  const int mine = per + (xcd < rem ? 1 : 0), at = geo.flip ? mine - 1 - (bb >> 3) : bb >> 3;
  const uint32_t q = uint32_t(xcd * per + (xcd < rem ? xcd : rem) + at) * 256u + threadIdx.x;
  if constexpr (F::kMixed && V == 1) {
    // rows of odd length: a byte pair may cross a row's end, so a thread owns one pair in storage
    // order and looks up each cell's neighbours
    const uint32_t i0 = 2 * q, un = uint32_t(n);
    if (i0 >= un) return;
    const bool two = i0 + 1 < un;
    const uint32_t i1 = two ? i0 + 1 : i0;
    const uint32_t row = geo.row.quot(i0);
    int x[2], y[2], z[2];
    x[0] = int(i0 - row * geo.row.d);
    z[0] = int(geo.rows.quot(row));
    y[0] = int(row - uint32_t(z[0]) * geo.rows.d);
    x[1] = x[0] + (two ? 1 : 0);
    y[1] = y[0];
    z[1] = z[0];
    if (x[1] == nx) {
      x[1] = 0;
      if (++y[1] == ny) {
        y[1] = 0;
        ++z[1];
      }
    }
    const uint32_t ux = uint32_t(nx);
    float v[2][7];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t i = k ? i1 : i0;
      v[k][6] = cin[i];
      v[k][0] = cin[x[k] == 0 ? i + ux - 1u : i - 1u];
      v[k][1] = cin[x[k] == nx - 1 ? i + 1u - ux : i + 1u];
      v[k][2] = cin[y[k] == 0 ? i + plane - ux : i - ux];
      v[k][3] = cin[y[k] == ny - 1 ? i + ux - plane : i + ux];
      v[k][4] = cin[z[k] == 0 ? (NOFLUX ? i : i + un - plane) : i - plane];
      v[k][5] = cin[z[k] == nz - 1 ? (NOFLUX ? i : i + plane - un) : i + plane];
    }
    const uint32_t f = load_flags<2>(packed, i0);
    const uint32_t f0 = f & 3u, f1 = two ? f >> 2 : f0;
    const uint32_t cw = comp_bytes(cin, n)[q];
    if (f0 == 0 || f1 == 0) return;
    uint32_t w = 0;
    float o[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float Dp = phase_d<float, P>(dc, k ? f1 : f0);
      BulkAcc<F> acc;
      acc.first(v[k][0] - v[k][6], Dp);
#pragma unroll
      for (int e = 1; e < 6; ++e) acc.add(v[k][e] - v[k][6], Dp);
      CompCode qo;
      o[k] = mixed_step(v[k][6], acc.result(dc.r, Dp * dc.r), comp_unpack(cw >> (4 * k)),
                        comp_hash(i0 + uint32_t(k), dc.key), qo);
      w |= (uint32_t(qo) & 15u) << (4 * k);
    }
    cout[i0] = o[0];
    if (two) cout[i1] = o[1];
    comp_bytes(cout, n)[q] = uint8_t(two ? w : w & 15u);
    return;
  } else {
  const uint32_t row = geo.row.quot(q);
  const int x0 = int(q - row * geo.row.d) * V;
  const int zc = int(geo.rows.quot(row));
  const int y = int(row - uint32_t(zc) * geo.rows.d);
  const int z0 = zc * U;
  if (z0 >= nz) return;
  const int nv = min(U, nz - z0);
  const uint32_t oc = uint32_t(x0) + uint32_t(nx) * uint32_t(y);
  const uint32_t oym = y == 0 ? oc + plane - uint32_t(nx) : oc - uint32_t(nx);
  const uint32_t oyp = y == ny - 1 ? oc + uint32_t(nx) - plane : oc + uint32_t(nx);
  const uint32_t oxm = x0 == 0 ? oc + uint32_t(nx) - 1u : oc - 1u;
  const uint32_t oxp = x0 + V >= nx ? oc - uint32_t(x0) : oc + uint32_t(V);
  const int zm = z0 == 0 ? (NOFLUX ? 0 : nz - 1) : z0 - 1;
  const int zl = z0 + nv - 1;
  const int zp = zl == nz - 1 ? (NOFLUX ? zl : 0) : zl + 1;
  Run<C, V> c[U], ym[U], yp[U];
  C xm[U], xp[U];
  uint32_t fl[U], cw[U];
  const Run<C, V> lo = load_run<C, V>(cin + long(plane) * zm + oc);
  const Run<C, V> hi = load_run<C, V>(cin + long(plane) * zp + oc);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const long base = long(plane) * min(z0 + u, zl);
    const C *pl = cin + base;
    fl[u] = load_flags<V>(packed, uint32_t(base) + oc);
    c[u] = load_run<C, V>(pl + oc);
    ym[u] = load_run<C, V>(pl + oym);
    yp[u] = load_run<C, V>(pl + oyp);
    xm[u] = pl[oxm];
    xp[u] = pl[oxp];
    if constexpr (F::kMixed) {
      const uint8_t *cb = comp_bytes(cin, n) + ((base + oc) >> 1);
      if constexpr (V == 4) cw[u] = *reinterpret_cast<const uint16_t *>(cb);
      else cw[u] = *cb;
    }
  }
  // differences along z and along x are shared by the two cells they separate: a - b == -(b - a)
  A dz[V];
#pragma unroll
  for (int v = 0; v < V; ++v) dz[v] = A(c[0].v[v]) - A(lo.v[v]);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (u >= nv) break;
    A o[V];
    uint32_t w = 0;
    const uint32_t i0 = plane * uint32_t(z0 + u) + oc;
    A dx = A(c[u].v[0]) - A(xm[u]);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const A Dp = phase_d<A, P>(dc, (fl[u] >> (2 * v)) & 3u);
      const A m = A(c[u].v[v]);
      BulkAcc<F> acc;
      acc.first(-dx, Dp);
      dx = (v == V - 1 ? A(xp[u]) : A(c[u].v[v + 1 < V ? v + 1 : v])) - m;
      acc.add(dx, Dp);
      acc.add(A(ym[u].v[v]) - m, Dp);
      acc.add(A(yp[u].v[v]) - m, Dp);
      acc.add(-dz[v], Dp);
      dz[v] = A(u == nv - 1 ? hi.v[v] : c[u + 1 < U ? u + 1 : u].v[v]) - m;
      acc.add(dz[v], Dp);
      const A del = acc.result(dc.r, Dp * dc.r);
      if constexpr (F::kMixed) {
        CompCode qo;
        o[v] = mixed_step(m, del, comp_unpack(cw[u] >> (4 * v)), comp_hash(i0 + uint32_t(v), dc.key), qo);
        w |= (uint32_t(qo) & 15u) << (4 * v);
      } else {
        o[v] = m + del;
      }
    }
    C *dst = cout + long(i0);
    if constexpr (F::kMixed) {
      // a byte pair holding a listed cell belongs to the listed part
      uint8_t *cb = comp_bytes(cout, n) + (i0 >> 1);
      const bool a = (fl[u] & 3u) != 0 && (fl[u] & 12u) != 0;
      if constexpr (V == 4) {
        const bool d = (fl[u] & 0x30u) != 0 && (fl[u] & 0xc0u) != 0;
        if (a && d) {
          VecA<A, 4> t;
#pragma unroll
          for (int v = 0; v < 4; ++v) t.v[v] = o[v];
          *reinterpret_cast<VecA<A, 4> *>(dst) = t;
          *reinterpret_cast<uint16_t *>(cb) = uint16_t(w);
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if (h == 0 ? a : d) {
              dst[2 * h] = o[2 * h];
              dst[2 * h + 1] = o[2 * h + 1];
              cb[h] = uint8_t(w >> (8 * h));
            }
        }
      } else if (a) {
        VecA<A, 2> t;
        t.v[0] = o[0];
        t.v[1] = o[1];
        *reinterpret_cast<VecA<A, 2> *>(dst) = t;
        *cb = uint8_t(w);
      }
    } else if constexpr (V == 2) {
      if ((fl[u] & 3u) != 0 && (fl[u] & 12u) != 0) {
        VecA<A, 2> t;
        t.v[0] = o[0];
        t.v[1] = o[1];
        *reinterpret_cast<VecA<A, 2> *>(dst) = t;
      } else {
        if (fl[u] & 3u) dst[0] = o[0];
        if (fl[u] & 12u) dst[1] = o[1];
      }
    } else {
      if (fl[u]) dst[0] = o[0];
    }
  }
  }
}

}  // namespace pfamd
