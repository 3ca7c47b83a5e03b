// Device helpers of the kernels that update four consecutive z cells (a quad) per lane: the forward,
// batch and reverse sweeps of fwd_kernels.hip and the adjoint passes of adj_kernels.hip. Every field
// array moves as dwordx4, the z neighbours inside a quad come from the lane's own registers. Per cell the
// arithmetic is that of the one-cell sweeps, in the same order, so results are bit-identical.
//
// Rows of nz cells with nz not a multiple of 4 (RAG): the row's last quad starts at nz - 4 and so
// repeats up to 3 cells of the quad before it, the `sm` leading cells that its lane leaves out of its
// stores. Of the arrays a sweep writes the lane may read these cells before or after the other lane has
// stored them, so their values are unspecified: nothing computed from them may reach a cell that the lane
// stores, nor a record, a snapshot of a written field or the state of a pole. (A sweep reads only a lane's own
// cells of the arrays it writes, so kept cells never depend on them.) Accesses are then aligned to
// 4 bytes only, which global dwordx4 accesses allow.
#pragma once
#include "engine_common.h"
#include "stencil.h"

namespace fdtdx {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

template <bool RAG = false>
__device__ __forceinline__ f4v ld4(const float* p) {
  if constexpr (RAG) return *reinterpret_cast<const f4u*>(p);
  else return *reinterpret_cast<const f4v*>(p);
}

__device__ __forceinline__ void st4(float* p, f4v v) { *reinterpret_cast<f4v*>(p) = v; }

// Store of the cells e >= sm of a quad.
template <bool RAG>
__device__ __forceinline__ void st4m(float* p, f4v v, int sm) {
  if constexpr (!RAG) {
    st4(p, v);
  } else if (sm == 0) {
    *reinterpret_cast<f4u*>(p) = v;
  } else {
#pragma unroll
    for (int e = 1; e < 4; ++e)
      if (e >= sm) p[e] = v[e];
  }
}

constexpr uint32_t kSlabBits = (1u << FDTDX_MAX_CPML) - 1u;
constexpr uint32_t kAdeBits = ((1u << FDTDX_MAX_ADE) - 1u) << kMaskAde;
constexpr uint32_t kSnapBit = 1u << kMaskSnap;

// Quad of this lane in quad tile lb: cells (i, j, k0 .. k0 + 3) at offsets o .. o + 3, the first sm
// of which it leaves out of its stores.
__device__ __forceinline__ bool quad_of(const StepStatic& P, long long lb, int& i, int& j, int& k0, int& sm,
                                        long long& o) {
  if (lb >= P.vnblocks) return false;
  i = (int)(lb / P.vbpp);
  const int p = (int)(lb - (long long)i * P.vbpp) * kBlock + threadIdx.x;
  if (p >= P.ny * P.nzq) return false;
  perm_quad(P, p, j, k0, sm);
  o = (long long)i * P.plane + (long long)j * P.nz + k0;
  return true;
}

// One-sided derivatives of the four cells of a quad, one vector per (axis, component) pair that
// feeds a CPML slab: curl H uses (dx Hz, dx Hy), (dy Hx, dy Hz), (dz Hy, dz Hx), curl E the same
// pairs of E (the order of pml_pair).
struct QuadDeriv {
  f4v x1, x2, y1, y2, z1, z2;
};

// Per-axis CPML of a quad (StepStatic::cax): the quad meets at most one slab per axis, the x slab
// fixed by i, the y slab by j and the z slab by k0 (a quad across a z-slab edge updates the cells
// inside the slab one by one). Every psi load is issued before any is used (quad_slab_loads, ahead
// of the field loads), then the corrections are added x, y, z, i.e. in slab order (quad_slab_apply)
// with cpml_slab's arithmetic. Descriptor fields are read for both sides of an axis (wave-uniform)
// and selected per lane.
struct QuadSlabs {
  bool in[3], hi[3];  // the quad meets the axis's slab; of its max side
  unsigned zm;        // cells of the quad inside its z slab (bit e: cell k0 + e)
  f4v p1[3], p2[3];   // psi1, psi2 of the quad in that slab (zero for cells outside it)
};

// Descriptor fields of the slab of one side of axis AX (wave-uniform), and the float offset of psi1
// of cell (i, j, k0) in it (for the z axis k0 - lo may be negative or reach past the slab when the
// quad straddles a slab edge; only the cells inside are addressed).
template <int W, int AX>
__device__ __forceinline__ long long quad_psi_offset(const StepStatic& P, bool hi, int i, int j, int k0, int& dep,
                                                     long long& cells, const float*& cf, int& L, int& kap,
                                                     int& aligned) {
  const StepStatic::AxSlab& A = P.axd[AX][0];
  const StepStatic::AxSlab& B = P.axd[AX][1];
  const int lo = side_of(hi, B.lo, A.lo);
  L = side_of(hi, B.L, A.L);
  cells = side_of(hi, B.cells, A.cells);
  cf = side_of(hi, B.coef, A.coef) + (W ? 3 * L : 0);
  kap = side_of(hi, B.kappa_one, A.kappa_one);
  aligned = side_of(hi, B.aligned, A.aligned);
  dep = (AX == 0 ? i : (AX == 1 ? j : k0)) - lo;
  const long long base = side_of(hi, B.psi_off, A.psi_off) + (W ? 2 * cells : 0);
  if (AX == 0) return base + (long long)dep * P.plane + (long long)j * P.nz + k0;
  if (AX == 1) return base + ((long long)i * L + dep) * P.nz + k0;
  return base + ((long long)i * P.ny + j) * L + dep;
}

template <int W, int AX, bool RAG>
__device__ __forceinline__ void quad_slab_load(const StepStatic& P, const float* psi, int i, int j, int k0,
                                               QuadSlabs& S) {
  const StepStatic::AxSlab& A = P.axd[AX][0];
  const StepStatic::AxSlab& B = P.axd[AX][1];
  if (AX == 2) {  // a quad may straddle a z-slab edge (the plan keeps it off the other slab)
    S.hi[AX] = k0 + 3 >= B.lo && B.lo < B.hi;
    S.in[AX] = S.hi[AX] || k0 < A.hi;
    if (!S.in[AX]) return;
    const int lo = side_of(S.hi[AX], B.lo, A.lo), hi = side_of(S.hi[AX], B.hi, A.hi);
    S.zm = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) S.zm |= (k0 + e >= lo && k0 + e < hi) ? (1u << e) : 0u;
  } else {
    const int c = AX == 0 ? i : j;
    S.hi[AX] = c >= B.lo && c < B.hi;
    S.in[AX] = S.hi[AX] || (c >= A.lo && c < A.hi);
    if (!S.in[AX]) return;
  }
  int dep, L, kap, aligned;
  long long cells;
  const float* cf;
  const long long q = quad_psi_offset<W, AX>(P, S.hi[AX], i, j, k0, dep, cells, cf, L, kap, aligned);
  if (AX != 2 || (S.zm == 15u && (RAG || aligned))) {
    S.p1[AX] = ld4<RAG>(psi + q);
    S.p2[AX] = ld4<RAG>(psi + q + cells);
  } else {
    f4v a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if ((S.zm >> e) & 1u) {
        a[e] = psi[q + e];
        b[e] = psi[q + e + cells];
      }
    S.p1[AX] = a;
    S.p2[AX] = b;
  }
}

template <int W, bool RAG>
__device__ __forceinline__ void quad_slab_loads(const StepStatic& P, const float* psi, int i, int j, int k0,
                                                QuadSlabs& S) {
  quad_slab_load<W, 0, RAG>(P, psi, i, j, k0, S);
  quad_slab_load<W, 1, RAG>(P, psi, i, j, k0, S);
  quad_slab_load<W, 2, RAG>(P, psi, i, j, k0, S);
}

// Writes the advanced psi of the cells e >= sm to psi_out.
template <int W, int AX, bool RAG>
__device__ __forceinline__ void quad_slab_axis(const StepStatic& P, const QuadSlabs& S, float* psi_out, int i, int j,
                                               int k0, int sm, const QuadDeriv& d, f4v& cx, f4v& cy, f4v& cz) {
  if (!S.in[AX]) return;
  int dep, L, kap, aligned;
  long long cells;
  const float* cf;
  const long long q = quad_psi_offset<W, AX>(P, S.hi[AX], i, j, k0, dep, cells, cf, L, kap, aligned);
  const bool whole = AX != 2 || S.zm == 15u;
  // depths of the four cells (z: clamped into the slab for the cells outside it)
  int de[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) de[e] = AX != 2 ? dep : (dep + e < 0 ? 0 : (dep + e >= L ? L - 1 : dep + e));
  // z slabs with edges on quad boundaries: the quad's four depths are dep .. dep + 3 with dep and L
  // multiples of 4, so each coefficient vector is one aligned dwordx4 (unaligned rows: any whole quad)
  const bool zvec = AX == 2 && whole && (RAG || aligned);
  f4v b, a;
  if (zvec) {
    b = ld4<RAG>(cf + dep);
    a = ld4<RAG>(cf + L + dep);
  } else if (AX == 2) {
    b = f4v{cf[de[0]], cf[de[1]], cf[de[2]], cf[de[3]]};
    a = f4v{cf[L + de[0]], cf[L + de[1]], cf[L + de[2]], cf[L + de[3]]};
  } else {
    const float bv = cf[dep], av = cf[L + dep];
    b = f4v{bv, bv, bv, bv};
    a = f4v{av, av, av, av};
  }
  const f4v d1 = AX == 0 ? d.x1 : (AX == 1 ? d.y1 : d.z1);
  const f4v d2 = AX == 0 ? d.x2 : (AX == 1 ? d.y2 : d.z2);
  const f4v n1 = b * S.p1[AX] + a * d1;
  const f4v n2 = b * S.p2[AX] + a * d2;
  f4v r1 = n1, r2 = n2;
  if (!kap) {  // 1/kappa - 1
    const float* km = cf + 2 * L;
    f4v k;
    if (zvec) k = ld4<RAG>(km + dep);
    else k = f4v{km[de[0]], km[de[1]], km[de[2]], km[de[3]]};
    r1 = k * d1 + n1;
    r2 = k * d2 + n2;
  }
  if (AX != 2 || zvec) {
    st4m<RAG>(psi_out + q, n1, sm);
    st4m<RAG>(psi_out + q + cells, n2, sm);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!((S.zm >> e) & 1u)) {  // outside the slab: no correction (an exact zero)
        r1[e] = 0.f;
        r2[e] = 0.f;
        continue;
      }
      if (e >= sm) {
        psi_out[q + e] = n1[e];
        psi_out[q + e + cells] = n2[e];
      }
    }
  }
  // curl[(a+1)%3] += -corr1, curl[(a+2)%3] += corr2
  if (AX == 0) {
    cy = cy + (-r1);
    cz = cz + r2;
  } else if (AX == 1) {
    cz = cz + (-r1);
    cx = cx + r2;
  } else {
    cx = cx + (-r1);
    cy = cy + r2;
  }
}

template <int W, bool RAG>
__device__ __forceinline__ void quad_slab_apply(const StepStatic& P, const QuadSlabs& S, float* psi_out, int i, int j,
                                                int k0, int sm, const QuadDeriv& d, f4v& cx, f4v& cy, f4v& cz) {
  quad_slab_axis<W, 0, RAG>(P, S, psi_out, i, j, k0, sm, d, cx, cy, cz);
  quad_slab_axis<W, 1, RAG>(P, S, psi_out, i, j, k0, sm, d, cx, cy, cz);
  quad_slab_axis<W, 2, RAG>(P, S, psi_out, i, j, k0, sm, d, cx, cy, cz);
}

// The correction with psi frozen (the reverse run, PML.py:181-182) of the preloaded slabs, x, y, z.
template <int W, int AX, bool RAG>
__device__ __forceinline__ void quad_frozen_axis(const StepStatic& P, const QuadSlabs& S, int i, int j, int k0,
                                                 const QuadDeriv& d, f4v& cx, f4v& cy, f4v& cz) {
  if (!S.in[AX]) return;
  f4v r1 = S.p1[AX], r2 = S.p2[AX];  // zero for the cells outside a z slab
  int dep, L, kap, aligned;
  long long cells;
  const float* cf;
  quad_psi_offset<W, AX>(P, S.hi[AX], i, j, k0, dep, cells, cf, L, kap, aligned);
  if (!kap) {
    const f4v d1 = AX == 0 ? d.x1 : (AX == 1 ? d.y1 : d.z1);
    const f4v d2 = AX == 0 ? d.x2 : (AX == 1 ? d.y2 : d.z2);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (AX == 2 && !((S.zm >> e) & 1u)) continue;
      const float km = cf[2 * L + (AX == 2 ? dep + e : dep)];
      r1[e] = km * d1[e] + r1[e];
      r2[e] = km * d2[e] + r2[e];
    }
  }
  if (AX == 0) {
    cy = cy + (-r1);
    cz = cz + r2;
  } else if (AX == 1) {
    cz = cz + (-r1);
    cx = cx + r2;
  } else {
    cx = cx + (-r1);
    cy = cy + r2;
  }
}

template <int W, bool RAG>
__device__ __forceinline__ void quad_slab_frozen(const StepStatic& P, const QuadSlabs& S, int i, int j, int k0,
                                                 const QuadDeriv& d, f4v& cx, f4v& cy, f4v& cz) {
  quad_frozen_axis<W, 0, RAG>(P, S, i, j, k0, d, cx, cy, cz);
  quad_frozen_axis<W, 1, RAG>(P, S, i, j, k0, d, cx, cy, cz);
  quad_frozen_axis<W, 2, RAG>(P, S, i, j, k0, d, cx, cy, cz);
}

// The cells [a0, a1) of a quad, as one access where that is all of it.
__device__ __forceinline__ f4v ld4p(const float* p, int a0, int a1) {
  if (a1 - a0 == 4) return ld4<true>(p);
  f4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (e >= a0 && e < a1) v[e] = p[e];
  return v;
}

__device__ __forceinline__ void st4p(float* p, f4v v, int a0, int a1) {
  if (a1 - a0 == 4) {
    *reinterpret_cast<f4u*>(p) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (e >= a0 && e < a1) p[e] = v[e];
}

// Conductivity of a quad (loss_x and the update of update_E_cell / update_H_cell): f the field before
// the step, t = (c curl) inv, n the lossless result, replaced for the cells inside the box.
template <int W>
__device__ __forceinline__ void quad_loss(const StepStatic& P, int i, int j, int k0, const f4v* inv, const f4v* f,
                                          const f4v* t, f4v* n) {
  const LossK& L = P.loss[W];
  if (i < L.lo[0] || i >= L.hi[0] || j < L.lo[1] || j >= L.hi[1] || k0 + 3 < L.lo[2] || k0 >= L.hi[2]) return;
  const long long q = ((long long)(i - L.lo[0]) * L.by + (j - L.lo[1])) * L.bz + (k0 - L.lo[2]);
  // cells outside the box: zero conductivity, which leaves n as it is
  const int a0 = max(0, L.lo[2] - k0), a1 = min(4, L.hi[2] - k0);
  const f4v c = {P.c, P.c, P.c, P.c}, one = {1.f, 1.f, 1.f, 1.f};
  f4v sg;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (a == 0 || L.comps == 3) sg = ld4p(L.sig + a * L.cells + q, a0, a1);
    f4v x = (W == 0 ? ((c * sg) * P.eta0) * inv[a] : ((c * sg) / P.eta0) * inv[a]) / 2.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = e >= a0 && e < a1 ? x[e] : 0.f;  // also where inv is not finite
    const f4v g = (one - x) * f[a];
    n[a] = (W == 0 ? g + t[a] : g - t[a]) / (one + x);
  }
}

// Lorentz and Drude poles of a quad (the recurrence of update_E_cell): en += ie sum_p (P^n - P_hat) for
// the cells e >= sm inside each box; eo is E^n. ie (at the quad) is read again here: few quads have
// poles, and twelve registers held for them would cost every other quad a wave. Box edges and widths
// have no alignment, so whole quads move with 4-byte aligned accesses.
template <int EC>
__device__ __forceinline__ void quad_ade(const StepStatic& P, float* ade, const float* ie, uint32_t m, int n, int i,
                                         int j, int k0, int sm, const f4v* eo, f4v* en) {
#pragma unroll 1
  for (uint32_t mm = (m >> kMaskAde) & ((1u << P.nade) - 1u); mm; mm &= mm - 1u) {
    const AdeK& A = P.ade[__builtin_ctz(mm)];
    if (i < A.lo[0] || i >= A.hi[0] || j < A.lo[1] || j >= A.hi[1]) continue;
    const int a0 = max(sm, A.lo[2] - k0), a1 = min(4, A.hi[2] - k0);
    if (a0 >= a1) continue;
    const long long q = ((long long)(i - A.lo[0]) * A.by + (j - A.lo[1])) * A.bz + (k0 - A.lo[2]);
    // three slots: P^n in slot n%3, P^{n-1} in (n+2)%3, P^{n+1} written to (n+1)%3
    const long long cells = A.cells, slot = (long long)A.poles * 3 * cells;
    const long long coef = (long long)A.poles * A.ccomp * cells;
    const float* cur = ade + A.state_off + (long long)(n % 3) * slot + q;
    const float* prv = ade + A.state_off + (long long)((n + 2) % 3) * slot + q;
    float* nxt = ade + A.state_off + (long long)((n + 1) % 3) * slot + q;
    f4v dl[3];
#pragma unroll 1
    for (int p = 0; p < A.poles; ++p) {
      f4v c1, c2, c3;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (a == 0 || A.ccomp == 3) {
          const float* cf = A.coef + ((long long)p * A.ccomp + a) * cells + q;
          c1 = ld4p(cf, a0, a1);
          c2 = ld4p(cf + coef, a0, a1);
          c3 = ld4p(cf + 2 * coef, a0, a1);
        }
        const long long si = ((long long)p * 3 + a) * cells;
        const f4v pc = ld4p(cur + si, a0, a1), pp = ld4p(prv + si, a0, a1);
        const f4v ph = (c1 * pc + c2 * pp) + c3 * eo[a];
        dl[a] = p == 0 ? pc - ph : dl[a] + (pc - ph);
        st4p(nxt + si, ph, a0, a1);
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const f4v inv = ld4<true>(ie + (EC == 3 ? a * P.N : 0));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e >= a0 && e < a1) en[a][e] = en[a][e] + inv[e] * dl[a][e];
    }
  }
}

// Conducting faces of field W (0: E, PEC; 1: H, PMC) in the updated quad f (apply_walls). In registers
// ahead of the store: a face normal to z meets the end of every row, where reading the stored quad back in
// four rounds cost more than the sweep itself. us per step of a grid between two PEC faces normal
// to z, rounds / here / one cell per lane: 800x800x20 240 / 179 / 190, 400x400x8 26.6 / 20.3 / 21.6,
// 300x300x150 (four faces, y and z) 225 / 207 / 216.
template <int W>
__device__ __forceinline__ void quad_walls(const StepStatic& P, uint32_t m, int i, int j, int k0, f4v* f) {
#pragma unroll 1
  for (uint32_t mm = (m & P.vwall[W]) >> kMaskWall; mm; mm &= mm - 1u) {
    const WallK& w = P.wall[__builtin_ctz(mm)];
    const int d = w.index - (w.axis == 0 ? i : (w.axis == 1 ? j : k0));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool on = w.axis == 2 ? d == e : d == 0;
#pragma unroll
      for (int a = 0; a < 3; ++a) f[a][e] = on && w.axis != a ? 0.f : f[a][e];
    }
  }
}

// Sources of field W (0: E; 1: H) in the updated quad f (source_one, in list order), ahead of quad_walls and
// the store: profile and inverse material move as vectors, inv (at the quad, comps components; null: 1) is
// read again here rather than held. m: the tile's mask. INV: the reverse run's sources (negated),
// added before the half-step is undone. Tiles with sources ran one cell per lane in launches of their own
// at first (6 to 9 us each whatever the grid), then read the quad back after the store in four rounds, the
// end of a launch of one wave of blocks. us per step, launches / rounds / here: two plane waves in 128x120x100
// 60 / 45 / 41; rounds / here: 128x128x64 plane wave 35.1 / 30.6, 301x277x150 236 / 229. Rows of nz % 4 != 0
// cells, one cell per lane / rounds / here: four plane waves in 128x120x99 47 / 54 / 47.5, 141^3 53 / 54.6 / 52.
template <int W, bool INV = false>
__device__ __forceinline__ void quad_sources(const StepStatic& P, uint32_t m, const float* inv, int comps, int n,
                                             int i, int j, int k0, f4v* f) {
#pragma unroll 1
  for (uint32_t mm = (m & P.vpoint[W]) >> kMaskSrc; mm; mm &= mm - 1u) {
    const SrcK& S = P.src[__builtin_ctz(mm)];
    if (i < S.lo[0] || i >= S.hi[0] || j < S.lo[1] || j >= S.hi[1] || k0 + 3 < S.lo[2] || k0 >= S.hi[2]) continue;
    const int a0 = max(0, S.lo[2] - k0), a1 = min(4, S.hi[2] - k0);
    auto add = [&](int c, f4v v) {  // as source_one: zero is added to the other components
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = e >= a0 && e < a1;
#pragma unroll
        for (int a = 0; a < 3; ++a) f[a][e] = in ? f[a][e] + (a == c ? v[e] : 0.f) : f[a][e];
      }
    };
    if (S.kind == FDTDX_SRC_POINT) {
      const float v = INV ? -S.table[n] : S.table[n];
      add(S.comp, f4v{v, v, v, v});
      continue;
    }
    const long long q = ((long long)(i - S.lo[0]) * S.py + (j - S.lo[1])) * S.pz + (k0 - S.lo[2]);
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
      const int tc = S.target[t], sc = S.src[t];
      f4v x = (ld4p(S.profile + sc * S.pcells + q, a0, a1) * S.table[sc * P.T + n]) * P.c;
      if (inv) x = x * ld4<true>(inv + (comps == 3 ? tc : 0) * P.N);
      add(tc, (INV ? -S.sign[t] : S.sign[t]) * x);
    }
  }
}

// collect_interfaces (update.py:1140-1178, fdtd/misc.py:10-35): the float32 E and H of a cell on
// a slab's interface plane into step n's record slot.
__device__ __forceinline__ void record_iface(const StepStatic& P, uint32_t m, char* record, int i, int j, int k,
                                             float ex, float ey, float ez, float hx, float hy, float hz) {
#pragma unroll
  for (int s = 0; s < FDTDX_MAX_CPML; ++s) {
    if (s >= P.nslab) break;
    if (!((m >> s) & 1u)) continue;
    const SlabK& sl = P.slab[s];
    const int coord = sl.axis == 0 ? i : (sl.axis == 1 ? j : k);
    if (coord != sl.iface) continue;
    const long long pc = (long long)sl.pn0 * sl.pn1;
    const long long q = sl.axis == 0 ? (long long)j * P.nz + k : (sl.axis == 1 ? (long long)i * P.nz + k : (long long)i * P.ny + j);
    float* fe = (float*)(record + sl.rec_off_E);
    float* fh = (float*)(record + sl.rec_off_H);
    fe[q] = ex; fe[pc + q] = ey; fe[2 * pc + q] = ez;
    fh[q] = hx; fh[pc + q] = hy; fh[2 * pc + q] = hz;
  }
}

}  // namespace fdtdx
