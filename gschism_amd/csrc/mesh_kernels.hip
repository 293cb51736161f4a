// mesh_kernels.hip -- gfx950 kernels of the per-step mesh work: vertical levels and wet/dry,
// ELM backtracking, RHS producers, wave-equation assembly with essential BCs, elevation update.
//
// Arithmetic follows the reference's operation order term by term (no contraction: the library
// is built with -ffp-contract=off), so the CPU oracle reproduces every result bit for bit.
#include <hip/hip_runtime.h>

#include "device.h"
#include "reduce.h"

namespace gsh {

#define GSH_BT_WALK_CAP 1
#define GSH_BT_ITER38 2
#define GSH_BT_STUCK 4
#define GSH_BT_OPEN_EXIT 8
#define GSH_BT_SLIDE 16

typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr double kSmall = 1.0e-7;  // meshdata.h:10

// Node::compZCoord (meshdata.cu:1744-1807) at level k of a wet node with elevation eta, depth h
// and bottom level kb; sigmaTransitionDepth (:1647) is min(h, h_s). ivcor=2 (SZ: Z levels, the
// level at -min(h, h_s), S levels) and ivcor=1 (one sigma per level, or per node and level).
__device__ __forceinline__ double z_wet(const DMesh& m, int node, double eta, double h, int kb, int k) {
  const int nv = m.nvrt;
  if (m.vmode == 2) {
    const double hmod2 = fmin(h, m.h_s);
    if (k == nv - 1) return eta;
    if (k == m.izlev) return -hmod2;
    if (k == kb) return -h;
    if (k < m.izlev) return m.ztot[k];
    const int ks = k - m.izlev;
    const double sg = m.ssig[ks];
    if (hmod2 <= m.h_c) return sg * (hmod2 + eta) + eta;
    return eta * (1.0 + sg) + m.h_c * sg + (hmod2 - m.h_c) * m.cs[ks];
  }
  if (k <= kb) return -h;
  if (k == nv - 1) return eta;
  const double sg = m.vmode == 1 ? m.sig_node[(int64_t)node * nv + k] : m.sigma[k];
  return (eta + h) * sg + eta;
}

// compZCoord (meshdata.cu:1744-1807): z of level k at a node (0 when the node is dry).
__device__ __forceinline__ double zcoord(const DMesh& m, double h0, int node, int k) {
  const double eta = m.eta2[node], h = m.depth[node];
  if (eta + h <= h0) return 0.0;  // isDry2
  return z_wet(m, node, eta, h, m.kb[node], k);
}

// ---------------------------------------------------------------- packed geometry (mesh creation)
// DMesh::area_inv, side_geo (the side's unit normal as populateSides forms it, meshdata.cu:2283-2287)
// and ball_rec (side c of an element lies opposite its corner c).
__global__ void k_pack_geometry(DMesh m, double2* __restrict__ area_inv, double4* __restrict__ side_geo,
                                int4* __restrict__ ball_rec, int nball) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m.ne) {
    const double a = m.area[i];
    area_inv[i] = make_double2(a, 1.0 / a);
  }
  if (i < m.ns) {
    const int4 sr = m.side[i];
    const double vx = -(m.y[sr.x] - m.y[sr.y]), vy = m.x[sr.x] - m.x[sr.y];
    const double l = sqrt(vx * vx + vy * vy);
    side_geo[i] = make_double4(vx / l, vy / l, m.side_len[i], (double)sr.z);
  }
  if (i < nball) {
    const int e = m.ball_elem[i], l = m.ball_loc[i];
    const int* es = reinterpret_cast<const int*>(m.elem + 2 * (int64_t)e) + 3;
    ball_rec[i] = make_int4(e, es[l], es[l == 2 ? 0 : l + 1], es[l == 0 ? 2 : l - 1]);
  }
}

void launch_pack_geometry(const DMesh& m, double2* area_inv, double4* side_geo, int4* ball_rec, int nball,
                          hipStream_t st) {
  const int count = max(nball, max(m.ne, m.ns));
  hipLaunchKernelGGL(k_pack_geometry, dim3((count + 255) / 256), dim3(256), 0, st, m, area_inv, side_geo, ball_rec,
                     nball);
}

// ---------------------------------------------------------------- a3: levels and wet/dry
// ul0ComputeDryElements (meshdata.cu:5550-5580)
__global__ void k_elem_levels(DMesh m, double h0) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m.ne) return;
  const int4 r = m.elem[2 * e];
  const int nd[3] = {r.x, r.y, r.z};
  bool dry = false;
  for (int j = 0; j < 3; ++j) dry = dry || (m.eta2[nd[j]] + m.depth[nd[j]] <= h0);
  m.elem_wet[e] = dry ? 0 : 1;
  int kb = 0;
  if (!dry) kb = min(min(m.kb[nd[0]], m.kb[nd[1]]), m.kb[nd[2]]);
  m.elem_kb[e] = kb;
}

// ul0ComputeDryNodes (meshdata.cu:5596-5612)
__global__ void k_node_wet(DMesh m) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.n) return;
  int8_t wet = 0;
  for (int j = m.ball_ptr[i]; j < m.ball_ptr[i + 1]; ++j)
    if (m.elem_wet[m.ball_elem[j]]) {
      wet = 1;
      break;
    }
  m.node_wet[i] = wet;
  m.eta_lev[i] = m.eta2[i];
}

// ul0UpdateSides / ul0UpdateSides2 (meshdata.cu:5679-5760): side kb, zc, wet flag. One thread per
// side (g sides per workgroup) computes its levels into LDS (the node values are read once per side); the workgroup then
// stores its sides' zc rows, one contiguous span of HBM, with flat coalesced stores. Dry sides
// keep their zc, as in the reference.
constexpr int kLevelThreads = 128;

__global__ void __launch_bounds__(kLevelThreads) k_side_levels(DMesh m, double h0, int g) {
  extern __shared__ double lz[];  // [g][nv | 1]
  __shared__ int8_t lwet[kLevelThreads];
  const int nv = m.nvrt, zs = nv | 1;
  const int s0 = blockIdx.x * g;
  const int gc = min(g, m.ns - s0);
  const int t = threadIdx.x;
  if (t < gc) {
    const int s = s0 + t;
    const int4 r = m.side[s];
    const bool wet = m.elem_wet[r.z] || (r.w >= 0 && m.elem_wet[r.w]);
    const int kb1 = m.kb[r.x], kb2 = m.kb[r.y];
    const int kb = wet ? min(kb1, kb2) : 0;
    if (wet) {
      double* z = lz + t * zs;
      for (int k = 0; k < kb; ++k) z[k] = 0.0;
      for (int k = kb; k < nv; ++k)
        z[k] = 0.5 * (zcoord(m, h0, r.x, max(k, kb1)) + zcoord(m, h0, r.y, max(k, kb2)));
    }
    lwet[t] = wet ? 1 : 0;
    m.side_kb[s] = kb;
    m.side_wet[s] = wet ? 1 : 0;
  }
  __syncthreads();
  const int total = gc * nv;
  const float inv = 1.0f / (float)nv;
  double* zc = m.zc + (int64_t)s0 * nv;
  for (int i = t; i < total; i += kLevelThreads) {
    // side j = i / nv from a float reciprocal (exact for i < 2^17), corrected either way
    int j = (int)(((float)i + 0.5f) * inv);
    int k = i - j * nv;
    if (k < 0) {
      --j;
      k += nv;
    }
    if (k >= nv) {
      ++j;
      k -= nv;
    }
    if (lwet[j]) zc[i] = lz[j * zs + k];
  }
}

void launch_levels(const DMesh& m, const StepArgs& a, hipStream_t st) {
  if (m.ne > 0) hipLaunchKernelGGL(k_elem_levels, dim3((m.ne + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a.h0);
  if (m.n > 0) hipLaunchKernelGGL(k_node_wet, dim3((m.n + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m);
  if (m.ns > 0) {
    // sides per workgroup: one per thread, at most 32 KB of LDS
    const int g = max(1, min(kLevelThreads, 32 * 1024 / (8 * (m.nvrt | 1))));
    hipLaunchKernelGGL(k_side_levels, dim3((m.ns + g - 1) / g), dim3(kLevelThreads), (size_t)8 * g * (m.nvrt | 1), st,
                       m, a.h0, g);
  }
}

// ---------------------------------------------------------------- a4-a7: ELM backtracking
__device__ __forceinline__ double signed_area(double p1x, double p1y, double p2x, double p2y, double p3x,
                                              double p3y) {
  return 0.5 * ((p1x - p3x) * (p2y - p3y) - (p2x - p3x) * (p1y - p3y));
}

// Node ids and coordinates of one element, as the walk leaves them for the interpolation.
struct ElemGeom {
  int n0, n1, n2;
  int s0, s1, s2;  // sides opposite the corners
  double x0, y0, x1, y1, x2, y2;
};

// Ids are non-negative int32 wherever they index (every -1 is tested first), so the hot gathers
// index with unsigned 32-bit arithmetic (2 id + 1 < 2^32): one address instruction per load.
__device__ __forceinline__ unsigned ux(int i) { return (unsigned)i; }

__device__ __forceinline__ ElemGeom elem_geom(const DMesh& m, int e) {
  const int4 r = m.elem[2u * ux(e)], q = m.elem[2u * ux(e) + 1u];
  const double2 p0 = m.nrec[2u * ux(r.x)], p1 = m.nrec[2u * ux(r.y)], p2 = m.nrec[2u * ux(r.z)];
  return {r.x, r.y, r.z, r.w, q.x, q.y, p0.x, p0.y, p1.x, p1.y, p2.x, p2.y};
}

// A node's elevation, depth, total depth H = eta + h and bottom level, in registers. One sigma per
// level: a dry node's record is (0, 0) (k_pack_nodes), which makes every level 0 as zcoord does.
struct NodeZ {
  double eta, h, H;
  int kb;
};

constexpr int kKbMask = 0xffff;  // DMesh::nkz: kb below, flag above (nvrt <= 1024)

// F: the mesh has kb = 0 at every node and its last sigma is exactly 0 (DMesh::flat).
template <bool F>
__device__ __forceinline__ NodeZ node_z(const DMesh& m, int node) {
  const double2 q = m.nrec[2u * ux(node) + 1u];
  return {q.x, q.y, q.x + q.y, F ? 0 : m.kb[ux(node)]};
}

// a / b with y = 1 / b correctly rounded, correctly rounded as the division is: two Newton
// corrections of a y (Markstein, IBM J. Res. Dev. 34 (1990) 111-119: the second one, from a quotient
// within an ulp, rounds correctly). Five operations instead of the eleven of a division. (A zero
// quotient may differ in its sign; quotients whose remainder underflows are not met: a is an
// element area or a part of one.)
__device__ __forceinline__ double div_by(double a, double b, double y) {
  const double q0 = a * y;
  const double q1 = __builtin_fma(__builtin_fma(-b, q0, a), y, q0);
  return __builtin_fma(__builtin_fma(-b, q1, a), y, q1);
}

// a / 3.0, correctly rounded as the division is, in four operations instead of eleven: a RN(1/3) is
// within an ulp, one Newton correction then rounds correctly (Markstein; its remainder is a multiple
// of the smallest subnormal, so exact at any size), and the fixup gives the division's zeros,
// infinities and NaN.
__device__ __forceinline__ double third(double a) {
  constexpr double y = 1.0 / 3.0;
  const double q = a * y;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-3.0, q, a), y, q), 3.0, a);
}

// LDS-staged element patch (k_backtrack with ST = true): what the walk reads of an element and the
// vertical search of its nodes, for the elements on both sides of each of the workgroup's sides and
// their neighbours, in one record, in an LDS table keyed by element id (open addressing, linear
// probing). The interpolation's area and reciprocal come from DMesh::area_inv, once per element
// entered (BtCell). An element outside the patch is read from global memory as before, so the values
// and results are those of the unstaged kernel.
struct StElem {
  double x[3], y[3];    // corners in node order n0, n1, n2
  double eta[3], h[3];  // eta2 and depth of the corners (VM = 0)
  int n[3], s[3];       // node ids; sides opposite the corners
  int ekb, kb[3];       // element bottom level; the corners' kb
};
constexpr int kStSlots = 128;  // table size (a power of two)
constexpr int kStCand = 96;    // at most this many candidates, so a free slot always ends a probe

__device__ __forceinline__ unsigned st_hash(int e) { return ((unsigned)e * 2654435761u) >> 25; }

// slot of element e, or -1 when it is not staged
__device__ __forceinline__ int st_find(const int* key, int e) {
  unsigned h = st_hash(e);
  for (int p = 0; p < kStSlots; ++p) {
    const int k = key[h];
    if (k == e) return (int)h;
    if (k < 0) return -1;
    h = (h + 1) & (kStSlots - 1);
  }
  return -1;
}

__device__ __forceinline__ ElemGeom st_geom(const StElem& r) {
  return {r.n[0], r.n[1], r.n[2], r.s[0], r.s[1], r.s[2], r.x[0], r.y[0], r.x[1], r.y[1], r.x[2], r.y[2]};
}

__device__ __forceinline__ NodeZ st_node_z(const StElem& r, int c) {
  return {r.eta[c], r.h[c], r.eta[c] + r.h[c], r.kb[c]};
}

// Fills the table for sides s_first .. s_first + nsides - 1: candidate j of a side is one of
// its two elements (j = 0, 4) or that element's neighbour across its side j & 3 - 1.
__device__ void st_build(const DMesh& m, int* key, StElem* rec, int s_first, int nsides) {
  for (int i = threadIdx.x; i < kStSlots; i += blockDim.x) key[i] = -1;
  __syncthreads();
  const int i = threadIdx.x;
  if (i < min(nsides * 8, kStCand)) {
    const int4 sr = m.side[s_first + i / 8];
    const int j = i % 8, q = j & 3;
    int e = (j & 4) ? sr.w : sr.z;
    if (e >= 0 && q > 0) {
      const int4 r0 = m.elem[2 * e], r1 = m.elem[2 * e + 1];
      const int es = q == 1 ? r0.w : (q == 2 ? r1.x : r1.y);
      const int4 o = m.side[es];
      e = (o.z == e) ? o.w : o.z;
    }
    if (e >= 0) {
      unsigned h = st_hash(e);
      for (int p = 0; p < kStSlots; ++p) {
        const int old = atomicCAS(&key[h], -1, e);
        if (old == -1 || old == e) break;
        h = (h + 1) & (kStSlots - 1);
      }
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < kStSlots; t += blockDim.x) {
    const int e = key[t];
    if (e < 0) continue;
    const int4 r0 = m.elem[2 * e], r1 = m.elem[2 * e + 1];
    StElem& R = rec[t];
    const int nn[3] = {r0.x, r0.y, r0.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double2 p = m.nrec[2 * nn[c]], z = m.nrec[2 * nn[c] + 1];
      R.x[c] = p.x;
      R.y[c] = p.y;
      R.eta[c] = z.x;
      R.h[c] = z.y;
      R.kb[c] = m.kb[nn[c]];
      R.n[c] = nn[c];
    }
    R.s[0] = r0.w;
    R.s[1] = r1.x;
    R.s[2] = r1.y;
    R.ekb = m.elem_kb[e];
  }
  __syncthreads();
}

// zcoord(node, max(M, kb)) with sM = sigma[M] (one sigma per level): for M <= kb that is the bed
// -h, above kb level M. F: the last sigma, 0, gives H 0 + eta = eta without a select.
template <bool F>
__device__ __forceinline__ double zlev(const NodeZ& q, double sM, int M, int nv) {
  const double z = q.H * sM + q.eta;
  const double zs = (!F && M == nv - 1) ? q.eta : z;
  return (M <= q.kb) ? -q.h : zs;
}

// z of level M at the point with shape coordinates s0..s2 (the vertical bracket search's probe).
// One sigma per level (VM = 0) reads it once per probe from sig (LDS); otherwise each node's level
// max(M, kb) comes from its column zn (VM = 1, k_pack_levels) or from z_wet (VM = 2).
template <bool F>
struct ZSigma {
  NodeZ q0, q1, q2;
  const double* sig;
  int nv;
  __device__ __forceinline__ double3 nodes(int M) const {
    const double sM = sig[F ? M : max(M, 0)];
    return {zlev<F>(q0, sM, M, nv), zlev<F>(q1, sM, M, nv), zlev<F>(q2, sM, M, nv)};
  }
  __device__ __forceinline__ double operator()(double s0, double s1, double s2, int M) const {
    const double sM = sig[F ? M : max(M, 0)];
    return s0 * zlev<F>(q0, sM, M, nv) + s1 * zlev<F>(q1, sM, M, nv) + s2 * zlev<F>(q2, sM, M, nv) + 0.0;
  }
};
struct ZColumns {
  const DMesh& m;
  int n0, n1, n2;
  __device__ __forceinline__ double level(int node, int M) const {
    return m.zn[(uint64_t)ux(node) * ux(m.nvrt) + ux(max(M, 0))];
  }
  __device__ __forceinline__ double3 nodes(int M) const { return {level(n0, M), level(n1, M), level(n2, M)}; }
  __device__ __forceinline__ double operator()(double s0, double s1, double s2, int M) const {
    return s0 * level(n0, M) + s1 * level(n1, M) + s2 * level(n2, M) + 0.0;
  }
};

struct ZLevels {  // the nodes' records, read once per interpolation
  const DMesh& m;
  int n0, n1, n2;
  double2 q0, q1, q2;  // eta, depth
  int kb0, kb1, kb2;
  bool d0, d1, d2;     // dry
  __device__ __forceinline__ double level(int node, const double2& q, int kb, bool dry, int M) const {
    const double z = (M <= kb) ? -q.y : z_wet(m, node, q.x, q.y, kb, M);
    return dry ? 0.0 : z;
  }
  __device__ __forceinline__ double operator()(double s0, double s1, double s2, int M) const {
    return s0 * level(n0, q0, kb0, d0, M) + s1 * level(n1, q1, kb1, d1, M) + s2 * level(n2, q2, kb2, d2, M) + 0.0;
  }
};

// The vertical bracket of height pz: weights w1 of level L, w2 of level R. hint: the lower level of
// the previous point's bracket (updated here). L0, R0: the search's ends; bed: the highest level that
// is every node's bed (below L0: no level searched is). z: the probe. mono: z is non-decreasing in the level.
// With mono the search starts from the previous bracket, checked with the exact level z values: a
// bracket z_h < pz < z_(h+1) is the unique one the bisection below would end in, with the same zL
// and zR; otherwise one step down or up. A point at or below the bed, next to it (h <= bed, where
// z_h is z_L0), or at or above the surface takes the end that the full search finds first. A wave
// holds the levels of about two sides, the bed's and the surface's among them, so without these two
// rules every wave ran the full search's probes in every substep. (1,048,576 nodes x 31 levels, one
// sigma per level: 9.72 -> 8.58 ms a pass with the F variant and div_by; SZ grid 301x173 602 -> 282 us
// and per-node sigma 417x263 1419 -> 823 us, both with k_pack_levels, whose full search had evaluated
// the level functions at every probe.)
template <class Z>
__device__ __forceinline__ void z_bracket(const Z& z, double s0, double s1, double s2, double pz, int L0, int bed,
                                          int R0, bool mono, int& hint, int& L, int& R, double& w1, double& w2) {
  L = L0;
  R = R0;
  bool found = false;
  if (mono) {
    const int h = min(max(hint, L0), R0 - 1);
    const double zh = z(s0, s1, s2, h), zh1 = z(s0, s1, s2, h + 1);
    double zL = zh, zR = zh1;
    bool inside = false;
    if (zh < pz && pz < zh1) {
      L = h, R = h + 1, inside = true;
    } else if (pz <= zh && h <= bed) {
      w1 = 1.0;
      w2 = 0.0;
      return;
    } else if (pz >= zh1 && h + 1 == R0 && zh < zh1) {
      w1 = 0.0;
      w2 = 1.0;
      return;
    } else if (pz < zh && h > L0) {
      const double zd = z(s0, s1, s2, h - 1);
      if (zd < pz) L = h - 1, R = h, zL = zd, zR = zh, inside = true;
    } else if (pz > zh1 && h + 2 <= R0) {
      const double zu = z(s0, s1, s2, h + 2);
      if (pz < zu) L = h + 1, R = h + 2, zL = zh1, zR = zu, inside = true;
    }
    if (inside) {
      w2 = (pz - zL) / (zR - zL);
      w1 = 1.0 - w2;
      hint = L;
      found = true;
    }
  }
  if (found) return;
  double zL = z(s0, s1, s2, L), zR = z(s0, s1, s2, R);
  if (pz <= zL) {
    w1 = 1.0;
    w2 = 0.0;
  } else if (pz >= zR) {
    w1 = 0.0;
    w2 = 1.0;
  } else {
    while (R - L > 1) {
      const int M = (L + R) / 2;
      const double zM = z(s0, s1, s2, M);
      if (zM < pz) {
        L = M;
        zL = zM;
      } else {
        R = M;
        zR = zM;
      }
    }
    w2 = (pz - zL) / (zR - zL);
    w1 = 1.0 - w2;
    hint = L;
  }
}

// What the last interpolation of a start point read: the element, the z of its nodes at the two levels
// of the vertical bracket and the velocities there. A substep that stays in its prism reads nothing but
// the element's area: every operand is here, in the operations of the full search.
// LV: the velocities (36 registers' worth) lie in LDS and the area is read again, which leaves four waves
// a SIMD; otherwise all of it is in registers, for three. With three waves the full search, which every
// substep pays that enters a new element, was slower on one sigma than without anything kept: 700x500 nodes
// x 31 levels, 15 s substeps of flows up to 1 m/s, ms without / kept in registers / kept with LV:
//   one sigma, dx 1000 m 4.32 / 3.45 / 3.16, 50 m 5.82 / 6.80 / 5.97, 10 m 8.86 / 10.9 / 9.35
//   per-node sigma       5.33 / 3.60 / 3.65        7.16 / 7.71 / 7.75       12.5 / 14.2 / 13.9
// (before brackets were kept either: one sigma 5.17, 6.57, 9.60, per-node 9.52, 11.1, 14.7). 1,048,576
// nodes x 31 levels 8.58 ms with nothing kept, 7.48 in registers (16.8 at four waves, which spill), 6.90 LV.
constexpr int kCellVel = 18;  // (u, v, w) of nodes 0-2 at the lower level, then at the upper one
template <bool LV>
struct BtCell {
  int e = -1;         // -1: none
  int br = -1;        // the bracket's levels, (L + 1) << 10 | R (nvrt <= 1024); -1: not kept
  double2 area;       // (LV: read each time)
  double3 zL, zR;     // per node, where the column's levels do not decrease
  double v[LV ? 1 : kCellVel];
  double* lv;         // LV: the thread's column of LDS, kCellVel values 256 apart
  __device__ __forceinline__ double get(int i) const { return LV ? lv[256 * i] : v[LV ? 0 : i]; }
  __device__ __forceinline__ void put(int i, double x) {
    if (LV)
      lv[256 * i] = x;
    else
      v[LV ? 0 : i] = x;
  }
};

// Element::interpolateVelocities for triangles, ics=1 (meshdata.cu:1209-1291) with
// computeShapeCoords(fiAnywhere) (meshdata.cu:990-1043); g is element e's geometry.
// hint: the lower level of the previous vertical bracket (updated here).
// rc: element e's staged record (ST), else NULL.
template <int VM, bool ST, bool F, bool LV>
__device__ void interp_velocity(const DMesh& m, const double* sig, double h0, int e, const ElemGeom& g,
                                const StElem* rc, BtCell<LV>& c, double px, double py, double pz, double& uo, double& vo,
                                double& wo, int& hint) {
  const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
  const double x0 = g.x0, y0 = g.y0, x1 = g.x1, y1 = g.y1, x2 = g.x2, y2 = g.y2;
  const bool entered = c.e != e;
  if (entered) {
    c.e = e;
    c.br = -1;
  }
  if (LV || entered) c.area = m.area_inv[ux(e)];
  const double a0 = signed_area(px, py, x1, y1, x2, y2), a1 = signed_area(x0, y0, px, py, x2, y2);
  double s0 = div_by(a0, c.area.x, c.area.y);
  double s1 = div_by(a1, c.area.x, c.area.y);
  double s2 = 1.0 - s0 - s1;
  const double tmin = fmin(s0, fmin(s1, s2));
  if (tmin < 0.0) {
    const double aa = -tmin + 1.0e-8;
    const double bb = 1.0 / (s0 + s1 + s2 + 3.0 * aa);
    s0 = (s0 + aa) * bb;
    s1 = (s1 + aa) * bb;
    s2 = (s2 + aa) * bb;
  }
  const int nv = m.nvrt;
  const bool st = ST && rc;
  // F: level 0 is the bed, as -1 is
  const int R0 = nv - 1;
  double w1 = 1.0, w2 = 0.0;
  bool hit = false;
  if (c.br >= 0) {
    // the kept bracket: strictly inside two neighbouring levels, or the whole column (L0, R0) with the
    // point at or beyond an end: then z_bracket ends in it, with the same weights
    const double zL = s0 * c.zL.x + s1 * c.zL.y + s2 * c.zL.z + 0.0, zR = s0 * c.zR.x + s1 * c.zR.y + s2 * c.zR.z + 0.0;
    const bool whole = (c.br & 1023) > (c.br >> 10);  // R - L > 1
    if (!whole) {
      hit = zL < pz && pz < zR;
      if (hit) {
        w2 = (pz - zL) / (zR - zL);
        w1 = 1.0 - w2;
      }
    } else if (pz <= zL) {
      hit = true;
    } else if (pz >= zR) {
      hit = true;
      w1 = 0.0;
      w2 = 1.0;
    }
  }
  if (!hit) {
    int L, R, kb0, kb1, kb2;
    bool mono = true;
    const int L0 = F ? 0 : (st ? rc->ekb : m.elem_kb[ux(e)]) - 1;
    if constexpr (VM == 0) {
      const ZSigma<F> z{st ? st_node_z(*rc, 0) : node_z<F>(m, n0), st ? st_node_z(*rc, 1) : node_z<F>(m, n1),
                        st ? st_node_z(*rc, 2) : node_z<F>(m, n2), sig, nv};
      kb0 = z.q0.kb, kb1 = z.q1.kb, kb2 = z.q2.kb;
      z_bracket(z, s0, s1, s2, pz, L0, min(kb0, min(kb1, kb2)), R0, true, hint, L, R, w1, w2);
      c.zL = z.nodes(L);
      c.zR = z.nodes(R);
    } else if constexpr (VM == 2) {
      const double2 q0 = m.nrec[2u * ux(n0) + 1u], q1 = m.nrec[2u * ux(n1) + 1u], q2 = m.nrec[2u * ux(n2) + 1u];
      kb0 = m.kb[ux(n0)], kb1 = m.kb[ux(n1)], kb2 = m.kb[ux(n2)];
      const ZLevels z{m, n0, n1, n2, q0, q1, q2, kb0, kb1, kb2, q0.x + q0.y <= h0, q1.x + q1.y <= h0, q2.x + q2.y <= h0};
      mono = false;
      z_bracket(z, s0, s1, s2, pz, L0, 0, R0, false, hint, L, R, w1, w2);
    } else {
      // kb with a flag where the node's column is not non-decreasing (k_pack_levels)
      const int f0 = m.nkz[ux(n0)], f1 = m.nkz[ux(n1)], f2 = m.nkz[ux(n2)];
      kb0 = f0 & kKbMask, kb1 = f1 & kKbMask, kb2 = f2 & kKbMask;
      const ZColumns z{m, n0, n1, n2};
      mono = !((f0 | f1 | f2) & ~kKbMask);
      z_bracket(z, s0, s1, s2, pz, L0, min(kb0, min(kb1, kb2)), R0, mono, hint, L, R, w1, w2);
      c.zL = z.nodes(L);
      c.zR = z.nodes(R);
    }
    c.br = mono ? (L + 1) << 10 | R : -1;
    // the three nodes' level rows (64-bit row offsets), then two levels of each
    const double4* U = reinterpret_cast<const double4*>(m.uvw);
    auto at = [&](int node, int level, int kb) {
      return U[(uint64_t)ux(node) * ux(nv) + ux(F ? level : max(level, kb))];
    };
    const double4 q[6] = {at(n0, L, kb0), at(n1, L, kb1), at(n2, L, kb2), at(n0, R, kb0), at(n1, R, kb1), at(n2, R, kb2)};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      c.put(3 * i, q[i].x);
      c.put(3 * i + 1, q[i].y);
      c.put(3 * i + 2, q[i].z);
    }
  }
  auto mean = [&](int i) { return s0 * c.get(i) + s1 * c.get(i + 3) + s2 * c.get(i + 6) + 0.0; };
  const double uL = mean(0), vL = mean(1), uR = mean(9), vR = mean(10), wL = mean(2), wR = mean(11);
  uo = w1 * uL + w2 * uR;
  vo = w1 * vL + w2 * vR;
  wo = w1 * wL + w2 * wR;
}

// Leaded celestial walk (meshdata.cu:85-127) with Element::computePredicates (meshdata.cu:651-746).
// Corner j of a triangle is getNodeInOrder(j) = nodes[(j+1)%3]; walk side j is element side j.
// geo_valid: geo already holds element cur (the previous walk's final element), so the first
// step reads nothing. On return, geo holds the geometry of the final element cur.
// ST: slot is element cur's staged slot (-1: not staged), kept with geo.
template <bool ST>
__device__ __forceinline__ void walk_geom(const DMesh& m, const int* key, const StElem* rec, int cur, ElemGeom& geo,
                                          int& slot) {
  if (ST) {
    slot = st_find(key, cur);
    geo = slot >= 0 ? st_geom(rec[slot]) : elem_geom(m, cur);
  } else {
    geo = elem_geom(m, cur);
  }
}

template <bool ST>
__device__ bool celestial_walk(const DMesh& m, const int* key, const StElem* rec, int& cur, double x0x, double x0y,
                               double xtx, double xty, int& last_cross, int& status, ElemGeom& geo, int& slot,
                               bool geo_valid) {
  double fac = 0.00001;
  for (int iter = 0; iter < 40; ++iter) {
    if (iter > 0 || !geo_valid) walk_geom<ST>(m, key, rec, cur, geo, slot);
    const double C0x = geo.x1, C0y = geo.y1;  // corner j is node (j + 1) % 3
    const double C1x = geo.x2, C1y = geo.y2;
    const double C2x = geo.x0, C2y = geo.y0;
    const double vx = xtx - x0x, vy = xty - x0y;
    const double d0 = vx * (C0x - x0x) + vy * (C0y - x0y);
    const double d1 = vx * (C1x - x0x) + vy * (C1y - x0y);
    const double d2 = vx * (C2x - x0x) + vy * (C2y - x0y);
    double maxp = fmax(d0, d1);
    maxp = fmax(maxp, d2);
    // fmin(1, (maxp / vv) 1.00001) is 1 whenever maxp > 2 vv (the rounded quotient is then at
    // least 2; vv = 0 gives +inf as well), the usual case of a step shorter than the element:
    // the division runs only otherwise (NaN and overflow included), with the same result
    const double vv = vx * vx + vy * vy;
    double lead = 1.0;
    if (!(maxp > 2.0 * vv)) lead = fmin(1.0, (maxp / vv) * 1.00001);
    fac = fmax(1.00001 * fac, lead);
    const double ix = x0x + (xtx - x0x) * fac, iy = x0y + (xty - x0y) * fac;
    const double s0x = C1x - C0x, s0y = C1y - C0y;
    const double s1x = C2x - C1x, s1y = C2y - C1y;
    const double s2x = C0x - C2x, s2y = C0y - C2y;
    const bool left0 = (s0x * (iy - C0y) - s0y * (ix - C0x)) > -kSmall;
    const bool left1 = (s1x * (iy - C1y) - s1y * (ix - C1x)) > -kSmall;
    const bool left2 = (s2x * (iy - C2y) - s2y * (ix - C2x)) > -kSmall;
    // a side is an exit candidate only if the point is not left of it: with all three left
    // tests passed the walk ends here (the usual case), without the obtuse and bisector tests
    if (left0 && left1 && left2) return true;
    const bool obt0 = (s0x * s1x + s0y * s1y) > 0.0;
    const bool obt1 = (s1x * s2x + s1y * s2y) > 0.0;
    const bool obt2 = (s2x * s0x + s2y * s0y) > 0.0;
    const bool bis0 = ((ix - C1x) * (s0x + s1x) + (iy - C1y) * (s0y + s1y)) < 0.0;
    const bool bis1 = ((ix - C2x) * (s1x + s2x) + (iy - C2y) * (s1y + s2y)) < 0.0;
    const bool bis2 = ((ix - C0x) * (s2x + s0x) + (iy - C0y) * (s2y + s0y)) < 0.0;
    const bool v0 = !left0 && (!obt0 || bis0);
    const bool v1 = !left1 && (!obt1 || bis1);
    const bool v2 = !left2 && (!obt2 || bis2);
    if (!(v0 || v1 || v2)) return true;
    // the three side ids as opaque register values: a select among the struct's fields would
    // otherwise become an indexed load from a stack copy of it
    int gs0 = geo.s0, gs1 = geo.s1, gs2 = geo.s2;
    asm volatile("" : "+v"(gs0), "+v"(gs1), "+v"(gs2));
    const int side = v0 ? gs0 : (v1 ? gs1 : gs2);
    last_cross = side;
    const int4 sr = m.side[ux(side)];
    const int nxt = (sr.z == cur) ? sr.w : sr.z;
    if (nxt < 0 || !m.elem_wet[ux(nxt)]) return false;
    cur = nxt;
  }
  status |= GSH_BT_WALK_CAP;
  walk_geom<ST>(m, key, rec, cur, geo, slot);
  return true;
}

// Side::btrack (meshdata.cu:1449-1629). Returns the final velocity and the foot element.
template <int VM, bool ST, bool F, bool LV>
__device__ void btrack(const DMesh& m, const double* sig, double* lv, const int* key, const StElem* rec, const StepArgs& a, int s,
                       int k, double dtbk, int cur, double& ux, double& uy, int& foot, int& status) {
  const double h0 = a.h0;
  double x0x = m.side_cx[s], x0y = m.side_cy[s], x0z = m.zc[(int64_t)s * m.nvrt + k];
  double time_rm = a.dt;
  int still = 0;  // iterations on end, not counting the first, that left time_rm as it was
  const int4 sr = m.side[s];
  const double4* U = reinterpret_cast<const double4*>(m.uvw);
  double uix = m.su2[2 * ((int64_t)s * m.nvrt + k)], uiy = m.su2[2 * ((int64_t)s * m.nvrt + k) + 1];
  double uiz = 0.5 * (U[(int64_t)sr.x * m.nvrt + k].z + U[(int64_t)sr.y * m.nvrt + k].z);
  double xtx = -1.0e25, xty = -1.0e25, xtz = -1.0e25;
  int iter = 0;
  int hint = k;  // lower level of the last vertical bracket; the start point lies at level k
  ElemGeom geo;  // set by every walk before its first use
  int slot = -1;  // geo's staged slot (ST)
  bool geo_valid = false;
  BtCell<LV> cell;
  cell.lv = lv;
  bool interpolated = false;  // (uix, uiy) is the interpolated velocity at the last point
  while (true) {
    interpolated = false;
    const double dtb = fmin(dtbk, time_rm);
    xtx = x0x - dtb * uix;
    xty = x0y - dtb * uiy;
    xtz = x0z - dtb * uiz;
    int last = -1;
    const bool found = celestial_walk<ST>(m, key, rec, cur, x0x, x0y, xtx, xty, last, status, geo, slot, geo_valid);
    geo_valid = true;
    const StElem* rc = (ST && slot >= 0) ? rec + slot : nullptr;
    // the reference compares time_rm with that of three iterations before (1e10 s before the first); it
    // never grows, so it is not less after two iterations on end that left it as it was
    if (still == 2) {
      xtx = x0x;
      xty = x0y;
      xtz = x0z;
      status |= GSH_BT_STUCK;
      break;
    }
    if (!found) {
      const int4 cs = m.side[last];
      const double2 P1 = m.nrec[2 * cs.x], P2 = m.nrec[2 * cs.y];
      const double p1x = P1.x, p1y = P1.y, p2x = P2.x, p2y = P2.y;
      const double v1x = xtx - x0x, v1y = xty - x0y;
      const double v2x = p2x - p1x, v2y = p2y - p1y;
      const double denom = v2x * v1y - v2y * v1x;
      double t, sp;
      if (fabs(denom) < kSmall) {
        t = fmin(fmax(((xtx - p1x) * v2x + (xty - p1y) * v2y) / (v2x * v2x + v2y * v2y), 0.0), 1.0);
        if (t < 0.0000000001) t = 0.0;
        if (t > 0.9999999999) t = 1.0;
        sp = fmin(fmax(((p1x + t * v2x - x0x) * v1x + (p1y + t * v2y - x0y) * v1y) / (v1x * v1x + v1y * v1y), 0.0),
                  1.0);
      } else {
        t = fmin(fmax(((x0x - p1x) * v1y - (x0y - p1y) * v1x) / denom, 0.0), 1.0);
        if (t < 0.0000000001) t = 0.0;
        if (t > 0.9999999999) t = 1.0;
        sp = fmin(fmax(((p1x + t * v2x - x0x) * v1x + (p1y + t * v2y - x0y) * v1y) / (v1x * v1x + v1y * v1y), 0.0),
                  1.0);
        if (sp < 0.0000000001) sp = 0.0;
      }
      const double before = time_rm;
      time_rm -= sp * dtb;
      still = (iter > 0 && time_rm == before) ? still + 1 : 0;
      const double nz = x0z + sp * (xtz - x0z);
      xtx = p1x + t * v2x;
      xty = p1y + t * v2y;
      xtz = nz;
      if (m.side_type[last] == 2) {
        status |= GSH_BT_OPEN_EXIT;
        break;
      }
      const double len = sqrt(v2x * v2x + v2y * v2y);
      const double tx = v2x / len, ty = v2y / len;
      double iu, iv, iw;
      interp_velocity<VM, ST, F, LV>(m, sig, h0, cur, geo, rc, cell, xtx, xty, xtz, iu, iv, iw, hint);
      const double d = iu * tx + iv * ty;
      uix = tx * d;
      uiy = ty * d;
      uiz = iw;
      status |= GSH_BT_SLIDE;
    } else {
      const double before = time_rm;
      time_rm -= dtb;
      still = (iter > 0 && time_rm == before) ? still + 1 : 0;
      interp_velocity<VM, ST, F, LV>(m, sig, h0, cur, geo, rc, cell, xtx, xty, xtz, uix, uiy, uiz, hint);
      interpolated = true;
    }
    if (time_rm <= 0.0) break;
    if (uix * uix + uiy * uiy <= a.velmin2) {
      ux = uix;
      uy = uiy;
      foot = cur;
      return;
    }
    x0x = xtx;
    x0y = xty;
    x0z = xtz;
    ++iter;
    if (iter == 38) {
      status |= GSH_BT_ITER38;
      ux = uix;
      uy = uiy;
      foot = cur;
      return;
    }
  }
  // the velocity at the last point: already interpolated unless the walk slid, stuck or left the mesh
  // there
  ux = uix;
  uy = uiy;
  if (!interpolated) {
    double iw;
    interp_velocity<VM, ST, F, LV>(m, sig, h0, cur, geo, (ST && slot >= 0) ? rec + slot : nullptr, cell, xtx, xty, xtz, ux,
                               uy, iw, hint);
  }
  foot = cur;
}

// backtrackAllNodes (meshdata.cu:3547-3660), one thread per (side, level): consecutive
// lanes are consecutive levels of one side, so the nodal [node][level] gathers of a wave
// fall on a few contiguous cache lines.
// LV: BtCell's velocities in LDS. VM: 0, one sigma per level (kept in LDS) and levels that do not
// decrease in any wet column; 1, each node's column (DMesh::vmode 1 and 2); 2, each node's levels evaluated
// at each probe, always searched in full (short lists of vmode 1 and 2, and vmode 0 where levels may decrease).
// ST: the workgroup first stages its element patch in LDS (all sides and levels, no list).
// F: a mesh with kb = 0 at every node whose last sigma is 0 (VM = 0).
template <int VM, bool ST, bool F, bool LV>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LV || VM == 2 ? 4 : 3, 8)))
k_backtrack(DMesh m, StepArgs a, const int32_t* list_side, const int32_t* list_lev, int32_t count) {
  extern __shared__ double bt_lds[];  // LV: kCellVel x 256; VM = 0: the sigma levels
  double* sig = bt_lds + (LV ? kCellVel * 256 : 0);
  __shared__ int st_key[ST ? kStSlots : 1];
  __shared__ StElem st_rec[ST ? kStSlots : 1];
  if (VM == 0) {
    for (int j = threadIdx.x; j < m.nvrt; j += blockDim.x) sig[j] = m.sigma[j];
    __syncthreads();
  }
  if (ST) {  // the workgroup's sides: from its first to its last (side, level) pair
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x;
    const int64_t tl = min(t0 + (int64_t)blockDim.x, (int64_t)m.ns * m.nvrt) - 1;
    const int s_first = (int)(t0 / m.nvrt), s_last = (int)(tl / m.nvrt);
    st_build(m, st_key, st_rec, s_first, s_last - s_first + 1);
  }
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int s, k;
  if (list_side) {
    if (t >= count) return;
    s = list_side[t];
    k = list_lev[t];
  } else {
    if (t >= (int64_t)m.ns * m.nvrt) return;
    s = (t < 0xffffffffll) ? (int)((uint32_t)t / (uint32_t)m.nvrt) : (int)(t / m.nvrt);
    k = (int)(t - (int64_t)s * m.nvrt);
  }
  const int64_t idx = (int64_t)s * m.nvrt + k;
  const double ux0 = m.su2[2 * idx], uy0 = m.su2[2 * idx + 1];
  double bx = ux0, by = uy0;
  int foot = -1, status = 0;
  if (m.side_wet[s] && k >= m.side_kb[s] && !(ux0 * ux0 + uy0 * uy0 <= a.velmin2)) {
    const int4 sr = m.side[s];
    const double4* U = reinterpret_cast<const double4*>(m.uvw);
    double suma = 0.0;
    int icount = 0;
    for (int l = 0; l < 2; ++l) {
      const int e = (l == 0) ? sr.z : sr.w;
      if (e < 0) continue;
      ++icount;
      const int4 r = m.elem[2 * e];
      const double4 q0 = U[(int64_t)r.x * m.nvrt + k], q1 = U[(int64_t)r.y * m.nvrt + k],
                    q2 = U[(int64_t)r.z * m.nvrt + k];
      const double* g = m.gradphi + 6 * (int64_t)e;
      const double gux = q0.x * g[0] + q1.x * g[2] + q2.x * g[4];
      const double guy = q0.x * g[1] + q1.x * g[3] + q2.x * g[5];
      const double gvx = q0.y * g[0] + q1.y * g[2] + q2.y * g[4];
      const double gvy = q0.y * g[1] + q1.y * g[3] + q2.y * g[5];
      suma += a.dt * sqrt((gux * gux + guy * guy) + (gvx * gvx + gvy * gvy));
    }
    const int nd = (int)(suma / icount) * 4;
    const int ndelt = max(a.ndelt_min, min(nd, a.ndelt_max));
    const double dtbk = a.dt / ndelt;
    const int start = m.elem_wet[sr.z] ? sr.z : sr.w;
    btrack<VM, ST, F, LV>(m, sig, bt_lds + threadIdx.x, st_key, st_rec, a, s, k, dtbk, start, bx, by, foot, status);
  }
  m.btu[2 * idx] = bx;
  m.btu[2 * idx + 1] = by;
  m.foot[idx] = foot;
  m.bstatus[idx] = status;
}

// Packs (x, y) and (eta2, depth) of every node next to each other for the backtracking gathers.
// One sigma per level: (0, 0) for a dry node, whose levels are then all 0 (node_z).
__global__ void k_pack_nodes(DMesh m, double h0) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.n) return;
  const double eta = m.eta2[i], h = m.depth[i];
  m.nrec[2 * i] = make_double2(m.x[i], m.y[i]);
  m.nrec[2 * i + 1] = (m.vmode == 0 && eta + h <= h0) ? make_double2(0.0, 0.0) : make_double2(eta, h);
  if (m.zn) m.nkz[i] = m.kb[i];
}

// The z columns of the backtracking's vertical search on per-node sigma and SZ grids: zn[node][k] is
// zcoord(node, max(k, kb)); a node whose column decreases anywhere gets a flag beside its kb. A probe
// of the search is then three loads instead of three evaluations of the level functions, and starts
// from the previous point's bracket as on one sigma per level. Bound by its stores: 13.5 us for
// 109,671 nodes, against the 600 us that the kept columns save there.
__global__ void k_pack_levels(DMesh m, double h0) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nv = (uint32_t)m.nvrt;
  if (t >= (uint64_t)m.n * nv) return;
  const int i = (t < 0xffffffffull) ? (int)((uint32_t)t / nv) : (int)(t / nv);
  const int k = (int)(t - (uint64_t)i * nv);
  const double eta = m.eta2[i], h = m.depth[i];
  const int kb = m.kb[i];
  auto level = [&](int M) {
    if (eta + h <= h0) return 0.0;
    return M <= kb ? -h : z_wet(m, i, eta, h, kb, M);
  };
  const double z = level(k);
  m.zn[t] = z;
  if (k > 0 && !(level(k - 1) <= z)) atomicOr(&m.nkz[i], kKbMask + 1);
}

// Workgroups from which the fourth wave a SIMD of the LV form pays for its LDS trips: three waves hold 768
// on the chip. One sigma, register form / LV, flows that stay in their elements and that leave one each
// substep: 60x40x11 (303 workgroups) 45 / 49 and 119 / 126 us, 110x80x12 (1,220) 71 / 71 and 193 / 190,
// 120x90x14 (1,750) 87 / 87 and 240 / 224. Columns, whose probes are loads and whose search spills at four
// waves, stay in registers (BtCell has the figures).
constexpr unsigned kBtFill = 1536;

void launch_backtrack(const DMesh& mesh, const StepArgs& a, const int32_t* ls, const int32_t* ll, int32_t count,
                      hipStream_t st) {
  DMesh m = mesh;
  // Columns cost one evaluation per node and level, a start point without them several per substep and a
  // longer search. Lists, levels evaluated / columns: 52,073 nodes x 24 levels 300 start points 98 / 77 us, x 60
  // 64 of them 67 / 66; 350,000 x 31 4,000 of them 118 / 119, 256,000 612 / 402 (SZ 451 / 421); 1,400,000 x 20
  // 64,000 of them 233 / 312, 256,000 686 / 540 (SZ 521 / 564).
  const int64_t items = (int64_t)m.n * m.nvrt;
  if (ls && items > (4 << 20) && count < items / 96) m.zn = nullptr;
  if (m.n > 0) hipLaunchKernelGGL(k_pack_nodes, dim3((m.n + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a.h0);
  const int64_t total = ls ? (int64_t)count : (int64_t)m.ns * m.nvrt;
  if (total <= 0) return;
  if (m.zn) {
    const int64_t nz = (int64_t)m.n * m.nvrt;
    hipLaunchKernelGGL(k_pack_levels, dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, st, m, a.h0);
  }
  const dim3 grid((unsigned)((total + 255) / 256));
  const bool stage = m.bt_stage != 0 && !ls;
  // One sigma per level: a wet node's levels do not decrease where 0 <= h0 < H and every sigma between
  // bed and surface lies in [-1, 0], which VM = 0 relies on. Outside that, VM = 2 searches in full.
  const bool sigma = m.vmode == 0 && m.sig_mono && a.h0 >= 0.0;
  const size_t lds_sig = sigma ? 8 * (size_t)m.nvrt : 0;
  auto go = [&](auto ker, size_t lds) { hipLaunchKernelGGL(ker, grid, dim3(256), lds, st, m, a, ls, ll, count); };
  if (!sigma && !m.zn) return go(k_backtrack<2, false, false, false>, 0);
  if (stage) {
    if (sigma)
      go(k_backtrack<0, true, false, false>, lds_sig);
    else
      go(k_backtrack<1, true, false, false>, 0);
    return;
  }
  if (!sigma) return go(k_backtrack<1, false, false, false>, 0);
  const bool lv = grid.x > kBtFill;
  auto pick = [&](auto ldsv, auto regv) {
    if (lv)
      go(ldsv, lds_sig + 8 * kCellVel * 256);
    else
      go(regv, lds_sig);
  };
  if (m.flat)
    pick(k_backtrack<0, false, true, true>, k_backtrack<0, false, true, false>);
  else
    pick(k_backtrack<0, false, false, true>, k_backtrack<0, false, false, false>);
}

// ---------------------------------------------------------------- nodal velocities
// zeroNodalVelocities, computeNodalVerticalVelocities1/2 and computeNodalHorizontalVelocities1/2
// (meshdata.cu:5765-5929) for triangles, ics=1, indvel <= 0. The reference scatters each
// element's contributions to its nodes with atomicAdd; here one thread per (node, level) gathers
// them over the node's ball in ball order, so the sums are deterministic:
//   w2[k] = (1 / sum area_e) * sum w_e[k] area_e                 over all ball elements, k >= kb
//   u2[k] = (sum clamp(u_s2 + u_s3 - u_s1)[k]) * (1 / count)     over the wet ball elements, k >= kb
// (s1 the element side opposite the node, s2 and s3 the following ones; count = wet elements;
// zero below kb and where no wet element touches the node). The level index is the fastest, so a
// wave reads consecutive levels of the same side and element rows.
__device__ __forceinline__ double clamp_vel(double x, double hi) { return fmin(fmax(x, -hi), hi); }

// Each ball is counter-clockwise, so the spoke s2 of one entry is the next entry's s3 (ball_rec.w
// holds the first entry's s3): a node with m elements reads 2 m + 1 side rows instead of 3 m.
// The workgroup's threads cover the levels of a few consecutive nodes, whose balls are one
// contiguous range of the ball arrays: its entries (record, and the area, negative where the
// element is dry) are staged in LDS once, up to kNvCap of them (the rest read from global memory,
// the same values), so each (node, level) thread only gathers its level's w and u2, kNvBatch entries'
// loads at a time. Bound by the first-level cache: its misses stall it 60 % of the time (215,683 nodes
// x 31 levels: 240 -> 205 us, 3.1 TB/s; 3 entries at a time 213, 2 230; workgroups of consecutive
// nodes on one XCD 210).
constexpr int kNvCap = 512;
constexpr int kNvBatch = 4;  // ball entries whose loads are in flight together

__global__ void __launch_bounds__(256) k_nodal_velocity(DMesh m, double rx, double ry) {
  __shared__ int4 Lrec[kNvCap];
  __shared__ double Larea[kNvCap];
  __shared__ f64x2 Lout[512];
  const uint64_t t0 = (uint64_t)blockIdx.x * blockDim.x;
  const uint32_t nv = (uint32_t)m.nvrt;
  const uint64_t total = (uint64_t)m.n * nv;
  auto node_of = [&](uint64_t tt) { return (tt < 0xffffffffull) ? (int)((uint32_t)tt / nv) : (int)(tt / nv); };
  const int ifirst = node_of(t0), ilast = node_of(min(t0 + blockDim.x, total) - 1);
  const int jb = m.ball_ptr[ifirst];
  const int nst = min(m.ball_ptr[ilast + 1] - jb, kNvCap);
  auto area_of = [&](int e) {
    const double a = m.area[e];
    const int wet = m.elem_wet[e];
    return wet ? a : -a;
  };
  for (int q = threadIdx.x; q < nst; q += blockDim.x) {
    const int4 r = m.ball_rec[jb + q];
    Lrec[q] = r;
    Larea[q] = area_of(r.x);
  }
  const uint64_t t = min(t0 + threadIdx.x, total - 1);
  const int i = node_of(t);
  const int k = (int)(t - (uint64_t)i * nv);
  const int j0 = m.ball_ptr[i], j1 = m.ball_ptr[i + 1];
  const bool node_wet = m.node_wet[i] != 0;
  const bool above = k >= m.kb[i];
  __syncthreads();
  const double2* su = reinterpret_cast<const double2*>(m.su2) + k;
  const double* ew = m.ew + k;
  // one pass over the ball; each sum keeps its own ball-order sequence of additions
  double asum = 0.0, ws = 0.0, sx = 0.0, sy = 0.0;
  int count = 0;
  auto pass = [&](auto rec, auto area) {
    if (j0 >= j1) return;
    double2 u3 = su[(int64_t)rec(j0).w * nv];
    for (int j = j0; j < j1; j += kNvBatch) {
      double2 u1[kNvBatch] = {}, u2[kNvBatch] = {};
      double w[kNvBatch] = {};
#pragma unroll
      for (int q = 0; q < kNvBatch; ++q)
        if (j + q < j1) {
          const int4 r = rec(j + q);
          u1[q] = su[(int64_t)r.y * nv];
          u2[q] = su[(int64_t)r.z * nv];
          w[q] = ew[(int64_t)r.x * nv];
        }
#pragma unroll
      for (int q = 0; q < kNvBatch; ++q)
        if (j + q < j1) {
          const double as = area(j + q), a = fabs(as);
          asum += a;
          ws += w[q] * a;
          if (as > 0.0 && node_wet) {
            ++count;
            sx += clamp_vel(u2[q].x + u3.x - u1[q].x, rx);
            sy += clamp_vel(u2[q].y + u3.y - u1[q].y, ry);
          }
          u3 = u2[q];
        }
    }
  };
  // levels below the node's bed are 0 and read nothing
  if (!above) {
  } else if (j1 - jb <= nst)
    pass([&](int j) { return Lrec[j - jb]; }, [&](int j) { return Larea[j - jb]; });
  else
    pass([&](int j) { return m.ball_rec[j]; }, [&](int j) { return area_of(m.ball_rec[j].x); });
  double ux = 0.0, uy = 0.0, w = 0.0;
  if (above) {
    w = (1.0 / asum) * ws;
    if (count > 0) {
      ux = sx * (1.0 / count);
      uy = sy * (1.0 / count);
    }
  }
  // a lane's record is 32 bytes: through LDS each store of a wave covers one contiguous KB (two
  // stores of every other 16 bytes write each line twice)
  f64x2* mine = Lout + 128 * (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  mine[2 * lane] = f64x2{ux, uy};
  mine[2 * lane + 1] = f64x2{w, 0.0};
  wave_lds_sync();
  const uint64_t c0 = 2 * t0 + 128 * (threadIdx.x >> 6) + lane;
  f64x2* out = reinterpret_cast<f64x2*>(m.uvw);
  if (c0 < 2 * total) out[c0] = mine[lane];
  if (c0 + 64 < 2 * total) out[c0 + 64] = mine[lane + 64];
}

void launch_nodal_velocity(const DMesh& m, double rmaxvel, hipStream_t st) {
  const int64_t total = (int64_t)m.n * m.nvrt;
  if (total > 0)
    hipLaunchKernelGGL(k_nodal_velocity, dim3((unsigned)((total + kTpb - 1) / kTpb)), dim3(kTpb), 0, st, m, rmaxvel,
                       rmaxvel * 1.013);
}

// ---------------------------------------------------------------- a8-a10, elevation BC
// computeVerticallyIntegratedVelocity (meshdata.cu:4459-4476) and
// computeVegetationAndDragParameters for iveg=0, nchi=0 (meshdata.cu:4615-4725).
// A workgroup takes g consecutive sides: the sides' zc and velocity rows are one contiguous
// span of HBM each, which the workgroup copies into LDS with flat coalesced loads; one thread
// per side then sums its levels in the reference's order from LDS, and the velocity rows are
// replaced by the btu rows for the second integral. Row strides in LDS are odd so the
// per-side reads spread over the banks.
// Row g = i / row_len and column j from a float reciprocal (exact here: i < 2^20, row_len <=
// 2048); the two corrections keep it exact whatever the rounding.
__device__ __forceinline__ int split_row(int i, float inv, int row_len, int& j) {
  int g = (int)(((float)i + 0.5f) * inv);
  j = i - g * row_len;
  if (j < 0) {
    --g;
    j += row_len;
  }
  if (j >= row_len) {
    ++g;
    j -= row_len;
  }
  return g;
}

// Each thread issues its loads 8 at a time before the LDS writes, so a small workgroup still
// keeps enough loads in flight.
__device__ __forceinline__ void stage_rows(double* __restrict__ dst, int stride, const double* __restrict__ src,
                                           int row_len, int rows) {
  constexpr int B = 8;
  const int total = rows * row_len;
  const float inv = 1.0f / (float)row_len;
  for (int base = threadIdx.x; base < total; base += B * blockDim.x) {
    double v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int i = base + u * blockDim.x;
      v[u] = i < total ? src[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int i = base + u * blockDim.x;
      if (i < total) {
        int j;
        const int g = split_row(i, inv, row_len, j);
        dst[g * stride + j] = v[u];
      }
    }
  }
}

__global__ void __launch_bounds__(256) k_side_rhs(DMesh m, StepArgs a, int g) {
  extern __shared__ double lds[];
  const int nv = m.nvrt;
  const int zs = nv | 1, us = (2 * nv) | 1;
  double* Lz = lds;           // [g][zs]: zc
  double* Lu = lds + g * zs;  // [g][us]: side velocity u2, then btu
  const int s0 = blockIdx.x * g;
  const int gc = min(g, m.ns - s0);
  stage_rows(Lz, zs, m.zc + (int64_t)s0 * nv, nv, gc);
  stage_rows(Lu, us, m.su2 + 2 * (int64_t)s0 * nv, 2 * nv, gc);
  __syncthreads();
  const int t = threadIdx.x;
  const bool mine = t < gc;
  const int s = s0 + t;
  bool wet = false;
  int kb = 0;
  double Ux = 0.0, Uy = 0.0;
  const double* zc = Lz + t * zs;
  const double* u = Lu + t * us;
  if (mine) {
    wet = m.side_wet[s] != 0;
    if (wet) {
      kb = m.side_kb[s];
      for (int k = kb; k < nv - 1; ++k) {
        const double ucx = 0.5 * (u[2 * k] + u[2 * (k + 1)]);
        const double ucy = 0.5 * (u[2 * k + 1] + u[2 * (k + 1) + 1]);
        const double dz = zc[k + 1] - zc[k];
        Ux += dz * ucx;
        Uy += dz * ucy;
      }
    }
  }
  __syncthreads();
  stage_rows(Lu, us, m.btu + 2 * (int64_t)s0 * nv, 2 * nv, gc);
  __syncthreads();
  if (!mine) return;
  double hhat = 0.0, chi = 0.0;
  if (wet) {
    const int4 r = m.side[s];
    const double htot = 0.5 * (m.eta2[r.x] + m.eta2[r.y]) + 0.5 * (m.depth[r.x] + m.depth[r.y]);
    const double* bt = u;
    // the side's share of computeElemAverageGhat (meshdata.cu:6183-6424): vertical integral of btu,
    // the same for both elements of the side
    double usx = 0.0, usy = 0.0;
    if (kb == nv - 2) {
      const double dz = zc[nv - 1] - zc[nv - 2];
      usx += bt[2 * (nv - 1)] * dz;
      usy += bt[2 * (nv - 1) + 1] * dz;
    } else {
      for (int k = kb + 1; k < nv; ++k) {
        const double dz = zc[k] - zc[k - 1];
        usx += (bt[2 * k] + bt[2 * (k - 1)]) / 2.0 * dz;
        usy += (bt[2 * k + 1] + bt[2 * (k - 1) + 1]) / 2.0 * dz;
      }
    }
    m.side_us[2 * s] = usx;
    m.side_us[2 * s + 1] = usy;
    const double bx = bt[2 * (kb + 1)], by = bt[2 * (kb + 1) + 1];
    const double vmag1 = sqrt(bx * bx + by * by);
    const double cd = 0.5 * (m.cd[r.x] + m.cd[r.y]);
    const double chi2 = cd * vmag1;
    chi = chi2;
    if (kb == nv - 2) {
      const double fricH = htot + chi2 * a.dt;
      hhat = htot * htot / fricH;
    } else {
      hhat = htot - chi * a.dt;
      if (a.ihhat == 1) hhat = fmax(0.0, hhat);
    }
  }
  m.sU[2 * s] = Ux;
  m.sU[2 * s + 1] = Uy;
  m.hhat[s] = hhat;
  m.chi[s] = chi;
}

// computeElemAverageGhat (meshdata.cu:6183-6424) for the barotropic, ics=1, iveg=0 subset with
// no Coriolis, wind stress, horizontal viscosity, atmospheric pressure or tidal potential:
// those terms are identically zero here and are kept as explicit zero operands.
__global__ void k_elem_ghat(DMesh m, StepArgs a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m.ne) return;
  double gx = 0.0, gy = 0.0;
  if (m.elem_wet[e]) {
    const int nv = m.nvrt;
    const int4 r0 = m.elem[2 * e], r1 = m.elem[2 * e + 1];
    const int sides[3] = {r0.w, r1.x, r1.y};
    const double dt = a.dt;
    for (int j = 0; j < 3; ++j) {
      const int s = sides[j];
      const int4 sr = m.side[s];
      const double chi = m.chi[s];
      const double htot = 0.5 * (m.eta2[sr.x] + m.eta2[sr.y]) + 0.5 * (m.depth[sr.x] + m.depth[sr.y]);
      const int kb = m.side_kb[s];
      double cff1, cff2, cff3;
      if (kb == nv - 2) {
        cff1 = m.hhat[s] / htot;
        cff2 = 0.0;
        cff3 = 0.0;
      } else {
        cff1 = 1.0;
        cff2 = 1.0;
        cff3 = 0.0;
      }
      const double* bt = m.btu + 2 * (int64_t)s * nv;
      const double usx = m.side_us[2 * s], usy = m.side_us[2 * s + 1];  // from k_side_rhs
      gx += cff1 * usx - cff3 * 0.0;
      gy += cff1 * usy - cff3 * 0.0;
      const double ubx = bt[2 * (kb + 1)], uby = bt[2 * (kb + 1) + 1];
      gx -= chi * dt * cff2 * ubx + dt * cff1 * 0.0;
      gy -= chi * dt * cff2 * uby + dt * cff1 * 0.0;
    }
    gx = (1.0 / 3) * gx;
    gy = (1.0 / 3) * gy;
  }
  m.ghat1[2 * e] = gx;
  m.ghat1[2 * e + 1] = gy;
}

// Elevation BC type of node i: its own (GSH_F_ETYPE) or, where never set, the step parameter.
__device__ __forceinline__ int node_etype(const DMesh& m, const StepArgs& a, int i) {
  const int t = m.etype[i];
  return t < 0 ? a.iettype : t;
}

// computeElevationBoundaryConditions (meshdata.cu:4276-4339) for node types 1-5: eth for 1, 2, 4,
// the tidal constituents for 3, both for 5; no ramp-down of an initial elevation
// (nramp_elev = 0), no loading tide, no inverse barometric term. Type 0 leaves elbc as it is.
__global__ void k_elbc(DMesh m, StepArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.n) return;
  if (!m.open_bnd[i]) return;
  const int iettype = node_etype(m, a, i);
  const double eic = 0.0;
  const double r_eic = (1.0 - a.ramp) * eic;
  const double r_eth = a.ramp * m.eth[i];
  double r_eta1_bar = 0.0;
  if (iettype == 3 || iettype == 5) {
    const double pi = 3.14159265358979323846;
    for (int j = 0; j < m.nbfr; ++j) {
      const double amig = m.tide[j], ff = m.tide[m.nbfr + j], face = m.tide[2 * m.nbfr + j];
      const double efa = m.efa[(int64_t)i * m.nbfr + j], emo = m.emo[(int64_t)i * m.nbfr + j];
      const int ncyc = (int)(amig * a.time / (2.0 * pi));
      const double arg = amig * a.time - (2.0 * pi) * ncyc + face - efa;
      r_eta1_bar += a.ramp * ff * emo * cos(arg);
    }
  }
  switch (iettype) {
    case 1:
    case 2:
    case 4: m.elbc[i] = r_eic + r_eth; break;
    case 3: m.elbc[i] = r_eic + r_eta1_bar; break;
    case 5: m.elbc[i] = r_eic + r_eta1_bar + r_eth; break;
    default: break;
  }
}

void launch_rhs(const DMesh& m, const StepArgs& a, hipStream_t st) {
  if (m.n > 0) hipLaunchKernelGGL(k_elbc, dim3((m.n + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a);
  if (m.ns > 0) {
    // sides per workgroup: as many as fit 16 KB of LDS (measured best against 4-64 KB at 1M
    // sides x 31 levels), at most one per thread
    const int row = 8 * ((m.nvrt | 1) + ((2 * m.nvrt) | 1));
    const int g = max(1, min(kTpb, (16 * 1024) / row));
    hipLaunchKernelGGL(k_side_rhs, dim3((unsigned)((m.ns + g - 1) / g)), dim3(kTpb), (size_t)g * row, st, m, a, g);
  }
  if (m.ne > 0) hipLaunchKernelGGL(k_elem_ghat, dim3((m.ne + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a);
}

// ---------------------------------------------------------------- momentum (the step after the solve)
// Side::grad2 (meshdata.cu:1363-1398) of eta1 over the side's elements that are wet (isDry of
// the last level update) and of eta2 over those wet by eta2 (Element::isDry2, meshdata.cu:774-778:
// a node with eta2 + depth <= h0 makes its element dry), each the mean of the element gradients
// (Element::grad2, meshdata.h:1105-1114). Lane c of the side's two (adjacent) lanes reads and forms
// element c's gradients; the lanes then exchange the components the other one sums.
struct SideElem {  // element c of a side: its gradient coefficients, its nodes and whether it is wet
  bool there, wet;
  double2 p[3];
  double f1[3], f2[3], h[3];
};

__device__ __forceinline__ SideElem side_elem_load(const DMesh& m, int e) {
  SideElem q;
  q.there = e >= 0;
  e = max(e, 0);
  const int4 r0 = m.elem[2 * (int64_t)e];
  const double2* gp = reinterpret_cast<const double2*>(m.gradphi) + 3 * (int64_t)e;
  q.wet = m.elem_wet[e] != 0;
  const int nd[3] = {r0.x, r0.y, r0.z};
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    q.p[j] = gp[j];
    q.f1[j] = m.eta1[nd[j]];
    q.f2[j] = m.eta2[nd[j]];
    q.h[j] = m.depth[nd[j]];
  }
  return q;
}

// The mean over the elements of one component; x, y: this lane's element's gradient, in: it counts.
__device__ __forceinline__ double side_grad_mean(double x, double y, bool in, int c) {
  const double own = c ? y : x, other = __shfl_xor(c ? x : y, 1, 64);
  const bool oin = __shfl_xor((int)in, 1, 64) != 0;
  const bool in0 = c ? oin : in, in1 = c ? in : oin;
  double g = 0.0;
  if (in0) g += c ? other : own;
  if (in1) g += c ? own : other;
  const int n = (int)in0 + (int)in1;
  return n > 0 ? g * (1.0 / n) : g;
}

__device__ __forceinline__ void side_eta_grads(const SideElem& q, double h0, int c, double& g1, double& g2) {
  const double x1 = q.f1[0] * q.p[0].x + q.f1[1] * q.p[1].x + q.f1[2] * q.p[2].x;
  const double y1 = q.f1[0] * q.p[0].y + q.f1[1] * q.p[1].y + q.f1[2] * q.p[2].y;
  g1 = side_grad_mean(x1, y1, q.there && q.wet, c);
  const bool dry2 = q.f2[0] + q.h[0] <= h0 || q.f2[1] + q.h[1] <= h0 || q.f2[2] + q.h[2] <= h0;
  const double x2 = q.f2[0] * q.p[0].x + q.f2[1] * q.p[1].x + q.f2[2] * q.p[2].x;
  const double y2 = q.f2[0] * q.p[0].y + q.f2[1] * q.p[1].y + q.f2[2] * q.p[2].y;
  g2 = side_grad_mean(x2, y2, q.there && !dry2, c);
}

// solveMomentumEquations (meshdata.cu:5074-5352) for one side, barotropic, itur=0 (dfv = dfv0),
// iveg=0, ics=1, imm=0 and no Coriolis, wind, horizontal viscosity, pressure or tidal potential
// (zero terms omitted), then applyMomentumBC for land sides (meshdata.cu:5356-5446, islip=0).
// zc and u are the side's rows in LDS; u holds btu on entry and u2 on exit. The 3D case is
// tridag_sch<2> (meshdata.cu:3665-3711) with the coefficients formed on the fly: the forward
// sweep keeps u_j in the btu slot k-1 and gam_j in the zc slot k-1 (both dead once row j is
// formed), and the back substitution moves each result up one slot, clamped.
// Component c (0: x, 1: y) of one side's momentum solve, by one of the side's two lanes (adjacent
// lanes of one wave): both lanes compute the shared coefficients identically (the Thomas pivots,
// written to the same zc slots with the same values, in lockstep) and each solves its own
// component. The free-slip projection needs both components and runs in lane 0 after a wave
// fence. Every value has the operands and order of the one-lane form.
// Few waves fit (24 bytes of LDS per side and level), so a wave must not wait for LDS at each level:
// both sweeps read kMomAhead levels before the arithmetic that needs them.
constexpr int kMomAhead = 4;

struct MomSide {  // what a side's solve reads besides its rows
  int kb;
  bool wet;
  double g1, g2, grav3, Cd, hhat, chi;  // g1, g2: the lane's component of the two gradients
};

__device__ __forceinline__ void momentum_side(int nv, const StepArgs& a, const MomSide& q, int c, double* zc, double* u) {
  const int kb = q.kb;
  const double rc = c ? a.rmaxvel * 1.013 : a.rmaxvel;
  if (!q.wet) {
    for (int k = 0; k < nv; ++k) u[2 * k + c] = 0.0;
    return;
  }
  const double dt = a.dt, th = a.theta;
  if (kb == nv - 2) {
    const double htot = zc[nv - 1] - zc[kb];
    const double hc = u[2 * (nv - 1) + c] + dt * (0.0 - q.grav3 * ((1.0 - th) * q.g1 + th * q.g2));
    const double vc = fmin(fmax(hc * q.hhat / htot, -rc), rc);
    for (int k = 0; k < nv; ++k) u[2 * k + c] = vc;
  } else {
    const double G = q.grav3 * (th * q.g2 + (1.0 - th) * q.g1);
    const double td = dt * a.dfv0;
    // dz/6, dz/3 and dt dfv0 / dz of layer (k, k+1); the next row reuses them for its layer
    // (k-1, k), whose dz is the same difference of the same two levels. dz/6 = (dz/3) 0.5
    // exactly: halving commutes with rounding for normal values.
    double z0 = zc[kb + 1], zp = zc[kb + 2];                                        // zc[k], zc[k+1]
    double bm = u[2 * kb + c], b0 = u[2 * (kb + 1) + c], bp = u[2 * (kb + 2) + c];  // btu of this component
    // row kb + 1 (never the top one)
    double dzp = zp - z0;
    double tp = td / dzp, d3p = third(dzp), d6p = d3p * 0.5;
    double bet = (d3p + tp) + dt * q.chi;
    double cprev = d6p - tp;
    double up = (-(0.5 * dzp) * dt * G + d6p * (2.0 * b0 + bp)) / bet;
    u[2 * kb + c] = up;
    z0 = zp, bm = b0, b0 = bp;
    // rows kb + 2 .. nv - 2
    for (int k0 = kb + 2; k0 < nv - 1; k0 += kMomAhead) {
      double zb[kMomAhead], bb[kMomAhead];
#pragma unroll
      for (int j = 0; j < kMomAhead; ++j) {
        const int k = min(k0 + 1 + j, nv - 1);
        zb[j] = zc[k];
        bb[j] = u[2 * k + c];
      }
#pragma unroll
      for (int j = 0; j < kMomAhead; ++j) {
        const int k = k0 + j;
        if (k < nv - 1) {
          zp = zb[j];
          bp = bb[j];
          const double dz_1 = zp - z0;
          const double tq = td / dz_1, d3 = third(dz_1), d6 = d3 * 0.5;
          const double aj = d6p - tp;
          const double bj = (d3 + tq) + (d3p + tp);
          double r = -(0.5 * (dz_1 + dzp)) * dt * G;
          r += d6 * (2.0 * b0 + bp);
          r += d6p * (2.0 * b0 + bm);
          const double gam = cprev / bet;
          bet = bj - aj * gam;
          up = (r - aj * up) / bet;
          zc[k - 1] = gam;
          u[2 * (k - 1) + c] = up;
          cprev = d6 - tq;
          dzp = dz_1, tp = tq, d3p = d3, d6p = d6;
          z0 = zp, bm = b0, b0 = bp;
        }
      }
    }
    // row nv - 1
    {
      const double aj = d6p - tp, bj = d3p + tp;
      double r = -(0.5 * dzp) * dt * G;
      r += d6p * (2.0 * b0 + bm);
      const double gam = cprev / bet;
      bet = bj - aj * gam;
      up = (r - aj * up) / bet;
      zc[nv - 2] = gam;
    }
    // back substitution: u_j (slot kb + j) -= gam_{j+1} (zc slot kb + j + 1) u_{j+1}, each value
    // clamped into the slot above, whose own value has been read
    u[2 * (nv - 1) + c] = fmin(fmax(up, -rc), rc);
    for (int k0 = nv - 3; k0 >= kb; k0 -= kMomAhead) {
      double gb[kMomAhead], ub[kMomAhead];
#pragma unroll
      for (int j = 0; j < kMomAhead; ++j) {
        const int k = max(k0 - j, kb);
        gb[j] = zc[k + 1];
        ub[j] = u[2 * k + c];
      }
#pragma unroll
      for (int j = 0; j < kMomAhead; ++j) {
        const int k = k0 - j;
        if (k >= kb) {
          up = ub[j] - gb[j] * up;
          u[2 * (k + 1) + c] = fmin(fmax(up, -rc), rc);
        }
      }
    }
  }
  // bottom condition, imm = 0
  if (q.Cd == 0.0) {
    u[2 * kb + c] = u[2 * (kb + 1) + c];
  } else if (kb < nv - 2) {
    u[2 * kb + c] = 0.0;
  }
  for (int k = 0; k < kb; ++k) u[2 * k + c] = 0.0;
}

// The free-slip projection of a land side (side_type 1), both components, by the side's lane 0
// after both lanes' momentum_side.
__device__ void momentum_free_slip(const DMesh& m, int s, double* u) {
  if (m.side_type[s] != 1) return;
  const int nv = m.nvrt;
  const int kb = m.side_kb[s];
  const int4 sr = m.side[s];
  // free slip: the tangential component, t = (-n.y, n.x), n from populateSides (meshdata.cu:2283-2287)
  const double vx = -(m.y[sr.x] - m.y[sr.y]), vy = m.x[sr.x] - m.x[sr.y];
  const double len = sqrt(vx * vx + vy * vy);
  const double nx = vx / len, ny = vy / len;
  const double tx = -ny, ty = nx;
  for (int k = kb; k < nv; ++k) {
    const double vtan = u[2 * k] * tx + u[2 * k + 1] * ty;
    u[2 * k] = vtan * tx;
    u[2 * k + 1] = vtan * ty;
  }
}

// A wave takes g <= 32 consecutive sides: their zc and btu rows come into LDS with flat coalesced
// loads, two lanes per side solve in LDS (one component each), the u2 rows leave with flat stores.
// 24 KB of LDS allow six waves on a CU, so what a wave waits for is what the kernel takes: all its
// loads (kMomItems of either array per lane, and the records of its sides) are in flight together
// (of 25 us a wave, 16 went into loads waited for in turn; 645,122 sides x 31 levels: 387 -> 186 us,
// 4.3 TB/s; now half the time is the serial sweep, four divisions a level).
// Strides: zs odd and us = 2 zs spread the sides' reads of one level over the banks.
// NI, the items of either array per lane, is a power of two up to kMomItems with g sides' rows in 64 NI
// items: 32 sides of few levels would otherwise read and write their last item many times over, at two
// waves a SIMD (156,000 sides, 16 items / as many as they need: 2 levels 16.7 / 11.1 us, 5 levels 21.1 /
// 15.8, 8 levels 25.6 / 19.9; 840,000 sides x 16 levels 149 with 8 items).
constexpr int kMomItems = 16;
constexpr int kMomLds = 24 * 1024;

template <int NI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, NI < kMomItems ? 8 : 2)))
k_momentum(DMesh m, StepArgs a, int g) {
  extern __shared__ double lds[];
  const int nv = m.nvrt, zs = nv | 1, us = 2 * zs;
  double* Lu = lds;
  double* Lz = lds + g * us;
  const int s0 = blockIdx.x * g;
  const int gc = min(g, m.ns - s0);
  const int total = gc * nv;  // <= 64 NI
  const int t = threadIdx.x, sl = t >> 1, c = t & 1;
  const float inv = 1.0f / (float)nv;
  const double* zc = m.zc + (int64_t)s0 * nv;
  const f64x2* btu = reinterpret_cast<const f64x2*>(m.btu) + (int64_t)s0 * nv;
  const int s = s0 + min(sl, gc - 1);
  const int4 sr = m.side[s];
  __builtin_amdgcn_sched_barrier(0);  // the compiler would move each load down to its use
  double z[NI];
  f64x2 b[NI];
  // past the end the last item is read and written again
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int i = min(t + 64 * j, total - 1);
    z[j] = zc[i];
    b[j] = btu[i];
  }
  __builtin_amdgcn_sched_barrier(0);
  const SideElem el = side_elem_load(m, c ? sr.w : sr.z);
  MomSide q;
  q.kb = m.side_kb[s];
  q.wet = m.side_wet[s] != 0;
  q.hhat = m.hhat[s];
  q.chi = m.chi[s];
  const double gr0 = m.grav2[sr.x], gr1 = m.grav2[sr.y], cd0 = m.cd[sr.x], cd1 = m.cd[sr.y];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    int k;
    const int r = split_row(min(t + 64 * j, total - 1), inv, nv, k);
    Lz[r * zs + k] = z[j];
    *reinterpret_cast<f64x2*>(Lu + r * us + 2 * k) = b[j];
  }
  q.grav3 = 0.5 * (gr0 + gr1);
  q.Cd = 0.5 * (cd0 + cd1);
  side_eta_grads(el, a.h0, c, q.g1, q.g2);
  wave_lds_sync();
  if (sl < gc) momentum_side(nv, a, q, c, Lz + sl * zs, Lu + sl * us);
  wave_lds_sync();
  if (sl < gc && c == 0) momentum_free_slip(m, s0 + sl, Lu + sl * us);
  wave_lds_sync();
  f64x2* out = reinterpret_cast<f64x2*>(m.su2) + (int64_t)s0 * nv;
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int i = t + 64 * j;
    if (i < total) {
      int k;
      const int r = split_row(i, inv, nv, k);
      out[i] = *reinterpret_cast<const f64x2*>(Lu + r * us + 2 * k);
    }
  }
}

// shapiroFilter1 + shapiroFilter2 (meshdata.cu:5456-5518) in one pass that writes every side's
// final u2 into `out` (the caller then swaps it with u2). For a wet internal side, level k > kb
// takes bcc[k] = u2[k] + shapiro0 (0.25 sum_j u2_j[kin_j] - u2[k]) over its four neighbours
// Side::neigh(j) (meshdata.h:1409-1422: the sides before (j = 0, 1) and after (j = 2, 3) it in
// elements 0 and 1, summed in that order; kin_j = max(k, kb_j + 1) for a wet neighbour); a 2D
// side's bottom slot takes bcc[kb+1] (recomputed by its own thread, the same bits); levels below
// kb - 1 become 0; every other value, and boundary and dry sides, pass through unchanged.
// A workgroup takes 256 kShItems consecutive (side, level) items. Each side's record (kb, its four
// neighbours and the lowest level each contributes, kb_j + 1 for a wet neighbour) is read once into
// LDS, a chain of three loads; then each thread has the five u2 loads of its kShItems items in flight
// together. A side that passes through is its own four neighbours: no branch between the loads.
// 645,122 sides x 31 levels: 274 -> 136 us, 4.7 TB/s of rows read once and written once (one item a
// thread 264, two 196, three 142, six 151).
constexpr int kShItems = 4;

__global__ void __launch_bounds__(256) k_shapiro(DMesh m, double shapiro0, double* __restrict__ out) {
  extern __shared__ int4 Lsh[];  // per side: neighbours, their lowest levels, (kb, filtered, -, -)
  const int nv = m.nvrt;
  const int64_t t0 = (int64_t)blockIdx.x * (256 * kShItems);
  const int64_t total = (int64_t)m.ns * nv;
  // a 32-bit division below 2^32 (the 64-bit one is a long instruction sequence)
  auto side_of = [&](int64_t tt) { return (tt < 0xffffffffll) ? (int)((uint32_t)tt / (uint32_t)nv) : (int)(tt / nv); };
  const int sfirst = side_of(t0), nsd = side_of(min(t0 + 256 * kShItems, total) - 1) - sfirst + 1;
  const int off = (int)(t0 - (int64_t)sfirst * nv);
  for (int q = threadIdx.x; q < nsd; q += blockDim.x) {
    const int sd = sfirst + q;
    // all loads of a step together: the values are combined without branches
    const int4 g4 = reinterpret_cast<const int4*>(m.side_nbr)[sd];  // -1 on boundary sides
    const int kb = m.side_kb[sd], wet = m.side_wet[sd];
    int4 nb = g4.x >= 0 ? g4 : make_int4(sd, sd, sd, sd);
    const int w0 = m.side_wet[nb.x], w1 = m.side_wet[nb.y], w2 = m.side_wet[nb.z], w3 = m.side_wet[nb.w];
    const int k0 = m.side_kb[nb.x], k1 = m.side_kb[nb.y], k2 = m.side_kb[nb.z], k3 = m.side_kb[nb.w];
    const bool filtered = wet && g4.x >= 0;
    auto low = [](int w, int k) { return ((k + 1) & -w) | (w - 1); };  // w ? k + 1 : -1
    int4 kin = make_int4(low(w0, k0), low(w1, k1), low(w2, k2), low(w3, k3));
    if (!filtered) {
      nb = make_int4(sd, sd, sd, sd);
      kin = make_int4(-1, -1, -1, -1);
    }
    Lsh[3 * q] = nb;
    Lsh[3 * q + 1] = kin;
    Lsh[3 * q + 2] = make_int4(kb, filtered, 0, 0);
  }
  __syncthreads();
  const double2* u2 = reinterpret_cast<const double2*>(m.su2);
  double2* o = reinterpret_cast<double2*>(out);
  const float inv = 1.0f / (float)nv;
  double2 v[kShItems][5];
  int kk[kShItems], kbf[kShItems];
#pragma unroll
  for (int j = 0; j < kShItems; ++j) {
    const int i = (int)min((int64_t)threadIdx.x + 256 * j, total - 1 - t0);
    int k;
    const int q = split_row(off + i, inv, nv, k);
    const int4 nb = Lsh[3 * q], kin = Lsh[3 * q + 1], f = Lsh[3 * q + 2];
    // the level whose filtered value this slot takes
    const int kf = (f.y && f.x == nv - 2 && k >= f.x) ? f.x + 1 : k;
    v[j][0] = u2[(int64_t)nb.x * nv + max(kf, kin.x)];
    v[j][1] = u2[(int64_t)nb.y * nv + max(kf, kin.y)];
    v[j][2] = u2[(int64_t)nb.z * nv + max(kf, kin.z)];
    v[j][3] = u2[(int64_t)nb.w * nv + max(kf, kin.w)];
    v[j][4] = u2[(int64_t)(sfirst + q) * nv + kf];
    kk[j] = k;
    kbf[j] = f.y ? f.x : 0x7fffffff;
  }
#pragma unroll
  for (int j = 0; j < kShItems; ++j) {
    const int64_t t = t0 + threadIdx.x + 256 * j;
    if (t >= total) break;
    // u2 + shapiro0 (sum of the four neighbours' u2 / 4 - u2), neighbour j at level max(kf, kb_j + 1)
    // when wet, in Side::neigh order
    double sx = 0.0, sy = 0.0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      sx += v[j][h].x;
      sy += v[j][h].y;
    }
    const double2 u = v[j][4];
    const int k = kk[j], kb = kbf[j];
    double2 r = make_double2(u.x + shapiro0 * (0.25 * sx - u.x), u.y + shapiro0 * (0.25 * sy - u.y));
    if (kb == 0x7fffffff || k == kb - 1 || (k == kb && kb < nv - 2))
      r = u;
    else if (k < kb - 1)
      r = make_double2(0.0, 0.0);
    o[t] = r;
  }
}

void launch_shapiro(const DMesh& m, double shapiro0, double* out, hipStream_t st) {
  const int64_t total = (int64_t)m.ns * m.nvrt;
  if (total <= 0) return;
  constexpr int kItems = 256 * kShItems;
  const size_t lds = 3 * sizeof(int4) * ((kItems - 1) / m.nvrt + 2);  // the sides that a workgroup's items touch
  hipLaunchKernelGGL(k_shapiro, dim3((unsigned)((total + kItems - 1) / kItems)), dim3(256), lds, st, m, shapiro0, out);
}

void launch_momentum(const DMesh& m, const StepArgs& a, hipStream_t st) {
  if (m.ns <= 0) return;
  // sides per wave: one per two lanes, as many as 24 KB of LDS and kMomItems loads a lane hold
  const int row = 24 * (m.nvrt | 1);
  const int g = max(1, min(32, min(kMomLds / row, 64 * kMomItems / m.nvrt)));
  auto go = [&](auto ker) {
    hipLaunchKernelGGL(ker, dim3((unsigned)((m.ns + g - 1) / g)), dim3(64), (size_t)g * row, st, m, a, g);
  };
  const int items = (g * m.nvrt + 63) / 64;
  if (items <= 2)
    go(k_momentum<2>);
  else if (items <= 4)
    go(k_momentum<4>);
  else if (items <= 8)
    go(k_momentum<8>);
  else
    go(k_momentum<kMomItems>);
}

// ---------------------------------------------------------------- vertical velocity
// computeVerticalVelocity (meshdata.cu:5978-6102), triangles, ics=1, imm=0: element w from the
// flux balance of its prisms, bottom up, with the levels of the last level update (node z from
// the elevation of that update, side zc and kb) and the side velocities u2. A workgroup takes E
// elements. Phase 1, one thread per (element, level l): the side fluxes of layer (l, l+1), the
// horizontal flux through the face at level l+1 and that face's n_z A (Element::n,
// meshdata.cu:559-631); phase 2, one thread per element: the running top flux
// top_l = -side_l - bottom_l, bottom_l+1 = -top_l, in the reference's order; phase 3, one thread
// per (element, level): w = (top - horizontal) / (n_z A), stored with coalesced writes.
// 55 % of the time is VALU issue (a square root, four divisions and the geometry of each face), the
// rest the three loads one after the other before phase 1's values are there: the side normals come
// from the mesh (DMesh::side_geo), the level function has no branches (VM), and the bottom velocity
// is phase 1's own (645,122 sides x 31 levels: 308 -> 219 us, 2.2 TB/s).

// Per-element values that every level of phase 1 reads: node positions and level data, side
// normals (populateSides, meshdata.cu:2283-2287), orientation signs, lengths and bottom levels.
struct VvElem {
  double px[3], py[3], eta[3], h[3];
  double snx[3], sny[3], sign[3], slen[3];
  double area;
  int nkb[3], s[3], skb[3], dry[3], nd[3];
  int kb;  // the element's bottom level, nvrt when it is dry
};

template <int VM>
__global__ void __launch_bounds__(256) k_vertical_velocity(DMesh m, double h0, int E) {
  extern __shared__ double lds[];
  const int nv = m.nvrt, nvp = nv - 1;
  double* Lsf = lds;            // [E][nvp]: side flux of layer (l, l+1), then the top flux
  double* Lth = Lsf + E * nvp;  // [E][nvp]: horizontal flux through the face at level l+1
  double* Lden = Lth + E * nvp; // [E][nvp]: n_z A of that face
  double* Lbw = Lden + E * nvp; // [E]: w at the element's bottom level
  VvElem* Lel = reinterpret_cast<VvElem*>(Lbw + E);  // [E]
  const int e0 = blockIdx.x * E;
  const int ec = min(E, m.ne - e0);
  // three threads per element, thread j taking corner j and side j
  for (int t = threadIdx.x; t < 3 * ec; t += blockDim.x) {
    const int el = t / 3, j = t - 3 * el;
    const int e = e0 + el;
    VvElem& q = Lel[el];
    const int* er = reinterpret_cast<const int*>(m.elem + 2 * (int64_t)e);  // nodes 0-2, sides 0-2
    const int i = er[j], s = er[3 + j];
    const double4 sg = m.side_geo[s];
    const double eta = m.eta_lev[i], h = m.depth[i];
    q.px[j] = m.x[i];
    q.py[j] = m.y[i];
    q.eta[j] = eta;
    q.h[j] = h;
    q.nkb[j] = m.kb[i];
    q.nd[j] = i;
    q.dry[j] = eta + h <= h0;  // isDry2 at the level update
    q.snx[j] = sg.x;
    q.sny[j] = sg.y;
    q.slen[j] = sg.z;
    q.sign[j] = sg.w == (double)e ? 1.0 : -1.0;
    q.s[j] = s;
    q.skb[j] = m.side_kb[s];
    const int wet = m.elem_wet[e], kb = m.elem_kb[e];
    const double area = m.area[e];
    if (j == 0) {
      q.area = area;
      q.kb = wet ? kb : nv;
    }
  }
  __syncthreads();
  const float inv = 1.0f / (float)nvp;
  for (int idx = threadIdx.x; idx < ec * nvp; idx += blockDim.x) {
    int l;
    const int el = split_row(idx, inv, nvp, l);
    const VvElem& q = Lel[el];
    if (l < q.kb) continue;
    double2 ut[3], ul[3];
    double zt[3], zl[3], sg[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      // the face's sigma: its level's, its nodes' from their beds up, or (SZ) its sigma, C and Z level
      if (VM == 0) sg[j] = m.sigma[l + 1];
      if (VM == 1) sg[j] = m.sig_node[(int64_t)q.nd[j] * nv + max(l + 1, q.nkb[j])];
      if (VM == 2) sg[j] = j == 0 ? m.ssig[max(l + 1 - m.izlev, 0)] : (j == 1 ? m.cs[max(l + 1 - m.izlev, 0)] : m.ztot[min(l + 1, m.izlev)]);
      const int64_t row = (int64_t)q.s[j] * nv;
      const int kt = max(l + 1, q.skb[j]), kl = max(l, q.skb[j]);
      const double2* u2 = reinterpret_cast<const double2*>(m.su2) + row;
      ut[j] = u2[kt];
      ul[j] = u2[kl];
      zt[j] = m.zc[row + kt];
      zl[j] = m.zc[row + kl];
    }
    if (l == q.kb) {
      // w at the bottom: -grad(h) . u there (kl is then the side's own bottom level)
      const double* gp = m.gradphi + 6 * (int64_t)(e0 + el);
      const double ghx = q.h[0] * gp[0] + q.h[1] * gp[2] + q.h[2] * gp[4];
      const double ghy = q.h[0] * gp[1] + q.h[1] * gp[3] + q.h[2] * gp[5];
      const double ubx = third(ul[0].x + ul[1].x + ul[2].x + 0.0), uby = third(ul[0].y + ul[1].y + ul[2].y + 0.0);
      const double bottomW = -(ghx * ubx + ghy * uby);
      Lbw[el] = 0.0 + bottomW;
    }
    // the face at level l+1 (node levels clamped to each node's bed), zcoord of the level update
    double pz[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double eta = q.eta[j], h = q.h[j];
      const int k = max(l + 1, q.nkb[j]);
      double z;
      if (VM == 2) {  // z_wet's SZ branch as selects
        const double hm = fmin(h, m.h_s);
        const double zs = hm <= m.h_c ? sg[0] * (hm + eta) + eta : eta * (1.0 + sg[0]) + m.h_c * sg[0] + (hm - m.h_c) * sg[1];
        z = k < m.izlev ? sg[2] : zs;
        z = k == q.nkb[j] ? -h : z;
        z = k == m.izlev ? -hm : z;
        z = k == nv - 1 ? eta : z;
      } else {
        z = (eta + h) * sg[j] + eta;
        z = k <= q.nkb[j] ? -h : (k == nv - 1 ? eta : z);
      }
      pz[j] = q.dry[j] ? 0.0 : z;
    }
    const double n20x = q.px[2] - q.px[0], n20y = q.py[2] - q.py[0], n20z = pz[2] - pz[0];
    const double n10x = q.px[1] - q.px[0], n10y = q.py[1] - q.py[0], n10z = pz[1] - pz[0];
    const double nx = (n10y) * (n20z) - (n20y) * (n10z);
    const double ny = (n20x) * (n10z) - (n10x) * (n20z);
    const double nz = 2.0 * q.area;
    const double len = sqrt(nx * nx + ny * ny + nz * nz);
    const double ta = 0.5 * len;
    const double inv_len = 1.0 / len;
    const double tnx = nx * inv_len, tny = ny * inv_len, tnz = nz * inv_len;
    double sf = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double ucx = 0.5 * (ut[j].x + ul[j].x), ucy = 0.5 * (ut[j].y + ul[j].y);
      const double sideArea = q.slen[j] * (zt[j] - zl[j]);
      sf += q.sign[j] * (ucx * q.snx[j] + ucy * q.sny[j]) * sideArea;
    }
    const double utx = third(ut[0].x + ut[1].x + ut[2].x + 0.0), uty = third(ut[0].y + ut[1].y + ut[2].y + 0.0);
    Lsf[idx] = sf;
    Lth[idx] = (utx * tnx + uty * tny) * ta;
    Lden[idx] = tnz * ta;
  }
  __syncthreads();
  if (threadIdx.x < ec) {
    const int el = threadIdx.x;
    // the running sums in level order; the side fluxes of 8 levels are read ahead so that
    // the dependent additions do not wait for LDS one at a time
    double bottom = 0.0;
    double* row = Lsf + el * nvp;
    for (int l0 = Lel[el].kb; l0 < nvp; l0 += 8) {
      double f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = (l0 + u < nvp) ? row[l0 + u] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (l0 + u < nvp) {
          const double top = -f[u] - bottom;
          row[l0 + u] = top;
          bottom = -top;
        }
    }
  }
  __syncthreads();
  double* w = m.ew + (int64_t)e0 * nv;
  const float invn = 1.0f / (float)nv;
  for (int idx = threadIdx.x; idx < ec * nv; idx += blockDim.x) {
    int k;
    const int el = split_row(idx, invn, nv, k);
    const int kb = Lel[el].kb;
    double v = 0.0;
    if (k == kb) {
      v = Lbw[el];
    } else if (k > kb) {
      const int j = el * nvp + k - 1;
      v = (Lsf[j] - Lth[j]) / Lden[j];
    }
    w[idx] = v;
  }
}

void launch_vertical_velocity(const DMesh& m, double h0, hipStream_t st) {
  if (m.ne <= 0 || m.nvrt < 2) return;
  const int nvp = m.nvrt - 1;
  // elements per workgroup: four (element, level) items a thread, within 32 KB of LDS (215,683 nodes x
  // 31 levels: one item 359 us, two 238, four 219, eight 224); one item where four would leave fewer
  // than two workgroups a CU (24 x 16 nodes x 8 levels 9.1 us with four, 5.8 with one; 200 x 80 x 31,
  // just above the line, 20.0 and 24.4)
  const size_t per_elem = 8 * (3 * (size_t)nvp + 1) + sizeof(VvElem);
  auto elems = [&](int items) { return max(1, min(items * 256 / nvp, (int)((32 * 1024) / per_elem))); };
  // two elements on more than 512 levels: phase 2 is one thread per element, and of workgroups of one
  // element registers let only five onto a CU (18,802 elements x 700 levels 622 us with one, 442 with two)
  const int two = 2 * per_elem <= 64 * 1024 ? 2 : 1;
  const int E = m.ne >= 512 * elems(4) ? max(two, elems(4)) : elems(1);
  const size_t lds = per_elem * E;
  auto go = [&](auto ker) { hipLaunchKernelGGL(ker, dim3((unsigned)((m.ne + E - 1) / E)), dim3(256), lds, st, m, h0, E); };
  if (m.vmode == 0)
    go(k_vertical_velocity<0>);
  else if (m.vmode == 1)
    go(k_vertical_velocity<1>);
  else
    go(k_vertical_velocity<2>);
}

// ---------------------------------------------------------------- a11+a12: assembly + BC
// setupCoefficientMatrixAndRHS for triangles, imm=0 (meshdata.cu:3182-3311), fused with
// setEssentialBC (meshdata.cu:4400-4446), in two passes. k_elem_assemble evaluates, once per
// element and corner id1, the terms the reference adds when node nodes[id1] visits the element
// in its ball: the three matrix entries (diagonal, next, previous corner) and the five RHS
// increments in their order (advective/ghat term, eta terms of corners 0-2, volume source).
// k_assemble then gives each node its CSR row (node-gather, no atomics) by adding those terms
// over its ball in ball order, so every sum has the reference's operands and order.
// Open nodes of elevation type 0 (no essential BC) add the boundary integral I_5; I_3 is zero
// because every open boundary here has flow type ifltype = 0 (meshdata.cu:3373-3470).
__global__ void __launch_bounds__(256) k_elem_assemble(DMesh m, StepArgs a) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= m.ne) return;
  const int4 r0 = m.elem[2 * e], r1 = m.elem[2 * e + 1];
  const int nd[3] = {r0.x, r0.y, r0.z};
  const int sd[3] = {r0.w, r1.x, r1.y};
  const double dt = a.dt, th = a.theta;
  const double grav3 = (m.grav2[nd[0]] + m.grav2[nd[1]] + m.grav2[nd[2]] + 0.0) / 3;
  const double hhatb = (m.hhat[sd[0]] + m.hhat[sd[1]] + m.hhat[sd[2]] + 0.0) / 3;
  const double area = m.area[e];
  const double Ux = (m.sU[2 * sd[0]] + m.sU[2 * sd[1]] + m.sU[2 * sd[2]] + 0.0) / 3;
  const double Uy = (m.sU[2 * sd[0] + 1] + m.sU[2 * sd[1] + 1] + m.sU[2 * sd[2] + 1] + 0.0) / 3;
  const double* g = m.gradphi + 6 * (int64_t)e;
  double gp[6];
  for (int l = 0; l < 6; ++l) gp[l] = g[l];
  const double ghx = m.ghat1[2 * e], ghy = m.ghat1[2 * e + 1];
  const double px[3] = {m.x[nd[0]], m.x[nd[1]], m.x[nd[2]]}, py[3] = {m.y[nd[0]], m.y[nd[1]], m.y[nd[2]]};
  const double eta[3] = {m.eta2[nd[0]], m.eta2[nd[1]], m.eta2[nd[2]]};
  const double wet = m.elem_wet[e] ? 1.0 : 0.0;
  const double src = (dt / 3) * m.vsource[e];
  const double fric = grav3 * th * (1.0 - th) * dt * dt * hhatb;
  const double c = grav3 * th * th * dt * dt * hhatb;
  double2* out = reinterpret_cast<double2*>(m.econ + 24 * (int64_t)e);
  for (int id1 = 0; id1 < 3; ++id1) {
    const double g1x = gp[2 * id1], g1y = gp[2 * id1 + 1];
    const double I41 = g1x * Ux + g1y * Uy;
    const double I42 = g1x * ghx + g1y * ghy;
    const double adv = dt * area * ((1 - th) * I41 + th * I42);
    const int id2 = (id1 + 1) % 3, id3 = (id1 + 2) % 3;
    const double x0x = px[id1], x0y = py[id1];
    const double x1x = px[id2], x1y = py[id2];
    const double x2x = px[id3], x2y = py[id3];
    const double ipp_ii = (1.0 / 6.0) * area, ipp_ij = (1.0 / 12.0) * area, ipp_ik = (1.0 / 12.0) * area;
    const double ax = x2x - x1x, ay = x2y - x1y;
    const double igpgp_ii = ((1.0 / 4.0) / area) * (ax * ax + ay * ay);
    const double igpgp_ij = ((1.0 / 4.0) / area) * (ax * (x0x - x2x) + ay * (x0y - x2y));
    const double igpgp_ik = -igpgp_ii - igpgp_ij;
    double q[3];
    for (int l = 0; l < 3; ++l) {
      const double ipp = ((id1 == l) ? (2.0 / 12.0) : (1.0 / 12.0)) * area;
      const double igpgp = area * (g1x * gp[2 * l] + g1y * gp[2 * l + 1]);
      q[l] = (eta[l] + 0.0) * ipp - eta[l] * fric * igpgp * wet;
    }
    out[4 * id1 + 0] = make_double2(ipp_ii + c * igpgp_ii, ipp_ij + c * igpgp_ij);
    out[4 * id1 + 1] = make_double2(ipp_ik + c * igpgp_ik, adv);
    out[4 * id1 + 2] = make_double2(q[0], q[1]);
    out[4 * id1 + 3] = make_double2(q[2], src);
  }
}

// Row accumulation for k_assemble: in LDS for rows of up to kRowLds entries, in the CSR values
// themselves for longer rows; both add the same terms in the same order.
constexpr int kRowLds = 16;

template <class Row>
__device__ __forceinline__ double assemble_row(const DMesh& m, const StepArgs& a, int i, int len, int diag, Row rv) {
  for (int k = 0; k < len; ++k) rv(k) = 0.0;
  double qel = 0.0;
  const double2* con = reinterpret_cast<const double2*>(m.econ);
  for (int j = m.ball_ptr[i]; j < m.ball_ptr[i + 1]; ++j) {
    const int64_t base = 4 * (3 * (int64_t)m.ball_elem[j] + m.ball_loc[j]);
    const double2 c0 = con[base], c1 = con[base + 1], c2 = con[base + 2], c3 = con[base + 3];
    qel += c1.y;
    rv(diag) += c0.x;
    rv(m.ball_slot[2 * j]) += c0.y;
    rv(m.ball_slot[2 * j + 1]) += c1.x;
    qel += c2.x;
    qel += c2.y;
    qel += c3.x;
    qel += c3.y;
  }
  // I_5 of an open node without an essential BC (meshdata.cu:3373-3380, 3457-3463): its two
  // boundary sides (open or land, ascending side index), the non-dry ones.
  if (m.open_bnd[i] && node_etype(m, a, i) == 0) {
    const int2 bs = m.node_bside[i];
    const int sl[2] = {bs.x, bs.y};
    for (int l = 0; l < 2; ++l) {
      const int s = sl[l];
      if (s < 0 || !m.side_wet[s]) continue;
      const int4 sr = m.side[s];
      const double vx = -(m.y[sr.x] - m.y[sr.y]), vy = m.x[sr.x] - m.x[sr.y];
      const double ql = sqrt(vx * vx + vy * vy);
      const double Unbar = m.sU[2 * s] * (vx / ql) + m.sU[2 * s + 1] * (vy / ql);
      qel -= 0.5 * (1.0 - a.theta) * a.dt * m.side_len[s] * Unbar;
    }
  }
  if (m.open_bnd[i] && node_etype(m, a, i) != 0) {
    for (int k = 0; k < len; ++k) rv(k) = 0.0;
    rv(diag) = 1.0;
    qel = m.elbc[i];
  } else {
    for (int j = m.nbr_ptr[i]; j < m.nbr_ptr[i + 1]; ++j) {
      const int nb = m.nbr_node[j];
      if (m.open_bnd[nb] && node_etype(m, a, nb) != 0) {
        const int sl = m.csr_slot[j];
        qel -= rv(sl) * m.elbc[nb];
        rv(sl) = 0.0;
      }
    }
  }
  return qel;
}

__global__ void __launch_bounds__(256) k_assemble(DMesh m, StepArgs a, double* __restrict__ val,
                                                  double* __restrict__ b) {
  __shared__ double rows[kRowLds][256];  // entry k of thread t's row at rows[k][t]
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.n) return;
  const int row = m.indptr[i];
  const int len = m.indptr[i + 1] - row;
  const int diag = m.diag_off[i];
  double qel;
  if (len <= kRowLds) {
    const int t = threadIdx.x;
    qel = assemble_row(m, a, i, len, diag, [&](int k) -> double& { return rows[k][t]; });
    for (int k = 0; k < len; ++k) val[row + k] = rows[k][t];
  } else {
    double* rv = val + row;
    qel = assemble_row(m, a, i, len, diag, [&](int k) -> double& { return rv[k]; });
  }
  b[i] = qel;
}

void launch_assemble(const DMesh& m, const StepArgs& a, double* val, double* b, hipStream_t st) {
  if (m.ne > 0) hipLaunchKernelGGL(k_elem_assemble, dim3((m.ne + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a);
  if (m.n > 0) hipLaunchKernelGGL(k_assemble, dim3((m.n + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, a, val, b);
}

// rollUpElevation + updateElevation (meshdata.cu:3538-3544, 4449-4456)
__global__ void k_update_elevation(DMesh m, const double* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m.n) return;
  m.eta1[i] = m.eta2[i];
  m.eta2[i] = x[i];
}

void launch_update_elevation(const DMesh& m, const double* x, hipStream_t st) {
  if (m.n > 0) hipLaunchKernelGGL(k_update_elevation, dim3((m.n + kTpb - 1) / kTpb), dim3(kTpb), 0, st, m, x);
}

}  // namespace gsh
