// pcg_kernels.hip -- Jacobi-preconditioned CG for gfx950 in two fused phases per iteration.
//
// The reference issues four launches per iteration (f_update_p, cuSPARSE SpMV, f_dot,
// f_update_xrz; pcg_loop.cpp:367-403) and sums dot products with one atomicAdd per block
// (pcg_solver.py:134-167), so its results are not reproducible. Here every iteration is
//   phase A  beta; p_new = z + beta p_old (own row and, on the fly, every column of the
//            stencil); q = A p_new (rows summed in column order); p.q
//   phase B  alpha; x += alpha p; r -= alpha q; z = invD r; r.r, r.z; stopping test
// with the same scalar recurrences as the reference (f_update_p / f_update_xrz,
// pcg_solver.py:208-276).
//
// Dot products use one fixed tree. A tile of 256*R rows is summed per thread over its R rows
// (thread tau takes rows tile*256R + 256 j + tau), then by a wave64 shuffle tree, then as
// (w0 + w1) + (w2 + w3) over the 4 waves; every consumer workgroup sums the tile partials with
// the same tree (thread t takes partials t, t+256, ...). A single-writer-per-scalar scheme with
// device-scope counters was measured slower: thousands of workgroups serialize on one atomic
// address across the XCDs. Results are bitwise reproducible and independent of how many
// workgroups run concurrently.
//
// A workgroup finds its system and tile through a launch table, so one launch advances any
// number of independent systems (batched and served solves); finished systems drop out
// through their device-side `done` flag.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.h"
#include "reduce.h"

namespace gsh {

template <class VT>
struct SysView {
  int n, ntiles;
  gptr<const int32_t> rowptr, col, diag;
  gptr<const int16_t> cdel;
  gptr<const VT> val;
  gptr<const double> b, h0, h1, h2;
  gptr<VT> x, r, z, pa, pb, q, invd;
  gptr<double> part_rr, part_rz, part_pq, part_bb;
  gptr<PcgState> st;
  bool has_hist, has_cdel;
};

template <class VT>
__device__ __forceinline__ SysView<VT> view(const PcgSys<VT>& S) {
  SysView<VT> v;
  v.n = S.n;
  v.ntiles = S.ntiles;
  v.rowptr = G(S.rowptr);
  v.col = G(S.col);
  v.diag = G(S.diag);
  v.has_cdel = S.cdel != nullptr;
  v.cdel = G(S.cdel);
  v.val = G(S.val);
  v.b = G(S.b);
  v.has_hist = S.h0 != nullptr;
  v.h0 = G(S.h0);
  v.h1 = G(S.h1);
  v.h2 = G(S.h2);
  v.x = G(S.x);
  v.r = G(S.r);
  v.z = G(S.z);
  v.pa = G(S.pa);
  v.pb = G(S.pb);
  v.q = G(S.q);
  v.invd = G(S.invd);
  v.part_rr = G(S.part_rr);
  v.part_rz = G(S.part_rz);
  v.part_pq = G(S.part_pq);
  v.part_bb = G(S.part_bb);
  v.st = G(S.st);
  return v;
}

// ------------------------------------------------------------------ state reset
// rtols (device, may be NULL): per-system relative tolerances instead of rtol.
template <class VT>
__global__ void k_pcg_reset(const PcgSys<VT>* sys, int nsys, double rtol, int maxiter, int check_every,
                            const double* __restrict__ rtols) {
  const int sidx = blockIdx.x * blockDim.x + threadIdx.x;
  if (sidx >= nsys) return;
  if (rtols) rtol = rtols[sidx];
  gptr<PcgState> st = G(sys[sidx].st);
  st->k = 0;
  st->kk = 0;
  st->done = -1;
  st->zero = 0;
  st->maxiter = maxiter;
  st->check_every = check_every;
  st->rtol = rtol;
  st->atol2 = 0.0;
  st->rr_last = -1.0;
  st->bb = 0.0;
  st->rho[0] = 0.0;
  st->rho[1] = 0.0;
  st->gave_up = 0;
}

// ------------------------------------------------------------------ CSR row sums (block staged)
// Sums row i = r0 + threadIdx.x of A*v, v(c) given by `vf`, in column order. The chunk's
// products are staged in LDS with coalesced loads of val/col when they fit.
template <class VT, class VF>
__device__ __forceinline__ VT csr_chunk(gptr<const int32_t> rowptr, gptr<const int32_t> col, gptr<const VT> val,
                                        int n, int r0, VT* lds, VF vf) {
  const int i = r0 + threadIdx.x;
  const int rend = min(r0 + kTpb, n);
  const int s0 = rowptr[r0], e0 = rowptr[rend];
  VT acc = (VT)0;
  if (e0 - s0 <= kSpmvLdsCap) {
    for (int k = s0 + threadIdx.x; k < e0; k += kTpb) lds[k - s0] = val[k] * vf(col[k]);
    __syncthreads();
    if (i < n) {
      const int a = rowptr[i], b = rowptr[i + 1];
      for (int k = a; k < b; ++k) acc += lds[k - s0];
    }
    __syncthreads();
  } else if (i < n) {
    const int a = rowptr[i], b = rowptr[i + 1];
    for (int k = a; k < b; ++k) acc += val[k] * vf(col[k]);
  }
  return acc;
}

// ------------------------------------------------------------------ init
// extrapolateGuess + computeResiduals + computeInvDiag + f_init (pcg_solver.py:881-938, 172-182):
// x = 3 x0 - 3 x1 + x2; r = b - A x; invD = 1/diag; z = invD r; p_old = 0; partials of r.r, r.z, b.b.
template <class VT, int R>
__global__ void __launch_bounds__(256) k_pcg_init(const PcgSys<VT>* __restrict__ sys,
                                                  const TileRef* __restrict__ tiles) {
  __shared__ double red[4];
  __shared__ VT lds[kSpmvLdsCap];
  const TileRef tr = tiles[xcd_block(blockIdx.x, gridDim.x)];
  const SysView<VT> S = view(sys[tr.sys]);
  const int n = S.n;
  const gptr<const double> h0 = S.h0, h1 = S.h1, h2 = S.h2;
  const bool hist = S.has_hist;
  auto xe = [&](int c) -> VT {
    if (!hist) return (VT)0;
    return (VT)((3.0 * h0[c] - 3.0 * h1[c]) + h2[c]);
  };
  double rr = 0.0, rz = 0.0, bb = 0.0;
  const int base = tr.tile * kTpb * R;
  for (int j = 0; j < R; ++j) {
    const int r0 = base + j * kTpb;
    if (r0 >= n) break;
    const VT q = csr_chunk<VT>(S.rowptr, S.col, S.val, n, r0, lds, xe);
    const int i = r0 + threadIdx.x;
    if (i < n) {
      const VT xi = xe(i);
      S.x[i] = xi;
      const VT inv = (VT)(1.0 / (double)S.val[S.diag[i]]);
      S.invd[i] = inv;
      const double bi = S.b[i];
      const VT ri = (VT)(bi - (double)q);
      const VT zi = inv * ri;
      S.r[i] = ri;
      S.z[i] = zi;
      S.pb[i] = (VT)0;
      rr += (double)ri * (double)ri;
      rz += (double)ri * (double)zi;
      bb += bi * bi;
    }
  }
  rr = block_tree(rr, red);
  rz = block_tree(rz, red);
  bb = block_tree(bb, red);
  if (threadIdx.x == 0) {
    S.part_rr[tr.tile] = rr;
    S.part_rz[tr.tile] = rz;
    S.part_bb[tr.tile] = bb;
  }
}

// ------------------------------------------------------------------ phase A
// f_update_p + SpMV + f_dot (pcg_solver.py:208-249): beta = rz(k-1)/rz(k-2) (0 at k = 0),
// p = z + beta p, q = A p, p.q.
//
// Each wave owns the 64 consecutive rows r0w..r0w+63 of a sub-round (thread tau = 64w + lane
// handles row base + 256 j + tau, the rows of the fixed reduction order). The wave loads the
// chunk's nonzeros coalesced (lane l takes entries s0 + l + 64 m) together with the z and p_old
// gathers; the products go to the wave's LDS slice and each lane sums its own row in column
// order. Columns are read as int16 offsets from the chunk's first row when they fit.
//
// W: a workgroup of 256 R threads, one row each, the tile's p.q summed in the R-rows-per-thread order
// (tile_tree_wide), so results equal the 256-thread form's bit for bit. The 256-thread form walks
// its R sub-rounds one after another, each waiting for entries and then gathers; the wide form has
// all 4 R chunks of a tile in flight, which a system of few tiles needs (launch_pcg_phase).
//
// What the two forms load first differs. The wide one, a single wait chain per thread, requests the
// row pointers before the done test and every column before the first gather. The narrow one runs
// where many waves share a SIMD, and among a batch's finished systems: it tests done first, and its
// FP32 chunk takes each entry's column and gathers together, which keeps it at 71 registers and 7
// waves a SIMD (with every column held at once 76 and 6: batched mixed Jacobi solves of 16 x 501,264
// rows 19.3 ms against 16.8, of 96 systems of 5,000 to 200,000 rows 12.6 against 11.8).
template <class VT, bool W>
struct Chunk {
  // nonzeros of a 64-row chunk held in registers, per lane. The narrow form sums a longer chunk row by
  // row; the wide one, whose four times as many rows in flight then ran the caches over (500,000 rows of
  // 15 entries 156 us an iteration against 62), takes it in pieces (50 us).
  static constexpr int kM = W ? kWideChunk / 64 : 10, kCap = 64 * kM;
  int s0, e0;
  VT v[kM], zc[kM], pc[kM];
};

template <class VT>
__device__ __forceinline__ int col_of(const SysView<VT>& S, int kk, int base64) {
  return S.has_cdel ? base64 + (int)S.cdel[kk] : S.col[kk];
}

// s0, e0: the chunk's first entry and the entry after its last (rowptr at r0w and r0w + 64)
template <class VT, bool W>
__device__ __forceinline__ void load_chunk(const SysView<VT>& S, gptr<const VT> po, int r0w, int lane, int s0, int e0,
                                           Chunk<VT, W>& c) {
  c.s0 = s0;
  c.e0 = e0;
  if (c.e0 - c.s0 > c.kCap) return;
  if constexpr (!W) {
#pragma unroll
    for (int m = 0; m < c.kM; ++m) {
      const int kk = c.s0 + lane + 64 * m;
      if (kk < c.e0) {
        const int col = col_of(S, kk, r0w);
        c.v[m] = S.val[kk];
        c.zc[m] = S.z[col];
        c.pc[m] = po[col];
      }
    }
    return;
  }
  int col[c.kM];
#pragma unroll
  for (int m = 0; m < c.kM; ++m) {
    const int kk = c.s0 + lane + 64 * m;
    if (kk < c.e0) {
      col[m] = col_of(S, kk, r0w);
      c.v[m] = S.val[kk];
    }
  }
#pragma unroll
  for (int m = 0; m < c.kM; ++m) {
    const int kk = c.s0 + lane + 64 * m;
    if (kk < c.e0) {
      c.zc[m] = S.z[col[m]];
      c.pc[m] = po[col[m]];
    }
  }
}

template <class VT, int R, bool W>
__device__ __forceinline__ void pcg_phase_a_body(const SysView<VT>& S, int tile, double* red, VT* lds) {
  constexpr int kCap = Chunk<VT, W>::kCap, J = W ? 1 : R;
  gptr<PcgState> st = S.st;
  const int n = S.n;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int base = tile * kTpb * R;
  if (!W && load_done(st) >= 0) return;
  // FP64: the row pointers of every sub-round first: they depend on nothing, so each sub-round's
  // chunk then waits for two memory steps (entries, then gathers) instead of three. FP32 loads them
  // per sub-round: its registers would otherwise drop it from 7 to 5 waves per SIMD, which its
  // batched launches of small systems need more.
  constexpr bool kPre = W || sizeof(VT) == 8;
  int cs0[J], ce0[J], ra[J], rb[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r0w = base + j * kTpb + w * 64;
    cs0[j] = ce0[j] = ra[j] = rb[j] = 0;
    if (kPre && r0w < n) {
      cs0[j] = S.rowptr[r0w];
      ce0[j] = S.rowptr[min(r0w + 64, n)];
      const int i = r0w + lane;
      if (i < n) {
        ra[j] = S.rowptr[i];
        rb[j] = S.rowptr[i + 1];
      }
    }
  }
  if (W && load_done(st) >= 0) return;
  const int k = st->k;
  const gptr<VT> pn = (k & 1) ? S.pb : S.pa;
  const gptr<const VT> po = (k & 1) ? S.pa : S.pb;
  // a sub-round's first and end entries and the thread's row range (FP32: loaded here)
  auto rows_of = [&](int j, int r0w) {
    if (!kPre) {
      cs0[j] = S.rowptr[r0w];
      ce0[j] = S.rowptr[min(r0w + 64, n)];
      const int i = r0w + lane;
      if (i < n) {
        ra[j] = S.rowptr[i];
        rb[j] = S.rowptr[i + 1];
      }
    }
  };
  const gptr<const VT> z = S.z;
  Chunk<VT, W> c;
  const int r00 = base + w * 64;
  VT zi0 = 0, pi0 = 0;  // the thread's own row (wide form: its only one)
  if (r00 < n) {
    rows_of(0, r00);
    load_chunk(S, po, r00, lane, cs0[0], ce0[0], c);
    if (W && r00 + lane < n) {
      zi0 = z[r00 + lane];
      pi0 = po[r00 + lane];
    }
  }
  const double rz_cur = W ? final_reduce_lo(S.part_rz, S.ntiles, red) : final_reduce(S.part_rz, S.ntiles, red);
  double beta = 0.0;
  if (k > 0) {
    const double rz_old = st->rho[(k - 1) & 1];
    beta = (rz_old == 0.0) ? 0.0 : rz_cur / rz_old;
  }
  if (tile == 0) {
    // workgroup 0: atol = rtol ||b|| at k = 0 (pcg_solver.py:928-930, 1089-1095), otherwise the
    // stopping test of iteration k-1 (pcg_loop.cpp:405-412)
    if (k == 0) {
      const double bb = W ? final_reduce_lo(S.part_bb, S.ntiles, red) : final_reduce(S.part_bb, S.ntiles, red);
      if (threadIdx.x == 0) {
        const double atol = st->rtol * sqrt(bb);
        st->bb = bb;
        st->atol2 = atol * atol;
        if (atol == 0.0) {
          st->zero = 1;
          st->done = 0;
        }
      }
    } else {
      const int it = k - 1;
      if ((it + 1) % st->check_every == 0 || it == st->maxiter - 1) {
        const double rr = W ? final_reduce_lo(S.part_rr, S.ntiles, red) : final_reduce(S.part_rr, S.ntiles, red);
        if (threadIdx.x == 0) {
          st->rr_last = rr;
          if (rr <= st->atol2) st->done = k;
        }
      }
    }
    if (threadIdx.x == 0) {
      st->rho[k & 1] = rz_cur;
      st->kk = k;
    }
  }
  const VT bv = (VT)beta;
  VT* my = lds + w * kCap;
  double pq = 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r0w = base + j * kTpb + w * 64;
    if (r0w >= n) break;
    if (j > 0) {
      rows_of(j, r0w);
      load_chunk(S, po, r0w, lane, cs0[j], ce0[j], c);
    }
    const int i = r0w + lane;
    VT q = (VT)0;
    if (c.e0 - c.s0 <= kCap) {
#pragma unroll
      for (int m = 0; m < c.kM; ++m) {
        const int kk = c.s0 + lane + 64 * m;
        if (kk < c.e0) my[kk - c.s0] = c.v[m] * (c.zc[m] + bv * c.pc[m]);
      }
      wave_lds_sync();
      if (i < n) {
        const int a = ra[j], b = rb[j];
        for (int kk = a; kk < b; ++kk) q += my[kk - c.s0];
      }
      wave_lds_sync();
    } else if (W) {
      // a longer chunk in pieces, each loaded as a chunk is and summed by the rows that it holds entries of
      for (int p0 = c.s0; p0 < c.e0; p0 += kCap) {
        Chunk<VT, W> d;
        const int p1 = min(p0 + kCap, c.e0);
        load_chunk(S, po, r0w, lane, p0, p1, d);
#pragma unroll
        for (int m = 0; m < d.kM; ++m) {
          const int kk = p0 + lane + 64 * m;
          if (kk < p1) my[kk - p0] = d.v[m] * (d.zc[m] + bv * d.pc[m]);
        }
        wave_lds_sync();
        const int a = max(ra[j], p0), b = min(rb[j], p1);
        for (int kk = a; kk < b; ++kk) q += my[kk - p0];
        wave_lds_sync();
      }
    } else if (i < n) {
      const int a = ra[j], b = rb[j];
      for (int kk = a; kk < b; ++kk) {
        const int col = col_of(S, kk, r0w);
        q += S.val[kk] * (z[col] + bv * po[col]);
      }
    }
    if (i < n) {
      const VT pi = (W ? zi0 : z[i]) + bv * (W ? pi0 : po[i]);
      pn[i] = pi;
      S.q[i] = q;
      const double t = (double)pi * (double)q;
      if (W)
        pq = t;
      else
        pq += t;
    }
  }
  // the wide form's row values pass through the first 64 words of each wave's own product slice
  if (W)
    pq = tile_tree_wide<R, kCap * (int)sizeof(VT) / 8>(pq, reinterpret_cast<double*>(lds), red);
  else
    pq = block_tree(pq, red);
  if (threadIdx.x == 0) S.part_pq[tile] = pq;
}

// The launch table names each workgroup's system and tile; one system (tiles = NULL) needs none.
template <class VT, int R, bool W>
__global__ void __launch_bounds__(W ? kTpb * R : kTpb) k_pcg_phase_a(const PcgSys<VT>* __restrict__ sys,
                                                                     const TileRef* __restrict__ tiles) {
  __shared__ double red[4];
  __shared__ __align__(8) VT lds[(W ? 4 * R : 4) * Chunk<VT, W>::kCap];
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const TileRef tr = tiles ? tiles[b] : TileRef{0, b};
  pcg_phase_a_body<VT, R, W>(view(sys[tr.sys]), tr.tile, red, lds);
}

// ------------------------------------------------------------------ phase B
// f_update_xrz (pcg_solver.py:253-276): alpha = rz / pq (0 if pq == 0). The row loads are
// issued before the scalar reduction, which only the arithmetic waits for. W as in phase A.
template <class VT, int R, bool W>
__device__ __forceinline__ void pcg_phase_b_body(const SysView<VT>& S, int tile, double* red, double* lrows) {
  constexpr int J = W ? 1 : R;
  gptr<PcgState> st = S.st;
  const int n = S.n;
  const int base = tile * kTpb * R;
  if (!W && load_done(st) >= 0) return;
  VT xv[J], pv[J], rv[J], qv[J], dv[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = base + j * kTpb + threadIdx.x;
    if (i < n) {
      xv[j] = S.x[i];
      rv[j] = S.r[i];
      qv[j] = S.q[i];
      dv[j] = S.invd[i];
    }
  }
  if (W && load_done(st) >= 0) return;
  const int k = st->kk;
  const gptr<const VT> p = (k & 1) ? S.pb : S.pa;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = base + j * kTpb + threadIdx.x;
    if (i < n) pv[j] = p[i];
  }
  const double pq = W ? final_reduce_lo(S.part_pq, S.ntiles, red) : final_reduce(S.part_pq, S.ntiles, red);
  const double rz = st->rho[k & 1];
  const double alpha = (pq != 0.0) ? rz / pq : 0.0;
  if (tile == 0 && threadIdx.x == 0) st->k = k + 1;
  const VT av = (VT)alpha;
  double rr = 0.0, rzs = 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = base + j * kTpb + threadIdx.x;
    if (i < n) {
      S.x[i] = xv[j] + av * pv[j];
      const VT ri = rv[j] - av * qv[j];
      const VT zi = dv[j] * ri;
      S.r[i] = ri;
      S.z[i] = zi;
      const double a = (double)ri * (double)ri, b = (double)ri * (double)zi;
      if (W) {
        rr = a;
        rzs = b;
      } else {
        rr += a;
        rzs += b;
      }
    }
  }
  if (W) {
    rr = tile_tree_wide<R>(rr, lrows, red);
    rzs = tile_tree_wide<R>(rzs, lrows, red);
  } else {
    rr = block_tree(rr, red);
    rzs = block_tree(rzs, red);
  }
  if (threadIdx.x == 0) {
    S.part_rr[tile] = rr;
    S.part_rz[tile] = rzs;
  }
}

template <class VT, int R, bool W>
__global__ void __launch_bounds__(W ? kTpb * R : kTpb) k_pcg_phase_b(const PcgSys<VT>* __restrict__ sys,
                                                                     const TileRef* __restrict__ tiles) {
  __shared__ double red[4];
  __shared__ double lrows[W ? kTpb * R : 1];
  const TileRef tr = tiles ? tiles[blockIdx.x] : TileRef{0, (int)blockIdx.x};
  pcg_phase_b_body<VT, R, W>(view(sys[tr.sys]), tr.tile, red, lrows);
}

// ------------------------------------------------------------------ whole solve in one launch
// Many iterations of one small system in one launch: one workgroup of 256 R threads per tile, one
// row per thread. The row's matrix entries, x, r, z and the inverse diagonal stay in registers, p of
// the tile and of the rows its columns reach (the halo: within the matrix bandwidth of the tile)
// in LDS, where every workgroup updates its own copy of the halo's p from z. So per iteration the
// workgroups exchange two tile sums (p.q; r.r and r.z) and z of the halo. Arithmetic, partial trees
// and stopping rule are those of the two phases, and so are the bits.
//
// The exchange: agent-scope relaxed atomic stores and loads, which no XCD's L2 answers from a stale
// line. A double travels as two 64-bit words of (epoch, 32 bits), each word whole in itself; every
// workgroup polls all tiles' words until they carry the exchange's epoch, which is both the sum's
// transport and the grid barrier, in one trip. z is performed (s_waitcnt) before the r.r, r.z words
// that announce it. The words of p.q are not overwritten before all have read them: the next p.q
// comes after an r.r, r.z exchange, which each workgroup enters when it has read p.q, and likewise
// the other way round.
//
// Why: an iteration of the phases on a small system is two launches, each of which waits for its
// dispatch and for five dependent loads before its first product: 12-15 us at 384 to 66,887 rows,
// where the matrix and vectors would take 1-3 us from the caches. Here (us per iteration, R = 4):
// 384 rows (one workgroup, no exchange) 4.2 against 12.4 with the solve's set-up, 16,000 rows 6.1
// against 15.1, 66,887 rows 6.6 against 14.8, 128,000 rows 7.0 against 17. Up to kRunTiles
// workgroups: an exchange takes 1.2 us among 32, 2.3 among 128, and at one workgroup of 1,024 threads
// per CU two such launches are resident together on 256 CUs (the host admits no more than a workgroup
// a CU, RunSlots). A launch whose workgroups do not become resident together all the same (another
// process's solve) gives up after `polls` polls and leaves the solve to the phases.
constexpr int kRunRow = 12;     // entries of a row held in registers
constexpr int kRunWin = 6144;   // p of the tile and its halo, words of LDS

// The tile partials of N sums at once, in the R-rows-per-thread order (tile_tree_wide), returned to
// every thread. rows: N x 256 R words, red: N x 4. With drain, the workgroup's earlier stores are
// performed when it returns.
template <int R, int N>
__device__ __forceinline__ void run_tile_sums(double (&v)[N], double* rows, double* red, bool drain) {
  const int tid = threadIdx.x, w = tid >> 6;
#pragma unroll
  for (int a = 0; a < N; ++a) rows[a * kTpb * R + tid] = v[a];
  __syncthreads();
  if (tid < kTpb) {
#pragma unroll
    for (int a = 0; a < N; ++a) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < R; ++j) acc += rows[a * kTpb * R + j * kTpb + tid];
      acc = wave_tree(acc);
      if ((tid & 63) == 0) red[4 * a + w] = acc;
    }
  }
  if (drain) wait_stores();
  __syncthreads();
#pragma unroll
  for (int a = 0; a < N; ++a) v[a] = (red[4 * a] + red[4 * a + 1]) + (red[4 * a + 2] + red[4 * a + 3]);
}

// Sums over the T <= 128 tile partials (thread t holds tile t's) in final_reduce's order.
template <int N>
__device__ __forceinline__ void run_totals(double (&v)[N], double* red) {
  const int tid = threadIdx.x, w = tid >> 6;
  if (w < 4) {
#pragma unroll
    for (int a = 0; a < N; ++a) {
      const double u = wave_tree(0.0 + v[a]);
      if ((tid & 63) == 0) red[4 * a + w] = u;
    }
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < N; ++a) v[a] = (red[4 * a] + red[4 * a + 1]) + (red[4 * a + 2] + red[4 * a + 3]);
}

// Publishes this tile's N partials (v, the same in every thread) and returns in v of thread t < T
// tile t's, 0 in the others. False in a thread that gave up.
template <int N>
__device__ __forceinline__ bool run_exchange(double (&v)[N], gptr<uint64_t> words, int tile, int T, uint32_t epoch,
                                             int polls) {
  const int tid = threadIdx.x;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  if (tid < 2 * N) {
    double x = v[0];
#pragma unroll
    for (int a = 1; a < N; ++a)
      if ((tid >> 1) == a) x = v[a];
    st_agent(words + (int64_t)tile * 2 * N + tid, run_word(x, tid & 1, epoch));
  }
  bool ok = true;
  if (tid < T) {
    uint64_t u[2 * N] = {};
    for (int spin = 0;; ++spin) {
      if (spin == polls) {
        ok = false;
        break;
      }
#pragma unroll
      for (int a = 0; a < 2 * N; ++a) u[a] = ld_agent((gptr<const uint64_t>)words + (int64_t)tid * 2 * N + a);
      bool all = true;
#pragma unroll
      for (int a = 0; a < 2 * N; ++a) all = all && (uint32_t)(u[a] >> 32) == epoch;
      if (all) break;
    }
#pragma unroll
    for (int a = 0; a < N; ++a) v[a] = run_value(u[2 * a], u[2 * a + 1]);
  } else {
#pragma unroll
    for (int a = 0; a < N; ++a) v[a] = 0.0;
  }
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  return ok;
}

// words: 6 x 128 exchange words of the solver; epoch0: the launch's first epoch, above every earlier
// launch's; band: the largest |column - row|; iters: iterations at most; polls: run_exchange's bound.
template <class VT, int R, bool SOLO>
__global__ void __launch_bounds__(kTpb * R) k_pcg_run(const PcgSys<VT>* __restrict__ sys, uint64_t* __restrict__ words_,
                                                      uint32_t epoch0, int band, int iters, int polls) {
  constexpr int kRows = kTpb * R;
  __shared__ double red[8], redt[8], rows[2 * kRows];
  __shared__ int stuck;
  __shared__ VT win[SOLO ? kRows : kRunWin];
  const SysView<VT> S = view(*sys);
  gptr<PcgState> st = S.st;
  const gptr<uint64_t> wpq = G(words_), wrr = wpq + 2 * kRunTiles;
  const int n = S.n, T = S.ntiles, tile = blockIdx.x, tid = threadIdx.x;
  const int base = tile * kRows, i = base + tid;
  const bool in = i < n;
  const int lo = SOLO ? 0 : max(0, base - band), hi = SOLO ? n : min(n, base + kRows + band);
  const int below = base - lo, halo = (hi - lo) - (min(n, base + kRows) - base);
  // halo word h: rows below the tile, then rows above it
  auto halo_row = [&](int h) { return h < below ? lo + h : base + kRows + (h - below); };
  if (tid == 0) stuck = 0;
  if (load_done(st) >= 0) return;
  const int check_every = st->check_every, maxiter = st->maxiter;
  int k = st->k;
  const gptr<const VT> pold = (k & 1) ? S.pa : S.pb;
  VT v[kRunRow];
  int c[kRunRow];
  VT x = 0, r = 0, z = 0, p = 0, invd = 0;
  int len = 0;
  if (in) {
    const int a = S.rowptr[i];
    len = S.rowptr[i + 1] - a;
#pragma unroll
    for (int m = 0; m < kRunRow; ++m) {
      v[m] = 0;
      c[m] = i - lo;
      if (m < len) {
        v[m] = S.val[a + m];
        c[m] = S.col[a + m] - lo;
      }
    }
    x = S.x[i];
    r = S.r[i];
    z = S.z[i];
    p = pold[i];
    invd = S.invd[i];
    win[i - lo] = p;
  }
  if (!SOLO)
    for (int h = tid; h < halo; h += kRows) {
      const int row = halo_row(h);
      win[row - lo] = pold[row];
    }
  double rz_cur, rz_old = 0.0, rr_last = st->rr_last, atol2;
  double part[2] = {tid < T ? S.part_rz[tid] : 0.0, (k == 0 && tid < T) ? S.part_bb[tid] : 0.0};
  run_totals(part, redt);
  rz_cur = part[0];
  int done = -1;
  if (k == 0) {  // atol = rtol ||b|| (pcg_solver.py:928-930, 1089-1095)
    const double atol = st->rtol * sqrt(part[1]);
    atol2 = atol * atol;
    if (tile == 0 && tid == 0) {
      st->bb = part[1];
      st->atol2 = atol2;
      if (atol == 0.0) {
        st->zero = 1;
        st->done = 0;
      }
    }
    if (atol == 0.0) return;
  } else {
    atol2 = st->atol2;
    rz_old = st->rho[(k - 1) & 1];
  }
  uint32_t epoch = epoch0;
  double t2[2] = {0.0, 0.0};
  for (int it = 0; it < iters; ++it) {
    // phase A(k): p = z + beta p on the window, q = A p
    const VT bv = (VT)((k > 0 && rz_old != 0.0) ? rz_cur / rz_old : 0.0);
    if (!SOLO)
      for (int h0 = tid; h0 < halo; h0 += 4 * kRows) {
        VT zh[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int h = h0 + u * kRows;
          // the first launch iteration reads what an earlier launch stored, all others a neighbour's
          zh[u] = h < halo ? ld_agent((gptr<const VT>)S.z + halo_row(h)) : (VT)0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int h = h0 + u * kRows;
          if (h < halo) {
            const int j = halo_row(h) - lo;
            win[j] = zh[u] + bv * win[j];
          }
        }
      }
    if (in) {
      p = z + bv * p;
      win[i - lo] = p;
    }
    __syncthreads();
    VT q = 0;
    if (in) {
      VT pw[kRunRow];
#pragma unroll
      for (int m = 0; m < kRunRow; ++m) pw[m] = win[c[m]];
#pragma unroll
      for (int m = 0; m < kRunRow; ++m)
        if (m < len) q += v[m] * pw[m];
    }
    double t1[1] = {in ? (double)p * (double)q : 0.0};
    run_tile_sums<R>(t1, rows, red, false);
    if (!SOLO) {
      if (!run_exchange(t1, wpq, tile, T, epoch, polls)) stuck = 1;
    } else if (tid != 0) {
      t1[0] = 0.0;
    }
    run_totals(t1, redt);
    // phase B(k)
    const double pq = t1[0];
    const VT av = (VT)((pq != 0.0) ? rz_cur / pq : 0.0);
    t2[0] = t2[1] = 0.0;
    if (in) {
      x = x + av * p;
      r = r - av * q;
      z = invd * r;
      if (!SOLO) st_agent(S.z + i, z);
      t2[0] = (double)r * (double)r;
      t2[1] = (double)r * (double)z;
    }
    run_tile_sums<R>(t2, rows, red, !SOLO);
    double s2[2] = {t2[0], t2[1]};
    if (!SOLO) {
      if (!run_exchange(s2, wrr, tile, T, epoch, polls)) stuck = 1;
    } else if (tid != 0) {
      s2[0] = s2[1] = 0.0;
    }
    run_totals(s2, redt);
    if (!SOLO && stuck) break;  // set before run_totals' barrier, so the same in every thread
    ++epoch;
    rz_old = rz_cur;
    rz_cur = s2[1];
    ++k;
    if (k % check_every == 0 || k == maxiter) {
      rr_last = s2[0];
      if (rr_last <= atol2) {
        done = k;
        break;
      }
    }
  }
  if (!SOLO && stuck) {
    if (tid == 0) st->gave_up = 1;
    return;
  }
  if (in) {
    S.x[i] = x;
    S.r[i] = r;
    S.z[i] = z;
    ((k & 1) ? S.pa : S.pb)[i] = p;
  }
  if (tid == 0) {
    S.part_rr[tile] = t2[0];
    S.part_rz[tile] = t2[1];
    if (tile == 0) {
      st->rho[(k - 1) & 1] = rz_old;
      st->rr_last = rr_last;
      st->k = k;
      st->kk = k - 1;
      if (done >= 0) st->done = done;
    }
  }
}

// ------------------------------------------------------------------ window-end stopping test
// The test of iteration k-1 normally runs at the start of phase A(k); at the end of a window of
// launches this kernel runs it (one workgroup per system) so the host sees the flag at once.
// Phase A(k) repeats the same test on the same partials, so running both is harmless.
template <class VT>
__global__ void __launch_bounds__(256) k_pcg_check(const PcgSys<VT>* __restrict__ sys) {
  __shared__ double red[4];
  const SysView<VT> S = view(sys[blockIdx.x]);
  gptr<PcgState> st = S.st;
  if (load_done(st) >= 0) return;
  const int k = st->k;
  if (k < 1) return;
  const int it = k - 1;
  if (!((it + 1) % st->check_every == 0 || it == st->maxiter - 1)) return;
  const double rr = final_reduce(S.part_rr, S.ntiles, red);
  if (threadIdx.x == 0) {
    st->rr_last = rr;
    if (rr <= st->atol2) st->done = k;
  }
}

// ------------------------------------------------------------------ finish
// atol == 0: x = 0 (pcg_solver.py:1089-1095).
template <class VT, int R>
__global__ void __launch_bounds__(256) k_pcg_finish(const PcgSys<VT>* __restrict__ sys,
                                                    const TileRef* __restrict__ tiles) {
  const TileRef tr = tiles[blockIdx.x];
  const SysView<VT> S = view(sys[tr.sys]);
  if (!S.st->zero) return;
  const int base = tr.tile * kTpb * R;
  for (int j = 0; j < R; ++j) {
    const int i = base + j * kTpb + threadIdx.x;
    if (i < S.n) S.x[i] = (VT)0;
  }
}

// ------------------------------------------------------------------ true residual
// checkSolution (pcg_solver.py:1127-1143): r = b - A x; partials of r.r and b.b.
template <int R>
__global__ void __launch_bounds__(256) k_true_residual(const PcgSys<double>* __restrict__ sys,
                                                       const TileRef* __restrict__ tiles,
                                                       const double* __restrict__ xv_, double* __restrict__ rvec_) {
  __shared__ double red[4];
  __shared__ double lds[kSpmvLdsCap];
  const TileRef tr = tiles[xcd_block(blockIdx.x, gridDim.x)];
  const SysView<double> S = view(sys[tr.sys]);
  const int n = S.n;
  const gptr<const double> xv = G(xv_);
  const gptr<double> rvec = G(rvec_);
  const bool want_r = rvec_ != nullptr;
  auto xf = [&](int c) -> double { return xv[c]; };
  double rr = 0.0, bb = 0.0;
  const int base = tr.tile * kTpb * R;
  for (int j = 0; j < R; ++j) {
    const int r0 = base + j * kTpb;
    if (r0 >= n) break;
    const double q = csr_chunk<double>(S.rowptr, S.col, S.val, n, r0, lds, xf);
    const int i = r0 + threadIdx.x;
    if (i < n) {
      const double ri = S.b[i] - q;
      if (want_r) rvec[i] = ri;
      rr += ri * ri;
      bb += S.b[i] * S.b[i];
    }
  }
  rr = block_tree(rr, red);
  bb = block_tree(bb, red);
  if (threadIdx.x == 0) {
    S.part_rr[tr.tile] = rr;
    S.part_bb[tr.tile] = bb;
  }
}

// Batched r = b - A x (x = S.x, r written to S.r) over a launch table; partials of r.r and b.b.
template <int R>
__global__ void __launch_bounds__(256) k_residual_batch(const PcgSys<double>* __restrict__ sys,
                                                        const TileRef* __restrict__ tiles) {
  __shared__ double red[4];
  __shared__ double lds[kSpmvLdsCap];
  const TileRef tr = tiles[xcd_block(blockIdx.x, gridDim.x)];
  const SysView<double> S = view(sys[tr.sys]);
  const int n = S.n;
  const gptr<const double> xv = S.x;
  auto xf = [&](int c) -> double { return xv[c]; };
  double rr = 0.0, bb = 0.0;
  const int base = tr.tile * kTpb * R;
  for (int j = 0; j < R; ++j) {
    const int r0 = base + j * kTpb;
    if (r0 >= n) break;
    const double q = csr_chunk<double>(S.rowptr, S.col, S.val, n, r0, lds, xf);
    const int i = r0 + threadIdx.x;
    if (i < n) {
      const double bi = S.b[i];
      const double ri = bi - q;
      S.r[i] = ri;
      rr += ri * ri;
      bb += bi * bi;
    }
  }
  rr = block_tree(rr, red);
  bb = block_tree(bb, red);
  if (threadIdx.x == 0) {
    S.part_rr[tr.tile] = rr;
    S.part_bb[tr.tile] = bb;
  }
}

// Per-system totals of the r.r and b.b partials: out[2 i], out[2 i + 1] (one workgroup per system).
__global__ void __launch_bounds__(256) k_reduce_systems(const PcgSys<double>* __restrict__ sys,
                                                        double* __restrict__ out) {
  __shared__ double red[4];
  const PcgSys<double>& S = sys[blockIdx.x];
  double a, b;
  final_reduce2(G((const double*)S.part_rr), G((const double*)S.part_bb), S.ntiles, red, a, b);
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = a;
    out[2 * blockIdx.x + 1] = b;
  }
}

// x64 += d32 for every system of a launch table (sys64[i].x, sys32[i].x).
template <int R>
__global__ void __launch_bounds__(256) k_refine_batch(const PcgSys<double>* __restrict__ sys64,
                                                      const PcgSys<float>* __restrict__ sys32,
                                                      const TileRef* __restrict__ tiles) {
  const TileRef tr = tiles[blockIdx.x];
  const gptr<double> x = G(sys64[tr.sys].x);
  const gptr<const float> d = G((const float*)sys32[tr.sys].x);
  const int n = sys64[tr.sys].n;
  const int base = tr.tile * kTpb * R;
  for (int j = 0; j < R; ++j) {
    const int i = base + j * kTpb + threadIdx.x;
    if (i < n) x[i] = x[i] + (double)d[i];
  }
}

__global__ void k_reduce_pair(const double* __restrict__ pa, const double* __restrict__ pb, int T,
                              double* __restrict__ out) {
  __shared__ double red[4];
  double a, b;
  final_reduce2(G(pa), G(pb), T, red, a, b);
  if (threadIdx.x == 0) {
    out[0] = a;
    out[1] = b;
  }
}

// ------------------------------------------------------------------ mixed precision helpers
__global__ void k_cast_values(const double* __restrict__ in, float* __restrict__ out, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) out[i] = (float)in[i];
}

__global__ void k_refine_update(double* __restrict__ x, const float* __restrict__ d, int32_t n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = x[i] + (double)d[i];
}

__global__ void k_copy_f64(double* __restrict__ dst, const double* __restrict__ src, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) dst[i] = src[i];
}

__global__ void k_fill_f64(double* __restrict__ dst, double v, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) dst[i] = v;
}

// ------------------------------------------------------------------ launch wrappers
#define GSH_DISPATCH_R(rpt, KER, VT, ...)                                              \
  switch (rpt) {                                                                       \
    case 1: hipLaunchKernelGGL((KER<VT, 1>), __VA_ARGS__); break;                      \
    case 2: hipLaunchKernelGGL((KER<VT, 2>), __VA_ARGS__); break;                      \
    case 8: hipLaunchKernelGGL((KER<VT, 8>), __VA_ARGS__); break;                      \
    default: hipLaunchKernelGGL((KER<VT, 4>), __VA_ARGS__); break;                     \
  }

template <class VT>
void launch_pcg_reset(const PcgSys<VT>* sys, int nsys, double rtol, int maxiter, int check_every, hipStream_t s,
                      const double* rtols) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(k_pcg_reset<VT>, dim3((nsys + 63) / 64), dim3(64), 0, s, sys, nsys, rtol, maxiter, check_every,
                     rtols);
}

template <class VT>
void launch_pcg_init(const PcgSys<VT>* sys, const TileRef* tiles, int ntiles, int rpt, hipStream_t s) {
  if (ntiles <= 0) return;
  GSH_DISPATCH_R(rpt, k_pcg_init, VT, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles);
}

// Calls f with R as a constant.
template <class F>
static void with_rpt(int rpt, F&& f) {
  switch (rpt) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 8: f(std::integral_constant<int, 8>()); break;
    default: f(std::integral_constant<int, 4>()); break;
  }
}

// With e0/e1 the runtime stamps the kernel's start and end (hipExtLaunchKernelGGL), for profiling;
// without them a plain launch, which stream capture records.
template <class... A>
static void launch_stamped(void (*ker)(A...), int grid, int block, hipStream_t s, hipEvent_t e0, hipEvent_t e1,
                           A... a) {
  if (e0 || e1)
    hipExtLaunchKernelGGL(ker, dim3(grid), dim3(block), 0, s, e0, e1, 0, a...);
  else
    hipLaunchKernelGGL(ker, dim3(grid), dim3(block), 0, s, a...);
}

// Wide workgroups (R = 2, 4) up to 512 tiles: below that the tiles' serial
// sub-rounds leave the chip waiting, above it the narrow form's row pointers, loaded ahead for R
// sub-rounds, keep more in flight per register. Microseconds per Jacobi iteration, wide against
// narrow, at R = 4: 16,000 rows 15.1 against 24.3, 66,887 14.8 against 24.2, 501,264 (490 tiles) 30.0
// against 33.5, 1,048,576 (1,024 tiles) 53.7 against 42.3; at R = 2: 66,887 13.2 against 16.3,
// 501,264 (980 tiles) 28.7 against 26.0.
// At R = 4 a workgroup's 16 waves fill a CU's registers, so more than 256 tiles come in two rounds; where
// the chunks also take two pieces each (577 to 832 entries) the narrow form is faster there: 293 tiles
// of 10 entries a row 39.4 against 36.4, of 13 44.5 against 41.2, of 14 46.1 against 46.2; 254 tiles of 10
// entries a row 24.3 against 34.0. FP32 up to 16 entries a row.
constexpr int kWideTiles = 512, kWideTilesLong = 256;

template <class VT>
void launch_pcg_phase(int which, const PcgSys<VT>* sys, const TileRef* tiles, int ntiles, int rpt, hipStream_t s,
                      int chunk, hipEvent_t e0, hipEvent_t e1) {
  if (ntiles <= 0) return;
  with_rpt(rpt, [&](auto r) {
    constexpr int R = decltype(r)::value;
    auto run = [&](auto wide) {
      constexpr bool W = decltype(wide)::value;
      launch_stamped(which == 0 ? k_pcg_phase_a<VT, R, W> : k_pcg_phase_b<VT, R, W>, ntiles, W ? kTpb * R : kTpb, s, e0,
                     e1, sys, tiles);
    };
    if constexpr (R == 2 || R == 4)
      if (ntiles <= ((R == 4 && chunk > kWideChunk && chunk <= (sizeof(VT) == 8 ? kWideLong : kWideLong32)) ? kWideTilesLong : kWideTiles))
        return run(std::true_type());
    run(std::false_type());
  });
}

template <class VT>
void launch_pcg_iter(const PcgSys<VT>* sys, const TileRef* tiles, int ntiles, int rpt, hipStream_t s, int chunk) {
  launch_pcg_phase<VT>(0, sys, tiles, ntiles, rpt, s, chunk);
  launch_pcg_phase<VT>(1, sys, tiles, ntiles, rpt, s, chunk);
}

bool pcg_run_fits(int ntiles, int rpt, int max_row, int band) {
  return ntiles >= 1 && ntiles <= kRunTiles && (rpt == 1 || rpt == 2 || rpt == 4) && max_row <= kRunRow &&
         (ntiles == 1 || kTpb * rpt + 2 * (int64_t)band <= kRunWin);
}

template <class VT>
void launch_pcg_run(const PcgSys<VT>* sys, int ntiles, int rpt, uint64_t* words, uint32_t epoch, int band, int iters,
                    int polls, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  with_rpt(rpt, [&](auto r) {
    constexpr int R = decltype(r)::value;
    if constexpr (R <= 4) {
      if (ntiles == 1)
        launch_stamped(k_pcg_run<VT, R, true>, 1, kTpb * R, s, e0, e1, sys, words, epoch, band, iters, polls);
      else
        launch_stamped(k_pcg_run<VT, R, false>, ntiles, kTpb * R, s, e0, e1, sys, words, epoch, band, iters, polls);
    }
  });
}

template <class VT>
void launch_pcg_check(const PcgSys<VT>* sys, int nsys, hipStream_t s) {
  if (nsys <= 0) return;
  hipLaunchKernelGGL(k_pcg_check<VT>, dim3(nsys), dim3(kTpb), 0, s, sys);
}

template <class VT>
void launch_pcg_finish(const PcgSys<VT>* sys, const TileRef* tiles, int ntiles, int rpt, hipStream_t s) {
  if (ntiles <= 0) return;
  GSH_DISPATCH_R(rpt, k_pcg_finish, VT, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles);
}

template void launch_pcg_reset<double>(const PcgSys<double>*, int, double, int, int, hipStream_t, const double*);
template void launch_pcg_reset<float>(const PcgSys<float>*, int, double, int, int, hipStream_t, const double*);
template void launch_pcg_init<double>(const PcgSys<double>*, const TileRef*, int, int, hipStream_t);
template void launch_pcg_init<float>(const PcgSys<float>*, const TileRef*, int, int, hipStream_t);
template void launch_pcg_iter<double>(const PcgSys<double>*, const TileRef*, int, int, hipStream_t, int);
template void launch_pcg_iter<float>(const PcgSys<float>*, const TileRef*, int, int, hipStream_t, int);
template void launch_pcg_phase<double>(int, const PcgSys<double>*, const TileRef*, int, int, hipStream_t, int, hipEvent_t,
                                       hipEvent_t);
template void launch_pcg_phase<float>(int, const PcgSys<float>*, const TileRef*, int, int, hipStream_t, int, hipEvent_t,
                                       hipEvent_t);
template void launch_pcg_run<double>(const PcgSys<double>*, int, int, uint64_t*, uint32_t, int, int, int, hipStream_t, hipEvent_t,
                                     hipEvent_t);
template void launch_pcg_run<float>(const PcgSys<float>*, int, int, uint64_t*, uint32_t, int, int, int, hipStream_t, hipEvent_t,
                                    hipEvent_t);
template void launch_pcg_check<double>(const PcgSys<double>*, int, hipStream_t);
template void launch_pcg_check<float>(const PcgSys<float>*, int, hipStream_t);
template void launch_pcg_finish<double>(const PcgSys<double>*, const TileRef*, int, int, hipStream_t);
template void launch_pcg_finish<float>(const PcgSys<float>*, const TileRef*, int, int, hipStream_t);

void launch_true_residual(const PcgSys<double>* sys, const TileRef* tiles, int ntiles, int rpt, const double* xv,
                          double* rvec, hipStream_t s) {
  if (ntiles <= 0) return;
  switch (rpt) {
    case 1: hipLaunchKernelGGL(k_true_residual<1>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles, xv, rvec); break;
    case 2: hipLaunchKernelGGL(k_true_residual<2>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles, xv, rvec); break;
    case 8: hipLaunchKernelGGL(k_true_residual<8>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles, xv, rvec); break;
    default: hipLaunchKernelGGL(k_true_residual<4>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles, xv, rvec); break;
  }
}

void launch_residual_batch(const PcgSys<double>* sys, const TileRef* tiles, int ntiles, int rpt, hipStream_t s) {
  if (ntiles <= 0) return;
  switch (rpt) {
    case 1: hipLaunchKernelGGL(k_residual_batch<1>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles); break;
    case 2: hipLaunchKernelGGL(k_residual_batch<2>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles); break;
    case 8: hipLaunchKernelGGL(k_residual_batch<8>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles); break;
    default: hipLaunchKernelGGL(k_residual_batch<4>, dim3(ntiles), dim3(kTpb), 0, s, sys, tiles); break;
  }
}

void launch_reduce_systems(const PcgSys<double>* sys, int nsys, double* out, hipStream_t s) {
  if (nsys > 0) hipLaunchKernelGGL(k_reduce_systems, dim3(nsys), dim3(kTpb), 0, s, sys, out);
}

void launch_refine_batch(const PcgSys<double>* sys64, const PcgSys<float>* sys32, const TileRef* tiles, int ntiles,
                         int rpt, hipStream_t s) {
  if (ntiles <= 0) return;
  switch (rpt) {
    case 1: hipLaunchKernelGGL(k_refine_batch<1>, dim3(ntiles), dim3(kTpb), 0, s, sys64, sys32, tiles); break;
    case 2: hipLaunchKernelGGL(k_refine_batch<2>, dim3(ntiles), dim3(kTpb), 0, s, sys64, sys32, tiles); break;
    case 8: hipLaunchKernelGGL(k_refine_batch<8>, dim3(ntiles), dim3(kTpb), 0, s, sys64, sys32, tiles); break;
    default: hipLaunchKernelGGL(k_refine_batch<4>, dim3(ntiles), dim3(kTpb), 0, s, sys64, sys32, tiles); break;
  }
}

void launch_reduce_pair(const double* pa, const double* pb, int ntiles, double* out2, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce_pair, dim3(1), dim3(kTpb), 0, s, pa, pb, ntiles, out2);
}

void launch_cast_values(const double* in, float* out, int64_t count, hipStream_t s) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_cast_values, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, in, out, count);
}

void launch_refine_update(double* x64, const float* d32, int32_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_refine_update, dim3((n + 255) / 256), dim3(256), 0, s, x64, d32, n);
}

void launch_copy_f64(double* dst, const double* src, int64_t count, hipStream_t s) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_copy_f64, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, dst, src, count);
}

void launch_fill_f64(double* dst, double v, int64_t count, hipStream_t s) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, dst, v, count);
}

}  // namespace gsh
