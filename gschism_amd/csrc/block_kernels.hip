// block_kernels.hip -- Jacobi PCG of a block of M systems that share one CSR pattern (ensemble
// members of one mesh: per-member matrix values and right-hand sides), on gfx950.
//
// Layout: every vector is [row][member] and the values are [entry][member], so the M members of
// one row are M consecutive words (M a power of two). A workgroup takes a tile of
// kBlkTile = 512 rows and W = min(M, 8 or 16) of its members (blk_wide): its lanes are W members of
// 64 / W consecutive rows, so a gather is 64- or 128-byte segments and the row pointers and columns
// are read once for W members. Each member keeps the reference's recurrences (pcg_solver.py:172-276, 881-947,
// 1075-1124; pcg_loop.cpp:361-413) and its own stopping rule; a member that has stopped keeps its
// solution and drops out of the loads.
//
// Dot products (FP64) are summed in one fixed order, restated by the oracle (or_pcg_block): slot s
// of 256 / M adds the products of the tile's rows s, s + S, s + 2 S, ... (S = 256 / M) to 0.0 in that
// order; the tile partial of member m adds the S slot sums to 0.0 in slot order; the reduction
// kernel (1024 threads, RS = 1024 / M slots per member) has slot r add the tile partials r, r + RS,
// ... to 0.0 and then adds the RS slot sums to 0.0 in slot order. The order fixes which rows form
// one chain of additions, not who multiplies: all 512 rows' products go to LDS with every load in
// flight, and W S threads then add them from there.
//
// Each iteration is four launches: phase A (p update, SpMV, p.q partials), the p.q reduction
// (alpha), phase B (x, r, z updates, r.r and r.z partials) and their reduction (stopping test,
// beta). Splitting a tile over members and rows instead of giving each of 256 threads its slot's
// whole chain of rows (J = 128 rows one after another at M = 64, on n / 512 workgroups) takes phase A
// from 501 to 27 us and phase B from 85 to 17 us at 16,000 rows x 64 members, where the vectors and
// values (115 MB) sit in the last-level cache; what bounds them now is that cache's rate.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "device.h"
#include "reduce.h"

namespace gsh {

constexpr int kBlkRows = 4;  // rows of a thread in flight
template <int W>
constexpr int kBlkThreads = W == 16 ? 512 : (W == 8 ? 1024 : 256);

// A thread's place: member m, tile, and the rows rl, rl + L, ... of the tile.
struct BlkPlace {
  int M, lm, lw, tile, w, m, rl, L;
};
template <int W>
__device__ __forceinline__ BlkPlace blk_place(int M) {
  BlkPlace q;
  q.M = M;
  q.lm = __builtin_ctz(M);
  q.lw = min(q.lm, __builtin_ctz(W));
  const int b = xcd_block(blockIdx.x, gridDim.x);  // a tile's parts and its neighbours on one XCD (shared L2)
  q.tile = b >> (q.lm - q.lw);
  q.w = (int)threadIdx.x & ((1 << q.lw) - 1);
  q.m = ((b - (q.tile << (q.lm - q.lw))) << q.lw) + q.w;
  q.rl = (int)threadIdx.x >> q.lw;
  q.L = kBlkThreads<W> >> q.lw;
  return q;
}

// 0.0 + f(0) + f(1) + ... + f(n - 1), n below 16 or a multiple of it, f a value in LDS: 16 are read
// ahead of their additions, without selects, which took longer than the additions (k_blk_reduce on
// 958 tiles of one member 23.7 us against 13.1).
template <class F>
__device__ __forceinline__ double blk_chain(int n, F&& f) {
  constexpr int B = 16;
  double x = 0.0;
  if (n < B) {
    for (int i = 0; i < n; ++i) x += f(i);
    return x;
  }
  for (int i0 = 0; i0 < n; i0 += B) {
    double v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) v[u] = f(i0 + u);
#pragma unroll
    for (int u = 0; u < B; ++u) x += v[u];
  }
  return x;
}

// The tile partial of each member of the workgroup from the rows' products in pr ([row][W]), which
// every thread passes after its own are written. A row beyond n or of a stopped member has the
// product +0.0, and a sum that started at 0.0 is never -0.0, so adding it changes no bit.
__device__ __forceinline__ void blk_tile_sum(const BlkPlace& q, const double* pr, double* slot,
                                             double* __restrict__ part) {
  const int SS = kTpb >> q.lm, J = kBlkTile / kTpb << q.lm;
  __syncthreads();
  if (q.rl < SS) slot[threadIdx.x] = blk_chain(J, [&](int j) { return pr[((q.rl + SS * j) << q.lw) + q.w]; });
  __syncthreads();
  if (q.rl == 0)
    part[(int64_t)q.tile * q.M + q.m] = blk_chain(SS, [&](int r) { return slot[(r << q.lw) + q.w]; });
}

// ---------------------------------------------------------------- init
// cold start: x = 0, r = b, invD = 1 / diag, z = invD r, p_old = 0; partials of b.b and r.z
template <class VT, int W>
__global__ void __launch_bounds__(kBlkThreads<W>) k_blk_init(BlkSys<VT> S) {
  __shared__ double pr[2][kBlkTile * W], slot[2][kTpb];
  const BlkPlace q = blk_place<W>(S.M);
  for (int r = q.rl; r < kBlkTile; r += q.L) {
    const int i = q.tile * kBlkTile + r;
    double bb = 0.0, rz = 0.0;
    if (i < S.n) {
      const int64_t e = (int64_t)i * q.M + q.m;
      const VT inv = (VT)(1.0 / (double)S.val[(int64_t)S.diag[i] * q.M + q.m]);
      const double bi = S.b[e];
      const VT ri = (VT)bi;
      const VT zi = inv * ri;
      S.invd[e] = inv;
      S.x[e] = (VT)0;
      S.r[e] = ri;
      S.z[e] = zi;
      S.pb[e] = (VT)0;
      bb = bi * bi;
      rz = (double)ri * (double)zi;
    }
    pr[0][(r << q.lw) + q.w] = bb;
    pr[1][(r << q.lw) + q.w] = rz;
  }
  blk_tile_sum(q, pr[0], slot[0], S.part_a);
  blk_tile_sum(q, pr[1], slot[1], S.part_b);
}

// ---------------------------------------------------------------- phase A
// Row sum of a_ij (z_j + beta p_j) in column order: the columns of 8 entries are loaded together,
// then their values and gathers, so a row waits for two memory steps per 8 entries, not per entry.
template <class VT>
__device__ __forceinline__ VT blk_row(const BlkSys<VT>& S, const VT* __restrict__ po, VT beta, int a, int b, int m,
                                      int M) {
  constexpr int B = 8;
  VT qv = (VT)0;
  for (int k0 = a; k0 < b; k0 += B) {
    int c[B];
    VT v[B], z[B], p[B];
#pragma unroll
    for (int u = 0; u < B; ++u) c[u] = k0 + u < b ? S.col[k0 + u] : -1;
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (c[u] >= 0) {
        const int64_t g = (int64_t)c[u] * M + m;
        v[u] = S.val[(int64_t)(k0 + u) * M + m];
        z[u] = S.z[g];
        p[u] = po[g];
      }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (c[u] >= 0) qv += v[u] * (z[u] + beta * p[u]);
  }
  return qv;
}

// beta (set by the previous reduction) -> p = z + beta p_old, q = A p, partials of p.q
template <class VT, int W>
__global__ void __launch_bounds__(kBlkThreads<W>) k_blk_a(BlkSys<VT> S, int it) {
  __shared__ double pr[kBlkTile * W], slot[kTpb];
  const BlkPlace q = blk_place<W>(S.M);
  const BlkState st = S.st[q.m];
  const VT beta = (VT)st.beta;
  const VT* __restrict__ po = (it & 1) ? S.pa : S.pb;
  VT* __restrict__ pn = (it & 1) ? S.pb : S.pa;
  for (int r0 = q.rl; r0 < kBlkTile; r0 += kBlkRows * q.L) {
    // every row pointer first: they depend on nothing
    int a[kBlkRows], b[kBlkRows];
#pragma unroll
    for (int u = 0; u < kBlkRows; ++u) {
      const int r = r0 + u * q.L, i = q.tile * kBlkTile + r;
      const bool in = st.done < 0 && r < kBlkTile && i < S.n;
      a[u] = in ? S.rowptr[i] : 0;
      b[u] = in ? S.rowptr[i + 1] : 0;
    }
#pragma unroll
    for (int u = 0; u < kBlkRows; ++u) {
      const int r = r0 + u * q.L, i = q.tile * kBlkTile + r;
      if (r >= kBlkTile) break;
      double pq = 0.0;
      if (st.done < 0 && i < S.n) {
        const int64_t e = (int64_t)i * q.M + q.m;
        const VT pi = S.z[e] + beta * po[e];
        const VT qv = blk_row(S, po, beta, a[u], b[u], q.m, q.M);
        pn[e] = pi;
        S.q[e] = qv;
        pq = (double)pi * (double)qv;
      }
      pr[(r << q.lw) + q.w] = pq;
    }
  }
  blk_tile_sum(q, pr, slot, S.part_a);
}

// ---------------------------------------------------------------- phase B
// x += alpha p, r -= alpha q, z = invD r; partials of r.r and r.z
template <class VT, int W>
__global__ void __launch_bounds__(kBlkThreads<W>) k_blk_b(BlkSys<VT> S, int it) {
  __shared__ double pr[2][kBlkTile * W], slot[2][kTpb];
  const BlkPlace q = blk_place<W>(S.M);
  const BlkState st = S.st[q.m];
  const VT alpha = (VT)st.alpha;
  const VT* __restrict__ p = (it & 1) ? S.pb : S.pa;
  for (int r0 = q.rl; r0 < kBlkTile; r0 += kBlkRows * q.L) {
    // the rows' loads first: a store between them would order the next row's loads after it
    VT xv[kBlkRows], pv[kBlkRows], rv[kBlkRows], qv[kBlkRows], dv[kBlkRows];
#pragma unroll
    for (int u = 0; u < kBlkRows; ++u) {
      const int r = r0 + u * q.L, i = q.tile * kBlkTile + r;
      if (st.done < 0 && r < kBlkTile && i < S.n) {
        const int64_t e = (int64_t)i * q.M + q.m;
        xv[u] = S.x[e];
        pv[u] = p[e];
        rv[u] = S.r[e];
        qv[u] = S.q[e];
        dv[u] = S.invd[e];
      }
    }
#pragma unroll
    for (int u = 0; u < kBlkRows; ++u) {
      const int r = r0 + u * q.L, i = q.tile * kBlkTile + r;
      if (r >= kBlkTile) break;
      double rr = 0.0, rz = 0.0;
      if (st.done < 0 && i < S.n) {
        const int64_t e = (int64_t)i * q.M + q.m;
        S.x[e] = xv[u] + alpha * pv[u];
        const VT ri = rv[u] - alpha * qv[u];
        const VT zi = dv[u] * ri;
        S.r[e] = ri;
        S.z[e] = zi;
        rr = (double)ri * (double)ri;
        rz = (double)ri * (double)zi;
      }
      pr[0][(r << q.lw) + q.w] = rr;
      pr[1][(r << q.lw) + q.w] = rz;
    }
  }
  blk_tile_sum(q, pr[0], slot[0], S.part_a);
  blk_tile_sum(q, pr[1], slot[1], S.part_b);
}

// ---------------------------------------------------------------- reductions
// total of member m over the tile partials P[tile][M] in the block order (1024 threads)
__device__ __forceinline__ double blk_total(const double* __restrict__ P, int ntiles, int M, double* lds) {
  const int m = (int)threadIdx.x % M, r = (int)threadIdx.x / M, RS = 1024 / M;
  double u = 0.0;
  for (int t0 = r; t0 < ntiles; t0 += 8 * RS) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = (t0 + q * RS < ntiles) ? P[(int64_t)(t0 + q * RS) * M + m] : 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (t0 + q * RS < ntiles) u += v[q];
  }
  lds[threadIdx.x] = u;
  __syncthreads();
  // slots beyond the tiles hold +0.0, which changes no sum: the chain ends with the 16 that hold the last tile
  const int nr = RS < 16 ? RS : min(RS, (ntiles + 15) & ~15);
  const double t = r == 0 ? blk_chain(nr, [&](int q) { return lds[q * M + m]; }) : 0.0;
  __syncthreads();
  return t;
}

// which = 0: after init (atol from b.b, rz); 1: after phase A (alpha); 2: after phase B (stopping
// test of iteration it, beta of the next iteration)
__global__ void __launch_bounds__(1024) k_blk_reduce(BlkState* __restrict__ st, const double* __restrict__ pa,
                                                     const double* __restrict__ pb, int ntiles, int M, int which,
                                                     int it, double rtol, int maxiter, int check_every) {
  __shared__ double lds[1024];
  const double ta = blk_total(pa, ntiles, M, lds);
  const double tb = (which != 1) ? blk_total(pb, ntiles, M, lds) : 0.0;
  if ((int)threadIdx.x >= M) return;
  BlkState& S = st[threadIdx.x];
  if (which == 0) {
    const double atol = rtol * sqrt(ta);
    S.atol2 = atol * atol;
    S.rz_cur = tb;
    S.rz_old = 0.0;
    S.beta = 0.0;
    S.alpha = 0.0;
    S.rr_last = -1.0;
    S.zero = 0;
    S.done = -1;
    if (atol == 0.0) {  // pcg_solver.py:1089-1095: x = 0 after 0 iterations
      S.zero = 1;
      S.done = 0;
    }
    return;
  }
  if (S.done >= 0) return;
  if (which == 1) {
    S.alpha = (ta != 0.0) ? S.rz_cur / ta : 0.0;
    return;
  }
  S.rz_old = S.rz_cur;
  S.rz_cur = tb;
  if ((it + 1) % check_every == 0 || it == maxiter - 1) {
    S.rr_last = ta;
    if (ta <= S.atol2) S.done = it + 1;
  }
  S.beta = (S.rz_old == 0.0) ? 0.0 : S.rz_cur / S.rz_old;
}

// ---------------------------------------------------------------- layout helpers
// member m's CSR values and right-hand side into the block layout
__global__ void k_blk_put(double* __restrict__ vblk, double* __restrict__ bblk, const double* __restrict__ v,
                          const double* __restrict__ b, int64_t nnz, int n, int M, int m) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v && i < nnz) vblk[i * M + m] = v[i];
  if (b && i < n) bblk[i * M + m] = b[i];
}

// member m's solution out of the block layout
template <class VT>
__global__ void k_blk_get(double* __restrict__ x, const VT* __restrict__ xblk, int n, int M, int m) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = (double)xblk[(int64_t)i * M + m];
}

// ---------------------------------------------------------------- launchers
// Members of a workgroup: 16 where that still gives two workgroups per CU, else 8. With 16 a gather
// is a whole 128-byte line and the columns are read once for twice the members (305,500 rows x 64
// members: 830 us per iteration against 980; 30,000 x 256: 420 against 490); with 8 a small block
// fills twice the CUs (16,000 x 64: 54 us against 75). 512 threads measured best with 16 members,
// 1024 with 8. A block of one or two members takes a tile with 256 threads: most of 1024 would have
// no row of it (1,048,576 rows, with the chains of blk_chain, 100 us per iteration against 227).
template <class VT, class F>
static void blk_wide(const BlkSys<VT>& S, F&& launch) {
  constexpr int kFill = 512;  // workgroups
  if (S.M >= 16 && S.ntiles * (S.M / 16) >= kFill)
    launch(std::integral_constant<int, 16>(), dim3(S.ntiles * (S.M / 16)));
  else if (S.M > 2)
    launch(std::integral_constant<int, 8>(), dim3(S.ntiles * (S.M / std::min(S.M, 8))));
  else
    launch(std::integral_constant<int, 2>(), dim3(S.ntiles));
}
template <class VT>
void launch_blk_init(const BlkSys<VT>& S, hipStream_t st) {
  blk_wide(S, [&](auto w, dim3 grid) {
    constexpr int W = decltype(w)::value;
    hipLaunchKernelGGL((k_blk_init<VT, W>), grid, dim3(kBlkThreads<W>), 0, st, S);
  });
}
template <class VT>
void launch_blk_iter(const BlkSys<VT>& S, int it, double rtol, int maxiter, int check_every, hipStream_t st) {
  blk_wide(S, [&](auto w, dim3 grid) {
    constexpr int W = decltype(w)::value;
    hipLaunchKernelGGL((k_blk_a<VT, W>), grid, dim3(kBlkThreads<W>), 0, st, S, it);
    hipLaunchKernelGGL(k_blk_reduce, dim3(1), dim3(1024), 0, st, S.st, S.part_a, S.part_b, S.ntiles, S.M, 1, it, rtol,
                       maxiter, check_every);
    hipLaunchKernelGGL((k_blk_b<VT, W>), grid, dim3(kBlkThreads<W>), 0, st, S, it);
    hipLaunchKernelGGL(k_blk_reduce, dim3(1), dim3(1024), 0, st, S.st, S.part_a, S.part_b, S.ntiles, S.M, 2, it, rtol,
                       maxiter, check_every);
  });
}
template <class VT>
void launch_blk_reduce_init(const BlkSys<VT>& S, double rtol, hipStream_t st) {
  hipLaunchKernelGGL(k_blk_reduce, dim3(1), dim3(1024), 0, st, S.st, S.part_a, S.part_b, S.ntiles, S.M, 0, 0, rtol,
                     1, 1);
}
void launch_blk_put(double* vblk, double* bblk, const double* v, const double* b, int64_t nnz, int n, int M, int m,
                    hipStream_t st) {
  const int64_t cnt = nnz > n ? nnz : n;
  hipLaunchKernelGGL(k_blk_put, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, st, vblk, bblk, v, b, nnz, n, M, m);
}
template <class VT>
void launch_blk_get(double* x, const VT* xblk, int n, int M, int m, hipStream_t st) {
  hipLaunchKernelGGL(k_blk_get<VT>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, xblk, n, M, m);
}

template void launch_blk_init<double>(const BlkSys<double>&, hipStream_t);
template void launch_blk_iter<double>(const BlkSys<double>&, int, double, int, int, hipStream_t);
template void launch_blk_reduce_init<double>(const BlkSys<double>&, double, hipStream_t);
template void launch_blk_get<double>(double*, const double*, int, int, int, hipStream_t);

}  // namespace gsh
