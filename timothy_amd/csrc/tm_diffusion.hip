// The environment solve: one or more backward-Euler steps of
//   du/dt = D lap(u) - lambda u + s
// on the field grid, as the reference assembles it for HYPRE
// (src/environment.c:131-511):
//   z = D dt / res^2   (res^2 formed in FP32, grid_t.resolution being float),
//   (1 + 6 z + lambda dt) u_i - z sum_{neighbours j inside the grid} u_j = b_i,
//   b_i = u_old_i + z bc per grid face the node lies on (the six faces in the
//         order x-, x+, y-, y+, z-, z+) + s_i,
// i.e. Dirichlet faces with the field outside the grid held at bc.  The
// reference solves with HYPRE's PCG (BoomerAMG-preconditioned) to a relative
// residual of 1e-12 in at most 50 iterations; the matrix is symmetric,
// positive definite and strongly diagonally dominant with a constant
// diagonal, so Jacobi-preconditioned CG (plain CG scaled by that constant,
// with the same stopping norm) reaches the same solution to that tolerance.
//
// Matrix-free, nodes in the field's layout ([i][j][k], k fastest).  An
// iteration is two streaming kernels:
//   k_cg<DIR>     beta = rr_new / rr, p_new = r + beta p_old, partial sums of
//                 p_new . A p_new              (reads r, p; writes p: 24 B/node)
//   k_cg<UPDATE>  alpha = rr / pAp, x += alpha p, r -= alpha A p, partial sums
//                 of r . r              (reads p, x, r; writes x, r: 40 B/node)
// A p is formed twice from the stencil rather than stored and read (16 B/node
// less), and every workgroup adds the partial sums itself, in one fixed order,
// so that no launch stands between the two and results do not depend on
// timing.  The scalars live in device memory; once converged, the kernels of
// the remaining iterations return at once, so the host launches a few iterations
// ahead and reads the state once.
#include <mutex>
#include <type_traits>

#include "tm_internal.h"

namespace {

constexpr int MAXBLK = 4096;  // partial sums per reduction

struct CGState {
  double bb, tol2;
  double rr[2];  // residual norm before iteration k at [k & 1]
  double last;   // and after the last one checked
  unsigned long long iters;
  // 0, or one more than the pass that set it: pass 0 is k_cg_start, DIR and
  // UPDATE of iteration k are 2k + 1 and 2k + 2.  A pass stops for an earlier
  // pass's mark only, so all its waves agree, also where its own first
  // workgroup has set one meanwhile.
  unsigned int done;
  unsigned int pad;
};

// The host launches a few iterations ahead of the one that runs, which its
// direction pass names here, in pinned host memory; ENDED once there is none.
constexpr unsigned int ENDED = ~0u;
__device__ __forceinline__ void tell(unsigned int *progress, unsigned int what) {
  __hip_atomic_store(progress, what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// what the host reads of the state, in pinned host memory, once the stream is done
__device__ __forceinline__ void report(const CGState *st, CGState *host) {
  host->bb = st->bb;
  host->last = st->last;
  host->iters = st->iters;
  host->done = st->done;
}

struct Op {
  int64_t lx, ly, lz;
  double diag, z, zbc;
};

// sum over the workgroup's T threads, in all of them, always in the same
// order; sh: T / 64 doubles that nothing else uses until the next barrier
template <int T>
__device__ __forceinline__ double block_sum(double v, double *sh) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < T / 64; ++i) s += sh[i];
  return s;
}
template <int T>
__device__ __forceinline__ double sum_parts(const double *__restrict__ part, int n, double *sh) {
  double a = 0.0;
  for (int i = threadIdx.x; i < n; i += T) a += part[i];
  return block_sum<T>(a, sh);
}

// right-hand side at a node, in the reference's order: u_old, the faces x-,
// x+, y-, y+, z-, z+, then s
__device__ __forceinline__ double rhs(const Op &A, double u, int64_t i, int64_t j, int64_t k, const double *src,
                                      int64_t node) {
  if (i == 0) u += A.zbc;
  if (i == A.lx - 1) u += A.zbc;
  if (j == 0) u += A.zbc;
  if (j == A.ly - 1) u += A.zbc;
  if (k == 0) u += A.zbc;
  if (k == A.lz - 1) u += A.zbc;
  if (src) u += src[node];
  return u;
}

// The three streaming passes, marching along i: a workgroup owns an MJ x MK
// block of (j, k) columns over a run of planes (MK the next power of two from
// the grid's extent along k, 8 to 64: 512^2 x 3 with 8 x 64 took twice the time).  Per plane the operand of the
// stencil (x, p_new or p) is formed once per node, and once per node of the
// block's edge ring (which the neighbouring blocks also form), into LDS; the
// values of its own column one plane before and after stay in registers.
//   INIT    r = b - A x                  parts: r . r, b . b
//   DIR     p_new = r + beta p_old       parts: p_new . A p_new
//   UPDATE  x += alpha p, r -= alpha A p parts: r . r
// Odd passes take the blocks and planes in the opposite order (`down`): what
// the pass before touched last is then read first, from the 256 MB memory-side
// cache.
//
// Bound by the bytes: 256^3 takes 195 us an iteration, 64 B a node at 5.5 TB/s
// (some of it from that cache), where storing A p and the one-workgroup
// reductions between the kernels took 80 B and 280 us.  The loads of a plane
// go out two planes ahead, and those of the first planes before the scalars are
// known: without that 217 against 280 us at 256^3, and a kernel of a 32^3 grid,
// which is latency from end to end, 9 us instead of 6.5.  The 8 x 64 block in
// two workgroups a CU: 4 x 64 in four takes 205 us, 16 x 64 in one 189 us but
// 20 % more than 8 x 64 at 64^3 and below; one workgroup a CU takes 250 us,
// four 217 us.
// At most 80 registers (6 waves a SIMD), so that three workgroups fit where the
// runs ask for them: 200x201x203 5.7 against 6.7 ms with 81.
enum Pass { INIT, DIR, UPDATE };
struct Blocks {
  unsigned int nk, nj, run;  // blocks along k and j, planes a run
  unsigned int count;        // workgroups' worth of work: at most MAXBLK are launched
};
constexpr int MT = 512;

// What DIR and UPDATE start with: the scalar of the pass from the partial sums of
// the one before (sh: as for block_sum), or false where there is nothing to do.
template <int PASS>
__device__ __forceinline__ bool begin(int iter, CGState *st, const double *__restrict__ in, double *sh,
                                      unsigned int *progress, CGState *host, double &scale) {
  const unsigned int pass = 2u * (unsigned int)iter + (PASS == DIR ? 1u : 2u), mark = st->done;
  if constexpr (PASS == DIR) {
    if (iter > 0) {
      const double before = st->rr[(iter - 1) & 1], limit = st->tol2 * st->bb;
      const double rr = sum_parts<MT>(in, (int)gridDim.x, sh);
      if (mark && mark <= pass) return false;
      const bool end = rr <= limit;
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->rr[iter & 1] = rr;
        st->last = rr;
        st->iters = (unsigned long long)iter;
        if (end) {
          st->done = pass + 1u;
          report(st, host);
        }
        tell(progress, end ? ENDED : (unsigned int)iter);
      }
      if (end) return false;
      scale = rr / before;
    } else if (mark) {
      return false;
    }
  } else {
    const double rr = st->rr[iter & 1];
    const double pAp = sum_parts<MT>(in, (int)gridDim.x, sh);
    if (mark && mark <= pass) return false;
    if (!(pAp > 0.0)) {  // breakdown: the residual is zero (or the operator is not positive definite)
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->done = pass + 1u;
        report(st, host);
        tell(progress, ENDED);
      }
      return false;
    }
    scale = rr / pAp;
  }
  return true;
}

template <int PASS, int MK>
__global__ __launch_bounds__(MT, 6) void k_cg(Op A, const double *__restrict__ src, double *__restrict__ x,
                                           double *__restrict__ r, const double *__restrict__ pold,
                                           double *__restrict__ pnew, Blocks B, int iter,
                                           CGState *__restrict__ st, const double *__restrict__ in,
                                           double *__restrict__ out, double *__restrict__ out2,
                                           unsigned int *progress, CGState *host) {
  constexpr int MJ = MT / MK;
  constexpr int MHALO = 2 * MJ + 2 * MK;  // the edge ring without its corners
  static_assert(MHALO <= MT, "a thread forms one ring node");
  __shared__ double pl[2][MJ + 2][MK + 2];
  __shared__ double sh[2][MT / 64];
  constexpr bool down = PASS == UPDATE;
  constexpr int64_t d = down ? -1 : 1;
  const int64_t sx = A.ly * A.lz, sy = A.lz;
  const int tk = (int)threadIdx.x % MK, tj = (int)threadIdx.x / MK;
  // this thread's place on the edge ring, if any: (a, c) in the (MJ+2) x (MK+2) frame
  int ha = -1, hc = -1;
  {
    const int t = (int)threadIdx.x;
    if (t < MK) {
      ha = 0;
      hc = 1 + t;
    } else if (t < 2 * MK) {
      ha = MJ + 1;
      hc = 1 + t - MK;
    } else if (t < 2 * MK + MJ) {
      ha = 1 + t - 2 * MK;
      hc = 0;
    } else if (t < MHALO) {
      ha = 1 + t - 2 * MK - MJ;
      hc = MK + 1;
    }
  }
  double acc = 0.0, acc2 = 0.0;
  double scale = 0.0;  // beta or alpha
  const unsigned int b0 = (unsigned int)tm_xcd_block();
  for (unsigned int c = b0; c < B.count; c += gridDim.x) {
    const unsigned int b = down ? B.count - 1 - c : c;
    const unsigned int kt = b % B.nk, bj = b / B.nk, jt = bj % B.nj, seg = bj / B.nj;
    const int64_t i0 = (int64_t)seg * B.run, i1 = i0 + B.run < A.lx ? i0 + B.run : A.lx;
    const int64_t j = (int64_t)jt * MJ + tj, k = (int64_t)kt * MK + tk;
    const bool own = j < A.ly && k < A.lz;
    const int64_t hj = (int64_t)jt * MJ + ha - 1, hk = (int64_t)kt * MK + hc - 1;
    const bool halo = ha >= 0 && hj >= 0 && hj < A.ly && hk >= 0 && hk < A.lz;
    const int64_t col = j * sy + k, hcol = hj * sy + hk;
    const int64_t first = down ? i1 - 1 : i0, stop = down ? i0 - 1 : i1;
    // what the operand of the stencil is formed from: own column, edge ring
    struct Raw {
      double a, b, ha, hb;
    };
    auto load = [&](int64_t i) -> Raw {
      Raw w{0.0, 0.0, 0.0, 0.0};
      if (i < 0 || i >= A.lx) return w;
      const double *u = PASS == INIT ? x : PASS == UPDATE ? pold : r;
      if (own) w.a = u[i * sx + col];
      if (halo) w.ha = u[i * sx + hcol];
      if constexpr (PASS == DIR) {
        if (iter > 0) {
          if (own) w.b = pold[i * sx + col];
          if (halo) w.hb = pold[i * sx + hcol];
        }
      }
      return w;
    };
    auto form = [&](double u, double v) -> double {
      if constexpr (PASS == DIR) return iter > 0 ? u + scale * v : u;
      return u;
    };
    auto place = [&](int64_t i, const Raw &w) {
      if (own) pl[i & 1][tj + 1][tk + 1] = form(w.a, w.b);
      if (halo) pl[i & 1][ha][hc] = form(w.ha, w.hb);
    };
    // the first planes' loads go out before the scalars are known
    const Raw wb = load(first - d);
    Raw w = load(first);
    Raw wn = load(first + d);
    double xn = 0.0, rn = 0.0;
    if constexpr (PASS == UPDATE) {
      if (own) {
        xn = x[first * sx + col];
        rn = r[first * sx + col];
      }
    }
    if (c == b0) {
      if constexpr (PASS != INIT)
        if (!begin<PASS>(iter, st, in, sh[0], progress, host, scale)) return;
    } else {
      __syncthreads();  // the buffers' last readers are done
    }
    double behind = form(wb.a, wb.b), cur = form(w.a, w.b);
    place(first, w);
    for (int64_t i = first; i != stop; i += d) {
      const int64_t node = i * sx + col;
      w = wn;
      const double xv = xn, rv = rn;
      if (i + d != stop) {
        wn = load(i + d + d);
        if constexpr (PASS == UPDATE) {
          if (own) {
            xn = x[node + d * sx];
            rn = r[node + d * sx];
          }
        }
      }
      __syncthreads();  // plane i is in its buffer; the reads of plane i - d are done
      const double ahead = form(w.a, w.b);
      if (i + d != stop) place(i + d, w);
      if (own) {
        const int q = (int)(i & 1);
        double nb = 0.0;
        if (i > 0) nb += down ? ahead : behind;
        if (i < A.lx - 1) nb += down ? behind : ahead;
        if (j > 0) nb += pl[q][tj][tk + 1];
        if (j < A.ly - 1) nb += pl[q][tj + 2][tk + 1];
        if (k > 0) nb += pl[q][tj + 1][tk];
        if (k < A.lz - 1) nb += pl[q][tj + 1][tk + 2];
        const double ap = A.diag * cur - A.z * nb;
        if constexpr (PASS == INIT) {
          const double bv = rhs(A, cur, i, j, k, src, node);
          const double res = bv - ap;
          r[node] = res;
          acc += res * res;
          acc2 += bv * bv;
        } else if constexpr (PASS == DIR) {
          pnew[node] = cur;
          acc += cur * ap;
        } else {
          x[node] = xv + scale * cur;
          const double now = rv - scale * ap;
          r[node] = now;
          acc += now * now;
        }
      }
      behind = cur;
      cur = ahead;
    }
  }
  const double s = block_sum<MT>(acc, sh[1]);
  if (threadIdx.x == 0) out[b0] = s;
  if constexpr (PASS == INIT) {
    const double s2 = block_sum<MT>(acc2, sh[0]);
    if (threadIdx.x == 0) out2[b0] = s2;
  }
}

// The passes with a lane per node, for planes that would leave more than half the
// march's lanes idle.  The operand at a node and its six neighbours comes from
// memory, through the caches, which hold such planes.  Latency on small grids,
// then the loads' issue.  At most 1,024 workgroups, whose partial sums every one
// adds: with 2,048 100,000x3x3 takes 635 against 571 us.
constexpr int64_t NODE_BLOCKS = 1024;
template <int PASS>
__global__ __launch_bounds__(MT) void k_cg_nodes(Op A, const double *__restrict__ src, double *__restrict__ x,
                                                 double *__restrict__ r, const double *__restrict__ pold,
                                                 double *__restrict__ pnew, int64_t chunk, int iter,
                                                 CGState *__restrict__ st, const double *__restrict__ in,
                                                 double *__restrict__ out, double *__restrict__ out2,
                                                 unsigned int *progress, CGState *host) {
  __shared__ double sh[2][MT / 64];
  double scale = 0.0;  // beta or alpha
  if constexpr (PASS != INIT)
    if (!begin<PASS>(iter, st, in, sh[0], progress, host, scale)) return;
  const int64_t b0 = tm_xcd_block();
  const int64_t total = A.lx * A.ly * A.lz, lo = b0 * chunk, hi = lo + chunk < total ? lo + chunk : total;
  const int64_t sx = A.ly * A.lz, sy = A.lz;
  const double *const u = PASS == INIT ? x : PASS == UPDATE ? pold : r;
  auto at = [&](int64_t node) -> double {
    if constexpr (PASS == DIR) return iter > 0 ? u[node] + scale * pold[node] : u[node];
    return u[node];
  };
  double acc = 0.0, acc2 = 0.0;
  for (int64_t node = lo + threadIdx.x; node < hi; node += MT) {
    const int64_t i = node / sx, m = node - i * sx, j = m / sy, k = m - j * sy;
    const double cur = at(node);
    double nb = 0.0;
    if (i > 0) nb += at(node - sx);
    if (i < A.lx - 1) nb += at(node + sx);
    if (j > 0) nb += at(node - sy);
    if (j < A.ly - 1) nb += at(node + sy);
    if (k > 0) nb += at(node - 1);
    if (k < A.lz - 1) nb += at(node + 1);
    const double ap = A.diag * cur - A.z * nb;
    if constexpr (PASS == INIT) {
      const double bv = rhs(A, cur, i, j, k, src, node);
      const double res = bv - ap;
      r[node] = res;
      acc += res * res;
      acc2 += bv * bv;
    } else if constexpr (PASS == DIR) {
      pnew[node] = cur;
      acc += cur * ap;
    } else {
      x[node] += scale * cur;
      const double now = r[node] - scale * ap;
      r[node] = now;
      acc += now * now;
    }
  }
  const double s = block_sum<MT>(acc, sh[1]);
  if (threadIdx.x == 0) out[b0] = s;
  if constexpr (PASS == INIT) {
    const double s2 = block_sum<MT>(acc2, sh[0]);
    if (threadIdx.x == 0) out2[b0] = s2;
  }
}

__global__ __launch_bounds__(256) void k_cg_start(const double *__restrict__ part_rr,
                                                  const double *__restrict__ part_bb, int nblk, double tol,
                                                  int maxiter, CGState *st, unsigned int *progress, CGState *host) {
  __shared__ double sh[2][4];
  const double rr = sum_parts<256>(part_rr, nblk, sh[0]), bb = sum_parts<256>(part_bb, nblk, sh[1]);
  if (threadIdx.x == 0) {
    st->rr[0] = st->last = rr;
    st->bb = bb;
    st->tol2 = tol * tol;
    st->iters = 0;
    st->done = (rr <= st->tol2 * bb || maxiter <= 0) ? 1u : 0u;
    if (st->done) report(st, host);
    tell(progress, st->done ? ENDED : 0u);
  }
}

// after `iters` iterations: their residual, and whether to stop
__global__ __launch_bounds__(256) void k_cg_check(const double *__restrict__ part, int nblk, int iters, int maxiter,
                                                  CGState *st, CGState *host) {
  __shared__ double sh[4];
  if (st->done) return;  // (reported)
  const double rr = sum_parts<256>(part, nblk, sh);
  if (threadIdx.x == 0) {
    st->last = rr;
    st->iters = (unsigned long long)iters;
    if (rr <= st->tol2 * st->bb || iters >= maxiter) st->done = 1u;
    report(st, host);
  }
}

// The whole solve of a small grid in one workgroup: thread t holds x and r of
// nodes t + ST m in registers, the direction lies in LDS.
// Latency-bound: two barriers with a sum over 16 waves and one more an
// iteration, 3 to 6 us against 12 to 14 us for the two streaming kernels.  17^3
// with three iterations: 36 us a solve (62 us streaming); 22^3 with 100: 0.62
// ms (1.3 ms).  Ten nodes a thread is the limit, as more spill: 25^3 took 1.4 ms
// for 108 iterations, streaming 1.3 ms, and with three 92 us against 65 us.
constexpr int ST = 1024;
constexpr int64_t SMALL_NODES = 10 * ST;
template <int NPT>
__global__ __launch_bounds__(ST) void k_cg_small(Op A, const double *__restrict__ src, double *__restrict__ x,
                                                 double tol, int maxiter, int substeps, CGState *st) {
  __shared__ double p[ST * NPT];
  __shared__ double sh[3][ST / 64];
  const int lz = (int)A.lz, lyz = (int)(A.ly * A.lz), total = (int)(A.lx * lyz);
  double xv[NPT], rv[NPT];
  uint32_t in[NPT];  // which neighbours lie inside the grid: i-1, i+1, j-1, j+1, k-1, k+1
#pragma unroll
  for (int m = 0; m < NPT; ++m) {
    const int node = (int)threadIdx.x + ST * m;
    const int i = node / lyz, j = (node - i * lyz) / lz, k = node - i * lyz - j * lz;
    in[m] = (i > 0 ? 1u : 0u) | (i < (int)A.lx - 1 ? 2u : 0u) | (j > 0 ? 4u : 0u) | (j < (int)A.ly - 1 ? 8u : 0u) |
            (k > 0 ? 16u : 0u) | (k < lz - 1 ? 32u : 0u);
    xv[m] = node < total ? x[node] : 0.0;
  }
  auto apply = [&](int node, uint32_t w) -> double {
    double nb = 0.0;
    if (w & 1u) nb += p[node - lyz];
    if (w & 2u) nb += p[node + lyz];
    if (w & 4u) nb += p[node - lz];
    if (w & 8u) nb += p[node + lz];
    if (w & 16u) nb += p[node - 1];
    if (w & 32u) nb += p[node + 1];
    return A.diag * p[node] - A.z * nb;
  };
  const double tol2 = tol * tol;
  unsigned long long its = 0;
  double rr = 0.0, bb = 0.0;
  for (int s = 0; s < substeps; ++s) {
    __syncthreads();
#pragma unroll
    for (int m = 0; m < NPT; ++m) {
      const int node = (int)threadIdx.x + ST * m;
      if (node < total) p[node] = xv[m];
    }
    __syncthreads();
    double a = 0.0, c = 0.0;
#pragma unroll
    for (int m = 0; m < NPT; ++m) {
      const int node = (int)threadIdx.x + ST * m;
      rv[m] = 0.0;
      if (node < total) {
        const uint32_t w = in[m];
        double b = xv[m];
        if (!(w & 1u)) b += A.zbc;
        if (!(w & 2u)) b += A.zbc;
        if (!(w & 4u)) b += A.zbc;
        if (!(w & 8u)) b += A.zbc;
        if (!(w & 16u)) b += A.zbc;
        if (!(w & 32u)) b += A.zbc;
        if (src) b += src[node];
        rv[m] = b - apply(node, w);
        a += rv[m] * rv[m];
        c += b * b;
      }
    }
    rr = block_sum<ST>(a, sh[0]);
    bb = block_sum<ST>(c, sh[1]);
    double beta = 0.0;
    for (int it = 0; it < maxiter && !(rr <= tol2 * bb); ++it) {
#pragma unroll
      for (int m = 0; m < NPT; ++m) {
        const int node = (int)threadIdx.x + ST * m;
        if (node < total) p[node] = it > 0 ? rv[m] + beta * p[node] : rv[m];
      }
      __syncthreads();
      double ap[NPT];
      a = 0.0;
#pragma unroll
      for (int m = 0; m < NPT; ++m) {
        const int node = (int)threadIdx.x + ST * m;
        ap[m] = 0.0;
        if (node < total) {
          ap[m] = apply(node, in[m]);
          a += p[node] * ap[m];
        }
      }
      const double pAp = block_sum<ST>(a, sh[2]);
      if (!(pAp > 0.0)) break;
      const double alpha = rr / pAp;
      a = 0.0;
#pragma unroll
      for (int m = 0; m < NPT; ++m) {
        const int node = (int)threadIdx.x + ST * m;
        if (node < total) {
          xv[m] += alpha * p[node];
          rv[m] -= alpha * ap[m];
          a += rv[m] * rv[m];
        }
      }
      const double now = block_sum<ST>(a, sh[it & 1]);
      beta = now / rr;
      rr = now;
      ++its;
    }
  }
#pragma unroll
  for (int m = 0; m < NPT; ++m) {
    const int node = (int)threadIdx.x + ST * m;
    if (node < total) x[node] = xv[m];
  }
  if (threadIdx.x == 0) {
    st->bb = bb;
    st->last = rr;
    st->iters = its;
    st->done = 1u;
  }
}

}  // namespace

// doubles of work memory for a grid of `total` nodes: r and two directions;
// three arrays of partial sums; the state
static constexpr int64_t work_doubles(int64_t total) {
  return 3 * total + 3 * MAXBLK + (int64_t)((sizeof(CGState) + 7) / 8);
}

// The allocation-free entry point's work memory: one buffer per device, in
// the code object (the loader places it on every device the library runs
// on).  Host code never passes `scratch` itself to a kernel: on the host the
// name is a stand-in, not the device address.  The address is looked up
// once per device (tm_noalloc_init) and kept in scratch_addr.
constexpr int64_t SCRATCH_DOUBLES = work_doubles(TM_NOALLOC_MAX_NODES);
static __device__ __align__(256) double scratch[SCRATCH_DOUBLES];

constexpr int MAX_DEVICES = 64;
static std::mutex scratch_mu;
static double *scratch_addr[MAX_DEVICES];

// (j, k) blocks times runs of planes: the number of runs that takes the
// fullest of 256 CUs the fewest planes, each run costing RUN_COST planes more
// (it reads one more at either end, and every workgroup adds all the partial
// sums).  A CU needs two workgroups to be busy, so one counts as two.
static Blocks blocks_for(int64_t lx, int64_t ly, int64_t lz, int MK) {
  const int MJ = MT / MK;
  constexpr int64_t CUS = 256, FULL = 1024 / MT, MOST = 4 * FULL * CUS / 2, MIN_RUN = 2, RUN_COST = 3;
  Blocks B;
  B.nk = (unsigned int)((lz + MK - 1) / MK);
  B.nj = (unsigned int)((ly + MJ - 1) / MJ);
  const int64_t ncol = (int64_t)B.nk * B.nj;
  int64_t best = 0;
  for (int64_t nseg = 1; nseg == 1 || (nseg * MIN_RUN <= lx + 1 && nseg * ncol <= MOST); ++nseg) {
    const int64_t run = (lx + nseg - 1) / nseg, count = ncol * ((lx + run - 1) / run);
    const int64_t cost = std::max((count + CUS - 1) / CUS, FULL) * (run + RUN_COST);
    if (nseg > 1 && cost >= best) continue;
    best = cost;
    B.run = (unsigned int)run;
    B.count = (unsigned int)count;
  }
  return B;
}

// CG's bound on the iterations to a relative residual of tol, from the
// operator's least and greatest eigenvalue
static double iterations_for(const Op &A, double tol) {
  const double n = 2.0 * A.z * (cos(M_PI / (double)(A.lx + 1)) + cos(M_PI / (double)(A.ly + 1)) +
                                cos(M_PI / (double)(A.lz + 1)));
  const double k = sqrt((A.diag + n) / (A.diag - n));
  const double its = log(2.0 / std::max(tol, 1e-300)) / log((k + 1.0) / (k - 1.0));
  return its > 1.0 ? its : 1.0;  // (one also where there is no such number)
}

// the solve with its work arrays at `work` (work_doubles(total) doubles)
static tm_status run_diffusion(tm_ctx *c, double *work, const tm_grid *g, const tm_diffusion *d, const double *src,
                               double *field, int32_t *iterations, double *residual) {
  int64_t lx = g->localsize[0], ly = g->localsize[1], lz = g->localsize[2];
  const int64_t total = lx * ly * lz;
  // Axes of one node go to the front, where the passes march: the layout, the
  // order of a node's neighbours and its six equal face terms stay the same.
  for (int q = 0; q < 2 && lz == 1; ++q) {
    lz = ly;
    ly = lx;
    lx = 1;
  }
  if (ly == 1) std::swap(lx, ly);
  double *r = work, *p0 = r + total, *p1 = p0 + total;
  double *part = p1 + total, *part2 = part + MAXBLK, *partb = part2 + MAXBLK;
  CGState *st = (CGState *)(partb + MAXBLK);
  Op A;
  A.lx = lx;
  A.ly = ly;
  A.lz = lz;
  const float res2 = g->resolution * g->resolution;  // FP32 product, as the reference forms it
  A.z = d->diffusion * d->dt / (double)res2;
  A.diag = 1 + 6.0 * A.z + d->lambda * d->dt;
  A.zbc = A.z * d->boundary;
  int32_t it_total = 0;
  double last_res = 0.0;
  // the kernels report the state in pinned host memory set aside at tm_create
  CGState &h = *reinterpret_cast<CGState *>(c->h_flags + TM_HFLAGS_CG);
  auto read_state = [&]() -> tm_status {
    TM_HIP(c, hipGetLastError());
    TM_HIP(c, hipStreamSynchronize(c->stream));
    last_res = h.bb > 0.0 ? sqrt(h.last / h.bb) : sqrt(h.last);
    it_total += (int32_t)h.iters;
    return TM_OK;
  };
  if (total <= SMALL_NODES && d->substeps > 0) {
    auto kern = total <= ST * 5 ? k_cg_small<5> : k_cg_small<10>;
    kern<<<1, ST, 0, c->stream>>>(A, src, field, d->tol, d->maxiter, d->substeps, &h);
    TM_TRY(read_state());
  } else {
    const int mk = lz <= 8 ? 8 : lz <= 16 ? 16 : lz <= 32 ? 32 : 64;
    const Blocks B = blocks_for(lx, ly, lz, mk);
    // Where a plane fills less than half the lanes of its blocks, a lane per node.
    // Solves with a coupling of 0.5, march and lane per node: 100,000x3x3 (2 %) 5,950
    // and 571 us, 3,000x8x8 (12 %) 544 and 369, 4,000x9x33 (29 %) 1,190 and 971,
    // 2,000x33x33 (43 %) 1,456 and 1,374, 65^3 (46 %) 566 and 475, 5,000x12x20 (47 %)
    // 922 and 951; 10,000x16x16 (50 %) 1,315 and 1,399, 1,000x40x40 (62 %) 968 and
    // 1,204.
    const bool nodes = 2 * ly * lz < (int64_t)B.nk * B.nj * MT;
    // (whole rounds of a workgroup's nodes each)
    const int64_t rounds = (total + MT - 1) / MT, chunk = (rounds + NODE_BLOCKS - 1) / NODE_BLOCKS * MT;
    const int nblk = nodes ? (int)((total + chunk - 1) / chunk) : (int)std::min<unsigned int>(MAXBLK, B.count);
    // Iterations are launched until one of them is seen to have ended the solve,
    // three ahead of it up to CG's bound on their number and one beyond: enough
    // that the GPU does not wait for the host, and few that find the solve ended
    // (4.4 us a launch).  0.8 of the bound in one batch, then four at a time with a
    // wait after each, took 1.49 against 1.39 ms at 32^3 with 116 iterations and 340
    // against 211 us where 8 iterations end a solve of 96x80x112; the store costs
    // 1.5 us an iteration at 256^3.
    const int32_t bound = (int32_t)std::min(iterations_for(A, d->tol) + 1.0, 1e9);
    unsigned int *const progress = c->h_flags + TM_HFLAGS_PROGRESS;
    volatile unsigned int *const seen = progress;
    auto pass = [&](auto which, const double *source, double *x, double *p, double *next, int iter, const double *in,
                    double *out, double *out2) {
      constexpr int P = decltype(which)::value;
      if (nodes) {
        k_cg_nodes<P><<<nblk, MT, 0, c->stream>>>(A, source, x, r, p, next, chunk, iter, st, in, out, out2, progress, &h);
        return;
      }
      auto kern = mk == 8 ? k_cg<P, 8> : mk == 16 ? k_cg<P, 16> : mk == 32 ? k_cg<P, 32> : k_cg<P, 64>;
      kern<<<nblk, MT, 0, c->stream>>>(A, source, x, r, p, next, B, iter, st, in, out, out2, progress, &h);
    };
    constexpr std::integral_constant<int, INIT> init;
    constexpr std::integral_constant<int, DIR> direction;
    constexpr std::integral_constant<int, UPDATE> update;
    for (int s = 0; s < d->substeps; ++s) {
      const int32_t before = it_total;
      *seen = 0u;
      pass(init, src, field, nullptr, nullptr, 0, nullptr, part2, partb);
      k_cg_start<<<1, 256, 0, c->stream>>>(part2, partb, nblk, d->tol, d->maxiter, st, progress, &h);
      // the first direction is r; the two arrays then alternate
      double *pold = p0, *pnew = p1;
      int32_t launched = 0;
      unsigned int at = 0u;
      for (; launched < d->maxiter; ++launched) {
        if (launched == bound) {  // (next to no coupling: the bound is the number)
          k_cg_check<<<1, 256, 0, c->stream>>>(part2, nblk, launched, d->maxiter, st, &h);
          TM_TRY(read_state());
          at = h.done ? ENDED : 0u;
          if (at == ENDED) break;
        }
        at = *seen;
        for (unsigned int spin = 1; at != ENDED && launched > (int32_t)at + (launched < bound ? 3 : 1); ++spin) {
          if (spin % 4096 == 0 && hipStreamQuery(c->stream) != hipErrorNotReady) break;  // (an error)
          __builtin_ia32_pause();
          at = *seen;
        }
        if (at == ENDED) break;
        pass(direction, nullptr, nullptr, pold, pnew, launched, part2, part, nullptr);
        pass(update, nullptr, field, pnew, nullptr, launched, part, part2, nullptr);
        std::swap(pold, pnew);
      }
      if (at != ENDED && launched > 0)
        k_cg_check<<<1, 256, 0, c->stream>>>(part2, nblk, launched, d->maxiter, st, &h);
      it_total = before;
      TM_TRY(read_state());
    }
  }
  if (iterations) *iterations = it_total;
  if (residual) *residual = last_res;
  return TM_OK;
}

static_assert(sizeof(CGState) <= 4 * (TM_HFLAGS_PROGRESS - TM_HFLAGS_CG), "solver state fits the pinned words");

tm_status tm_run_diffusion(tm_ctx *c, const tm_grid *g, const tm_diffusion *d, const double *src, double *field,
                           int32_t *iterations, double *residual) {
  const int64_t total = g->localsize[0] * g->localsize[1] * g->localsize[2];
  TM_TRY(tm_ensure(c, &c->d_cg, c->cap_cg, work_doubles(total), "diffusion work arrays"));
  return run_diffusion(c, c->d_cg, g, d, src, field, iterations, residual);
}

tm_status tm_noalloc_init(tm_ctx *c) {
  // called by tm_create with c->device current
  if (c->device < 0 || c->device >= MAX_DEVICES) return tm_fail(c, TM_ERR_UNSUPPORTED, "device index too large");
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (scratch_addr[c->device]) return TM_OK;
  void *p = nullptr;
  TM_HIP(c, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) return tm_fail(c, TM_ERR_HIP, "no device address for the static work buffer");
  scratch_addr[c->device] = (double *)p;
  return TM_OK;
}

tm_status tm_run_diffusion_noalloc(tm_ctx *c, const tm_grid *g, const tm_diffusion *d, const double *src,
                                   double *field, int32_t *iterations, double *residual) {
  const int64_t total = g->localsize[0] * g->localsize[1] * g->localsize[2];
  if (total > TM_NOALLOC_MAX_NODES)
    return tm_fail(c, TM_ERR_INVALID, "tm_diffusion_step_noalloc: the grid has " + std::to_string(total) +
                                          " nodes, more than TM_NOALLOC_MAX_NODES (" +
                                          std::to_string((long long)TM_NOALLOC_MAX_NODES) +
                                          "); use tm_diffusion_step");
  double *work;
  {
    std::lock_guard<std::mutex> lock(scratch_mu);
    work = scratch_addr[c->device];
  }
  if (!work) return tm_fail(c, TM_ERR_STATE, "static work buffer not set up on this device");
  return run_diffusion(c, work, g, d, src, field, iterations, residual);
}
