// Neighbour stage: the cells whose leaf octants overlap a cell's query box (the
// reference's, with its strict overlap test), visited in descending Morton
// key -- the order the reference's LIFO DFS pops them (children pushed 0..7,
// src/potential.c:111-131).  By default a wave looks for the candidates of
// all its cells together (k_union, below).  With walk_coop or walk_f32 off one
// lane per cell walks its colony's radix tree (k_neighbors), read in the
// walk's own pre-order (built by k_wnodes): one 16-byte record per visited
// node, the next slot after a hit and the escape slot after a miss.
//
// Per cell p this yields:
//   N(p)    candidates q != p with sqrt((dx*dx+dy*dy)+dz*dz) <= h_p, stored in
//           visit order at nbr[tm_slot(p, k, cap)] (slot-major inside each
//           group of 64 cells, coalesced for the one-lane-per-cell pair
//           kernels), count[p]
//   mindist min distance over all candidates (src/potential.c:49), computed as
//           sqrt of the minimum squared distance (sqrt is monotone and
//           correctly rounded, so this is the minimum of the rounded roots)
//   qstar   the last candidate visited = minimum key, the one whose potential
//           the reference leaves in v (src/potential.c:124 assigns, not adds)
//   v       that potential, in the reference's FP64 expressions
// The cutoff test d <= h is evaluated exactly as d2 <= cut2, cut2 being the
// largest double whose correctly rounded root is <= h.
#include <type_traits>

#include "tm_internal.h"

namespace {

__device__ __forceinline__ uint32_t box_code(double v, double shift, double scale) {
  return (uint32_t)((v - shift) / scale * 536870912.0);
}

// potential() (src/potential.c:39-78) without its density/mindist side effects,
// in the reference's expressions and order
__device__ __forceinline__ double pot_fp64(double4 P, float yp, double4 Q, float yq, double h) {
  const double dx = P.x - Q.x, dy = P.y - Q.y, dz = P.z - Q.z;
  const double dist = sqrt((dx * dx + dy * dy) + dz * dz);
  if (!(dist <= h)) return 0.0;
  const double s1 = P.w, s2 = Q.w;
  const double xc = s1 + s2 - dist;
  if (xc <= 0.0) return 0.0;
  const double poisson = 0.33;
  const double D = 0.75 * ((1.0 - poisson * poisson) / (double)yp + (1.0 - poisson * poisson / (double)yq));
  const double r01 = (s1 * s1 - s2 * s2 + dist * dist) / (2.0 * dist);
  const double r02 = dist - r01;
  const double area = M_PI * ((s1 * s1 * (s1 - r01) - (s1 * s1 * s1 - r01 * r01 * r01) / 3.0) +
                              (s2 * s2 * (s2 - r02) - (s2 * s2 * s2 - r02 * r02 * r02) / 3.0));
  // pow(xc, 5/2) with integer 5/2 == 2 is xc*xc
  return (2.0 * (xc * xc) / (5.0 * D)) * sqrt((s1 * s2) / (s1 + s2)) + area * 0.1;
}

// reference squared distance, src/potential.c:49 order (contraction is off)
__device__ __forceinline__ double dist2_fp64(const double4 &P, const double4 &Q) {
  const double dx = P.x - Q.x, dy = P.y - Q.y, dz = P.z - Q.z;
  return (dx * dx + dy * dy) + dz * dz;
}

// lane moves within the wave (DPP): the lanes without a source get `old`
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xf, false);
}
// maximum over the wave's 64 lanes, all active
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, dpp<0x111>(0u, v));  // row_shr 1, 2, 4, 8
  v = max(v, dpp<0x112>(0u, v));
  v = max(v, dpp<0x114>(0u, v));
  v = max(v, dpp<0x118>(0u, v));
  v = max(v, dpp<0x142, 0xa>(0u, v));  // row_bcast 15 into rows 1 and 3
  v = max(v, dpp<0x143, 0xc>(0u, v));  // row_bcast 31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// maximum over each row of 16 lanes, in all of them
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
  v = max(v, dpp<0x128>(0u, v));  // row_ror 8, 4, 2, 1
  v = max(v, dpp<0x124>(0u, v));
  v = max(v, dpp<0x122>(0u, v));
  return max(v, dpp<0x121>(0u, v));
}
// set bits of m below this lane
__device__ __forceinline__ uint32_t mbcnt64(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// the value of the row's first lane
__device__ __forceinline__ float row_first(float v) {
  return __uint_as_float(dpp<0x150>(0u, __float_as_uint(v)));  // row_newbcast 0
}
// v[g] of row b of lanes becomes v[b] of row g
__device__ __forceinline__ void transpose4(uint32_t v[4]) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const auto r = __builtin_amdgcn_permlane32_swap(v[k], v[k + 2], false, false);
    v[k] = r[0];
    v[k + 2] = r[1];
  }
#pragma unroll
  for (int k = 0; k < 4; k += 2) {
    const auto r = __builtin_amdgcn_permlane16_swap(v[k], v[k + 1], false, false);
    v[k] = r[0];
    v[k + 1] = r[1];
  }
}
// mean over the lanes that are in
__device__ __forceinline__ float wave_mean(float v, bool in) {
  const uint64_t m = __ballot(in);
  v = in ? v : 0.f;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v / (float)__builtin_popcountll(m);
}
// minimum over the wave (no NaN)
__device__ __forceinline__ double wave_min_f64(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}
// orders the wave's LDS accesses before and after it
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A cell's query box as mx - 1 and mx - mn - 1 per axis.  The strict overlap
// of [mn, mx] with a region [lo, lo + s) on one axis, mx > lo and
// mn < lo + s, is (mx - 1 - lo) < (mx - mn - 1) + s in 32-bit unsigned
// arithmetic: the left side wraps past every right side when mx <= lo, and
// otherwise the two compares agree (mx >= mn: both codes are the same
// monotone map of x - h and x + h).
struct QBox {
  uint32_t ex0, ex1, ex2, dm0, dm1, dm2;
};
// query box, src/octree.c:246-266: ((x - h) - shift) / scale * 2^29
__device__ __forceinline__ QBox query_box(const double4 &P, double h, const double4 &A) {
  const uint32_t mn0 = box_code(P.x - h, A.x, A.w), mx0 = box_code(P.x + h, A.x, A.w);
  const uint32_t mn1 = box_code(P.y - h, A.y, A.w), mx1 = box_code(P.y + h, A.y, A.w);
  const uint32_t mn2 = box_code(P.z - h, A.z, A.w), mx2 = box_code(P.z + h, A.z, A.w);
  return QBox{mx0 - 1u, mx1 - 1u, mx2 - 1u, mx0 - mn0 - 1u, mx1 - mn1 - 1u, mx2 - mn2 - 1u};
}
__device__ __forceinline__ float volume(const QBox &b) {
  return (float)(b.dm0 + 1u) * (float)(b.dm1 + 1u) * (float)(b.dm2 + 1u);
}
// Morton order of two code triples (z, y, x within a level): the axis with the
// highest differing bit decides
__device__ __forceinline__ bool morton_less3(uint32_t ax, uint32_t ay, uint32_t az, uint32_t bx, uint32_t by,
                                             uint32_t bz) {
  const uint32_t dx = ax ^ bx, dy = ay ^ by, dz = az ^ bz;
  const bool y = (dz < dy) & (dz < (dz ^ dy));
  const uint32_t d = y ? dy : dz;
  const bool x = (d < dx) & (d < (d ^ dx));
  return x ? ax < bx : y ? ay < by : az < bz;
}
// a region: lower corner and sides in codes
struct Octant {
  uint32_t lx, ly, lz, sx, sy, sz;
};
__device__ __forceinline__ bool hits(const Octant &c, const QBox &b) {
  return (b.ex0 - c.lx < b.dm0 + c.sx) & (b.ex1 - c.ly < b.dm1 + c.sy) & (b.ex2 - c.lz < b.dm2 + c.sz);
}
// the region of a tree record
__device__ __forceinline__ Octant octant(const uint4 &a) {
  const uint32_t sx = 1u << ((a.x >> 29) | (((a.y >> 29) & 3u) << 3));
  return Octant{a.x & 0x1FFFFFFFu, a.y & 0x1FFFFFFFu,         a.z & 0x1FFFFFFFu,
                sx,                sx >> ((a.z >> 30) & 1u), sx >> ((a.z >> 29) & 1u)};
}
// the same of a leaf record (a cube)
__device__ __forceinline__ Octant leaf_octant(const uint4 &a) {
  const uint32_t s = 1u << ((a.x >> 29) | (((a.y >> 29) & 3u) << 3));
  return Octant{a.x & 0x1FFFFFFFu, a.y & 0x1FFFFFFFu, a.z & 0x1FFFFFFFu, s, s, s};
}

// the FP32 screening of one cell (see k_neighbors): thresholds, tin a further
// in_by inwards
struct Screen {
  float tin, tout, beta;
};
__device__ __forceinline__ Screen screen_of(const double4 &A, double cut2, double in_by) {
  Screen s;
  const double K = 1.7321 * (A.w * 1.2e-7 + 1e-44);
  const double hc = sqrt(cut2);
  double ti = (hc * (1.0 - 1e-15) - (K + in_by)) / (1.0 + 1e-7);
  ti = ti > 0.0 ? ti * ti / (1.0 + 3e-7) - 1e-44 : -1.0;
  // a threshold outside FP32's normal range decides nothing
  s.tin = (ti >= 1e-30 && ti <= 1e38) ? (float)(ti * (1.0 - 1e-6)) : -1.0f;
  double to = (hc * (1.0 + 1e-15) + K) / (1.0 - 1e-7);
  to = to * to * (1.0 + 3e-7) + 1e-44;
  // (overflow gives inf and NaN stays NaN: both decide nothing; below
  // FP32's normal range the threshold is raised, which only widens the
  // band read in FP64)
  s.tout = to < 1e-30 ? 1e-30f : (float)(to * (1.0 + 1e-6));
  s.beta = (float)((40500.0 * K * K + 1e-37) * (1.0 + 1e-6));
  return s;
}

// What every walk does last.  Pad each list to the longest one of its 64-cell
// slot group (this wave) with cell index n, the far-away stand-in record the
// build places after the cells: the pair kernels then read whole slot rows
// without per-lane tests, and a stand-in pair contributes exactly zero to the
// mixed sums (rows are written wave-wide, one 256-byte row per step).  Then
// the count, mindist, the last candidate and v, the potential with it
// (src/potential.c:124 assigns it per candidate; 0 beyond the cutoff and with
// no candidate); the records are read again here rather than kept through
// the walk.
template <int NW>
__device__ __forceinline__ void finish(int64_t p, bool live, uint32_t cnt, int32_t qs, double md2,
                                       const double4 *__restrict__ pos, const int32_t *__restrict__ ctype_s,
                                       const float *__restrict__ young_s, const TypeDev *__restrict__ types, int64_t n,
                                       int64_t cap, uint32_t *__restrict__ nbr, uint32_t *__restrict__ count,
                                       double *__restrict__ mindist, int32_t *__restrict__ qstar,
                                       double *__restrict__ vout, unsigned int *__restrict__ flags) {
  const uint32_t used = min(cnt, (uint32_t)cap);
  uint32_t g = used, lo = live ? used : 0xFFFFFFFFu;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    g = max(g, (uint32_t)__shfl_xor((int)g, o, 64));
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
  }
  if constexpr (NW > 1) {  // the group's cells lie in NW waves
    __shared__ uint32_t most[NW];
    if ((threadIdx.x & 63u) == 0) most[threadIdx.x >> 6] = g;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) g = max(g, most[w]);
  }
  for (uint32_t k = lo; k < g; ++k)
    if (live && k >= used) nbr[tm_slot(p, k, cap)] = (uint32_t)n;
  if (!live) return;
  count[p] = cnt;
  mindist[p] = qs >= 0 ? sqrt(md2) : 1.7976931348623157e308;
  qstar[p] = qs;
  const double4 P = pos[p];
  const double4 Qs = qs >= 0 ? pos[qs] : P;
  vout[p] = qs >= 0 ? pot_fp64(P, young_s[p], Qs, young_s[qs], types[ctype_s[p]].h) : 0.0;
  if (cnt > cap) atomicMax(flags + 1, cnt);
}

// WIN > 0: the workgroup first copies WIN consecutive slots of the
// pre-ordered tree, centred on the leaves of its own cells, into LDS; its
// walks read the nodes inside that window from LDS and the rest from memory.
// The cells of a workgroup are consecutive in Morton order, so their walks
// share many nodes near their own leaves (about half of all visits fall in
// 1024 slots around 256 cells), and a read from LDS spares the texture path
// the per-lane gather that bounds the walk.
// F32: candidates are screened with their FP32 positions relative to the
// colony's origin (16 bytes per candidate instead of 32); only a candidate
// whose FP32 distance cannot decide the cutoff, or that may hold the minimum
// distance, has its FP64 position read.  The results are those of the FP64
// walk (the bounds below are proved, not tuned):
//   stored values  |p~ - (P - A)| <= W (2^-24 + 2^-53) + 2^-150 per axis,
//                  W = the colony's largest extent >= |P - A|, so the FP32
//                  difference vector is within K = sqrt(3) * 1.2e-7 W
//                  (+1e-44) of the exact one after its own 2^-24 rounding,
//                  which is taken relative (1e-7) to the FP32 distance
//   FP32 sum       s~ = fma(dz, dz, fma(dy, dy, dx dx)): relative 3e-7,
//                  absolute 1e-44 from underflow
//   FP64 sum       the reference's d2 is within 1e-15 (relative) of the
//                  exact squared distance
// so with r~ = sqrt(s~), the reference's d2 lies in
//   [((r~ (1 - 1e-7) - K)+)^2 (1 - 1e-15), (r~ (1 + 1e-7) + K)^2 (1 + 1e-15)]
// (r~ widened by 3e-7 and 1e-44 as above).  tin / tout are the FP32 values
// of s~ below which d2 <= cut2 holds and above which it fails, each rounded
// inward by 1e-6; between them the candidate is read in FP64.  For the
// minimum, a candidate c cannot hold it when s~_c > 1.0002 s~_b + beta for
// a candidate b already seen: the bound above on both sides, with the cross
// term 4.02 K r~ <= 1e-4 r~^2 + 40401 K^2 (AM-GM), gives that threshold.
// The smallest FP32 distance is kept with its cell; the candidate that loses
// that place (the newcomer, or the one it displaces) is read in FP64 at once
// when it is still within reach of the smallest (rare), and the smallest is
// read in FP64 at the end.
template <int BS, int WIN, bool F32>
__global__ __launch_bounds__(BS) void k_neighbors(const double4 *__restrict__ pos, const float4 *__restrict__ posf,
                                                  const uint4 *__restrict__ code,
                                                  const int32_t *__restrict__ ctype_s,
                                                  const float *__restrict__ young_s,
                                                  const uint4 *__restrict__ wn,
                                                  const int64_t *__restrict__ col_off,
                                                  const double4 *__restrict__ aff,
                                                  const TypeDev *__restrict__ types, int64_t n, int64_t cap,
                                                  uint32_t *__restrict__ nbr,
                                                  uint32_t *__restrict__ count, double *__restrict__ mindist,
                                                  int32_t *__restrict__ qstar, double *__restrict__ vout,
                                                  unsigned int *__restrict__ flags) {
  const int64_t cell = tm_xcd_block() * BS + threadIdx.x;
  const bool live = cell < n;
  const int64_t p = live ? cell : n - 1;  // idle lanes only join the padding step below
  const double4 P = pos[p];
  const uint32_t cid = code[p].w;
  const double4 A = aff[cid];
  const TypeDev &T = types[ctype_s[p]];
  const double h = T.h;
  const double cut2 = T.cut2;
  const uint4 *winp = nullptr;
  const QBox box = query_box(P, h, A);
  // the window of slots staged in LDS: around the leaf slot of the
  // workgroup's middle cell, 2 s + 2 (e - k) for cell k of colony [s, e]
  // (up to its ancestor count), within the tree's 2 n - 1 slots
  uint32_t wlo = 0;
  if constexpr (WIN > 0) {
    __shared__ uint4 win[WIN];
    const int64_t km = min((int64_t)(tm_xcd_block() * BS + BS / 2), n - 1);
    const uint32_t cm = code[km].w;
    const int64_t cs = col_off[cm], ce = col_off[cm + 1] - 1;
    const int64_t nslot = 2 * n - 1;
    int64_t lo = 2 * cs + 2 * (ce - km) - WIN / 2;
    lo = max((int64_t)0, min(lo, nslot - WIN));
    wlo = (uint32_t)max((int64_t)0, lo);
    for (int i = threadIdx.x; i < WIN; i += BS) {
      const int64_t sl = (int64_t)wlo + i;
      win[i] = sl < nslot ? wn[sl] : make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
    winp = win;
  }
  // the colony's slots of the pre-ordered tree
  uint32_t node = live ? (uint32_t)(2 * col_off[cid]) : 0u;
  const uint32_t end = live ? (uint32_t)(2 * col_off[cid + 1] - 1) : 0u;
  uint32_t cnt = 0;
  int32_t qs = -1;
  double md2 = 1.0 / 0.0;
  // candidate q (its leaf octant overlaps the box, q != p) with its position
  // Q: distance, mindist, the last-visited candidate, and the list entry when
  // within the cutoff (returned as its slot, stored by the caller; -1 if none)
  using QRec = typename std::conditional<F32, float4, double4>::type;
  // FP32 screening state: the cell's FP32 relative position, the cutoff
  // thresholds, and the smallest FP32 distance so far with its cell
  float pfx = 0.f, pfy = 0.f, pfz = 0.f, tin = -1.f, tout = 0.f, beta = 0.f;
  float s1 = 1.0f / 0.0f;
  uint32_t c1 = 0xFFFFFFFFu;
  if constexpr (F32) {
    pfx = (float)(P.x - A.x);
    pfy = (float)(P.y - A.y);
    pfz = (float)(P.z - A.z);
    const Screen s = screen_of(A, cut2, 0.0);
    tin = s.tin;
    tout = s.tout;
    beta = s.beta;
  }
  // the reference's d2 of candidate q, read in FP64, into the minimum
  auto exact = [&](uint32_t q) -> double {
    const double d2 = dist2_fp64(P, pos[q]);
    md2 = d2 < md2 ? d2 : md2;
    return d2;
  };
  auto visit = [&](uint32_t q, const QRec &Q) -> int64_t {
    bool in;
    if constexpr (F32) {
      const float dx = pfx - Q.x, dy = pfy - Q.y, dz = pfz - Q.z;
      const float sq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
      if (sq <= tin) in = true;
      else if (sq > tout) in = false;
      else in = exact(q) <= cut2;
      // the smallest (selects); the one that loses it
      const bool lt = sq < s1;
      const float so = lt ? s1 : sq;
      const uint32_t co = lt ? c1 : q;
      s1 = lt ? sq : s1;
      c1 = lt ? q : c1;
      if (so <= fmaf(1.0002f, s1, beta)) {
        if (co != 0xFFFFFFFFu) (void)exact(co);
      }
    } else {
      const double d2 = dist2_fp64(P, Q);
      md2 = d2 < md2 ? d2 : md2;
      in = d2 <= cut2;
    }
    qs = (int32_t)q;
    int64_t slot = -1;
    if (in) {
      if (cnt < cap) slot = tm_slot(p, cnt, cap);
      ++cnt;
    }
    return slot;
  };
  // One record per node: after a hit the next slot (the first child, or for
  // a leaf the next node), after a miss the escape slot; slots only grow, so
  // the walk ends at the colony's last slot.  A candidate's record load is
  // issued when its leaf is found and consumed one node later, under the
  // next node's load; its list entry is stored after that node's loads are
  // issued, so waiting for them does not also wait for the store (vector
  // memory counters retire in order).  Candidates are still taken in visit
  // order.
  uint32_t pq = 0xFFFFFFFFu;  // the candidate whose record is in flight
  QRec Qp{};
  while (node < end) {
    uint4 a;
    if constexpr (WIN > 0) {
      const uint32_t wi = node - wlo;
      a = wi < (uint32_t)WIN ? winp[wi] : wn[node];
    } else {
      a = wn[node];
    }
    int64_t slot = -1;
    const uint32_t q = pq;
    if (pq != 0xFFFFFFFFu) {
      slot = visit(pq, Qp);
      pq = 0xFFFFFFFFu;
    }
    const bool hit = hits(octant(a), box);
    const bool leaf = (a.y & 0x80000000u) != 0u;
    const uint32_t next = (hit || leaf) ? node + 1 : a.w;
    if (next <= node || (leaf && a.w >= (uint32_t)n)) {  // a malformed tree: a well-formed one only moves forward
      if (slot >= 0) nbr[slot] = q;
      atomicOr(flags, (unsigned)TM_FLAG_WALK);
      break;
    }
    if (leaf && hit && a.w != (uint32_t)p) {
      if constexpr (F32) Qp = posf[a.w];
      else Qp = pos[a.w];
      pq = a.w;
    }
    if (slot >= 0) nbr[slot] = q;
    node = next;
  }
  if (pq != 0xFFFFFFFFu) {
    const int64_t slot = visit(pq, Qp);
    if (slot >= 0) nbr[slot] = pq;
  }
  if constexpr (F32) {
    // the smallest
    if (c1 != 0xFFFFFFFFu) (void)exact(c1);
  }
  finish<1>(p, live, cnt, qs, md2, pos, ctype_s, young_s, types, n, cap, nbr, count, mindist, qstar, vout, flags);
}

// The cooperative walk: a wave looks once for all cells that any of its own G
// may take, and its lanes pick theirs from those.  The per-lane walk above
// reads a tree record per node and lane (257 per cell in the 2M-cell Gaussian
// colony, 25 K vector instructions per wave of 64 cells); here a wave issues
// 12 K, and half of its loads fetch 64 consecutive records.
//
//   1. The wave's cells are cut in two at the highest Morton step between two
//      of them, and the union of either part's query boxes is formed (a run of
//      Morton order often lies in two places; one box over both held 1.7 times
//      as many candidates, and up to 33 K).  Each row of 16 lanes gets two
//      boxes the same way.
//   2. From the top of the tree of boxes (BvhNode) the wave finds the blocks
//      of 16 cells that overlap the two boxes, 64 nodes per load, then tests
//      their cells' leaf octants, four blocks per load, in descending Morton
//      order.  Every leaf that overlaps a cell's own box overlaps its part's
//      union, and boxes above it contain it, so none is missed.
//   3. The leaves found (547 per 64 cells at 2M) are staged in LDS, CB at a
//      time; each row keeps a list of those that overlap its own boxes (about
//      250; one byte each).
//   4. The last candidate of each lane (qstar) comes from its row's list, from
//      the end.
//   5. The entries within a lane's cutoff: FP32 squared distances of 16
//      entries to the row's 16 cells as outer products on the matrix cores,
//      with a margin that covers their rounding; the lane then takes those
//      marked, in order, with the FP32 screening of the per-lane walk: tin is
//      taken four code units further in, so that a candidate at most that far
//      away also overlaps the query box strictly (its code differs from both
//      corners'); between tin and tout the distance and the octant are
//      evaluated exactly.  Candidates beyond the cutoff matter only for qstar
//      and, where a cell has none within, for mindist.
//   6. mindist: the smallest FP32 distance and the second smallest are kept;
//      the first is read in FP64, and the cell's list once more where the
//      second is within reach of it.  A cell with candidates but none within
//      its cutoff takes the minimum over all of them, the wave's lanes sharing
//      the work: a few such cells two at a time over the candidates kept (or
//      alone down the tree, if there were more), from 14 in 64 or 8 in 32 on all
//      of them together over the group's blocks, with marks as in 5 by the
//      distance to the last candidate.  A pair costs 0.8 ns of a 2M-cell walk, a
//      cell alone 0.7 ns, all together 8 ns.  Steps of a ball at a volume fraction
//      of 0.08, where 53 % of the cells have no neighbour, without and with that
//      third way: 300 K cells 436 and 339 us, 2M 1,482 and 1,027; at 0.02 482 and
//      303, 1,607 and 967 us.
// A group whose cells lie in more places than two boxes serve (its queue full
// and the boxes more than `ratio` times the cells' own) is taken in parts, cut
// at the step; a wave's colonies are taken one after another.
//
// What bounds it: vector issue (80% of the SIMDs' cycles at 2M cells with the
// four waves per SIMD that 127 registers allow; the list entries cost 12 K
// instructions per wave), below about 500 K cells the longest wave, whose
// cells lie in many places: a wave then takes fewer cells (launch_union).
// Walk alone, per-lane before and this: 20 K-cell ball 119 and 43 us, 300 K
// ball 208 and 175 us, 2M Gaussian 1,729 and 862 us (three seeds: 843 to 897),
// 4M cells in 128 colonies 3,358 and 1,700 us, 3M of two types 3,605 and
// 1,580 us; and the build need not make the radix tree (130 us of 500 at 2M).
// Also measured: the per-lane walk's tree read 64 slots at a time in its
// pre-order (103 dependent loads per wave against 48 here) 450 us of a 1.46 ms
// walk; distances on the vector unit 5% slower at 2M; blocks of 32 cells 8%
// more loads.
constexpr int CB = 255;  // candidates staged at a time (a byte names one; 255 names none)
// FP32 rounding of |c|^2 + |p|^2 - 2 c.p (five products and sums, operands
// rounded to 2^-24) stays within 1.5e-6 (|c|^2 + |p|^2): the squares are
// taken 2^-18 too small
constexpr float LESS = 1.0f - 0x1p-18f;
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int BQ = 320;  // blocks queued (a node's 64 children must fit beside the ratio's)
constexpr int UC = 512;  // candidates of a wave kept for its cells without a neighbour

// For 16 entries c and a row's 16 cells p, the four rows at once, the signs of
// |c|^2 + |p|^2 - 2 c.p less a threshold, by five outer products: lane 16 g + j
// collects those of entries 4 g + k and cell j of row q in word q (mw: |p|^2 less
// the threshold).
__device__ __forceinline__ void marks(float x, float y, float z, float mx, float my, float mz, float mw,
                                      uint32_t (&near)[4]) {
  const float c2 = fmaf(z, z, fmaf(y, y, x * x));
  const bool fits = c2 < 1e37f;
  f32x16 d{};
  d = __builtin_amdgcn_mfma_f32_16x16x1f32(fits ? -2.0f * x : 0.f, mx, d, 0, 0, 0);
  d = __builtin_amdgcn_mfma_f32_16x16x1f32(fits ? -2.0f * y : 0.f, my, d, 0, 0, 0);
  d = __builtin_amdgcn_mfma_f32_16x16x1f32(fits ? -2.0f * z : 0.f, mz, d, 0, 0, 0);
  d = __builtin_amdgcn_mfma_f32_16x16x1f32(fits ? c2 * LESS : -1e38f, 1.0f, d, 0, 0, 0);
  d = __builtin_amdgcn_mfma_f32_16x16x1f32(1.0f, mw, d, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) near[q] = __builtin_amdgcn_alignbit(near[q], __float_as_uint(d[4 * q + k]), 31);
}

template <int G>
__global__ __launch_bounds__(4096 / G, 4) void k_union(
    const double4 *__restrict__ pos, const float4 *__restrict__ posf, const uint4 *__restrict__ code,
    const int32_t *__restrict__ ctype_s, const float *__restrict__ young_s, const uint4 *__restrict__ leaf,
    const BvhNode *__restrict__ bvh, Bvh tree, const int64_t *__restrict__ col_off, const double4 *__restrict__ aff,
    const TypeDev *__restrict__ types, int64_t n, int64_t cap, uint32_t *__restrict__ nbr,
    uint32_t *__restrict__ count, double *__restrict__ mindist, int32_t *__restrict__ qstar,
    double *__restrict__ vout, unsigned int *__restrict__ flags, uint32_t ratio) {
  constexpr int NW = 64 / G;     // waves per workgroup
  constexpr int BARE = G == 64 ? 13 : G == 32 ? 7 : 64;  // cells without a neighbour that are few
  constexpr int ROWS = G < 16 ? 1 : G / 16;  // rows of lanes with cells
  __shared__ uint4 crec_[NW][CB + 1];  // a staged candidate: its octant and cell, later its record and cell
  // per row of 16 lanes the staged candidates it may take, one byte each
  __shared__ __align__(16) uint32_t sub_[NW][4 * 64];
  __shared__ QBox rbox_[NW][2 * ROWS];  // per row its two boxes
  // blocks of 16 cells to look into; last their number, if these are all of the group's
  __shared__ uint32_t queue_[NW][BQ + 1];
  __shared__ uint32_t ucell_[NW][UC];   // the first candidates (cells)
  const uint32_t lane = threadIdx.x & 63u, row = lane >> 4, wv = threadIdx.x >> 6;
  uint4 *const crec = crec_[wv];
  uint32_t *const sub = sub_[wv];
  QBox *const rbox = rbox_[wv];
  uint32_t *const queue = queue_[wv];
  uint32_t *const ucell = ucell_[wv];
  uint8_t *const sub8 = reinterpret_cast<uint8_t *>(sub);
  const int64_t cell = tm_xcd_block() * 64 + G * (int64_t)wv + lane;
  const bool live = lane < (uint32_t)G && cell < n;
  const int64_t p = live ? cell : n - 1;  // idle lanes only join the wave-wide steps
  // values used once per group of cells, or rarely, are read again where they
  // are used rather than held in registers through the walk
  auto again = [&]() {
    int64_t v = p;
    asm volatile("" : "+v"(v));
    return v;
  };
  const uint32_t cid = code[p].w;
  QBox own;
  float pfx, pfy, pfz, tin, tout;
  {
    const double4 P = pos[p], A = aff[cid];
    const TypeDev &T = types[ctype_s[p]];
    own = query_box(P, T.h, A);
    pfx = (float)(P.x - A.x);
    pfy = (float)(P.y - A.y);
    pfz = (float)(P.z - A.z);
    // tin four code units further in, so that a candidate it accepts also
    // overlaps the query box; none is accepted where the coordinates are so
    // large beside W that FP64 rounding moves a code
    const double far = fmax(fmax(fabs(A.x), fabs(A.y)), fabs(A.z)) + A.w;
    const Screen s = screen_of(A, T.cut2, far <= A.w * 1048576.0 ? A.w * 0x1p-27 : 1.0 / 0.0);
    tin = s.tin;
    tout = s.tout;
  }
  auto dist2_f32 = [&](const float4 &Q) {
    const float dx = pfx - Q.x, dy = pfy - Q.y, dz = pfz - Q.z;
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  };
  uint32_t cnt = 0;
  int32_t qs = -1;
  double md2 = 1.0 / 0.0;
  uint64_t todo = __ballot(live), solo = 0;
  uint32_t upto = 64;  // lanes from here on wait (after a group that held too many candidates)
  while (todo) {
    // the group: the first waiting cell's colony, up to lane upto; or that
    // cell alone
    const uint32_t first = (uint32_t)__builtin_ctzll(todo);
    const uint32_t scid = (uint32_t)__builtin_amdgcn_readlane((int)cid, (int)first);
    const bool single = (solo >> first) & 1u;
    const bool mine = single ? lane == first : ((todo & ~solo) >> lane & 1u) && cid == scid && lane < upto;
    if (mine) {
      cnt = 0;
      qs = -1;
      md2 = 1.0 / 0.0;
    }
    // the smallest FP32 distance accepted by tin, with its cell, and the
    // second smallest
    float s1 = 1.0f / 0.0f, s2 = 1.0f / 0.0f;
    uint32_t c1 = 0xFFFFFFFFu;
    // the group cut at the highest Morton step between two of its cells, and
    // each row's cells at the row's: the place of the highest bit that differs
    // from the lane before (0: none)
    uint32_t step = 0;
    {
      const uint4 me = code[again()];
      const uint32_t ox = me.x ^ dpp<0x138>(0u, me.x), oy = me.y ^ dpp<0x138>(0u, me.y),
                     oz = me.z ^ dpp<0x138>(0u, me.z);  // wave_shr 1
      const uint32_t o = ox | oy | oz;
      if (mine && lane > first && o) {
        const uint32_t b = (uint32_t)tm_msb32(o);
        step = ((3u * b + ((oz >> b) & 1u ? 2u : (oy >> b) & 1u ? 1u : 0u) + 1u) << 6) | lane;
      }
    }
    const uint32_t wstep = wave_max_u32(step);
    const uint32_t rstep = row_max_u32((lane & 15u) ? step : 0u);
    const uint32_t wcut = wstep ? wstep & 63u : 64u, rcut = rstep ? rstep & 63u : 64u;
    auto box_of = [&](bool in, auto &&reduce) {
      QBox b;
      auto axis = [&](uint32_t ex, uint32_t dm, uint32_t &bex, uint32_t &bdm) {
        const uint32_t h = reduce(in ? ex + 1u : 0u), l = ~reduce(in ? ~(ex - dm) : 0u);
        bex = h - 1u;  // no cells: ex = 2^32 - 1, dm = 0, which overlaps nothing
        bdm = h - l - 1u;
      };
      axis(own.ex0, own.dm0, b.ex0, b.dm0);
      axis(own.ex1, own.dm1, b.ex1, b.dm1);
      axis(own.ex2, own.dm2, b.ex2, b.dm2);
      return b;
    };
    auto on_wave = [](uint32_t v) { return wave_max_u32(v); };
    auto on_row = [](uint32_t v) { return row_max_u32(v); };
    const QBox boxa = box_of(mine && lane < wcut, on_wave), boxb = box_of(mine && lane >= wcut, on_wave);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const QBox b = box_of(mine && (half ? lane >= rcut : lane < rcut), on_row);
      if ((lane & 15u) == 0 && row < (uint32_t)ROWS) rbox[2 * row + half] = b;
    }
    // the cell's side of the products below, relative to the row's first cell;
    // where FP32 cannot hold the squares everything is near
    const float ox = row_first(pfx), oy = row_first(pfy), oz = row_first(pfz);
    float mx = pfx - ox, my = pfy - oy, mz = pfz - oz, mw;
    {
      const float p2 = fmaf(mz, mz, fmaf(my, my, mx * mx));
      const bool fits = p2 < 1e37f && tout < 1e37f;
      mw = fits ? p2 * LESS - (tout * (1.0f + 1e-6f) + 1e-36f) : -1e38f;
      mx = fits ? mx : 0.f;
      my = fits ? my : 0.f;
      mz = fits ? mz : 0.f;
    }
    uint32_t nb = 0;  // staged candidates
    auto drain = [&]() {
      reinterpret_cast<uint4 *>(sub)[lane] = make_uint4(~0u, ~0u, ~0u, ~0u);
      wave_lds_sync();
      // the staged candidates of each row, in order: those that overlap one
      // of its two boxes
      float4 f[(CB + 64) / 64];
      uint32_t len[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int b = 0; b < (CB + 64) / 64; ++b) {
        f[b] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (64u * b < nb) {
          const uint32_t e = 64u * b + lane;
          const bool ok = e < nb;
          const uint4 r = crec[ok ? e : 0u];
          f[b] = posf[r.w];
          const Octant c = leaf_octant(r);
#pragma unroll
          for (int q = 0; q < ROWS; ++q) {
            uint32_t at = 2u * q;  // (opaque: two boxes in registers at a time, not all eight)
            asm volatile("" : "+v"(at));
            const bool h0 = hits(c, rbox[at]), h1 = hits(c, rbox[at + 1]);
            const bool hit = ok & (h0 | h1);
            const uint64_t m = __ballot(hit);
            if (hit) sub8[256 * q + len[q] + mbcnt64(m)] = (uint8_t)e;
            len[q] += (uint32_t)__builtin_popcountll(m);
          }
        }
      }
      wave_lds_sync();
      const uint32_t mylen = row == 0 ? len[0] : row == 1 ? len[1] : row == 2 ? len[2] : len[3];
      const uint8_t *const mysub = sub8 + 256 * row;
      // The last candidate so far: the row's list backwards to the first octant
      // that overlaps the lane's box.  An octant that does holds a code at or
      // above the box's lower corner on every axis, so its last key is no
      // smaller than that corner's: the octants of the list's end with smaller
      // ones are skipped by a binary search (the list's keys descend).
      {
        const uint32_t nx = own.ex0 - own.dm0, ny = own.ex1 - own.dm1, nz = own.ex2 - own.dm2;
        uint32_t at = 0;
#pragma unroll 1
        for (uint32_t b = 128; b > 0; b >>= 1) {
          const uint4 r = crec[mysub[min(at + b - 1, 255u)]];
          const Octant c = leaf_octant(r);
          const bool skip = morton_less3(c.lx + c.sx - 1, c.ly + c.sy - 1, c.lz + c.sz - 1, nx, ny, nz);
          at += ((at + b <= mylen) & !skip) ? b : 0u;
        }
        // upwards from there, as far as an octant's first key exceeds the
        // box's upper corner's
        bool want = mine & (at > 0);
        for (int k = 0; k < 8 && __ballot(want); ++k) {
          if (want) {
            --at;
            const uint4 r = crec[mysub[at]];
            const Octant c = leaf_octant(r);
            const bool hit = hits(c, own) & (r.w != (uint32_t)p);
            qs = hit ? (int32_t)r.w : qs;
            want = !hit & (at > 0) & !morton_less3(own.ex0, own.ex1, own.ex2, c.lx, c.ly, c.lz);
          }
        }
        // a lane that needs more steps has the rest searched by the whole
        // wave, 64 entries at a time
        for (uint64_t left = __ballot(want); left; left &= left - 1) {
          const int who = __builtin_ctzll(left);
          auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, who); };
          const QBox b{of(own.ex0), of(own.ex1), of(own.ex2), of(own.dm0), of(own.dm1), of(own.dm2)};
          const uint32_t wp = of((uint32_t)p);
          const uint8_t *const wsub = sub8 + 256 * (who >> 4);
          for (int k1 = (int)of(at); k1 > 0; k1 -= 64) {
            const int k = k1 - 64 + (int)lane;
            const uint4 r = crec[k >= 0 ? wsub[k] : CB];
            const uint64_t m = __ballot((k >= 0) & hits(leaf_octant(r), b) & (r.w != wp));
            if (m) {
              const int32_t q = __builtin_amdgcn_readlane((int)r.w, 63 - __builtin_clzll(m));
              if ((int)lane == who) qs = q;
              break;
            }
          }
        }
      }
      if (single) {
        // a cell alone: every staged candidate but itself is one of its own
        const int64_t pf = (int64_t)__builtin_amdgcn_readlane((int)p, (int)first);
        const double4 W = pos[pf];
        double least = 1.0 / 0.0;
        for (uint32_t e = lane; e < nb; e += 64) {
          const uint32_t q = crec[e].w;
          if (q != (uint32_t)pf) least = fmin(least, dist2_fp64(W, pos[q]));
        }
        least = wave_min_f64(least);
        if (mine) md2 = least < md2 ? least : md2;
      }
      wave_lds_sync();
      float4 *const cq = reinterpret_cast<float4 *>(crec);
#pragma unroll
      for (int b = 0; b < (CB + 64) / 64; ++b) {
        const uint32_t e = 64u * b + lane;
        if (e < nb) cq[e] = make_float4(f[b].x, f[b].y, f[b].z, __uint_as_float(crec[e].w));
      }
      if (lane == 0) cq[CB] = make_float4(1.0e15f, 1.0e15f, 1.0e15f, 0.f);  // far from every cell
      wave_lds_sync();
      const uint32_t most = max(max(len[0], len[1]), max(len[2], len[3]));
      for (uint32_t k0 = 0; k0 < most; k0 += 128) {
        // Which of the row's next 16 T entries may be within a lane's cutoff:
        // bit 31 - b of word g for entry 4 T g + b, b < 4 T.  The squared
        // distances of 16 entries to the row's 16 cells, for the four rows at
        // once, as |c|^2 + |p|^2 - 2 c.p by five outer products (relative to
        // the row's first cell); lane 16 g + j holds those of entries 4 g + k
        // of each row to the row's cell j, whose signs (less the threshold,
        // with a margin for the rounding) are collected per row and then
        // exchanged between the rows of lanes.
        const uint32_t T = min(8u, (most - k0 + 15) >> 4);
        uint32_t near[4] = {0u, 0u, 0u, 0u};
        const uint8_t *const mine8 = mysub + k0 + 4 * T * ((lane & 15u) >> 2) + (lane & 3u);
        float4 Qn = cq[mine8[0]];
#pragma unroll 1
        for (uint32_t t = 0; t < T; ++t) {
          const float4 Q = Qn;
          Qn = cq[mine8[4 * min(t + 1, T - 1)]];
          marks(Q.x - ox, Q.y - oy, Q.z - oz, mx, my, mz, mw, near);
        }
        transpose4(near);
#pragma unroll
        for (int q = 0; q < 4; ++q) near[q] = mine ? near[q] << (32u - 4u * T) : 0u;
        // those, in order
        uint32_t kb = k0;
        while (near[0] | near[1] | near[2] | near[3]) {
          if (near[0] == 0u) {
            near[0] = near[1];
            near[1] = near[2];
            near[2] = near[3];
            near[3] = 0u;
            kb += 4 * T;
          }
          if (near[0] != 0u) {
            const uint32_t j = (uint32_t)__clz((int)near[0]);
            near[0] ^= 0x80000000u >> j;
            const uint32_t e = mysub[kb + j];
            const float4 Q = cq[e];
            const uint32_t q = __float_as_uint(Q.w);
            if (q != (uint32_t)p && e != (uint32_t)CB) {
              const float sq = dist2_f32(Q);
              bool in = sq <= tin;
              if (in) {
                s2 = __builtin_amdgcn_fmed3f(s1, s2, sq);
                c1 = sq < s1 ? q : c1;
                s1 = fminf(s1, sq);
              } else {
                // the FP32 distance leaves the cutoff or the octant open
                const int64_t pa = again();
                const double d2 = dist2_fp64(pos[pa], pos[q]);
                in = d2 <= types[ctype_s[pa]].cut2 && hits(leaf_octant(leaf[q]), own);
                if (in) md2 = d2 < md2 ? d2 : md2;
              }
              if (in) {
                if (cnt < cap) nbr[tm_slot(p, cnt, cap)] = q;
                ++cnt;
              }
            }
          }
        }
      }
      wave_lds_sync();
      nb = 0;
    };
    // The colony's cells whose octants overlap one of the two boxes, in
    // descending order: the blocks of 16 cells that overlap, found from the
    // top of the tree of boxes down into a queue, then their cells, four
    // blocks at a time.  Bits of a mask are taken from the highest.
    const uint32_t s = (uint32_t)col_off[scid], e = (uint32_t)(col_off[scid + 1] - 1);
    // lane's child of the 64 of node g, and the children that overlap and hold
    // cells of the colony
    auto child = [&](const BvhNode *lv, uint32_t sh, uint32_t g) {
      const uint32_t lo = s >> sh, hi = e >> sh, i = 64u * g + lane;
      const BvhNode *const b = lv + min(max(i, lo), hi);
      const uint4 u = *reinterpret_cast<const uint4 *>(b);
      const uint2 v = *reinterpret_cast<const uint2 *>(&b->sy);
      return Octant{u.x, u.y, u.z, u.w, v.x, v.y};
    };
    auto overlapping = [&](const Octant &c, uint32_t sh, uint32_t g) -> uint64_t {
      const uint32_t i = 64u * g + lane;
      const bool ha = hits(c, boxa), hb = hits(c, boxb);
      return __ballot((i >= s >> sh) & (i <= e >> sh) & (ha | hb));
    };
    // (a level with a single node for the colony is not read)
    auto children = [&](const BvhNode *lv, uint32_t sh, uint32_t g) -> uint64_t {
      const uint32_t lo = s >> sh;
      return lo == e >> sh ? 1ull << (lo & 63u) : overlapping(child(lv, sh, g), sh, g);
    };
    auto top = [](uint64_t m) { return 63u - (uint32_t)__builtin_clzll(m); };
    uint64_t m3 = 0, m2 = 0, m1 = 0;
    uint32_t i3 = 0, i2 = 0, found = 0;
    int g3 = (int)(e >> 28);
    bool over = false;
    for (bool last = false, full = false; !last && !over; full = false) {
      uint32_t nq = 0;
      for (;;) {
        for (;;) {
          for (;;) {
            if (m1) {
              uint32_t i1 = 64u * i2 + top(m1);
              Octant next = child(bvh, 4, i1);
              do {
                const Octant c = next;
                const uint64_t m = m1 & ~(1ull << (i1 & 63u));
                const uint32_t j1 = 64u * i2 + (m ? top(m) : 0u);
                if (m) next = child(bvh, 4, j1);
                const uint64_t m0 = overlapping(c, 4, i1);
                const uint32_t k = (uint32_t)__builtin_popcountll(m0);
                full = nq + k > (uint32_t)BQ;
                if (full) break;
                if ((m0 >> lane) & 1u) queue[nq + k - 1 - mbcnt64(m0)] = 64u * i1 + lane;
                nq += k;
                m1 = m;
                i1 = j1;
              } while (m1);
            }
            if (full || !m2) break;
            i2 = 64u * i3 + top(m2);
            m2 &= ~(1ull << (i2 & 63u));
            m1 = children(bvh + tree.l1, 10, i2);
          }
          if (full || !m3) break;
          i3 = 64u * (uint32_t)(g3 + 1) + top(m3);
          m3 &= ~(1ull << (i3 & 63u));
          m2 = children(bvh + tree.l2, 16, i3);
        }
        if (full) break;
        last = g3 < (int)(s >> 28);
        if (last) break;
        m3 = children(bvh + tree.l3, 22, (uint32_t)g3);
        --g3;
      }
      // many blocks, and boxes much larger than the cells' own: the cells lie
      // in several places, and those before the cut are taken first
      if (wstep && nq > min(4u * ratio, (uint32_t)BQ - 64u) &&
          volume(boxa) + volume(boxb) > (float)ratio * wave_mean(volume(own), mine)) {
        over = true;
        break;
      }
      if (G > BARE) queue[BQ] = last && found == 0 && nb == 0 ? nq : 0u;
      wave_lds_sync();
      auto block = [&](uint32_t i) { return i + row < nq ? queue[i + row] : ~0u; };
      auto load = [&](uint32_t blk) {
        const uint32_t q = blk * 16u + (15u - (lane & 15u));
        const bool ok = (blk != ~0u) & (q >= s) & (q <= e);
        uint4 r = leaf[ok ? q : s];
        r.w = ok ? r.w : ~0u;
        return r;
      };
      uint4 rn = load(block(0));
      uint32_t bn = block(4);
      for (uint32_t i = 0;; i += 4) {
        const bool more = i < nq;
        const uint4 r = rn;
        rn = load(bn);
        bn = block(i + 8);
        const Octant c = leaf_octant(r);
        const bool ha = hits(c, boxa), hb = hits(c, boxb);
        const bool cand = (r.w != ~0u) & (ha | hb);  // none past the queue's end
        const uint64_t cm = __ballot(cand);
        const uint32_t k = (uint32_t)__builtin_popcountll(cm);
        if (nb + k > (uint32_t)CB || (!more && last && nb > 0)) drain();
        if (!more) break;
        if (cand) {
          const uint32_t at = mbcnt64(cm);
          crec[nb + at] = r;
          if (found + at < (uint32_t)UC) ucell[found + at] = r.w;
        }
        nb += k;
        found += k;
      }
    }
    if (over) {
      upto = wcut;
      continue;
    }
    upto = 64;
    const uint64_t group = __ballot(mine);
    todo &= ~group;
    solo &= ~group;
    // Cells with candidates but none within the cutoff: the minimum distance
    // takes every candidate.  Many such cells: together.  A few: two at a time,
    // the lanes taking the group's candidates; with more of those than are kept,
    // each is walked alone.
    uint64_t bare = single ? 0ull : __ballot(mine && cnt == 0 && qs >= 0);
    uint32_t blocks = 0;
    if (G > BARE && __builtin_popcountll(bare) > BARE) blocks = (uint32_t)__builtin_amdgcn_readfirstlane((int)queue[BQ]);
    if (blocks > 0) {
      // Over the group's blocks once more.  The last candidate bounds the
      // distance: of the cells that overlap the group's boxes those within its
      // reach are marked as above, and of them the candidates within reach of
      // the nearest so far are read in FP64.
      const bool in = (bare >> lane) & 1u;
      float least = 1.0f / 0.0f, beta = 0.f;
      if (in) {
        least = dist2_f32(posf[qs]);
        beta = screen_of(aff[cid], 1.0, 0.0).beta;
      }
      float nx = pfx - ox, ny = pfy - oy, nz = pfz - oz, nw;
      {
        const float p2 = fmaf(nz, nz, fmaf(ny, ny, nx * nx)), limit = fmaf(1.0002f, least, beta);
        const bool fits = p2 < 1e37f && limit < 1e37f;
        nw = fits ? p2 * LESS - (limit * (1.0f + 1e-6f) + 1e-36f) : -1e38f;
        nx = fits ? nx : 0.f;
        ny = fits ? ny : 0.f;
        nz = fits ? nz : 0.f;
      }
      float4 *const cq = reinterpret_cast<float4 *>(crec);
      for (uint32_t i = 0;; i += 4) {
        const uint32_t b = i + row < blocks ? queue[i + row] : ~0u, c = b * 16u + (lane & 15u);
        const bool more = i < blocks, ok = (b != ~0u) & (c >= s) & (c <= e);
        const uint4 r = leaf[ok ? c : s];
        const Octant o = leaf_octant(r);
        const bool ha = hits(o, boxa), hb = hits(o, boxb), cand = ok & (ha | hb);
        const uint64_t cm = __ballot(cand);
        const uint32_t k = (uint32_t)__builtin_popcountll(cm);
        if (nb + k > (uint32_t)CB || (!more && nb > 0)) {
          wave_lds_sync();
          for (uint32_t u = lane; u < ((nb + 15u) & ~15u); u += 64) {
            const uint32_t q = u < nb ? crec[u].w : 0u;
            const float4 P = u < nb ? posf[q] : make_float4(1.0e15f, 1.0e15f, 1.0e15f, 0.f);
            cq[u] = make_float4(P.x, P.y, P.z, __uint_as_float(q));
          }
          wave_lds_sync();
          for (uint32_t k0 = 0; k0 < nb; k0 += 128) {
            // bit 31 - b of word g: entry k0 + 16 (b / 4) + 4 g + b % 4
            const uint32_t T = min(8u, (nb - k0 + 15u) >> 4);
            uint32_t near[4] = {0u, 0u, 0u, 0u};
#pragma unroll 1
            for (uint32_t t = 0; t < T; ++t) {
              const float4 Q = cq[k0 + 16u * t + (lane & 15u)];
              marks(Q.x - ox, Q.y - oy, Q.z - oz, nx, ny, nz, nw, near);
            }
            transpose4(near);
#pragma unroll
            for (int q = 0; q < 4; ++q) near[q] = in ? near[q] << (32u - 4u * T) : 0u;
            uint32_t at = k0;
            while (near[0] | near[1] | near[2] | near[3]) {
              if (near[0] == 0u) {
                near[0] = near[1];
                near[1] = near[2];
                near[2] = near[3];
                near[3] = 0u;
                at += 4u;
              }
              if (near[0] != 0u) {
                const uint32_t j = (uint32_t)__clz((int)near[0]), u = at + 16u * (j >> 2) + (j & 3u);
                near[0] ^= 0x80000000u >> j;
                const float4 Q = cq[u];
                const uint32_t q = __float_as_uint(Q.w);
                const float sq = dist2_f32(Q);
                if (u < nb && q != (uint32_t)p && !(sq > fmaf(1.0002f, least, beta)) && hits(leaf_octant(leaf[q]), own)) {
                  const double d2 = dist2_fp64(pos[again()], pos[q]);
                  md2 = d2 < md2 ? d2 : md2;
                  least = fminf(least, sq);
                }
              }
            }
          }
          wave_lds_sync();
          nb = 0;
        }
        if (!more) break;
        if (cand) crec[nb + mbcnt64(cm)] = r;
        nb += k;
      }
    } else if (found > (uint32_t)UC) {
      todo |= bare;
      solo |= bare;
    } else if (bare) {
      wave_lds_sync();
      while (bare) {
        const int w0 = __builtin_ctzll(bare);
        bare &= bare - 1;
        const int w1 = bare ? __builtin_ctzll(bare) : w0;
        bare &= bare - 1;
        auto box_at = [&](int w) {
          auto of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, w); };
          return QBox{of(own.ex0), of(own.ex1), of(own.ex2), of(own.dm0), of(own.dm1), of(own.dm2)};
        };
        const QBox b0 = box_at(w0), b1 = box_at(w1);
        const uint32_t p0 = (uint32_t)__builtin_amdgcn_readlane((int)p, w0),
                       p1 = (uint32_t)__builtin_amdgcn_readlane((int)p, w1);
        const double4 W0 = pos[p0], W1 = pos[p1];
        double l0 = 1.0 / 0.0, l1 = 1.0 / 0.0;
#pragma unroll 2
        for (uint32_t k = lane; k < found; k += 64) {
          const uint32_t q = ucell[k];
          const Octant c = leaf_octant(leaf[q]);
          const bool h0 = hits(c, b0) & (q != p0), h1 = hits(c, b1) & (q != p1);
          if (h0 | h1) {
            const double4 Q = pos[q];
            if (h0) l0 = fmin(l0, dist2_fp64(W0, Q));
            if (h1) l1 = fmin(l1, dist2_fp64(W1, Q));
          }
        }
        l0 = wave_min_f64(l0);
        l1 = wave_min_f64(l1);
        if ((int)lane == w0) md2 = l0;
        else if ((int)lane == w1) md2 = l1;
      }
    }
    if (mine && c1 != 0xFFFFFFFFu) {
      // the smallest in FP64, and with it the others of the lane's list within
      // its reach
      const int64_t pa = again();
      const double4 P = pos[pa];
      const float reach = fmaf(1.0002f, s1, screen_of(aff[cid], 1.0, 0.0).beta);
      double d2 = dist2_fp64(P, pos[c1]);
      md2 = d2 < md2 ? d2 : md2;
      if (s2 <= reach) {
        for (uint32_t k = 0; k < min(cnt, (uint32_t)cap); ++k) {
          const uint32_t q = nbr[tm_slot(p, k, cap)];
          if (dist2_f32(posf[q]) <= reach) {
            d2 = dist2_fp64(P, pos[q]);
            md2 = d2 < md2 ? d2 : md2;
          }
        }
      }
    }
  }
  finish<NW>(again(), live, cnt, qs, md2, pos, ctype_s, young_s, types, n, cap, nbr, count, mindist, qstar, vout,
             flags);
}

template <int BS, int WIN>
void launch_walk(tm_ctx *c) {
  auto kern = c->walk_f32 ? k_neighbors<BS, WIN, true> : k_neighbors<BS, WIN, false>;
  kern<<<tm_blocks(c->n, BS), BS, 0, c->stream>>>(
      c->d_pos, c->d_posf, c->d_code, c->d_ctype_s, c->d_young_s, c->d_wn, c->d_col_off, c->d_aff, c->d_types, c->n,
      c->nbr_alloc, c->d_nbr, c->d_ncount, c->d_mind, c->d_qstar, c->d_v, c->d_flags);
}

// Cells per wave.  A wave costs about as much for 16 cells as 0.5 waves of
// 64, so 64 is best where the waves fill the chip several times over; below,
// the longest wave's time counts, and it falls with its cells.  Walk, us, with
// 8 / 16 / 32 / 64 cells: Gaussian 30 K cells 81 / 90 / 101 / 294, 65 K 138 /
// 116 / 173 / 339, 130 K - / 163 / 175 / 346, 260 K - / 275 / 215 / 343, 600 K
// - / 562 / 398 / 549, 1M - / 910 / 736 / 748; ball 1M - / 591 / 401 / 339.
int cells_per_wave(int64_t n) { return n <= 1 << 15 ? 8 : n <= 1 << 17 ? 16 : n <= 3 << 18 ? 32 : 64; }

// Whether a wave holds so many colonies, which it takes one after another, that
// a lane per cell is faster, its radix tree included.  FP64 steps, together and
// with a lane per cell: 65,536 colonies of 4 cells 632 and 459 us, of 12 789 and
// 611, of 24 939 and 899, of 28 1,016 and 992, of 32 996 and 1,084; 50,000 of 14
// (32 a wave) 671 and 534, 30,000 of 32 522 and 582; 50,000 of 2 (16 a wave) 478 and 361,
// 10,000 of 8 208 and 201, 3,000 of 16 157 and 184; 3,000 of 2 (8 a wave) 156 and 153,
// of 6 158 and 163.
bool many_colonies(int64_t n, int64_t ncol) {
  const int g = cells_per_wave(n);
  return ncol > 1 && n <= (g == 64 ? 28 : g / 2) * ncol;
}

template <int G>
void launch_union(tm_ctx *c) {
  k_union<G><<<tm_blocks(c->n, 64), 4096 / G, 0, c->stream>>>(
      c->d_pos, c->d_posf, c->d_code, c->d_ctype_s, c->d_young_s, c->d_leaf, c->d_bvh, bvh_of(c->n), c->d_col_off,
      c->d_aff, c->d_types, c->n, c->nbr_alloc, c->d_nbr, c->d_ncount, c->d_mind, c->d_qstar, c->d_v, c->d_flags,
      (uint32_t)c->walk_coop_ratio);
}

}  // namespace

// grows the neighbour lists and repeats the walk when a cell overflowed them
tm_status tm_run_neighbors(tm_ctx *c, bool check, bool tiles) {
  if (c->stage < 2) return tm_fail(c, TM_ERR_STATE, "tm_neighbors before tm_build");
  const int64_t n = c->n;
  if (n == 0) {
    c->stage = 3;
    return TM_OK;
  }
  c->tiles_ts = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    const int64_t need = tm_slot_elems(n, c->nbr_cap);
    if (c->nbr_elems < need || !c->d_nbr) {
      tm_free(c, c->d_nbr, true);
      c->d_nbr = nullptr;
      c->nbr_elems = 0;
      if (hipMalloc((void **)&c->d_nbr, sizeof(uint32_t) * (size_t)need) != hipSuccess) {
        c->d_nbr = nullptr;
        return tm_fail(c, TM_ERR_NOMEM, "hipMalloc failed: neighbour lists");
      }
      c->nbr_elems = need;
    }
    c->nbr_alloc = c->nbr_cap;
    const int bs = c->nbr_block;
    const bool coop = c->walk_coop && c->walk_f32 && !many_colonies(n, c->ncol);
    const int g = coop ? cells_per_wave(n) : 0;
    if (!coop) TM_TRY(tm_ensure_tree(c));
    if (g == 8) launch_union<8>(c);
    else if (g == 16) launch_union<16>(c);
    else if (g == 32) launch_union<32>(c);
    else if (g == 64) launch_union<64>(c);
    else if (bs == 64) launch_walk<64, 0>(c);
    else if (bs == 128) launch_walk<128, 0>(c);
    else if (c->walk_window == 2048 && 2 * n - 1 >= 2048) launch_walk<256, 2048>(c);
    else if (c->walk_window == 1280 && 2 * n - 1 >= 1280) launch_walk<256, 1280>(c);
    else if (c->walk_window == 1024 && 2 * n - 1 >= 1024) launch_walk<256, 1024>(c);
    else if (c->walk_window == 512 && 2 * n - 1 >= 512) launch_walk<256, 512>(c);
    else launch_walk<256, 0>(c);
    TM_HIP(c, hipGetLastError());
    // the tiles are made before the host knows that no list overflowed (then
    // both are repeated): one wait for both
    if (tiles) TM_TRY(tm_run_tiles(c, false));
    if (!check) break;
    TM_HIP(c, hipMemcpyAsync(c->h_flags, c->d_flags, 16 * sizeof(unsigned int), hipMemcpyDeviceToHost, c->stream));
    TM_HIP(c, hipStreamSynchronize(c->stream));
    if (c->h_flags[0] & TM_FLAG_DEGENERATE)
      return tm_fail(c, TM_ERR_DEGENERATE,
                     "two cells share location codes down to bit 1, or more than 64 lie within 2^-16 of their colony's "
                     "extent on every axis (duplicate or near-duplicate positions)");
    if (c->h_flags[0] & TM_FLAG_ROOT) return tm_fail(c, TM_ERR_STATE, "colony root not found in the radix tree");
    if (c->h_flags[0] & TM_FLAG_WALK) return tm_fail(c, TM_ERR_STATE, "malformed tree: walk left its node range");
    if (c->h_flags[0] & TM_FLAG_CTYPE) return tm_fail(c, TM_ERR_INVALID, "ctype out of range");
    const int64_t mx = c->h_flags[1];
    if (mx <= c->nbr_alloc) break;
    tm_graph_destroy(c);  // a captured graph has lists of the old length
    c->nbr_cap = (mx + 7) & ~7ll;  // grow to the largest count seen, rounded up
  }
  if (tiles && check) tm_size_tiles(c);
  c->lists_tiles = tm_tiles_serve(c);
  c->direct_sums = 0;
  c->stage = 3;
  return TM_OK;
}
