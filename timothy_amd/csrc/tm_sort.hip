// Device-wide exclusive scan and stable LSD radix sort of (u64 key, i32 value)
// pairs, 8-bit digits, for the Morton ordering of cells.
//
// Each pass: histogram per tile (LDS atomics) -> exclusive scan of the
// digit-major histogram (up to MEDIUM_N keys each tile of the scatter adds up
// histograms itself) -> stable scatter.  Stable ranks inside a tile
// come from 64-lane ballots: the lanes holding the same digit are found with
// eight ballots, the leader of each group advances a per-wave digit counter
// in LDS.
#include <type_traits>

#include "tm_internal.h"

namespace {

constexpr int RS_THREADS = 256;
constexpr int RS_GROUP = 32;  // tiles a group
// how the scatter finds a tile's first slot of a digit: from rows scanned by a
// kernel in between, from the tiles' histograms, from those of its group of
// tiles and the sums of the groups
enum Prefix { SCANNED, FEW, GROUPED };
constexpr int RS_WAVES = RS_THREADS / 64;

constexpr int SC_THREADS = 256;
constexpr int SC_ITEMS = 8;
constexpr int SC_TILE = SC_THREADS * SC_ITEMS;

// lanes of this wave that are valid and hold the same 8-bit digit
__device__ __forceinline__ unsigned long long tm_match8(uint32_t d, bool valid) {
  unsigned long long m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    bool bit = (d >> b) & 1u;
    unsigned long long bb = __ballot(bit);
    m &= bit ? bb : ~bb;
  }
  return m;
}

// zero: a histogram cleared for the pass after this one (or null)
template <int RS_ITEMS, Prefix P, typename K>
__global__ __launch_bounds__(RS_THREADS) void k_rs_hist(const K *__restrict__ keys, int64_t n, int shift,
                                                        uint32_t *__restrict__ hist, int nblocks,
                                                        uint32_t *__restrict__ group, uint32_t *__restrict__ zero) {
  constexpr int RS_TILE = RS_THREADS * RS_ITEMS;
  __shared__ uint32_t h[RS_WAVES][256];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int j = tid; j < RS_WAVES * 256; j += RS_THREADS) (&h[0][0])[j] = 0;
  if (P == FEW) zero[(int64_t)blockIdx.x * 256 + tid] = 0u;
  if (P == GROUPED && blockIdx.x % RS_GROUP == 0) zero[blockIdx.x / RS_GROUP * 256 + tid] = 0u;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * RS_TILE + (int64_t)w * (64 * RS_ITEMS);
  uint32_t dg[RS_ITEMS];  // all of this lane's digits are loaded before any is counted
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it) {
    const int64_t i = base + it * 64 + lane;
    dg[it] = i < n ? (uint32_t)((keys[i] >> shift) & 255u) : 0u;
  }
  // counts only (the ranks are the scatter's), so one LDS atomic per key
  // into this wave's histogram
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it)
    if (base + it * 64 + lane < n) atomicAdd(&h[w][dg[it]], 1u);
  __syncthreads();
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < RS_WAVES; ++k) s += h[k][tid];
  hist[P != SCANNED ? (int64_t)blockIdx.x * 256 + tid : (int64_t)tid * nblocks + blockIdx.x] = s;
  if (P == GROUPED && s) atomicAdd(group + blockIdx.x / RS_GROUP * 256 + tid, s);
}

// Exclusive scan of each digit's row of per-tile counts (one workgroup per
// digit), the row's total stored after the rows: the scatter adds the
// totals of the smaller digits itself.
__global__ __launch_bounds__(RS_THREADS) void k_rs_rowscan(uint32_t *__restrict__ hist, int nblocks) {
  __shared__ uint32_t wsum[RS_WAVES];
  const int d = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  uint32_t *row = hist + (int64_t)d * nblocks;
  const int per = (nblocks + RS_THREADS - 1) / RS_THREADS;
  const int b0 = tid * per, b1 = min(b0 + per, nblocks);
  uint32_t sum = 0;
  for (int b = b0; b < b1; ++b) sum += row[b];
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint32_t run = inc - sum, all = 0;
#pragma unroll
  for (int q = 0; q < RS_WAVES; ++q) {
    if (q < w) run += wsum[q];
    all += wsum[q];
  }
  for (int b = b0; b < b1; ++b) {
    const uint32_t v = row[b];
    row[b] = run;
    run += v;
  }
  if (tid == 0) hist[(int64_t)256 * nblocks + d] = all;
}

// The tile's keys are ranked stably (by digit, then input order), placed in
// LDS in that order, and written out from there: consecutive lanes write
// consecutive slots of one digit's run instead of 64 scattered records.
// next: the following pass's histogram, to which every key is added where it
// arrives (FEW; a pass is then one launch: 30K keys 8.5 against 9.5 us, while at
// 300K the atomics take 20 us and the kernel they replace 7); zero: the one
// after that, cleared.
template <int RS_ITEMS, Prefix P, typename K, typename O>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(const K *__restrict__ keys,
                                                           const int32_t *__restrict__ vals,
                                                           O *__restrict__ okeys, int32_t *__restrict__ ovals,
                                                           int64_t n, int shift, const uint32_t *__restrict__ offs,
                                                           int nblocks, const uint32_t *__restrict__ group,
                                                           uint32_t *__restrict__ next, uint32_t *__restrict__ zero) {
  constexpr int RS_TILE = RS_THREADS * RS_ITEMS;
  __shared__ uint32_t cnt[RS_WAVES][256];
  __shared__ uint32_t pre[RS_WAVES][256];
  __shared__ uint32_t gbase[256];
  __shared__ uint32_t tstart[256];  // first tile-local slot of each digit
  __shared__ uint32_t wsum[RS_WAVES];
  __shared__ K skey[RS_TILE];
  __shared__ int32_t sval[RS_TILE];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int j = tid; j < RS_WAVES * 256; j += RS_THREADS) (&cnt[0][0])[j] = 0;
  if (zero) zero[(int64_t)blockIdx.x * 256 + tid] = 0u;
  const int64_t tile0 = (int64_t)blockIdx.x * RS_TILE;
  const int64_t base = tile0 + (int64_t)w * (64 * RS_ITEMS);
  K k[RS_ITEMS];
  int32_t v[RS_ITEMS];
  uint32_t rank[RS_ITEMS];
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it) {
    const int64_t i = base + it * 64 + lane;
    const bool valid = i < n;
    k[it] = valid ? keys[i] : (K)0;
    v[it] = valid ? vals[i] : 0;
  }
  // this tile's first slot for digit tid: its keys in the tiles before (added
  // up here from the tiles' histograms, FEW, or from those of its group and the
  // sums of the groups before, GROUPED; or scanned by k_rs_rowscan) plus the keys
  // of all smaller digits (the digits' totals, scanned here)
  {
    uint32_t rt = 0, before = 0;
    // adds rows [0, end) to rt, those before `own` also to before
    auto add = [&](const uint32_t *__restrict__ rows, int end, int own) {
      for (int b = 0; b < end; b += 16) {
        uint32_t h[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) h[q] = b + q < end ? rows[(b + q) * 256 + tid] : 0u;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          rt += h[q];
          if (b + q < own) before += h[q];
        }
      }
    };
    if constexpr (P == FEW) {
      add(offs, nblocks, (int)blockIdx.x);
    } else if constexpr (P == GROUPED) {
      const int g = (int)blockIdx.x / RS_GROUP, in = (int)blockIdx.x % RS_GROUP;
      add(offs + (int64_t)g * RS_GROUP * 256, in, in);
      rt = 0;
      add(group, (nblocks + RS_GROUP - 1) / RS_GROUP, g);
    } else {
      rt = offs[(int64_t)256 * nblocks + tid];
      before = offs[(int64_t)tid * nblocks + blockIdx.x];
    }
    uint32_t inc = rt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t wb = 0;
#pragma unroll
    for (int q = 0; q < RS_WAVES; ++q)
      if (q < w) wb += wsum[q];
    gbase[tid] = before + wb + inc - rt;
    __syncthreads();
  }
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it) {
    const bool valid = base + it * 64 + lane < n;
    uint32_t d = (uint32_t)((k[it] >> shift) & 255u);
    unsigned long long peers = tm_match8(d, valid);
    uint32_t before = (uint32_t)__popcll(peers & tm_lanemask_lt());
    uint32_t c0 = valid ? cnt[w][d] : 0u;
    __builtin_amdgcn_wave_barrier();
    if (valid && before == 0) cnt[w][d] = c0 + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
    rank[it] = c0 + before;
  }
  __syncthreads();
  uint32_t total = 0;
  {
    uint32_t run = 0;
#pragma unroll
    for (int q = 0; q < RS_WAVES; ++q) {
      pre[q][tid] = run;
      run += cnt[q][tid];
    }
    total = run;
  }
  // exclusive scan of the digit totals over the 256 threads
  {
    uint32_t inc = total;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t wb = 0;
#pragma unroll
    for (int q = 0; q < RS_WAVES; ++q)
      if (q < w) wb += wsum[q];
    tstart[tid] = wb + inc - total;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it) {
    if (base + it * 64 + lane < n) {
      const uint32_t d = (uint32_t)((k[it] >> shift) & 255u);
      const uint32_t lp = tstart[d] + pre[w][d] + rank[it];  // < the tile's valid count
      skey[lp] = k[it];
      sval[lp] = v[it];
    }
  }
  __syncthreads();
  const int64_t valid_n = min((int64_t)RS_TILE, n - tile0);
  for (int j = tid; j < valid_n; j += RS_THREADS) {
    const K key = skey[j];
    const uint32_t d = (uint32_t)((key >> shift) & 255u);
    const int64_t pos = (int64_t)gbase[d] + (uint32_t)j - tstart[d];
    if (pos >= 0 && pos < n) {  // always true for a consistent histogram; keeps a bad scan from writing out of bounds
      okeys[pos] = (O)(sizeof(O) < sizeof(K) ? (uint64_t)key >> 32 : key);
      ovals[pos] = sval[j];
      if (P == FEW && next) {
        const uint32_t t1 = (uint32_t)pos / RS_TILE, d1 = (uint32_t)((key >> (shift + 8)) & 255u);
        atomicAdd(next + (int64_t)t1 * 256 + d1, 1u);
      }
    }
  }
}

// All passes of up to OT RS_ITEMS keys in one workgroup: the keys stay in
// registers and change places through LDS.  Missing keys are all ones, after
// the others in every pass.  Latency: one launch instead of seven; a build of 1K
// cells 48 -> 32 us, of 2K 52 -> 33, of 4K 55 -> 44 (8K, eight keys a thread, 58
// -> 63: not taken).
constexpr int OT = 1024, OW = OT / 64;
template <int RS_ITEMS>
__global__ __launch_bounds__(OT) void k_rs_one(const uint64_t *__restrict__ keys, int32_t *__restrict__ vals, int n,
                                               int lo_bit) {
  __shared__ uint32_t cnt[OW][256];
  __shared__ uint32_t tstart[256];
  __shared__ uint32_t wsum[4];
  __shared__ uint64_t skey[OT * RS_ITEMS];
  __shared__ uint16_t sval[OT * RS_ITEMS];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int base = w * (64 * RS_ITEMS) + lane;
  uint64_t k[RS_ITEMS];
  uint32_t v[RS_ITEMS], rank[RS_ITEMS];
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it) {
    const int i = base + it * 64;
    k[it] = i < n ? keys[i] : ~0ull;
    v[it] = i < n ? (uint32_t)vals[i] : 0u;
  }
  for (int shift = lo_bit; shift < 64; shift += 8) {
    for (int j = tid; j < OW * 256; j += OT) (&cnt[0][0])[j] = 0;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < RS_ITEMS; ++it) {
      const uint32_t d = (uint32_t)(k[it] >> shift) & 255u;
      const unsigned long long peers = tm_match8(d, true);
      const uint32_t before = (uint32_t)__popcll(peers & tm_lanemask_lt());
      const uint32_t c0 = cnt[w][d];
      __builtin_amdgcn_wave_barrier();
      if (before == 0) cnt[w][d] = c0 + (uint32_t)__popcll(peers);
      __builtin_amdgcn_wave_barrier();
      rank[it] = c0 + before;
    }
    __syncthreads();
    uint32_t total = 0, inc = 0;
    if (tid < 256) {
      uint32_t c[OW];
#pragma unroll
      for (int q = 0; q < OW; ++q) c[q] = cnt[q][tid];
#pragma unroll
      for (int q = 0; q < OW; ++q) {
        cnt[q][tid] = total;
        total += c[q];
      }
      inc = total;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
      }
      if (lane == 63) wsum[w] = inc;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t wb = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < w) wb += wsum[q];
      tstart[tid] = wb + inc - total;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < RS_ITEMS; ++it) {
      const uint32_t d = (uint32_t)(k[it] >> shift) & 255u;
      const uint32_t lp = tstart[d] + cnt[w][d] + rank[it];
      skey[lp] = k[it];
      sval[lp] = (uint16_t)v[it];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < RS_ITEMS; ++it) {
      k[it] = skey[base + it * 64];
      v[it] = sval[base + it * 64];
    }
  }
#pragma unroll
  for (int it = 0; it < RS_ITEMS; ++it)
    if (base + it * 64 < n) vals[base + it * 64] = (int32_t)v[it];
}

// ---- scan ----------------------------------------------------------------

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const int lane = __lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  return x;
}

// exclusive block scan of one value per thread; returns the block total in *tot
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t *tot) {
  __shared__ uint32_t ws[SC_THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t inc = wave_incl_scan(x);
  if (lane == 63) ws[w] = inc;
  __syncthreads();
  uint32_t wbase = 0, all = 0;
#pragma unroll
  for (int k = 0; k < SC_THREADS / 64; ++k) {
    uint32_t s = ws[k];
    if (k < w) wbase += s;
    all += s;
  }
  __syncthreads();
  *tot = all;
  return wbase + inc - x;
}

__global__ __launch_bounds__(SC_THREADS) void k_scan_reduce(const uint32_t *__restrict__ in, int64_t n,
                                                            uint32_t *__restrict__ sums) {
  const int64_t base = (int64_t)blockIdx.x * SC_TILE + (int64_t)threadIdx.x * SC_ITEMS;
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < SC_ITEMS; ++k)
    if (base + k < n) s += in[base + k];
  uint32_t tot;
  (void)block_excl_scan(s, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(SC_THREADS) void k_scan_apply(const uint32_t *__restrict__ in, int64_t n,
                                                           const uint32_t *__restrict__ sums_scanned,
                                                           uint32_t *__restrict__ out) {
  const int64_t base = (int64_t)blockIdx.x * SC_TILE + (int64_t)threadIdx.x * SC_ITEMS;
  uint32_t v[SC_ITEMS];
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < SC_ITEMS; ++k) {
    v[k] = (base + k < n) ? in[base + k] : 0u;
    s += v[k];
  }
  uint32_t tot;
  uint32_t run = block_excl_scan(s, &tot) + (sums_scanned ? sums_scanned[blockIdx.x] : 0u);
#pragma unroll
  for (int k = 0; k < SC_ITEMS; ++k) {
    if (base + k < n) out[base + k] = run;
    run += v[k];
  }
}

}  // namespace

// exclusive scan; `out` may alias `in`.  Uses c->d_scan as scratch.
tm_status tm_scan_u32(tm_ctx *c, const uint32_t *in, uint32_t *out, int64_t n) {
  if (n <= 0) return TM_OK;
  int64_t nb = (n + SC_TILE - 1) / SC_TILE;
  if (nb == 1) {
    k_scan_apply<<<1, SC_THREADS, 0, c->stream>>>(in, n, nullptr, out);
    TM_HIP(c, hipGetLastError());
    return TM_OK;
  }
  // scratch layout: level sums for up to three levels
  int64_t nb2 = (nb + SC_TILE - 1) / SC_TILE;
  int64_t need = nb + nb2 + 1;
  TM_TRY(tm_ensure(c, &c->d_scan, c->cap_scan, need, "scan scratch", c->graph_tree));
  uint32_t *sums = c->d_scan;
  uint32_t *sums2 = c->d_scan + nb;
  k_scan_reduce<<<(unsigned)nb, SC_THREADS, 0, c->stream>>>(in, n, sums);
  TM_HIP(c, hipGetLastError());
  if (nb2 == 1) {
    k_scan_apply<<<1, SC_THREADS, 0, c->stream>>>(sums, nb, nullptr, sums);
  } else {
    if (nb2 > SC_TILE) return tm_fail(c, TM_ERR_INVALID, "scan too large");
    k_scan_reduce<<<(unsigned)nb2, SC_THREADS, 0, c->stream>>>(sums, nb, sums2);
    k_scan_apply<<<1, SC_THREADS, 0, c->stream>>>(sums2, nb2, nullptr, sums2);
    k_scan_apply<<<(unsigned)nb2, SC_THREADS, 0, c->stream>>>(sums, nb, sums2, sums);
  }
  TM_HIP(c, hipGetLastError());
  k_scan_apply<<<(unsigned)nb, SC_THREADS, 0, c->stream>>>(in, n, sums, out);
  TM_HIP(c, hipGetLastError());
  return TM_OK;
}

// Keys a tile, by the number of keys.  A tile's items are ranked one after the
// other, so that few keys, whose passes are latency, take small tiles on more
// CUs; many keys take large ones, whose runs of a digit are written in longer
// pieces, and fewer of them to scan.  Times of a build, 4096 / 2048 / 1024 keys a
// tile, rows scanned: 300K cells 174 / 138 / 129 us, 800K 222 / 195 / 197, 1.2M
// 274 / 245 / 258, 2M 364 / 357 / 407, 6M 914 / 953 / 1115.
// The prefix of a tile: scanned / from all tiles' histograms / from its group's
// and the groups' sums: 4K cells 79 / 65 / 68 us, 30K 85 / 76 / 77, 65K 90 / 91 /
// 81 (82 with one launch a pass, which the second allows), 300K 125 / - / 114, 2M
// 331 / - / 313; 4096 keys a tile: 6M 838 / - / 853, 33M 4.80 / - / 5.69 ms.
constexpr int64_t FEW_N = 1 << 16, SMALL_N = 3 << 18, MEDIUM_N = 1 << 22;

static int64_t group_words(int64_t nblocks) { return (nblocks + RS_GROUP - 1) / RS_GROUP * 256; }

template <int ITEMS, Prefix P>
static tm_status sort_passes(tm_ctx *c, uint64_t *keys, int32_t *vals, int64_t n, int lo_bit) {
  const int64_t tile = RS_THREADS * ITEMS;
  const int nblocks = (int)((n + tile - 1) / tile);
  const int64_t row = (int64_t)256 * nblocks + 256;
  // this pass's histogram, and with FEW the next one's and the one to be
  // cleared; with GROUPED the groups' sums and the next pass's
  uint32_t *h0 = c->d_hist, *h1 = P == FEW ? h0 + row : nullptr, *h2 = P == FEW ? h1 + row : nullptr;
  uint32_t *g0 = P == GROUPED ? h0 + row : nullptr, *g1 = P == GROUPED ? g0 + group_words(nblocks) : nullptr;
  uint64_t *k0 = keys, *k1 = c->d_key_alt;
  int32_t *v0 = vals, *v1 = c->d_val_alt;
  for (int shift = lo_bit; shift < 64; shift += 8) {
    const bool count = P != FEW || shift == lo_bit, more = P == FEW && shift + 8 < 64;
    auto pass = [&](auto *in, auto *out, int at) {
      using K = std::remove_reference_t<decltype(*in)>;
      using O = std::remove_reference_t<decltype(*out)>;
      if (count)
        k_rs_hist<ITEMS, P, K>
            <<<nblocks, RS_THREADS, 0, c->stream>>>(in, n, at, h0, nblocks, g0, P == FEW ? h1 : g1);
      if (P == SCANNED) k_rs_rowscan<<<256, RS_THREADS, 0, c->stream>>>(h0, nblocks);
      k_rs_scatter<ITEMS, P, K, O><<<nblocks, RS_THREADS, 0, c->stream>>>(
          in, v0, out, v1, n, at, h0, nblocks, g0, more ? h1 : nullptr, more ? h2 : nullptr);
    };
    if (shift >= 32) pass((uint32_t *)k0, (uint32_t *)k1, shift - 32);
    else if (shift + 8 >= 32) pass(k0, (uint32_t *)k1, shift);
    else pass(k0, k1, shift);
    std::swap(h0, P == FEW ? h1 : h0);
    std::swap(h1, h2);
    std::swap(g0, g1);
    TM_HIP(c, hipGetLastError());
    std::swap(k0, k1);
    std::swap(v0, v1);
  }
  return TM_OK;
}

// Sizes the sort's workspace for n keys; the *words first words at the address
// returned must be zero when the sort starts.
tm_status tm_sort_prepare(tm_ctx *c, int64_t n, uint32_t **clear, int64_t *words) {
  const int64_t tile = RS_THREADS * (n <= SMALL_N ? 4 : n <= MEDIUM_N ? 8 : 16), nblocks = (n + tile - 1) / tile;
  const int64_t row = 256 * nblocks + 256, gw = n > FEW_N && n <= MEDIUM_N ? group_words(nblocks) : 0;
  TM_TRY(tm_ensure(c, &c->d_hist, c->cap_hist, n <= FEW_N ? 3 * row : row + 2 * gw, "radix histogram", true));
  *clear = c->d_hist + row;
  *words = gw;
  return TM_OK;
}

// Stable sort of (keys, vals) by key bits [lo_bit, 64) (lo_bit a multiple
// of 16, so the passes are even in number); the passes ping-pong through
// c->d_key_alt / d_val_alt.  vals, which starts as 0, 1, ..., n - 1, ends sorted;
// the keys' own order at the end is left open: once a pass has used the last bit
// below 32 it hands on the keys' upper halves only (16 instead of 24 bytes a key
// and pass, and less LDS; a build of 2M cells 312 -> 304 us, of 33M 4.33 -> 4.15
// ms).
tm_status tm_sort_pairs(tm_ctx *c, uint64_t *keys, int32_t *vals, int64_t n, int lo_bit) {
  if (n <= 1) return TM_OK;
  if (lo_bit < 0 || lo_bit >= 32 || lo_bit % 16) return tm_fail(c, TM_ERR_INVALID, "sort: lo_bit");
  if (n <= 4 * OT) {
    auto one = n <= 2 * OT ? k_rs_one<2> : k_rs_one<4>;
    one<<<1, OT, 0, c->stream>>>(keys, vals, (int)n, lo_bit);
    TM_HIP(c, hipGetLastError());
    return TM_OK;
  }
  if (n <= FEW_N) return sort_passes<4, FEW>(c, keys, vals, n, lo_bit);
  if (n <= SMALL_N) return sort_passes<4, GROUPED>(c, keys, vals, n, lo_bit);
  if (n <= MEDIUM_N) return sort_passes<8, GROUPED>(c, keys, vals, n, lo_bit);
  return sort_passes<16, SCANNED>(c, keys, vals, n, lo_bit);
}
