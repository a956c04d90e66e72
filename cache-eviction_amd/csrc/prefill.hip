// Chunked-prefill score tiles on MFMA (gfx950): exact probabilities with the
// sink in the normaliser, reduced per KV head over its query heads (sum or
// max) and over the chunk's queries, added to each key's slot score.
//
// Pass 1 (prefill_norm_kernel, prefill_merge_kernel) streams the visible keys past each query
// block once to get every (query, head) row's log-sum-exp, with the sink; pass 2
// (prefill_score_kernel) streams the queries past each key block, turns logits into probabilities
// with that normaliser and accumulates each key's sum (with a score delay d, only over the queries
// at least d entries after it). MFMA rows or columns are (query, head) pairs, the KV head's 8 query
// heads each, so none is padding: a 16-wide block holds two queries.
//
// Work per (query head, key) is one exp2 per pass, which bounds the kernels: v_exp_f32 takes 8.6
// cycles per wave instruction, FMA and add 2 to 4, and the card's power limit lowers the clock
// (1.9 GHz) over a launch of milliseconds.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "host.hpp"

namespace gse {

namespace pf {
constexpr int D = 64;
constexpr int GROUP = 8;
constexpr int QB = 64;          // queries per workgroup
constexpr int KT = 64;          // keys per tile (4 key-blocks of 16)
constexpr int KROW = D + 8;     // padded bf16 row of a staged key
// A row's reference follows its sums: past kMoveSum it moves up by a power of two (exponents near
// zero keep the exponential's argument exact), past kRescaleSum, near the overflow, to the tile's
// maximum.
constexpr float kMoveSum = 64.f;
constexpr float kRescaleSum = 0x1p64f;
}  // namespace pf

struct PrefillArgs {
  const uint16_t* q;
  int64_t q_st, q_sh;
  int64_t count;
  const uint16_t* k;
  int64_t kv_ss, kv_sh;
  const void* slots;
  int slots_dtype;
  int64_t total, prefix_len;
  const void* sinks;
  int sinks_dtype;
  int mode;
  float* scores;
  int64_t ssg, sss;
  int q_heads, kv_heads;
  float scale2;
  float* norm2;  // [count, q_heads] row normalisers in log2 units (sink included)
  int delay;     // pass 2 credits query i's keys k <= prefix_len + i - delay only
  int block_shift;  // kind 4: log2 of the block size
  // Pass 1's key ranges: at most `splits`, of at most `tiles` 64-key tiles; part[(range * count + query) *
  // q_heads + head] = (reference, sum of 2^(x - reference)) of the row over that range.
  float2* part;
  int splits, tiles;
  int qblock;  // pass 2: queries per workgroup
};

// ---------------------------------------------------------------------------
// Pass 1: row normalisers
// ---------------------------------------------------------------------------
// S^T = K . Q^T in 16x16x32 MFMAs: a lane holds 4 keys per key block of one (query, head) row, so a
// row needs one reference and one sum per lane, and its terms add up in the lane. A workgroup (8
// waves x 8 queries) takes one KV head, 64 queries and a range of at most `tiles` 64-key tiles of
// what they see; prefill_merge_kernel joins the ranges' (reference, sum) pairs and the sink.
// Bound by vector issue (one FMA, one exponential and one add per logit: 305 cycles per 1024
// logits and SIMD with their MFMAs) and, over a launch of milliseconds, by the card's power: that
// mix alone runs at 2.2 GHz, 139 ns per 1024 logits; 32x32x16 MFMAs take fewer issue slots but
// more power (156 ns), and the FMA with a vector instead of a scalar scale 147 ns. Against rows
// spread over 16 lanes (a running maximum per row and lane) with 2 waves per SIMD and whole causal
// ranges, means of 20 traced calls in a row, the join of the ranges included: 82 -> 51 us for the first
// 2048 tokens of a prompt, 738 -> 652 us for 1896 tokens after 30,720, 2.91 -> 2.54 ms for 8192 after
// 28,672. Single calls between waits run at another clock (790 us for the second), and another card's
// power limit made the passes 6 % slower.
namespace p1 {
constexpr int QW = 8;                // queries per wave: two column blocks of 4 queries x 8 heads
constexpr int WAVES = 8;
constexpr int THREADS = 64 * WAVES;
static_assert(QW * WAVES == pf::QB, "a workgroup's queries");
// Work items of a launch: about three rounds of the SLOTS workgroups that 256 CUs hold (2 each). Where
// these have FEW_TILES tiles or less each to do, whole rounds count: then the item length (at least
// MIN_TILES tiles) whose rounds take least, with the start of an item (its query and first key loads,
// some 4 us) counted as START tiles. Both passes of sums, without the rule -> with it, us: 2047 tokens
// without a prefix 87.2 -> 86.1, 1000 after 1000 67.8 -> 63.3, 400 after 4096 70.4 -> 64.9, 400 after 9000
// 120 -> 111; 1000 without a prefix 45.0 -> 44.9. Past that the rounds' count no longer decides (8192
// after 28,672: 5.45 ms, 5.8 with the fewest rounds).
constexpr int SLOTS = 512;
constexpr int ITEMS = 3 * SLOTS;
constexpr int FEW_TILES = 16;
constexpr int MIN_TILES = 4;
constexpr double START = 2.3;
}  // namespace p1

// Key ranges of a query block that sees ntiles tiles (equal ones, of at most `tiles` tiles).
GSE_DEVICE int key_ranges(int ntiles, int tiles) { return (ntiles + tiles - 1) / tiles; }

// Row block rb's fragments of a staged tile of 16-row blocks: lane (col, grp) holds dims [8*grp, +8)
// and [32 + 8*grp, +8) of row 16*rb + col.
GSE_DEVICE void fragments(const uint16_t* tile, int rb, int lane, bf16x8_t (&f)[2]) {
  const uint16_t* r = tile + (16 * rb + (lane & 15)) * pf::KROW + 8 * (lane >> 4);
  f[0] = as_bf16x8(*reinterpret_cast<const uint4*>(r));
  f[1] = as_bf16x8(*reinterpret_cast<const uint4*>(r + 32));
}

GSE_DEVICE f32x4_t dot64(const bf16x8_t (&a)[2], const bf16x8_t (&b)[2]) {
  return mfma16x16x32(a[1], b[1], mfma16x16x32(a[0], b[0], f32x4_t{0.f, 0.f, 0.f, 0.f}));
}

// Logits of keys past a lane's causal bound become -inf: register r of a block holds key first + r,
// dead when past `bound` (both relative to the same origin).
GSE_DEVICE void mask_keys(f32x4_t& d, int first, int bound) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (first + r > bound) d[r] = -INFINITY;
}

GSE_DEVICE float sum4(const f32x4_t& p) { return (p[0] + p[1]) + (p[2] + p[3]); }

// One tile of a wave: ts[rb] = the lane's sum of 2^(x * scale2 + nref[rb]) over its 16 keys, nref
// the negated reference, a whole number. When a sum passes kMoveSum, its row's reference takes the
// sum's exponent and both sums are scaled by that power of two (exact); when one passes kRescaleSum
// (rows whose first keys were all masked, or logits over 40 above them) the references of the
// wave's rows move to their tile maximum and the tile is formed again.
// MASKED: key 16*kb + r of the tile is dead past bound + 2*rb.
template <bool MASKED>
GSE_DEVICE void row_sum_tile(const uint16_t* kt, const bf16x8_t (&qf)[4][2], float (&nref)[4], float (&sum)[4],
                             float scale2, int bound, int lane) {
  using namespace pf;
  float ts[4];
  {
    // Units of two key blocks against one column block (2 queries); the next unit's MFMAs are
    // issued ahead of this one's vector work.
    bf16x8_t ka[2][2];
    f32x4_t dn[2];
    fragments(kt, 0, lane, ka[0]);
    fragments(kt, 1, lane, ka[1]);
    dn[0] = dot64(ka[0], qf[0]);
    dn[1] = dot64(ka[1], qf[0]);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int kp = u >> 2, rb = u & 3;
      f32x4_t d[2] = {dn[0], dn[1]};
      if (u == 3) {
        fragments(kt, 2, lane, ka[0]);
        fragments(kt, 3, lane, ka[1]);
      }
      if (u < 7) {
        dn[0] = dot64(ka[0], qf[(u + 1) & 3]);
        dn[1] = dot64(ka[1], qf[(u + 1) & 3]);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (MASKED) mask_keys(d[h], 32 * kp + 16 * h, bound + 2 * rb);
#pragma unroll
        for (int r = 0; r < 4; ++r) d[h][r] = fast_exp2(fmaf(d[h][r], scale2, nref[rb]));
      }
      const float t = sum4(d[0]) + sum4(d[1]);
      ts[rb] = kp == 0 ? t : ts[rb] + t;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  const float tsmax = fmaxf(fmaxf(ts[0], ts[1]), fmaxf(ts[2], ts[3]));
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(tsmax > kMoveSum) == 0, 1)) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) sum[rb] += ts[rb];
    return;
  }
  if (__builtin_amdgcn_ballot_w64(tsmax > kRescaleSum)) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      float tmax = -INFINITY;
#pragma unroll 1
      for (int kb = 0; kb < 4; ++kb) {
        bf16x8_t ka[2];
        fragments(kt, kb, lane, ka);
        f32x4_t d = dot64(ka, qf[rb]);
        if (MASKED) mask_keys(d, 16 * kb, bound + 2 * rb);
        tmax = fmaxf(fmaxf(tmax, fmaxf(d[0], d[1])), fmaxf(d[2], d[3]));
      }
      const float nr = fminf(nref[rb], -rintf(tmax * scale2));
      float t = 0.f;
#pragma unroll 1
      for (int kb = 0; kb < 4; ++kb) {
        bf16x8_t ka[2];
        fragments(kt, kb, lane, ka);
        f32x4_t d = dot64(ka, qf[rb]);
        if (MASKED) mask_keys(d, 16 * kb, bound + 2 * rb);
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = fast_exp2(fmaf(d[r], scale2, nr));
        t += sum4(d);
      }
      sum[rb] *= fast_exp2(nr - nref[rb]);
      nref[rb] = nr;
      ts[rb] = t;
    }
  }
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int e = ts[rb] > kMoveSum && ts[rb] <= kRescaleSum ? __builtin_amdgcn_frexp_expf(ts[rb]) : 0;
    nref[rb] -= float(e);
    sum[rb] = ldexpf(sum[rb] + ts[rb], -e);
  }
}

// Staging of a walk over 64-key tiles by 512 threads: thread t brings 16 bytes of key t/8. Tile t's
// K rows are loaded into registers during tile t - 2 and stored to LDS at the end of tile t - 1,
// and its slot indices are read two tiles before that, in two register sets alternating by tile
// parity (the walks are unrolled by two: copying one into the other would wait for the loads in
// flight into it). Keys past kend read slot 0's row (any valid row) and are masked.
struct KeyTiles {
  typedef uint16_t Tile[pf::KT * pf::KROW];
  const PrefillArgs& a;
  const int kend, lk, lp;
  const global_ptr<const uint16_t> base;
  uint4 row[2];     // row[p]: K rows of the tile of offset parity p in flight
  int32_t slot[2];  // slot[p]: slot of the next tile of parity p whose rows are not yet loaded

  GSE_DEVICE KeyTiles(const PrefillArgs& a_, int g, int kend_)
      : a(a_), kend(kend_), lk(threadIdx.x >> 3), lp(threadIdx.x & 7),
        base(as_global(a_.k) + int64_t(g) * a_.kv_sh + 8 * (threadIdx.x & 7)) {}
  GSE_DEVICE int32_t slot_at(int ti) const {
    const uint32_t key = uint32_t(ti) * pf::KT + lk;  // up to four tiles past kend < 2^31
    return key < uint32_t(kend) ? int32_t(load_index_dyn(a.slots, a.slots_dtype, key)) : 0;
  }
  GSE_DEVICE uint4 load(int32_t s) const { return gload16(base + int64_t(s) * a.kv_ss); }
  GSE_DEVICE void store(Tile& tile, const uint4& x) const { *reinterpret_cast<uint4*>(&tile[lk * pf::KROW + 8 * lp]) = x; }
  // Tile ti0 to LDS, the next ones on their way.
  GSE_DEVICE void start(int ti0, Tile (&tiles)[2]) {
    const int32_t s0 = slot_at(ti0), s1 = slot_at(ti0 + 1);
    slot[0] = slot_at(ti0 + 2);
    slot[1] = slot_at(ti0 + 3);
    const uint4 y = load(s0);
    row[1] = load(s1);
    store(tiles[0], y);
  }
  // At the start of tile ti, of parity p: tile ti + 2's rows and tile ti + 4's slots go out.
  GSE_DEVICE void ahead(int ti, int p) {
    row[p] = load(slot[p]);
    slot[p] = slot_at(ti + 4);
  }
  GSE_DEVICE void stage(int p, Tile (&tiles)[2]) { store(tiles[p], row[p]); }
};

// m + log2(l), rounded once: the exponent of l joins m without loss and only the mantissa's logarithm,
// in [-1, 0), is inexact (log2(l) itself, 6 to 16 for the sums here, is rounded to 2^-21 or 2^-20).
GSE_DEVICE float add_log2(float m, float l) {
  const float e = float(__builtin_amdgcn_frexp_expf(l));
  const float s = m + e, t = s - m;
  const float lost = (m - (s - t)) + (e - t);
  return s + (__log2f(__builtin_amdgcn_frexp_mantf(l)) + lost);
}

// A row's normaliser (log2 units) from its one pair and the sink.
GSE_DEVICE float row_norm(const PrefillArgs& a, int h, float ref, float sum) {
  const float sink2 = load_float_dyn(a.sinks, a.sinks_dtype, h) * kLog2e;
  const float m = fmaxf(ref, sink2);
  return add_log2(m, sum * fast_exp2(ref - m) + fast_exp2(sink2 - m));
}

__global__ __launch_bounds__(p1::THREADS, 4) void prefill_norm_kernel(PrefillArgs a) {
  using namespace pf;
  using p1::QW;
  __shared__ __attribute__((aligned(16))) KeyTiles::Tile ktile[2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block i: KV head i % kv_heads, then the query block from the end (the longest causal ranges
  // first), then the key range. Blocks go to an XCD's shader engines in turn, whatever these have
  // left to do, so ranges of different lengths must not alternate with the block index.
  const int nqb = int((a.count + QB - 1) / QB);
  const int g = blockIdx.x % a.kv_heads;
  const int item = blockIdx.x / a.kv_heads;
  const int split = item / nqb;
  const int64_t qb0 = int64_t(nqb - 1 - item % nqb) * QB;
  const int last_q = int((qb0 + QB < a.count ? qb0 + QB : a.count) - 1);
  const int kend = int(a.prefix_len) + last_q + 1;  // keys any query of the workgroup sees
  const int ntiles = (kend + KT - 1) / KT;
  const int ranges = key_ranges(ntiles, a.tiles);
  if (split >= ranges) return;
  const int ti0 = int(int64_t(ntiles) * split / ranges), ti1 = int(int64_t(ntiles) * (split + 1) / ranges);
  const int i0 = int(qb0) + QW * wave;  // this wave's first query
  const bool wave_live = i0 < a.count;
  const int wave_kend = int(a.prefix_len) + min(i0 + QW - 1, int(a.count) - 1) + 1;

  // B fragments: column col = lane%16 of block rb is query i0 + 2*rb + col/8, head g*8 + col%8.
  bf16x8_t qf[4][2];
  float nref[4], sum[4];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int64_t qi = i0 + 2 * rb + ((lane & 15) >> 3);
    const uint16_t* qp = a.q + qi * a.q_st + int64_t(g * GROUP + (lane & 7)) * a.q_sh + 8 * (lane >> 4);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      qf[rb][h] = qi < a.count ? as_bf16x8(*reinterpret_cast<const uint4*>(qp + 32 * h)) : bf16x8_t{};
    nref[rb] = 1e30f;  // finite, so fully masked rows give 2^(-inf) = 0, never NaN
    sum[rb] = 0.f;
  }
  const float scale2 = a.scale2;

  KeyTiles keys(a, g, kend);
  keys.start(ti0, ktile);
  // The query fragments are in registers before the walk starts: a wait for them inside the
  // loop would also wait for every load in flight at the top of each tile.
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    landed(qf[rb][0]);
    landed(qf[rb][1]);
  }
  __syncthreads();

  // The causal bound of the lane's row of block 0, from the lane's first key (4*grp) on.
  const int qpos = int(a.prefix_len) + i0 + ((lane & 15) >> 3) - 4 * (lane >> 4);
  {  // Each row's reference: the maximum over the range's first 32 keys.
    bf16x8_t ka[2][2];
    fragments(ktile[0], 0, lane, ka[0]);
    fragments(ktile[0], 1, lane, ka[1]);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      float m = -INFINITY;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4_t d = dot64(ka[h], qf[rb]);
        mask_keys(d, 16 * h, qpos + 2 * rb - ti0 * KT);
        m = fmaxf(m, fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3])));
      }
      m = xor32_max(xor16_max(m));
      nref[rb] = fminf(nref[rb], -rintf(m * scale2));
    }
  }

  // The tiles every wave sees whole (below the workgroup's first query) run in a loop of their
  // own with no causal mask (a wave past the chunk's end computes rows nobody reads, with zero
  // queries); the rest choose per wave.
  auto tile_step = [&](int ti, auto general, auto parity) {
    constexpr bool GENERAL = decltype(general)::value;
    constexpr int P = decltype(parity)::value;  // (ti - ti0) & 1
    keys.ahead(ti, P);
    const int t0 = ti * KT;
    if (!GENERAL)
      row_sum_tile<false>(ktile[P], qf, nref, sum, scale2, 0, lane);
    else if (wave_live && t0 < wave_kend)
      row_sum_tile<true>(ktile[P], qf, nref, sum, scale2, qpos - t0, lane);
    if (ti + 1 < ti1) keys.stage(1 - P, ktile);
    __syncthreads();
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  const int whole = int((a.prefix_len + qb0 + 1) / KT);  // tiles whose keys the first query sees
  const int common = ti0 + (max(min(ti1, whole) - ti0, 0) & ~1);
  int ti = ti0;
#pragma unroll 1
  for (; ti < common; ti += 2) {
    tile_step(ti, std::false_type{}, P0{});
    tile_step(ti + 1, std::false_type{}, P1{});
  }
#pragma unroll 1
  for (; ti < ti1; ti += 2) {
    tile_step(ti, std::true_type{}, P0{});
    if (ti + 1 < ti1) tile_step(ti + 1, std::true_type{}, P1{});
  }

  // The row's pair over the four lane groups.
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const float nr = -xor32_max(xor16_max(-nref[rb]));
    const float total = xor32_sum(xor16_sum(sum[rb] * fast_exp2(nr - nref[rb])));
    const int64_t qi = i0 + 2 * rb + ((lane & 15) >> 3);
    if (lane < 16 && qi < a.count) {
      const int h = g * GROUP + (lane & 7);
      if (a.splits == 1)
        a.norm2[qi * a.q_heads + h] = row_norm(a, h, -nr, total);
      else
        a.part[(split * a.count + qi) * a.q_heads + h] = float2{-nr, total};
    }
  }
}

// Row normalisers in log2 units of several ranges: thread = (query, head), joining the key ranges that hold keys of
// the row's query block and the sink.
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t n = a.count * a.q_heads;
  if (t >= n) return;
  const int64_t qb0 = t / a.q_heads / pf::QB * pf::QB;
  const int64_t kend = a.prefix_len + (qb0 + pf::QB < a.count ? qb0 + pf::QB : a.count);
  const int ranges = key_ranges(int((kend + pf::KT - 1) / pf::KT), a.tiles);
  float m = load_float_dyn(a.sinks, a.sinks_dtype, t % a.q_heads) * kLog2e, l = 1.f;
  for (int s0 = 0; s0 < ranges; s0 += 8) {  // eight ranges' loads in flight together
    float2 p[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = a.part[int64_t(min(s0 + j, ranges - 1)) * n + t];
    float mn = m;
#pragma unroll
    for (int j = 0; j < 8; ++j) mn = fmaxf(mn, p[j].x);
    l *= fast_exp2(m - mn);
#pragma unroll
    for (int j = 0; j < 8; ++j) l += s0 + j < ranges ? p[j].y * fast_exp2(p[j].x - mn) : 0.f;
    m = mn;
  }
  a.norm2[t] = add_log2(m, l);
}

// ---------------------------------------------------------------------------
// Pass 2: column sums
// ---------------------------------------------------------------------------
// A workgroup owns one KV head, 256 keys (4 waves x 64, their K fragments in registers) and
// a.qblock queries, which stream through LDS 8 at a time: a key's sum stays in a register over the
// whole walk and reaches the score table with one atomic per (key, query block), and no key index
// is read inside it. Sum mode forms S^T = K . Q^T (a lane holds 16 keys of one row: one normaliser,
// a sum per key), max mode S = Q . K^T (a lane holds 4 heads of a query for one key: the maximum
// over over the heads is in the lane and its neighbouring group). 4 waves per SIMD. Bound as pass 1;
// max mode takes one exponential per (query, key). Against query blocks of 64 walking the keys (column
// sums through LDS rings, two waves per SIMD), traced as pass 1: sums 74 -> 44 us for the first 2048
// tokens of a prompt, 3.01 -> 2.65 ms for 8192 after 28,672; maxima 1053 -> 494 us for 1896 after 30,720.
namespace p2 {
constexpr int KW = 64;  // keys per wave: two 32-key blocks
constexpr int WAVES = 4;
constexpr int KB = KW * WAVES;
constexpr int THREADS = 64 * WAVES;
constexpr int QT = 8;  // queries per tile (64 rows)
// Query blocks: about ITEMS workgroups, of at least 64 queries and at most MAX_QUERIES: a sum takes at
// most MAX_QUERIES / 4 additions in one register, so its rounding error stays near that of a sum over
// 64-query blocks. Two exceptions, by the workgroups that have keys to credit:
// - Fewer than FEW (7 for 4 CUs): a workgroup has its CU nearly to itself and its walk is the launch, so
//   the blocks shrink (to MIN_QUERIES, by a quarter at least) as long as there are no more than FEW. Both
//   passes, sums / maxima, us: 60 tokens without a prefix 24.0 -> 17.9 / 20.2 -> 15.8, 850 without one
//   38.3 -> 34.1 / 33.7 -> 31.8, 190 after 1000 32.8 -> 28.4 / 30.1 -> 27.9. With more of them shorter
//   walks no longer pay for their starts and atomics: 1000 without a prefix, 640 workgroups instead of
//   320, 44.6 -> 45.3 / 40.4 -> 45.4.
// - Blocks of 64 in up to 13/8 rounds of the SLOTS workgroups that run at once: longer ones in one round,
//   if they fill it (7/8): 2047 without a prefix 92.6 -> 86.4, 1000 after 2500 100.5 -> 95.9 / 90.7 -> 86.4;
//   not 300 after 9000 (872 workgroups) 85.2 -> 91.5. Maxima only from 5/4 rounds on: at 1152 workgroups
//   79.0 -> 80.1, at 1048 69.2 -> 70.5.
constexpr int SLOTS = 1024;  // 4 workgroups on each of 256 CUs
constexpr int ITEMS = 2 * SLOTS;
constexpr int FEW = 448;
constexpr int ROUND = SLOTS * 13 / 8;
constexpr int MIN_QUERIES = 32;
constexpr int MAX_QUERIES = 512;
}  // namespace p2

// A staged query tile against the wave's keys, sums: cs[kb][r] += the probabilities of key
// 16*kb + 4*(lane/16) + r in rows lane%16 of the column blocks (2 queries each). MASKED: key
// 16*kb + r is dead past bound + 2*cb.
template <bool MASKED>
GSE_DEVICE void column_sum_tile(const uint16_t* qt, const float* nt, const bf16x8_t (&kf)[4][2], f32x4_t (&cs)[4],
                                float scale2, int bound, int lane) {
#pragma unroll
  for (int c2 = 0; c2 < 4; c2 += 2) {
    bf16x8_t qf[2][2];
    float nn[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      fragments(qt, c2 + j, lane, qf[j]);
      nn[j] = nt[16 * (c2 + j) + (lane & 15)];
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      f32x4_t d[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) d[j] = dot64(kf[kb], qf[j]);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (MASKED) mask_keys(d[j], 16 * kb, bound + 2 * (c2 + j));
#pragma unroll
        for (int r = 0; r < 4; ++r) d[j][r] = fast_exp2(fmaf(d[j][r], scale2, nn[j]));
      }
      // The sums are formed here: otherwise the exponentials sink behind the tile's last MFMA, with
      // their logits.
#pragma unroll
      for (int r = 0; r < 4; ++r) cs[kb][r] = formed(cs[kb][r] + (d[0][r] + d[1][r]));
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The same, maxima over the KV head's query heads: a lane holds heads 4*(grp%2) + r of query grp/2
// of a row block (2 queries) for key col of a key block; the other four heads are in the
// neighbouring lane group. One swap joins them for two key blocks: cs[kp] += the largest probability
// of key 32*kp + 16*(grp%2) + col over the tile's queries of parity grp/2. The largest probability
// is 2^(largest exponent): one exponential per (query, key). MASKED: key 16*kb is dead past
// bound + 2*rb.
template <bool MASKED>
GSE_DEVICE void column_max_tile(const uint16_t* qt, const float* nt, const bf16x8_t (&kf)[4][2], float (&cs)[2],
                                float scale2, int bound, int lane) {
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    bf16x8_t qf[2];
    fragments(qt, rb, lane, qf);
    const f32x4_t nn = *reinterpret_cast<const f32x4_t*>(nt + 16 * rb + 4 * (lane >> 4));
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) {
      float y[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t d = dot64(qf, kf[2 * kp + h]);
        float x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = fmaf(d[r], scale2, nn[r]);
        y[h] = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
        if (MASKED && 32 * kp + 16 * h > bound + 2 * rb) y[h] = -INFINITY;
      }
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[0]), __float_as_uint(y[1]), false, false);
      cs[kp] = formed(cs[kp] + fast_exp2(vmax(__uint_as_float(r[0]), __uint_as_float(r[1]))));
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One value per lane out of N: lane bits select it, log2(N) exchanges (lane l ends with the sum over
// its exchange group of value l % N; N is 2^k, the group the N lanes around it).
template <int N>
GSE_DEVICE float scatter_sum(float (&v)[N], int lane) {
  if constexpr (N == 1) {
    return v[0];
  } else {
    float w[N / 2];
    const bool upper = lane & (N / 2);
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float keep = upper ? v[i + N / 2] : v[i], send = upper ? v[i] : v[i + N / 2];
      w[i] = keep + __shfl_xor(send, N / 2, kWave);
    }
    return scatter_sum(w, lane);
  }
}

template <bool MAX_MODE>
__global__ __launch_bounds__(p2::THREADS, 4) void prefill_score_kernel(PrefillArgs a) {
  using namespace pf;
  using namespace p2;
  __shared__ __attribute__((aligned(16))) uint16_t qtile[2][QT * GROUP * KROW];
  __shared__ __attribute__((aligned(16))) float ntile[2][QT * GROUP];  // negated normalisers
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Block i: KV head i % kv_heads, then the query block, then the key block (the first keys are
  // credited by most queries; the last by few).
  const int count = int(a.count);
  const int nqb = (count + a.qblock - 1) / a.qblock;
  const int g = blockIdx.x % a.kv_heads;
  const int item = blockIdx.x / a.kv_heads;
  const int k0 = item / nqb * KB, kw = k0 + KW * wave;
  const int qb0 = item % nqb * a.qblock;
  const int q1 = min(qb0 + a.qblock, count);
  const int bound0 = int(a.prefix_len) - a.delay;  // query i credits keys up to bound0 + i
  const int q0 = max(qb0, max(k0 - bound0, 0) / QT * QT);
  if (q0 >= q1) return;
  const int kend = min(int(a.total), bound0 + q1);  // keys the item credits

  // The wave's keys: lane (col, grp) holds dims [8*grp, +8) and [32 + 8*grp, +8) of keys
  // kw + 16*kb + col (past the list: its last key, never credited).
  bf16x8_t kf[4][2];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const uint32_t key = min(uint32_t(kw) + 16 * kb + (lane & 15), uint32_t(a.total) - 1);
    const int64_t s = load_index_dyn(a.slots, a.slots_dtype, key);
    const auto kp = as_global(a.k) + s * a.kv_ss + int64_t(g) * a.kv_sh + 8 * (lane >> 4);
    kf[kb][0] = as_bf16x8(gload16(kp));
    kf[kb][1] = as_bf16x8(gload16(kp + 32));
  }
  // Query tile load: thread t stages 16 bytes of rows t/8 (query q + row/8, head row%8) and t/8 + 32
  // (four queries on); the next tile is in flight while one computes. Rows past the chunk are zero
  // with normaliser +inf: probability 0.
  static_assert(THREADS * 2 == QT * GROUP * 8, "two pieces per thread");
  const int lr = threadIdx.x >> 3, lp = threadIdx.x & 7;
  const auto qbase = as_global(a.q) + int64_t(g * GROUP + (lr & 7)) * a.q_sh + 8 * lp;
  const auto nbase = as_global(a.norm2) + g * GROUP + (threadIdx.x & 7);
  auto load_q = [&](int q) {
    const int qi = q + (lr >> 3);
    return qi < count ? gload16(qbase + int64_t(qi) * a.q_st) : uint4{};
  };
  auto load_n = [&](int q) {
    const int qi = q + int(threadIdx.x >> 3);
    return threadIdx.x < QT * GROUP && qi < count ? -nbase[int64_t(qi) * a.q_heads] : -INFINITY;
  };
  auto store_tile = [&](int p, const uint4& x0, const uint4& x1, float n) {
    *reinterpret_cast<uint4*>(&qtile[p][lr * KROW + 8 * lp]) = x0;
    *reinterpret_cast<uint4*>(&qtile[p][(lr + 32) * KROW + 8 * lp]) = x1;
    if (threadIdx.x < QT * GROUP) ntile[p][threadIdx.x] = n;
  };
  store_tile(0, load_q(q0), load_q(q0 + QT / 2), load_n(q0));
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    landed(kf[kb][0]);
    landed(kf[kb][1]);
  }
  __syncthreads();

  f32x4_t sums[4] = {};
  float maxes[2] = {0.f, 0.f};
  const float scale2 = a.scale2;
  // The bound of the lane's row of a tile at query 0, from the lane's first key on.
  const int rel = bound0 - kw + (MAX_MODE ? (lane >> 5) - (lane & 15) : ((lane & 15) >> 3) - 4 * (lane >> 4));
  auto tile_step = [&](int q, int p, auto whole) {
    constexpr bool WHOLE = decltype(whole)::value;
    const uint4 x0 = load_q(q + QT), x1 = load_q(q + QT + QT / 2);
    const float n = load_n(q + QT);
    const int bound = rel + q;
    auto compute = [&](auto masked) {
      constexpr bool MASKED = decltype(masked)::value;
      if constexpr (MAX_MODE)
        column_max_tile<MASKED>(qtile[p], ntile[p], kf, maxes, scale2, bound, lane);
      else
        column_sum_tile<MASKED>(qtile[p], ntile[p], kf, sums, scale2, bound, lane);
    };
    if constexpr (WHOLE) {
      compute(std::false_type{});
    } else if (kw + KW - 1 <= bound0 + q) {
      compute(std::false_type{});
    } else if (kw <= bound0 + q + QT - 1) {
      compute(std::true_type{});
    }
    if (q + QT < q1) store_tile(p ^ 1, x0, x1, n);
    __syncthreads();
  };
  // Queries that credit every key of the workgroup run in a loop of their own.
  const int qw = min(q1, max(q0, (max(k0 + KB - 1 - bound0, 0) + QT - 1) / QT * QT));
  int q = q0, p = 0;
#pragma unroll 1
  for (; q < qw; q += QT, p ^= 1) tile_step(q, p, std::false_type{});
#pragma unroll 1
  for (; q < q1; q += QT, p ^= 1) tile_step(q, p, std::true_type{});

  // One lane per key, one atomic per lane.
  float total;
  int key;
  if constexpr (MAX_MODE) {
    const float t0 = xor32_sum(maxes[0]), t1 = xor32_sum(maxes[1]);  // both query parities
    total = lane < 32 ? t0 : t1;
    key = kw + lane;
  } else {
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = sums[i / 4][i % 4];
    total = scatter_sum(v, lane);  // lane % 16 selects the register
    key = kw + 16 * ((lane & 15) >> 2) + 4 * (lane >> 4) + (lane & 3);
  }
  if (key < kend)
    unsafeAtomicAdd(&a.scores[int64_t(g) * a.ssg + load_index_dyn(a.slots, a.slots_dtype, key) * a.sss], total);
}

// ---------------------------------------------------------------------------
// Block counters of a chunk (score kind 4)
// ---------------------------------------------------------------------------
// The second pass for score kind 4 (TEX:197's block counters; no reference code). A workgroup owns 64
// queries (8 per wave, 4 row blocks of (query, head) pairs) and a range of 256-key tiles. Per tile it
// walks the KV heads: K_g of the tile's keys goes through LDS (the next head's rows in flight), the
// wave's queries of that head come into registers a head ahead, and D = Q . K_g^T with pass 1's
// normalisers raises a running maximum of the log2 probability per (query, key) and lane. After the
// last head the lane's two head halves meet, then a block's keys (a butterfly over the low lane bits:
// blocks of at most 64 aligned entries lie in a 64-key group), and only then, 2^x increasing with x,
// one exponential per (query, block). Query i credits the whole blocks of keys < prefix_len + i + 1 -
// delay: every other maximum is dropped there, so the heads' walk needs no mask. The waves' credits
// meet in LDS and one thread per key adds them to the block's counter (KV head 0's score of its first
// slot).
// Bound by the matrix units beside vector issue: per 1024 logits 8 MFMAs (132 cycles), 16 FMAs and 8
// three-way maxima. 2048 queries after 12,288 keys, blocks of 4: 630 us with a wave per KV head and
// an LDS atomic maximum per lane and 16x16 block, 414 with plain LDS maxima and a barrier per 64
// keys, 314 us so (2.1 GHz: the power limit; 287 in a row, 597 the first form).
namespace pb {
constexpr int QB = pf::QB;      // queries per workgroup
constexpr int QW = 8;           // queries per wave
constexpr int WAVES = QB / QW;
constexpr int THREADS = 64 * WAVES;
constexpr int KT = 256;         // keys per tile
constexpr int KB = KT / 16;     // its 16-key blocks
constexpr int MAX_HEADS = 64;   // query heads
// Work items of a launch: some eight rounds of the one workgroup a CU holds.
constexpr int ITEMS = 2048;
}  // namespace pb

GSE_DEVICE float vmax3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// x of the lower and y of the upper lanes (by lane bit 5, resp. 4), each summed over that bit.
GSE_DEVICE float join32(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
GSE_DEVICE float join16(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename IdxT>
__global__ __launch_bounds__(pb::THREADS, 2) void prefill_block_kernel(PrefillArgs a) {
  using namespace pb;
  using pf::KROW;
  __shared__ __attribute__((aligned(16))) uint16_t ktile[2][KT * KROW];
  // Negated normalisers of the workgroup's queries (-inf past the chunk), rows padded by 16 bytes.
  __shared__ __attribute__((aligned(16))) float norms[QB][MAX_HEADS + 4];
  __shared__ float cols[WAVES][KT];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int shift = a.block_shift, block = 1 << shift;
  const IdxT* slots = static_cast<const IdxT*>(a.slots);
  const int count = int(a.count), heads = a.kv_heads;
  // Block i: the query block from the end (the longest causal ranges first), then the key range.
  const int nqb = (count + QB - 1) / QB;
  const int split = blockIdx.x / nqb;
  const int qb0 = (nqb - 1 - blockIdx.x % nqb) * QB;
  auto limit = [&](int i) {  // credited keys of query i
    return i < count ? block_step_limit(int(a.prefix_len) + i + 1, a.delay, shift) : 0;
  };
  const int kend = limit(min(qb0 + QB, count) - 1);
  const int ntiles = (kend + KT - 1) / KT;
  const int ranges = key_ranges(ntiles, a.tiles);
  if (split >= ranges) return;
  const int ti0 = int(int64_t(ntiles) * split / ranges), ti1 = int(int64_t(ntiles) * (split + 1) / ranges);
  const int i0 = qb0 + QW * wave;
  const bool live = i0 < count;
  int lim[4];  // of this lane's D rows: query i0 + 2*rb + grp/2, heads 4*(grp%2) + r
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) lim[rb] = limit(i0 + 2 * rb + (grp >> 1));

  // A fragments of head g: row col of block rb is query i0 + 2*rb + col/8, head g*8 + col%8.
  auto load_q = [&](int g, uint4 (&q)[4][2]) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      const int qi = min(i0 + 2 * rb + (col >> 3), count - 1);  // past the chunk: any row, its normaliser is +inf
      const auto qp = as_global(a.q) + qi * a.q_st + int64_t(g * pf::GROUP + (col & 7)) * a.q_sh + 8 * grp;
      q[rb][0] = gload16(qp);
      q[rb][1] = gload16(qp + 32);
    }
  };
  // Thread t stages 16 bytes of keys t/8 + 64*j. A tile's slots are read a tile ahead.
  const int lk = threadIdx.x >> 3, lp = threadIdx.x & 7;
  auto load_slots = [&](int ti, IdxT (&sl)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) sl[j] = slots[min(uint32_t(ti) * KT + 64 * j + lk, uint32_t(kend) - 1)];
  };
  const auto kbase = as_global(a.k) + 8 * lp;
  auto load_k = [&](int g, const IdxT (&sl)[4], uint4 (&x)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = gload16(kbase + int64_t(sl[j]) * a.kv_ss + int64_t(g) * a.kv_sh);
  };
  auto store_k = [&](int p, const uint4 (&x)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4*>(&ktile[p][(lk + 64 * j) * KROW + 8 * lp]) = x[j];
  };
  IdxT sl[4], sn[4];
  uint4 qf[4][2];
  {
    uint4 x[4];
    load_slots(ti0, sl);
    load_q(0, qf);
    for (int t = threadIdx.x; t < QB * heads * pf::GROUP; t += THREADS) {
      const int i = t / (heads * pf::GROUP), h = t % (heads * pf::GROUP);
      norms[i][h] = qb0 + i < count ? -a.norm2[int64_t(qb0 + i) * a.q_heads + h] : -INFINITY;
    }
    load_k(0, sl, x);
    store_k(0, x);
  }
  __syncthreads();

  int p = 0;
#pragma unroll 1
  for (int ti = ti0; ti < ti1; ++ti) {
    load_slots(ti + 1, sn);
    float y[4][KB];  // the lane's maximum over its heads of query i0 + 2*rb + grp/2, key 16*kb + col
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) y[rb][kb] = -INFINITY;
#pragma unroll 1
    for (int g = 0; g < heads; ++g, p ^= 1) {
      // The next head's rows and queries (the first of the next tile's after the last) go out.
      const bool wrap = g + 1 == heads, more = !wrap || ti + 1 < ti1;
      uint4 xn[4], qn[4][2];
      if (wrap)
        load_k(0, sn, xn);
      else
        load_k(g + 1, sl, xn);
      load_q(wrap ? 0 : g + 1, qn);
      if (live) {
        bf16x8_t qa[4][2];
        f32x4_t nn[4];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          qa[rb][0] = as_bf16x8(qf[rb][0]);
          qa[rb][1] = as_bf16x8(qf[rb][1]);
          nn[rb] = *reinterpret_cast<const f32x4_t*>(&norms[QW * wave + 2 * rb + (grp >> 1)][g * pf::GROUP + 4 * (grp & 1)]);
        }
        bf16x8_t kf[2][2];  // alternate by key block
        fragments(ktile[p], 0, lane, kf[0]);
        f32x4_t dn[2] = {dot64(qa[0], kf[0]), dot64(qa[1], kf[0])};
#pragma unroll
        for (int u = 0; u < 2 * KB; ++u) {  // units of two row blocks against a key block
          const int kb = u >> 1, rb = 2 * (u & 1), nkb = (u + 1) >> 1, nrb = 2 * ((u + 1) & 1);
          const f32x4_t d[2] = {dn[0], dn[1]};
          if ((u & 1) == 0 && kb + 1 < KB) fragments(ktile[p], kb + 1, lane, kf[(kb + 1) & 1]);
          if (u + 1 < 2 * KB) {  // the next unit's MFMAs ahead of this one's vector work
            dn[0] = dot64(qa[nrb], kf[nkb & 1]);
            dn[1] = dot64(qa[nrb + 1], kf[nkb & 1]);
          }
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float x[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = fmaf(d[j][r], a.scale2, nn[rb + j][r]);
            y[rb + j][kb] = vmax3(vmax3(y[rb + j][kb], x[0], x[1]), x[2], x[3]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (more) {
        store_k(p ^ 1, xn);
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
          qf[rb][0] = qn[rb][0];
          qf[rb][1] = qn[rb][1];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) sl[j] = sn[j];

    // Per (query, key) the maximum over all heads, of two key blocks at once: lane holds query i0 +
    // 2*rb + grp/2 and key 32*kp + in_pair.
    const int in_pair = 16 * (grp & 1) + col;
    const bool leads = (in_pair & (block - 1)) == 0;
#pragma unroll
    for (int kp = 0; kp < KB / 2; kp += 2) {
      float c[2] = {0.f, 0.f};
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        float z[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[rb][2 * (kp + h)]),
                                                          __float_as_uint(y[rb][2 * (kp + h) + 1]), false, false);
          z[h] = vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
          if (ti * KT + 32 * (kp + h) + in_pair >= lim[rb]) z[h] = -INFINITY;
        }
        for (int o = 1; o < block && o < 32; o <<= 1) {
          z[0] = fmaxf(z[0], __shfl_xor(z[0], o, kWave));
          z[1] = fmaxf(z[1], __shfl_xor(z[1], o, kWave));
        }
        if (block == 64) z[0] = fmaxf(z[0], z[1]);
        c[0] += leads ? fast_exp2(z[0]) : 0.f;
        c[1] += leads && block < 64 ? fast_exp2(z[1]) : 0.f;
      }
      cols[wave][32 * kp + lane] = join32(c[0], c[1]);  // both queries of a row block
    }
    __syncthreads();
    // The next tile's columns are written past its heads' barriers.
    const int key = ti * KT + int(threadIdx.x);
    if (int(threadIdx.x) < KT && key < kend && (key & (block - 1)) == 0) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += cols[w][threadIdx.x];
      if (v > 0.f) unsafeAtomicAdd(&a.scores[int64_t(slots[key]) * a.sss], v);
    }
  }
}

// ---------------------------------------------------------------------------
// Static regret diagnostic (pass 3)
// ---------------------------------------------------------------------------
constexpr int DIAG_MAX_SPECS = 8;
constexpr int FOLD = 4;  // tiles per fold of the waves' column sums: a key and table per thread
static_assert(2 * FOLD * pf::KT == p1::THREADS, "one (table, key) per thread");

struct DiagArgs {
  PrefillArgs p;         // q, keys, slots, sinks, scale, row normalisers of pass 1
  float* score_max;      // second score table (max over the KV head's query heads)
  const uint32_t* evicted;  // bit k of word w of (spec s, KV head g): key 32*w + k is evicted
  int n_specs;
  int64_t ev_ss, ev_sg;  // word strides of spec and KV head
  float* lost;           // lost[s * lost_ss + i] += ... for chunk query i
  int64_t lost_ss;
  float lost_scale;      // 1 / (query heads * full layers)
};

// Bit masks of the diagnostic's specs: words[(s * kv_heads + g) * n_words ..], bit k%32 of word k/32
// set when key k < n is not resident. One wave per 64 keys of a (spec, KV head).
__global__ __launch_bounds__(256) void pack_evicted_kernel(const uint8_t* resident, int64_t res_ss, int64_t res_sg,
                                                           int kv_heads, int64_t n, uint32_t* words,
                                                           int64_t n_words) {
  const int sg = blockIdx.y, s = sg / kv_heads, g = sg % kv_heads;
  const int64_t key = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const bool gone = key < n && !resident[s * res_ss + g * res_sg + key];
  const uint64_t bits = __builtin_amdgcn_ballot_w64(gone);
  const int lane = threadIdx.x & 63;
  const int64_t w = (key >> 6) * 2 + lane;
  if (lane < 2 && w < n_words) words[sg * n_words + w] = uint32_t(bits >> (32 * lane));
}

// Pass 3 of a diagnostic chunk: the exact probabilities of pass 1's normalisers, added to two
// position-indexed score tables (sum and max over each KV head's query heads, summed over the
// chunk's queries), and every spec's lost mass per query: the group-summed probability on
// keys the spec has evicted, summed over keys and KV heads, times lost_scale. Items as pass 1 (64
// queries, a range of key tiles), S = Q . K^T: a lane holds 4 heads of one query for one key, so a
// spec costs one FMA (with its 0/1 bit of the key) per 4 logits; column sums and maxima meet by lane
// swaps, then through a column per wave in LDS (float atomics there took 194 cycles each, half the
// kernel). NS, the number of specs, is a template argument: a run-time bound on
// the unrolled spec loop cost a branch per (spec, 16x16 block). Vector issue bound as pass 1; 2048
// queries after 14,336 keys, 4 specs: 1249 -> 619 us (20 calls in a row), 65 % of the cycles issuing (2 waves per SIMD).
template <int NS>
__global__ __launch_bounds__(p1::THREADS, NS == 0 ? 4 : 2) void diagnose_kernel(DiagArgs da) {
  using namespace pf;
  using p1::QW;
  const PrefillArgs& a = da.p;
  __shared__ __attribute__((aligned(16))) KeyTiles::Tile ktile[2];
  // Column sums and maxima of each wave, two rings of FOLD tiles: one fills while the other folds.
  __shared__ float cols[2][2][p1::WAVES][FOLD * KT];
  __shared__ uint32_t evicted[2][2 * DIAG_MAX_SPECS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int nqb = int((a.count + QB - 1) / QB);
  const int g = blockIdx.x % a.kv_heads;
  const int item = blockIdx.x / a.kv_heads;
  const int split = item / nqb;
  const int64_t qb0 = int64_t(nqb - 1 - item % nqb) * QB;
  const int last_q = int((qb0 + QB < a.count ? qb0 + QB : a.count) - 1);
  const int kend = int(a.prefix_len) + last_q + 1;
  const int ntiles = (kend + KT - 1) / KT;
  const int ranges = key_ranges(ntiles, a.tiles);
  if (split >= ranges) return;
  const int ti0 = int(int64_t(ntiles) * split / ranges), ti1 = int(int64_t(ntiles) * (split + 1) / ranges);
  const int i0 = int(qb0) + QW * wave;
  const bool wave_live = i0 < a.count;
  const int wave_kend = int(a.prefix_len) + min(i0 + QW - 1, int(a.count) - 1) + 1;

  // A fragments: row col of block rb is query i0 + 2*rb + col/8, head g*8 + col%8. The lane's D
  // rows: query i0 + 2*rb + grp/2, heads hq0 + r.
  const int hq0 = g * GROUP + 4 * (grp & 1);
  bf16x8_t qf[4][2];
  f32x4_t nn[4];  // negated normalisers (-inf past the chunk: probability 0)
  float lost[NS > 0 ? NS : 1][4];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int64_t qi = i0 + 2 * rb + (col >> 3), qd = i0 + 2 * rb + (grp >> 1);
    const uint16_t* qp = a.q + qi * a.q_st + int64_t(g * GROUP + (col & 7)) * a.q_sh + 8 * grp;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      qf[rb][h] = qi < a.count ? as_bf16x8(*reinterpret_cast<const uint4*>(qp + 32 * h)) : bf16x8_t{};
#pragma unroll
    for (int r = 0; r < 4; ++r) nn[rb][r] = qd < a.count ? -a.norm2[qd * a.q_heads + hq0 + r] : -INFINITY;
#pragma unroll
    for (int sp = 0; sp < NS; ++sp) lost[sp][rb] = 0.f;
  }
  KeyTiles keys(a, g, kend);
  // The specs' words of a tile travel with its K rows (as KeyTiles): thread t < 2 * NS brings half
  // t%2 of spec t/2. Loaded where they are used they would cost a memory latency per tile.
  const auto words = as_global(da.evicted) + int64_t(g) * da.ev_sg +
                     (int(threadIdx.x) < 2 * NS ? (threadIdx.x >> 1) * da.ev_ss + (threadIdx.x & 1) : 0);
  const int last_tile = ntiles - 1;
  auto load_words = [&](int ti) { return NS > 0 ? words[2 * min(ti, last_tile)] : 0u; };
  auto stage_words = [&](int p, uint32_t w) {
    if (int(threadIdx.x) < 2 * NS) evicted[p][threadIdx.x] = w;
  };
  uint32_t word[2] = {0u, load_words(ti0 + 1)};
  stage_words(0, load_words(ti0));
  keys.start(ti0, ktile);
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    landed(qf[rb][0]);
    landed(qf[rb][1]);
#pragma unroll
    for (int r = 0; r < 4; ++r) landed(nn[rb][r]);
  }
  __syncthreads();

  const int qpos = int(a.prefix_len) + i0 + (grp >> 1) - col;  // causal bound of block 0, from the lane's key
  const float scale2 = a.scale2;
  auto tile_step = [&](int ti, auto parity) {
    constexpr int P = decltype(parity)::value;  // (ti - ti0) & 1
    word[P] = load_words(ti + 2);
    keys.ahead(ti, P);
    const int t0 = ti * KT;
    float tsum = 0.f, tmax = 0.f;  // of key t0 + lane
    if (wave_live && t0 < wave_kend) {
      float cs[4] = {0.f, 0.f, 0.f, 0.f}, cm[2] = {0.f, 0.f};
      auto rows = [&](auto masked) {
        constexpr bool MASKED = decltype(masked)::value;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          bf16x8_t kf[2][2];
          float gone[NS > 0 ? NS : 1][2];  // 1 for the specs that evicted the lane's keys
#pragma unroll
          for (int h = 0; h < 2; ++h) fragments(ktile[P], 2 * kp + h, lane, kf[h]);
#pragma unroll
          for (int sp = 0; sp < NS; ++sp) {
            const uint32_t w = evicted[P][2 * sp + kp];
#pragma unroll
            for (int h = 0; h < 2; ++h) gone[sp][h] = float((w >> (16 * h + col)) & 1u);
          }
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) {
            float y[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              f32x4_t d = dot64(qf[rb], kf[h]);
              if (MASKED && 32 * kp + 16 * h > qpos - t0 + 2 * rb) d = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
              for (int r = 0; r < 4; ++r) d[r] = fast_exp2(fmaf(d[r], scale2, nn[rb][r]));
              const float psum = sum4(d);
              cs[2 * kp + h] += psum;
              y[h] = fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3]));
#pragma unroll
              for (int sp = 0; sp < NS; ++sp) lost[sp][rb] = fmaf(psum, gone[sp][h], lost[sp][rb]);
            }
            // The maximum over all 8 heads, for the two key blocks at once (as column_max_tile).
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[0]), __float_as_uint(y[1]), false, false);
            cm[kp] = formed(cm[kp] + vmax(__uint_as_float(r[0]), __uint_as_float(r[1])));
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      };
      if (t0 + KT - 1 > int(a.prefix_len) + i0)
        rows(std::true_type{});
      else
        rows(std::false_type{});
      // Lane l ends with key l: lane bit 4 selects the key block of a pair, bit 5 the pair.
      tsum = join32(join16(cs[0], cs[1]), join16(cs[2], cs[3]));
      tmax = join32(cm[0], cm[1]);
    }
    const int n = ti - ti0, ring = (n / FOLD) & 1, slot = n % FOLD;
    cols[ring][0][wave][slot * KT + lane] = tsum;
    cols[ring][1][wave][slot * KT + lane] = tmax;
    if (ti + 1 < ti1) {
      stage_words(1 - P, word[1 - P]);
      keys.stage(1 - P, ktile);
    }
    __syncthreads();
    if (slot == FOLD - 1 || ti + 1 == ti1) {
      // One thread per key and table. Diagnostic score tables are indexed by position (the chunk's
      // CSR column).
      const int table = threadIdx.x / (FOLD * KT), at = threadIdx.x % (FOLD * KT);
      const int key = (ti - slot) * KT + at;
      if (at < (slot + 1) * KT && key < kend) {
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < p1::WAVES; ++w) total += cols[ring][table][w][at];
        unsafeAtomicAdd((table ? da.score_max : a.scores) + int64_t(g) * a.ssg + key * a.sss, total);
      }
    }
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
#pragma unroll 1
  for (int ti = ti0; ti < ti1; ti += 2) {
    tile_step(ti, P0{});
    if (ti + 1 < ti1) tile_step(ti + 1, P1{});
  }

  if (NS > 0 && wave_live) {
    // Per spec and query: the lane's sum over its key columns (16 lanes) and the two head halves.
#pragma unroll
    for (int sp = 0; sp < NS; ++sp)
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        float v = lost[sp][rb];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, kWave);
        v = xor16_sum(v);
        const int64_t qi = i0 + 2 * rb + (grp >> 1);
        if (col == 0 && (grp & 1) == 0 && qi < a.count) atomicAdd(&da.lost[sp * da.lost_ss + qi], v * da.lost_scale);
      }
  }
}

}  // namespace gse

using namespace gse;

// Upper bound of the key ranges pass 1 wants for a chunk of `count` queries: launch_norms divides the
// item count by the mean tiles of a query block, at least half of the last one's.
static int64_t max_splits(int64_t count, int kv_heads) {
  const int64_t blocks = (count + pf::QB - 1) / pf::QB * kv_heads;
  return blocks > 0 ? 2 * p1::ITEMS / blocks + 2 : 0;
}

static int64_t norm_bytes(int64_t count, int q_heads) { return ((count * q_heads * 4 + 255) / 256) * 256; }

extern "C" int64_t gse_prefill_workspace_bytes(int64_t count, int q_heads) {
  // The normalisers, then pass 1's (reference, sum) pairs.
  const int64_t pairs = max_splits(count, q_heads / pf::GROUP) * count * q_heads * int64_t(sizeof(float2));
  return norm_bytes(count, q_heads) + ((pairs + 255) / 256) * 256;
}

// Pass 1 and the merge: row normalisers of a chunk into a.norm2. Fills in a's workspace pointers
// and the key ranges: as many as a workspace of at least the normalisers' bytes holds the pairs of
// (one range leaves none).
static int launch_norms(PrefillArgs& a, void* workspace, int64_t workspace_bytes, hipStream_t s) {
  a.norm2 = static_cast<float*>(workspace);
  a.part = reinterpret_cast<float2*>(static_cast<char*>(workspace) + norm_bytes(a.count, a.q_heads));
  const int64_t nqb = (a.count + pf::QB - 1) / pf::QB;
  const int64_t last = (a.total + pf::KT - 1) / pf::KT;
  const int64_t room = (workspace_bytes - norm_bytes(a.count, a.q_heads)) / (a.count * a.q_heads * int64_t(sizeof(float2)));
  const int64_t most = std::max<int64_t>(1, std::min({max_splits(a.count, a.kv_heads), room, last / p1::MIN_TILES}));
  // Tiles that query block b sees, and the launch's (by the mean block).
  auto sees = [&](int64_t b) { return (a.prefix_len + std::min((b + 1) * pf::QB, a.count) + pf::KT - 1) / pf::KT; };
  const int64_t work = (sees(0) + last + 1) / 2 * nqb * a.kv_heads;
  int64_t tiles = std::max<int64_t>((work + p1::ITEMS - 1) / p1::ITEMS, (last + most - 1) / most);
  if (work <= p1::FEW_TILES * p1::SLOTS) {
    double best = 0;
    for (int64_t n = 1; n <= most; n += 1 + n / 16) {
      const int64_t t = (last + n - 1) / n;
      int64_t items = 0;
      for (int64_t b = 0; b < nqb; ++b) items += (sees(b) + t - 1) / t;
      const double cost = double((items * a.kv_heads + p1::SLOTS - 1) / p1::SLOTS) * (double(t) + p1::START);
      if (n == 1 || cost < best) {
        best = cost;
        tiles = t;
      }
    }
  }
  a.tiles = int(tiles);
  a.splits = int((last + tiles - 1) / tiles);
  const int64_t blocks = nqb * a.kv_heads * a.splits;
  if (blocks >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "prefill: chunk too large");
  hipLaunchKernelGGL(prefill_norm_kernel, dim3(uint32_t(blocks)), dim3(p1::THREADS), 0, s, a);
  if (int rc = gse_launch_check("prefill pass 1")) return rc;
  if (a.splits == 1) return GSE_OK;
  const int64_t rows = a.count * a.q_heads;
  hipLaunchKernelGGL(prefill_merge_kernel, dim3(uint32_t((rows + 255) / 256)), dim3(256), 0, s, a);
  return gse_launch_check("prefill normalisers");
}

extern "C" int gse_prefill_scores(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                                  const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h, const void* slots,
                                  int slots_dtype, int64_t total, int64_t prefix_len, const void* sinks,
                                  int sinks_dtype, int mode, float* scores, int64_t scores_stride_g,
                                  int64_t scores_stride_s, int q_heads, int kv_heads, int head_dim, float sm_scale,
                                  void* workspace, int64_t workspace_bytes, gse_stream_t stream) {
  if (head_dim != pf::D || kv_heads < 1 || q_heads != pf::GROUP * kv_heads)
    return gse_fail(GSE_ESHAPE, "prefill: need head_dim 64 and q_heads == 8 * kv_heads");
  const int kind = mode & 0xf, block_shift = (mode >> GSE_SCORE_BLOCK_SHIFT) & 0xf;
  const int delay = mode >> GSE_SCORE_DELAY_SHIFT;
  if (kind != 1 && kind != 2 && kind != GSE_SCORE_KIND_BLOCK_STEP)
    return gse_fail(GSE_EINVAL, "prefill: score kind must be 1 (sum), 2 (max) or 4 (block counters)");
  if (kind != GSE_SCORE_KIND_BLOCK_STEP ? (mode & 0xf0) != 0 : block_shift > 6)
    return gse_fail(GSE_EINVAL, "prefill: bad block size bits");
  if (delay < 0) return gse_fail(GSE_EINVAL, "prefill: negative score delay");
  if (count < 0 || prefix_len < 0 || total != prefix_len + count)
    return gse_fail(GSE_EINVAL, "prefill: total must equal prefix_len + count");
  if (total >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "prefill: too many keys");
  if (count == 0) return GSE_OK;
  if (q_stride_t % 8 || q_stride_h % 8 || kv_stride_s % 8 || kv_stride_h % 8)
    return gse_fail(GSE_EINVAL, "prefill: strides must be multiples of 8 elements");
  if (!q || !k_pool || !slots || !sinks || !scores) return gse_fail(GSE_EINVAL, "prefill: null pointer");
  if (workspace_bytes < norm_bytes(count, q_heads)) return gse_fail(GSE_EWORKSPACE, "prefill: workspace too small");
  PrefillArgs a = {static_cast<const uint16_t*>(q), q_stride_t, q_stride_h, count,
                   static_cast<const uint16_t*>(k_pool), kv_stride_s, kv_stride_h, slots, slots_dtype, total,
                   prefix_len, sinks, sinks_dtype, kind, scores, scores_stride_g, scores_stride_s, q_heads, kv_heads,
                   sm_scale * kLog2e, static_cast<float*>(workspace), delay, block_shift};
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (kind == GSE_SCORE_KIND_BLOCK_STEP && q_heads > pb::MAX_HEADS)
    return gse_fail(GSE_ESHAPE, "prefill: block counters need kv_heads <= 8");
  if (int rc = launch_norms(a, workspace, workspace_bytes, s)) return rc;
  if (kind == GSE_SCORE_KIND_BLOCK_STEP) {
    const int64_t nqb = (count + pb::QB - 1) / pb::QB;
    const int64_t first = prefix_len / pb::KT + 1, last = (total + pb::KT - 1) / pb::KT;
    const int64_t work = (first + last + 1) / 2 * nqb;  // tiles of the launch
    const int64_t tiles = std::max<int64_t>(1, (work + pb::ITEMS - 1) / pb::ITEMS);
    a.tiles = int(tiles);  // of this pass's ranges (pass 1 and the merge are launched)
    const int64_t items = nqb * ((last + tiles - 1) / tiles);
    if (items >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "prefill: chunk too large");
    const dim3 bgrid{static_cast<uint32_t>(items)};
    if (slots_dtype == GSE_I64)
      hipLaunchKernelGGL(prefill_block_kernel<int64_t>, bgrid, dim3(pb::THREADS), 0, s, a);
    else
      hipLaunchKernelGGL(prefill_block_kernel<int32_t>, bgrid, dim3(pb::THREADS), 0, s, a);
    return gse_launch_check("prefill block counters");
  }
  const int64_t nkb = (total + p2::KB - 1) / p2::KB;
  const int64_t bound0 = prefix_len - delay;  // query i credits keys up to bound0 + i
  auto block_of = [&](int64_t n) {  // queries of one of n blocks
    return std::min<int64_t>(((count + n - 1) / n + p2::QT - 1) / p2::QT * p2::QT, p2::MAX_QUERIES);
  };
  // Workgroups that credit keys: the key blocks that only part of the chunk credits have fewer query blocks.
  auto live = [&](int64_t qblock) {
    const int64_t nq = (count + qblock - 1) / qblock;
    int64_t n = 0;
    for (int64_t k = 0; k < nkb && k * p2::KB - bound0 < count; ++k)
      n += std::max<int64_t>(0, nq - std::max<int64_t>(0, k * p2::KB - bound0) / qblock);
    return n * kv_heads;
  };
  const int64_t nqmax = (count + p2::MIN_QUERIES - 1) / p2::MIN_QUERIES;
  const int64_t common = std::min(std::max<int64_t>(1, p2::ITEMS / (nkb * kv_heads)), (nqmax + 1) / 2);
  const int64_t wgs = nkb * kv_heads <= p2::ROUND ? live(block_of(common)) : p2::ROUND + 1;
  int64_t blocks = common;
  if (wgs < p2::FEW) {
    for (int64_t n = nqmax; n > blocks && block_of(n) * 4 <= block_of(common) * 3; --n)
      if (live(block_of(n)) <= p2::FEW) blocks = n;
  } else if (common == (nqmax + 1) / 2 && wgs > (kind == 2 ? p2::SLOTS * 5 / 4 : p2::SLOTS) && wgs <= p2::ROUND) {
    int64_t n = common - 1;
    while (n > 1 && live(block_of(n)) > p2::SLOTS) --n;
    const int64_t one = n > 0 ? live(block_of(n)) : 0;
    if (one <= p2::SLOTS && one * 8 >= p2::SLOTS * 7) blocks = n;
  }
  a.qblock = int(block_of(blocks));
  const int64_t items = nkb * ((count + a.qblock - 1) / a.qblock) * kv_heads;
  if (items >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "prefill: chunk too large");
  if (kind == 2)
    hipLaunchKernelGGL(prefill_score_kernel<true>, dim3(uint32_t(items)), dim3(p2::THREADS), 0, s, a);
  else
    hipLaunchKernelGGL(prefill_score_kernel<false>, dim3(uint32_t(items)), dim3(p2::THREADS), 0, s, a);
  return gse_launch_check("prefill pass 2");
}

extern "C" int gse_diagnose_chunk(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                                  const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h, const void* slots,
                                  int slots_dtype, int64_t total, int64_t prefix_len, const void* sinks,
                                  int sinks_dtype, float* score_sum, float* score_max, int64_t scores_stride_g,
                                  int64_t scores_stride_s, const uint32_t* evicted, int n_specs,
                                  int64_t evicted_stride_s, int64_t evicted_stride_g, float* lost,
                                  int64_t lost_stride_s, float lost_scale, int q_heads, int kv_heads, int head_dim,
                                  float sm_scale, void* workspace, int64_t workspace_bytes, gse_stream_t stream) {
  if (head_dim != pf::D || kv_heads < 1 || q_heads != pf::GROUP * kv_heads)
    return gse_fail(GSE_ESHAPE, "diagnose: need head_dim 64 and q_heads == 8 * kv_heads");
  if (n_specs < 0 || n_specs > DIAG_MAX_SPECS) return gse_fail(GSE_EINVAL, "diagnose: 0..8 policy specs");
  if (count < 0 || prefix_len < 0 || total != prefix_len + count)
    return gse_fail(GSE_EINVAL, "diagnose: total must equal prefix_len + count");
  if (total >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "diagnose: too many keys");  // 32-bit key indexes
  if (count == 0) return GSE_OK;
  if (q_stride_t % 8 || q_stride_h % 8 || kv_stride_s % 8 || kv_stride_h % 8)
    return gse_fail(GSE_EINVAL, "diagnose: strides must be multiples of 8 elements");
  if (!q || !k_pool || !slots || !sinks || !score_sum || !score_max || !lost || (n_specs && !evicted))
    return gse_fail(GSE_EINVAL, "diagnose: null pointer");
  if (evicted_stride_g * 32 < ((total + 63) / 64) * 64)
    return gse_fail(GSE_EINVAL, "diagnose: evicted rows must cover the visible keys rounded up to 64");
  if (workspace_bytes < norm_bytes(count, q_heads)) return gse_fail(GSE_EWORKSPACE, "diagnose: workspace too small");
  DiagArgs da;
  da.p = {static_cast<const uint16_t*>(q), q_stride_t, q_stride_h, count, static_cast<const uint16_t*>(k_pool),
          kv_stride_s, kv_stride_h, slots, slots_dtype, total, prefix_len, sinks, sinks_dtype, 1, score_sum,
          scores_stride_g, scores_stride_s, q_heads, kv_heads, sm_scale * kLog2e, static_cast<float*>(workspace),
          /*delay=*/0, /*block_shift=*/0};  // the diagnostic scores every visible key
  da.score_max = score_max;
  da.evicted = evicted;
  da.n_specs = n_specs;
  da.ev_ss = evicted_stride_s;
  da.ev_sg = evicted_stride_g;
  da.lost = lost;
  da.lost_ss = lost_stride_s;
  da.lost_scale = lost_scale;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (int rc = launch_norms(da.p, workspace, workspace_bytes, s)) return rc;
  // launch_norms has set the key ranges and checked the grid.
  const dim3 grid{static_cast<uint32_t>((count + pf::QB - 1) / pf::QB * kv_heads * da.p.splits)};
  static void (*const kernels[])(DiagArgs) = {diagnose_kernel<0>, diagnose_kernel<1>, diagnose_kernel<2>,
                                              diagnose_kernel<3>, diagnose_kernel<4>, diagnose_kernel<5>,
                                              diagnose_kernel<6>, diagnose_kernel<7>, diagnose_kernel<8>};
  static_assert(sizeof(kernels) / sizeof(kernels[0]) == DIAG_MAX_SPECS + 1, "one instance per spec count");
  hipLaunchKernelGGL(kernels[n_specs], grid, dim3(p1::THREADS), 0, s, da);
  return gse_launch_check("diagnose pass 3");
}

extern "C" int gse_pack_evicted(const void* resident, int64_t resident_stride_s, int64_t resident_stride_g,
                                int n_specs, int kv_heads, int64_t n, uint32_t* words, int64_t n_words,
                                gse_stream_t stream) {
  if (n_specs < 0 || n_specs > DIAG_MAX_SPECS || kv_heads < 1 || kv_heads > 1024 || n < 0)
    return gse_fail(GSE_EINVAL, "pack: 0..8 policy specs, kv_heads in 1..1024");
  if (n_words < (n + 63) / 64 * 2) return gse_fail(GSE_EINVAL, "pack: words must cover the keys rounded up to 64");
  if (!n_specs || !n_words) return GSE_OK;
  if (!resident || !words) return gse_fail(GSE_EINVAL, "pack: null pointer");
  const int64_t blocks = (n_words + 7) / 8;  // 256 keys each
  if (blocks >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "pack: too many keys");
  hipLaunchKernelGGL(pack_evicted_kernel, dim3(uint32_t(blocks), n_specs * kv_heads), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), static_cast<const uint8_t*>(resident), resident_stride_s,
                     resident_stride_g, kv_heads, n, words, n_words);
  return gse_launch_check("pack evicted");
}
