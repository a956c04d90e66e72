// Static replay's layer difference (R:520-546): for every query of a prefill chunk, the
// relative L2 distance between the first full layer's attention output over the unevicted keys
// (a) and over each KV head's survivors (b), both with the sink in the normaliser:
//   error[i] = |b_i - a_i| / max(|a_i|, 1e-12), norms over all query heads x 64 dims.
//
// One launch computes both outputs (the longer one, over all keys, first) as partials over ranges of
// keys; a second kernel joins each query's ranges and the sink and takes the norms.
//
// Output kernel, per workgroup: one KV head, 32 queries (8 waves x 2 row-blocks) and a range of
// 64-key tiles. A row-block is 16 MFMA columns, (query, head) pairs: queries 2*rb and 2*rb + 1, the
// KV head's 8 query heads each. Per tile:
//   S^T = K . Q^T            4 key-blocks x 2 dim halves (v_mfma_f32_16x16x32_bf16)
//   online softmax           one running reference per column, moved lazily
//   O^T += V^T . P^T         V transposed through LDS (ds_read_b64_tr_b16); P split into
//                            bf16 hi + lo parts, so products carry ~16 mantissa bits of P
// K and V tiles go through LDS, double-buffered (threads 0-255 stage K, 256-511 stage V). Fragments
// are read from LDS where they are used, which leaves 128 registers and 4 waves per SIMD, so that
// one wave's MFMAs run beside another's vector work. Bound by the card's power: 24 MFMAs per 1024
// logits cost 200 ns per SIMD by themselves, their exponentials and splits 140 (1.95 GHz). Both
// outputs and the errors, 2048 queries after 16,384 keys (2048 retained): 1107 -> 1029 us (20 calls in a row); 150
// queries after 8192, whose 40 workgroups now split their keys: 276 -> 80 us; 17 after 28,672: 770 -> 66.
//
// Key columns: column c < n_retained is key row retained[g][c]; column c >= n_retained is key
// row tail0 + (c - n_retained). Query i sees columns <= prefix_len + i. With n_retained = 0 and
// tail0 = 0 that is plain causal attention over rows 0..prefix_len + i.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "host.hpp"

namespace gse {

namespace rp {
constexpr int D = 64;
constexpr int GROUP = 8;
constexpr int RB = 2;                    // row-blocks per wave
constexpr int WAVES = 8;
constexpr int QB = 2 * RB * WAVES;       // queries per workgroup (32)
constexpr int KT = 64;                   // keys per tile
constexpr int KROW = D + 8;              // padded bf16 row of a staged K row
constexpr int VROW = D + 16;             // padded bf16 row of a staged V row (transposed reads)
// A column's reference moves (to its maximum) when a lane's 16 terms sum past 2^8.
constexpr float kRescaleSum = 256.f;
// Work items per output: one round of the 512 workgroups the chip holds (2 per CU), of at least
// MIN_TILES tiles. A longer chunk's blocks take their whole causal range.
constexpr int ITEMS = 512;
constexpr int MIN_TILES = 4;
}  // namespace rp

// One of the two outputs.
struct ReplaySide {
  const int32_t* retained;  // [kv_heads][ret_sg] key rows of the first n_retained columns
  int64_t ret_sg, n_retained, tail0;
  int64_t prefix_len;
  // Partials of key range s: o[((s * count + i) * q_heads + h) * 64 ..] unnormalised, relative to
  // the reference m, and (m, l) with l the sum of the terms. With one range, o is the output itself
  // (ml unused).
  float* o;
  float2* ml;
};

struct ReplayArgs {
  const uint16_t* q;
  int64_t q_st, q_sh, count;
  const uint16_t* k;
  const uint16_t* v;
  int64_t kv_ss, kv_sh, rows;  // rows: key rows of k and v (out-of-range rows read row 0)
  const void* sinks;
  int sinks_dtype;
  int q_heads, kv_heads;
  float scale2;
  int splits;  // key ranges of a query block, fewer where they would fall below MIN_TILES tiles
  ReplaySide side[2];
};

// Key ranges of a query block that sees ntiles tiles.
GSE_DEVICE int replay_ranges(int ntiles, int splits) {
  const int most = (ntiles + rp::MIN_TILES - 1) / rp::MIN_TILES;
  return most < splits ? most : splits;
}
GSE_DEVICE int replay_tiles(const ReplaySide& a, int64_t count, int64_t qb0) {
  const int64_t kend = a.prefix_len + (qb0 + rp::QB < count ? qb0 + rp::QB : count);
  return int((kend + rp::KT - 1) / rp::KT);
}

// One 64-key tile for the wave's row-blocks. s[rb][kb][r] is S^T[key 16*kb + 4*grp + r][column].
// MASKED: key column t0 + 16*kb + 4*grp + r is dead for column `col`'s query when
// rel + 16*kb + r > 2*rb + col/8, with rel = t0 + 4*grp - (prefix_len + first query of the wave).
template <bool MASKED>
GSE_DEVICE void replay_tile(const bf16x8_t (&qa)[rp::RB][2], const uint16_t* kt, const uint16_t* vt,
                            float (&ref)[rp::RB], float (&lsum)[rp::RB], f32x4_t (&o)[rp::RB][4], float scale2,
                            int rel, int col, int grp) {
  using namespace rp;
  auto k_frag = [&](int kb, bf16x8_t (&f)[2]) {
    const uint16_t* kr = kt + (16 * kb + col) * KROW + 8 * grp;
    f[0] = as_bf16x8(*reinterpret_cast<const uint4*>(kr));
    f[1] = as_bf16x8(*reinterpret_cast<const uint4*>(kr + 32));
  };
  auto dot = [&](const bf16x8_t (&f)[2], int rb, int kb) {
    f32x4_t d = mfma16x16x32(f[1], qa[rb][1], mfma16x16x32(f[0], qa[rb][0], f32x4_t{0.f, 0.f, 0.f, 0.f}));
    if (MASKED)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rel + 16 * kb + r > 2 * rb + (col >> 3)) d[r] = -INFINITY;
    return d;
  };
  f32x4_t s[RB][4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    bf16x8_t kf[2];
    k_frag(kb, kf);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) s[rb][kb] = dot(kf, rb, kb);
    __builtin_amdgcn_sched_barrier(0);
  }
  uint4 hi[RB][2], lo[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    // p = 2^(x*scale2 - ref). A lane whose 16 values sum past kRescaleSum may hold one 2^8 above
    // the reference: then (rarely, wave-uniform) the reference moves to the column's maximum over
    // the tile, and the terms are formed again from the products. References are whole numbers, so
    // that what a move or the join of key ranges scales by is a power of two and exact.
    auto expo = [&]() {
      float t[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) s[rb][kb][r] = fast_exp2(fmaf(s[rb][kb][r], scale2, -ref[rb]));
        t[kb] = (s[rb][kb][0] + s[rb][kb][1]) + (s[rb][kb][2] + s[rb][kb][3]);
      }
      return (t[0] + t[1]) + (t[2] + t[3]);
    };
    float ps = expo();
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(ps <= kRescaleSum)) != 0, 0)) {
      float tmax = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        bf16x8_t kf[2];
        k_frag(kb, kf);
        s[rb][kb] = dot(kf, rb, kb);
        tmax = fmaxf(fmaxf(tmax, fmaxf(s[rb][kb][0], s[rb][kb][1])), fmaxf(s[rb][kb][2], s[rb][kb][3]));
      }
      tmax = rintf(xor32_max(xor16_max(tmax)) * scale2);  // the column's maximum over the tile (scale > 0)
      const float nr = fmaxf(ref[rb], tmax);
      const float corr = fast_exp2(ref[rb] - nr);
      ref[rb] = nr;
      lsum[rb] *= corr;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[rb][j] = o[rb][j] * corr;
      ps = expo();
    }
    lsum[rb] += ps;
    // P^T operands: half h covers key-blocks 2h and 2h + 1; k-element e maps to key-block
    // 2h + e/4, key 4*grp + e%4 (the layout of the V fragments). hi = p truncated to bf16 (v_perm of
    // the upper halves), lo = bf16(p - hi).
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t hw[4], lw[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float x0 = s[rb][2 * h + e / 4][e % 4], x1 = s[rb][2 * h + e / 4][e % 4 + 1];
        const uint32_t b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
        hw[e / 2] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        lw[e / 2] = pack_bf16x2(x0 - __uint_as_float(b0 & 0xffff0000u), x1 - __uint_as_float(b1 & 0xffff0000u));
      }
      hi[rb][h] = uint4{hw[0], hw[1], hw[2], hw[3]};
      lo[rb][h] = uint4{lw[0], lw[1], lw[2], lw[3]};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_sched_barrier(0);
  // V^T fragments of dim block j, half h: lane (dim 16*j + lane%16, group grp) holds keys
  // 32*h + 4*grp + e (e < 4) and 32*h + 16 + 4*grp + (e - 4).
  const uint16_t* vr = vt + (4 * grp + (col >> 2)) * VROW + 4 * (col & 3);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bf16x8_t va = join_bf16x8(ds_read_tr16(vr + 32 * h * VROW + 16 * j),
                                      ds_read_tr16(vr + (32 * h + 16) * VROW + 16 * j));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        o[rb][j] = mfma16x16x32(va, as_bf16x8(hi[rb][h]), o[rb][j]);
        o[rb][j] = mfma16x16x32(va, as_bf16x8(lo[rb][h]), o[rb][j]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

__global__ __launch_bounds__(64 * rp::WAVES, 4) void replay_output_kernel(ReplayArgs a) {
  using namespace rp;
  __shared__ __attribute__((aligned(16))) uint16_t ktile[2][KT * KROW];
  __shared__ __attribute__((aligned(16))) uint16_t vtile[2][KT * VROW];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  // Block i of an output: KV head i % kv_heads, then the query block, then the key range. The longer
  // half of the query blocks from the end, then the others from the front: where all run at once, two
  // per CU, the longest shares a CU with the shortest (2048 queries without a prefix: 98 -> 89 us).
  const int nqb = int((a.count + QB - 1) / QB);
  const int per_side = nqb * a.kv_heads * a.splits;
  const ReplaySide sd = int(blockIdx.x) >= per_side ? a.side[1] : a.side[0];
  const int item = blockIdx.x % per_side;
  const int g = item % a.kv_heads;
  const int split = item / a.kv_heads / nqb;
  const int order = item / a.kv_heads % nqb, half = (nqb + 1) / 2;
  const int64_t qb0 = int64_t(order < half ? nqb - 1 - order : order - half) * QB;
  const int ntiles = replay_tiles(sd, a.count, qb0);
  const int ranges = replay_ranges(ntiles, a.splits);
  if (split >= ranges) return;
  const int ti0 = int(int64_t(ntiles) * split / ranges), ti1 = int(int64_t(ntiles) * (split + 1) / ranges);
  const int i0 = int(qb0) + 2 * RB * wave;
  const int last_q = int((qb0 + QB < a.count ? qb0 + QB : a.count) - 1);
  const int kend = int(sd.prefix_len) + last_q + 1;  // columns any query of the workgroup sees
  const bool wave_live = i0 < a.count;
  const int wave_kend = int(sd.prefix_len) + min(i0 + 2 * RB - 1, int(a.count) - 1) + 1;

  // Q^T fragments: column col of row-block rb is query i0 + 2*rb + col/8, head g*8 + col%8;
  // lane group grp supplies dims [8*grp, +8) and [32 + 8*grp, +8).
  bf16x8_t qa[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int64_t qi = i0 + 2 * rb + col / 8;
    qa[rb][0] = bf16x8_t{};
    qa[rb][1] = bf16x8_t{};
    if (qi < a.count) {
      const uint16_t* qp = a.q + qi * a.q_st + int64_t(g * GROUP + col % 8) * a.q_sh + 8 * grp;
      qa[rb][0] = as_bf16x8(*reinterpret_cast<const uint4*>(qp));
      qa[rb][1] = as_bf16x8(*reinterpret_cast<const uint4*>(qp + 32));
    }
  }
  float ref[RB], lsum[RB];
  f32x4_t o[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    ref[rb] = -1e30f;  // finite: the first tile's rescale multiplies zeros by 2^(-huge) = 0
    lsum[rb] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[rb][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // Staging: thread t holds row (t/4) % 64, dims [16*(t%4), +16) of K (t < 256) or V. The next
  // tile's rows are loaded while a tile computes and stored to LDS at its end; the key rows of the
  // tile after that are read meanwhile, so no row load waits on the index load of the same tile.
  const bool stage_v = threadIdx.x >= 256;
  const int lk = (threadIdx.x >> 2) & 63, lp = threadIdx.x & 3;
  const uint16_t* src = stage_v ? a.v : a.k;
  // The retained row of column t0 + lk as loaded (unused for other columns): nothing reads it
  // until its tile's rows are loaded, so the index load is not waited for where it is issued.
  const int n_retained = int(sd.n_retained), tail0 = int(sd.tail0) - n_retained;
  auto row_at = [&](int t0) -> int32_t {
    const uint32_t c = uint32_t(t0) + lk;  // up to two tiles past kend < 2^31
    return c < uint32_t(kend) && c < uint32_t(n_retained) ? sd.retained[g * sd.ret_sg + c] : 0;
  };
  const int rows = int(a.rows < INT32_MAX ? a.rows : INT32_MAX);
  const auto base = as_global(src) + int64_t(g) * a.kv_sh + 16 * lp;
  auto load_rows = [&](int32_t retained_row, int t0, uint4 (&x)[2]) {
    const uint32_t c = uint32_t(t0) + lk;
    const int32_t row = c >= uint32_t(kend) ? 0 : c < uint32_t(n_retained) ? retained_row : tail0 + int32_t(c);
    const auto p = base + (uint32_t(row) < uint32_t(rows) ? row : 0) * a.kv_ss;
    x[0] = gload16(p);
    x[1] = gload16(p + 8);
  };
  auto store_rows = [&](int p, const uint4 (&x)[2]) {
    uint16_t* dst = stage_v ? &vtile[p][lk * VROW + 16 * lp] : &ktile[p][lk * KROW + 16 * lp];
    *reinterpret_cast<uint4*>(dst) = x[0];
    *reinterpret_cast<uint4*>(dst + 8) = x[1];
  };
  uint4 xk[2];  // rows of the next tile, in flight
  int32_t rk;   // key row of the tile after the current one (its rows not yet loaded)
  {
    const int32_t r0 = row_at(ti0 * KT);
    rk = row_at((ti0 + 1) * KT);
    load_rows(r0, ti0 * KT, xk);
    store_rows(0, xk);
  }
  // The query fragments are in registers before the walk starts: a wait for them inside the
  // loop would also wait for every load in flight at the top of each tile.
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    landed(qa[rb][0]);
    landed(qa[rb][1]);
  }
  __syncthreads();

  // One tile of the walk. The tiles every wave sees whole (below the workgroup's first query)
  // run in a loop of their own with no causal mask and no test of the wave's range (a wave
  // past the chunk's end computes columns nobody reads, with zero queries): a loop whose body
  // chooses between the masked and unmasked forms keeps each column's reference, sum and output
  // in different registers on the two sides and copies them back every tile.
  const int qpos0 = int(sd.prefix_len) + i0;  // the wave's first query's causal bound
  auto tile_step = [&](int ti, auto general, auto parity) {
    constexpr bool GENERAL = decltype(general)::value;
    constexpr int P = decltype(parity)::value;  // (ti - ti0) & 1
    const int t0 = ti * KT;
    load_rows(rk, t0 + KT, xk);
    rk = row_at(t0 + 2 * KT);
    if (!GENERAL)
      replay_tile<false>(qa, ktile[P], vtile[P], ref, lsum, o, a.scale2, 0, col, grp);
    else if (wave_live && t0 < wave_kend)
      replay_tile<true>(qa, ktile[P], vtile[P], ref, lsum, o, a.scale2, t0 + 4 * grp - qpos0, col, grp);
    if (ti + 1 < ti1) store_rows(1 - P, xk);
    __syncthreads();
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  // Tiles whole for every wave: keys up to the workgroup's first query's causal bound (an even
  // count, for the unrolled pairs).
  const int whole = int((sd.prefix_len + qb0 + 1) / KT);
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

  if (!wave_live) return;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int64_t qi = i0 + 2 * rb + (col >> 3);
    const float l = xor32_sum(xor16_sum(lsum[rb]));  // the column's sum over the four lane groups
    if (qi < a.count) {
      const int hq = g * GROUP + (col & 7);
      const int64_t at = (split * a.count + qi) * a.q_heads + hq;
      if (a.splits == 1) {
        const float sink2 = load_float_dyn(a.sinks, a.sinks_dtype, hq) * kLog2e;
        const float m = fmaxf(ref[rb], sink2), keep = fast_exp2(ref[rb] - m);
        const float inv = keep / (l * keep + fast_exp2(sink2 - m));
#pragma unroll
        for (int j = 0; j < 4; ++j) o[rb][j] = o[rb][j] * inv;
      } else if (grp == 0) {
        sd.ml[at] = float2{ref[rb], l};
      }
      float* op = sd.o + at * D + 4 * grp;
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4_t*>(op + 16 * j) = o[rb][j];
    }
  }
}

// Four output dims (piece 0..15 of 4) of head h of query i, from its key ranges and the sink: eight
// ranges' loads in flight together (a range past the last is read again with weight 0).
GSE_DEVICE float4 replay_join(const ReplayArgs& a, const ReplaySide& sd, int64_t i, int h, int piece) {
  if (a.splits == 1) return *reinterpret_cast<const float4*>(sd.o + (i * a.q_heads + h) * rp::D + 4 * piece);
  const int ranges = replay_ranges(replay_tiles(sd, a.count, i / rp::QB * rp::QB), a.splits);
  float m = -1e30f, l = 0.f;
  float4 o = {0.f, 0.f, 0.f, 0.f};
  constexpr int B = 8;
  for (int s0 = 0; s0 < ranges; s0 += B) {
    float2 ml[B];
    float4 x[B];
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int64_t at = (min(s0 + j, ranges - 1) * a.count + i) * a.q_heads + h;
      ml[j] = sd.ml[at];
      x[j] = *reinterpret_cast<const float4*>(sd.o + at * rp::D + 4 * piece);
    }
    float mn = m;
#pragma unroll
    for (int j = 0; j < B; ++j) mn = fmaxf(mn, ml[j].x);
    const float keep = fast_exp2(m - mn);
    l *= keep;
    o = {o.x * keep, o.y * keep, o.z * keep, o.w * keep};
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const float w = s0 + j < ranges ? fast_exp2(ml[j].x - mn) : 0.f;
      l += ml[j].y * w;
      o = {o.x + x[j].x * w, o.y + x[j].y * w, o.z + x[j].z * w, o.w + x[j].w * w};
    }
    m = mn;
  }
  // The sink joins last: the ranges' weights stay whole powers of two.
  const float inv = 1.f / (l + fast_exp2(load_float_dyn(a.sinks, a.sinks_dtype, h) * kLog2e - m));
  return {o.x * inv, o.y * inv, o.z * inv, o.w * inv};
}

// error[i] = |b_i - a_i| / max(|a_i|, 1e-12) over all heads and dims: a workgroup per query, 16
// threads per head. Without a second output (nothing evicted yet) the outputs coincide.
__global__ __launch_bounds__(1024) void replay_error_kernel(ReplayArgs a, int sides, float* error) {
  __shared__ float red[2][16];
  const int64_t i = blockIdx.x;
  float dd = 0.f, aa = 0.f;
  for (int t = threadIdx.x; t < a.q_heads * (rp::D / 4); t += blockDim.x) {
    const float4 x = replay_join(a, a.side[0], i, t >> 4, t & 15);
    const float4 y = sides > 1 ? replay_join(a, a.side[1], i, t >> 4, t & 15) : x;
    const float d0 = y.x - x.x, d1 = y.y - x.y, d2 = y.z - x.z, d3 = y.w - x.w;
    dd += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
    aa += (x.x * x.x + x.y * x.y) + (x.z * x.z + x.w * x.w);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    dd += __shfl_xor(dd, off, kWave);
    aa += __shfl_xor(aa, off, kWave);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = dd;
    red[1][threadIdx.x >> 6] = aa;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    dd = aa = 0.f;
    for (int w = 0; w < int(blockDim.x >> 6); ++w) {
      dd += red[0][w];
      aa += red[1][w];
    }
    error[i] = sqrtf(dd) / fmaxf(sqrtf(aa), 1e-12f);
  }
}

}  // namespace gse

using namespace gse;

static int replay_splits(int64_t count, int kv_heads) {
  const int64_t blocks = (count + rp::QB - 1) / rp::QB * kv_heads;
  return int(std::max<int64_t>(1, blocks > 0 ? rp::ITEMS / blocks : 1));
}

// One output over `splits` key ranges: the sums, then (of several ranges) the (m, l) pairs.
static int64_t replay_side_bytes(int64_t count, int q_heads, int splits) {
  const int64_t rows = splits * count * q_heads;
  return (rows * (rp::D * 4 + (splits > 1 ? int64_t(sizeof(float2)) : 0)) + 255) / 256 * 256;
}

extern "C" int64_t gse_replay_workspace_bytes(int64_t count, int q_heads) {
  return 2 * replay_side_bytes(count, q_heads, replay_splits(count, std::max(1, q_heads / rp::GROUP)));
}

extern "C" int gse_replay_layer_difference(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                                           const void* k_shadow, const void* v_shadow, int64_t kv_stride_s,
                                           int64_t kv_stride_h, int64_t shadow_rows, int64_t start,
                                           const int32_t* retained, int64_t retained_stride_g,
                                           int64_t retained_count, int64_t frontier, const void* sinks,
                                           int sinks_dtype, int q_heads, int kv_heads, int head_dim, float sm_scale,
                                           float* error, void* workspace, int64_t workspace_bytes,
                                           gse_stream_t stream) {
  if (head_dim != rp::D || kv_heads < 1 || q_heads != rp::GROUP * kv_heads)
    return gse_fail(GSE_ESHAPE, "replay: need head_dim 64 and q_heads == 8 * kv_heads");
  if (count < 0 || start < 0 || retained_count < 0 || frontier < 0)
    return gse_fail(GSE_EINVAL, "replay: negative count, start, retained_count or frontier");
  if (count == 0) return GSE_OK;
  if (retained_count > 0 && frontier > start)
    return gse_fail(GSE_EINVAL, "replay: the chunk must start at or after the frontier");
  if (shadow_rows < start + count) return gse_fail(GSE_EINVAL, "replay: the shadow must hold start + count rows");
  if (q_stride_t % 8 || q_stride_h % 8 || kv_stride_s % 8 || kv_stride_h % 8)
    return gse_fail(GSE_EINVAL, "replay: strides must be multiples of 8 elements");
  if (!q || !k_shadow || !v_shadow || !sinks || !error || (retained_count && !retained))
    return gse_fail(GSE_EINVAL, "replay: null pointer");
  if (retained_count && retained_stride_g < retained_count)
    return gse_fail(GSE_EINVAL, "replay: retained rows overlap");
  // A smaller workspace than gse_replay_workspace_bytes takes fewer key ranges; one needs the two outputs.
  int splits = replay_splits(count, kv_heads);
  while (splits > 1 && workspace_bytes < 2 * replay_side_bytes(count, q_heads, splits)) splits /= 2;
  if (workspace_bytes < 2 * replay_side_bytes(count, q_heads, splits))
    return gse_fail(GSE_EWORKSPACE, "replay: workspace too small");
  if (start + count >= (int64_t(1) << 31) || retained_count + start + count >= (int64_t(1) << 31))
    return gse_fail(GSE_EINVAL, "replay: too many keys");
  ReplayArgs a = {static_cast<const uint16_t*>(q), q_stride_t, q_stride_h, count,
                  static_cast<const uint16_t*>(k_shadow), static_cast<const uint16_t*>(v_shadow), kv_stride_s,
                  kv_stride_h, shadow_rows, sinks, sinks_dtype, q_heads, kv_heads, sm_scale * kLog2e,
                  splits, {}};
  const int sides = retained_count > 0 ? 2 : 1;
  const int64_t rows = a.splits * count * q_heads;
  for (int i = 0; i < 2; ++i) {
    a.side[i].o = reinterpret_cast<float*>(static_cast<char*>(workspace) + i * replay_side_bytes(count, q_heads, splits));
    a.side[i].ml = reinterpret_cast<float2*>(a.side[i].o + rows * rp::D);
  }
  // a: every key up to the query (columns are positions).
  a.side[0].prefix_len = start;
  // b: each head's retained positions, then positions frontier .. start + count - 1.
  a.side[1].retained = retained;
  a.side[1].ret_sg = retained_stride_g;
  a.side[1].n_retained = retained_count;
  a.side[1].tail0 = frontier;
  a.side[1].prefix_len = retained_count + start - frontier;
  const int64_t blocks = (count + rp::QB - 1) / rp::QB * kv_heads * a.splits * sides;
  if (blocks >= (int64_t(1) << 31)) return gse_fail(GSE_EINVAL, "replay: chunk too large");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(replay_output_kernel, dim3(uint32_t(blocks)), dim3(64 * rp::WAVES), 0, s, a);
  if (int rc = gse_launch_check("replay outputs")) return rc;
  const unsigned threads = unsigned(std::min(q_heads * rp::D / 4, 1024));  // a multiple of 128
  hipLaunchKernelGGL(replay_error_kernel, dim3(uint32_t(count)), dim3(threads), 0, s, a, sides, error);
  return gse_launch_check("replay error");
}
