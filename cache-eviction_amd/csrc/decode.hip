// Decode attention with sinks and the H2O score of decode queries (gfx950).
//
// decode_fused_kernel: attention over a balanced partition of the batch's keys.
//   The batch's resident keys form one range [0, T), T = indptr[bs] (the CSR
//   concatenates the sequences). Workgroup w of P takes [w*C, (w+1)*C) with
//   C = ceil(T / P), so every workgroup streams the same number of keys whatever
//   the sequence lengths; its range splits into segments at sequence ends and
//   each segment leaves one partial (o, m, l per head), slot (w + b) of the
//   partial buffer (w + b is unique: a later workgroup never starts in an
//   earlier sequence). The kernel writes nothing else, so the HBM stream it
//   drives is reads only.
//   Workgroups P.. of the launch (present when the step folds queues) add the
//   queued steps of the listed sequences' rows to the score table, with the long
//   flush's tiles (fold.hpp), while the attention workgroups stream K and V: the
//   fold is bound by its exponentials, the attention by HBM, and the attention
//   needs only part of the CUs to hold its bandwidth.
// decode_merge_kernel: folds a sequence's partials with the sink into o and the
//   normaliser, and appends the step's query, normaliser and list length to the
//   row's score queue (folded into the score table later by score_flush_kernel,
//   or by a later decode launch's fold workgroups); a queue folded by this launch
//   restarts with the step.
// decode_score_kernel: the score update of one query per sequence given its
//   final normaliser, one pass over K (GSE_SCORE_EAGER's second pass and the
//   reference's after_decode hook).
#include <algorithm>

#include "common.hpp"
#include "fold.hpp"

namespace gse {

constexpr int D = 64;        // head_dim
constexpr int GROUP = 8;     // query heads per KV head
constexpr int TILE = 64;     // keys per inner iteration (four 16-key MFMA sub-tiles)
constexpr int MAX_KVH = 8;   // waves per workgroup
constexpr int LDS_ROW = D + 16;  // padded bf16 row of the V staging tile (160 B: transposed reads spread over banks)
constexpr int KROW = D + 8;      // padded bf16 row of the K staging tile (144 B: the 16 keys an MFMA-layout read
                                 // addresses fall in distinct banks)
constexpr int PART = D + 4;     // floats per (segment, head) partial: o[64], m, l, pad (16-byte rows)
constexpr int FUSED_THREADS = 64 * MAX_KVH;
// Fold workgroups per folded row of a decode launch when the caller leaves the count to the
// library: a 63-step queue of a 32K-key row folds in about the attention's time of a batch of
// 1M keys on 32 CUs, and the attention holds its bandwidth on 192 of 256 CUs.
constexpr int FOLD_WORKGROUPS_PER_ROW = 32;

GSE_DEVICE uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

// Keys per workgroup for P workgroups over T keys (0 when T == 0).
GSE_DEVICE int fused_chunk(int T, int P) { return (T + P - 1) / P; }

// The other partition, for batches of few sequences: every workgroup's keys lie in one sequence. With
// C keys per workgroup, sequence b takes ceil(len_b / C) of them, at most P in all; lane b of a wave
// counts sequence b's. A workgroup that crosses into a second sequence starts its load pipeline again
// (some 3 us) and ends last; here the others' chunks grow by bs / P at most instead, which a stream
// bound by HBM hardly shows; and the bounds come in one vector load instead of a chain of scalar ones.
// C = ceil(T / (P - bs)) always fits. Where the even cut gives a workgroup at most one tile, a few keys
// more would cost it a second tile step (4 us): there C is one tile, or, if the lists' last tiles make
// that more than P workgroups, the cut is even (C = ceil(T / P), bounds from the lanes too).
// Replayed steps of 12 layers, cut evenly with the bounds from scalar loads -> so: 3 lists of 720 to
// 1200 keys 163 -> 137 us, 2 of 4000 181 -> 160 (202 in chunks of 66 keys), 8 of 3900 to 9200 387 ->
// 359, 16 of 2047 287 -> 269, 32 of 4097 634 -> 604, 2 of 32,765 393 -> 384. Not faster: the even cut of
// 4 lists of 16,379 keys in all 217 -> 221 (236 in chunks of 66), and lists of whole tiles, where no
// even chunk crosses (2 of 512: 122.5 -> 125.2; 560: 155 -> 130). One sequence keeps the scalar form
// (140 us against 147 at 2252 keys).
constexpr int SHARE_MAX_BS = 32;
struct Share {
  bool even;         // the even cut: workgroup w has keys [w * chunk, + chunk) of all lists
  int chunk;         // keys per workgroup
  int total;         // keys of all lists
  int start, end;    // the lane's sequence's list
  int mine, before;  // (not even) its workgroups, and those of the sequences before it
};
GSE_DEVICE Share sequence_shares(const int32_t* indptr, int bs, int P, int lane) {
  Share sh;
  sh.start = lane < bs ? indptr[lane] : 0;
  sh.end = lane < bs ? indptr[lane + 1] : 0;
  const int T = sh.total = __builtin_amdgcn_readlane(sh.end, bs - 1);
  auto cut = [&](int chunk) {  // the workgroups that chunks of this many keys take
    sh.chunk = chunk;
    sh.mine = (sh.end - sh.start + chunk - 1) / chunk;
    int upto = sh.mine;  // a scan over 32 lanes by row shifts, then lane 15's into the second row
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xf, 0xf, false);
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xf, 0xf, false);
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xf, 0xf, false);
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x118, 0xf, 0xf, false);
    upto += __builtin_amdgcn_update_dpp(0, upto, 0x142, 0xa, 0xf, false);
    sh.before = upto - sh.mine;
    return __builtin_amdgcn_readlane(upto, 31);
  };
  sh.even = false;
  const int fits = max(1, (T + P - bs - 1) / (P - bs));
  if (fits <= TILE || T > TILE * P) {
    cut(fits);
  } else if (cut(TILE) > P) {
    sh.even = true;
    sh.chunk = fused_chunk(T, P);
  }
  return sh;
}
constexpr int SHARE_MIN_WG = 8;  // workgroups per sequence: chunks grow by at most a seventh

// Largest b in [0, bs) with indptr[b] <= p (indptr non-decreasing, indptr[0] = 0 <= p).
GSE_DEVICE int seq_of(const int32_t* indptr, int bs, int p) {
  int lo = 0, hi = bs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (indptr[mid] <= p) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// Fused attention
// ---------------------------------------------------------------------------
struct FusedArgs {
  const uint16_t* q;
  int64_t q_sb, q_sh;
  const uint16_t* k;
  const uint16_t* v;
  int64_t kv_ss, kv_sh;
  const int32_t* indptr;
  const void* indices;
  float* part;  // [P + bs, q_heads, PART]
  int bs, q_heads, kv_heads;
  float scale2;  // sm_scale * log2(e)
  // Kept logits (optional): for a sequence whose row r has 0 <= lidx[r] < lrows, the raw q.k of
  // list entry c < lcap, head h = 8 * g + j goes to logits[((lidx[r] * kv_heads + g) * lcap + c) * 8 + j].
  float* logits;
  const int32_t* lidx;
  const void* rows;
  int rows_dtype;
  int lrows, lcap;
  // Attention workgroups; workgroups P.. fold the queues of the sequences fold_seq[0..n_fold)
  // (batch indices whose rows have score kind 1 or 2): this layer's entries [0, count) of
  // queue q [rows, cap, q_heads, D], norm [rows, cap, q_heads], lim [rows, cap], count [rows]
  // into scores[g * ssg + slot * sss].
  int P;
  bool whole_seq;  // workgroups by sequence_shares
  // Queue mode: the queue counts this launch advances for the merge's append (null otherwise), and
  // the rows' score words.
  int32_t* step_count;
  const int32_t* step_mode;
  const int32_t* fold_seq;
  int n_fold;
  const int32_t* mode;
  float* scores;
  int64_t ssg, sss;
  const uint16_t* qq;
  const float* qnorm;
  const int32_t* qlim;
  const int32_t* qcount;
  int cap;
  // The fold's totals: fold_buf[(i * kv_heads + g) * fold_stride + c] for list entry c <
  // fold_hdr[i] of fold sequence i (fold_stride = the launch's bound of list lengths).
  float* fold_buf;
  int* fold_hdr;
  int fold_stride;
};

// The list entries of fold sequence i that its queue scores: [0, the largest scored length),
// within the sequence's list and the totals buffer's stride; 0 when the row's kind is not 1 or 2
// or its queue is empty.
GSE_DEVICE int fold_extent(const FusedArgs& a, int i) {
  const int b = a.fold_seq[i];
  if (b < 0 || b >= a.bs) return 0;
  const int64_t row = load_index_dyn(a.rows, a.rows_dtype, b);
  const int word = a.mode[row];
  const int md = score_kind(word);
  const int m = min(a.qcount[row], a.cap);
  if ((md != 1 && md != 2) || m <= 0) return 0;
  int ext = 0;
  for (int q = 0; q < m; ++q) ext = max(ext, a.qlim[row * a.cap + q] - score_delay(word));
  ext = min(ext, a.indptr[b + 1] - a.indptr[b]);
  return min(ext, a.fold_stride);
}

// A decode launch's fold workgroups: workgroup P + f of F takes a contiguous range of the work
// items (fold sequence i, KV head g, chunk k of fl::CHUNK list entries), ordered by (i, g, k) so
// that consecutive items of a workgroup share their staged queue. An item is what one
// score_flush_kernel workgroup does, over the sequence's CSR list (fill's list of the row, of
// which every queued list is a prefix), except that its totals go to the fold buffer (4 KiB
// contiguous per item); workgroup P also writes each sequence's extent. LDS: the attention's K
// and V staging tiles.
template <typename IdxT>
GSE_DEVICE void fold_role(const FusedArgs& a, uint16_t* qs, float* ns) {
  int* lims = reinterpret_cast<int*>(ns + fl::MAX_QUEUE * fl::GROUP);
  int* pmin = lims + fl::MAX_QUEUE + 1;
  int* pmax = pmin + fl::MAX_QUEUE / 2;
  const int F = gridDim.x - a.P, f = blockIdx.x - a.P;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const IdxT* idx = static_cast<const IdxT*>(a.indices);
  // Items of fold sequence i (none for a batch index outside the launch's batch).
  auto chunks = [&](int i) {
    const int b = a.fold_seq[i];
    return b < 0 || b >= a.bs ? 0 : (a.indptr[b + 1] - a.indptr[b] + fl::CHUNK - 1) / fl::CHUNK;
  };
  int total = 0;
  for (int i = 0; i < a.n_fold; ++i) total += a.kv_heads * chunks(i);
  if (f == 0)
    for (int i = threadIdx.x; i < a.n_fold; i += blockDim.x) a.fold_hdr[i] = fold_extent(a, i);
  const int per = (total + F - 1) / F;
  const int it1 = min((f + 1) * per, total);
  int i = 0, base = 0, nch = a.n_fold > 0 ? chunks(0) : 0;
  int staged_i = -1, staged_g = -1, npairs = 0, maxlim = 0, md = 0;
  for (int it = f * per; it < it1; ++it) {
    while (it >= base + a.kv_heads * nch) {
      base += a.kv_heads * nch;
      nch = chunks(++i);
    }
    const int g = (it - base) / nch, k = (it - base) % nch;
    const int b = a.fold_seq[i];
    const int64_t row = load_index_dyn(a.rows, a.rows_dtype, b);
    if (i != staged_i || g != staged_g) {
      staged_i = i;
      staged_g = g;
      const int word = a.mode[row];
      md = score_kind(word);
      const int m = min(a.qcount[row], a.cap);
      maxlim = 0;
      if ((md == 1 || md == 2) && m > 0) {
        __syncthreads();  // the previous item's tiles have read the staged queue
        const int64_t e0 = row * a.cap;
        npairs = fold_stage(a.qq + e0 * a.q_heads * fl::D, a.qnorm + e0 * a.q_heads, a.qlim + e0, m, a.q_heads, g,
                            score_delay(word), qs, ns, lims, pmin, pmax);
        for (int q = 0; q < m; ++q) maxlim = lims[q] > maxlim ? lims[q] : maxlim;
        // Every queued list is a prefix of the current one; the clamps keep a list read within
        // the sequence and a total within the buffer whatever the queue holds (fold_extent).
        const int len = a.indptr[b + 1] - a.indptr[b];
        maxlim = min(min(maxlim, len), a.fold_stride);
      }
    }
    const int c0 = k * fl::CHUNK;
    if (c0 >= maxlim) continue;
    const int start = a.indptr[b];
    auto slot_of = [&](int c) { return int32_t(idx[start + c]); };
    const auto kp = as_global(a.k) + int64_t(g) * a.kv_sh + 8 * ((threadIdx.x & 63) >> 4);
    float* tot_row = a.fold_buf + (int64_t(i) * a.kv_heads + g) * a.fold_stride;
    auto put = [&](int c, int32_t, float tot) { tot_row[c] = tot; };
    if (md == 2)
      fold_tiles<true>(qs, ns, lims, pmin, pmax, npairs, c0, wave, maxlim, a.scale2, kp, a.kv_ss, slot_of, put);
    else
      fold_tiles<false>(qs, ns, lims, pmin, pmax, npairs, c0, wave, maxlim, a.scale2, kp, a.kv_ss, slot_of, put);
  }
}

// Advances the queue count of sequence w's row (and of sequences w + P, ...) by this step, for the
// merge to append at count - 1: the launch boundary orders it before the merge's reads, which took an
// arrival ticket per head group when the merge advanced the count itself (0.65 us per layer). A row
// whose queue this launch folds restarts in the merge instead.
GSE_DEVICE void count_steps(const FusedArgs& a, int w, int64_t row, int word) {
  if (!a.step_count || threadIdx.x != 0) return;
  for (int b = w; b < a.bs; b += a.P) {
    if (b != w) {
      row = load_index_dyn(a.rows, a.rows_dtype, b);
      word = a.step_mode[row];
    }
    const int md = score_kind(word);
    bool folded = false;
    for (int i = 0; i < a.n_fold; ++i) folded |= a.fold_seq[i] == b;
    if (scoring_kind(md) && !(folded && (md == 1 || md == 2))) atomicAdd(a.step_count + row, 1);
  }
}

// Per 64-key tile a wave (one KV head) computes S^T = K . Q^T with
// v_mfma_f32_16x16x32_bf16 ([16 keys x 16 columns] per sub-tile; columns 0-7 are
// the KV head's 8 query heads, 8-15 padding), an online softmax with a lazy
// rescale, and O^T += V^T . P^T with V transposed through LDS
// (ds_read_b64_tr_b16). Slot indices two tiles ahead and K/V rows one tile ahead
// are issued, unconditionally, before each tile's compute.
// K and V rows are read as whole 128-byte head rows, one row per 8 lanes, with
// nontemporal loads: a line split over two load instructions (the MFMA layout's
// 64 bytes of 16 keys each) has to be kept in L2 for its second reader, and
// streaming whole lines past the cache reads faster (a gather probe with this
// kernel's shape: 6.9 TB/s against 5.5-5.9 for the split form). K reaches the
// MFMA layout through a staging tile in LDS, as V reaches the transposed reads.
template <typename IdxT, bool KEEP>
__global__ __launch_bounds__(FUSED_THREADS) void decode_fused_kernel(FusedArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t vtile[MAX_KVH][TILE * LDS_ROW];
  __shared__ __attribute__((aligned(16))) uint16_t ktile[MAX_KVH][TILE * KROW];
  static_assert(sizeof(ktile) >= fl::STAGE_Q_BYTES, "a staged queue fits the K tile");
  static_assert(sizeof(vtile) >= fl::STAGE_N_BYTES + (2 * fl::MAX_QUEUE + 1) * 4, "and its scalars the V tile");
  if (int(blockIdx.x) >= a.P) {
    fold_role<IdxT>(a, &ktile[0][0], reinterpret_cast<float*>(&vtile[0][0]));
    return;
  }

  const int lane = threadIdx.x & 63;
  const int g = threadIdx.x >> 6;
  if (g >= a.kv_heads) return;
  const int col = lane & 15;
  const int grp = lane >> 4;
  const bool live_col = col < GROUP;
  const int hq = g * GROUP + (col & 7);

  // Key positions are CSR offsets (int32 in the CSR itself).
  const int P = a.P;
  const int w = blockIdx.x;
  // Workgroup w counts the step of sequence w (and w + P, ...): its row's score word is on its way
  // while the keys stream, and the count moves when they have.
  const bool counts = a.step_count && w < a.bs;
  const int64_t own_row = counts ? load_index_dyn(a.rows, a.rows_dtype, w) : 0;
  int p, p_end, b, seq_end;
  int64_t slot0 = w;  // the partial of this workgroup's segment in sequence b is slot0 + b
  auto idle = [&]() { count_steps(a, w, own_row, counts ? a.step_mode[own_row] : 0); };
  if (a.whole_seq) {
    const Share sh = sequence_shares(a.indptr, a.bs, P, lane);
    if (sh.even) {
      p = w * sh.chunk;
      p_end = min(p + sh.chunk, sh.total);
      if (p >= p_end) return idle();
      // The lists that start at or before p: the last of them holds it (lane 0's starts at 0).
      b = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < a.bs && sh.start <= p)) - 1;
      seq_end = __builtin_amdgcn_readlane(sh.end, b);
    } else {
      const uint64_t own = __builtin_amdgcn_ballot_w64(sh.before <= w && w < sh.before + sh.mine);
      if (!own) return idle();
      b = __builtin_ctzll(own);
      seq_end = __builtin_amdgcn_readlane(sh.end, b);
      p = __builtin_amdgcn_readlane(sh.start, b) + (w - __builtin_amdgcn_readlane(sh.before, b)) * sh.chunk;
      p_end = min(p + sh.chunk, seq_end);
      slot0 -= b;  // one segment: slot w
    }
  } else {
    const int T = a.indptr[a.bs];
    const int C = fused_chunk(T, P);
    p = w * C;
    p_end = p + C < T ? p + C : T;
    if (p >= p_end) return idle();
    b = seq_of(a.indptr, a.bs, p);
    seq_end = a.indptr[b + 1];
  }

  // Load i of a tile: lane l reads 16-byte piece l % 8 of the wave's head row of key 8 * i + l / 8.
  const int krow = lane >> 3, piece = lane & 7;
  const auto krs = slot_rsrc(a.k, a.kv_ss), vrs = slot_rsrc(a.v, a.kv_ss);
  const int lane_bytes = int(g * a.kv_sh * 2) + 16 * piece;
  uint16_t* vt = vtile[g];
  uint16_t* kt = ktile[g];
  const IdxT* idx = static_cast<const IdxT*>(a.indices);

  struct Tile {
    int32_t s[8];
    uint4 k[8], v[8];
  };

  const int own_word = counts ? a.step_mode[own_row] : 0;
  while (p < p_end) {
    while (seq_end <= p) seq_end = a.indptr[++b + 1];  // the next sequence, skipping empty ones
    const int s0 = p;
    const int s1 = seq_end < p_end ? seq_end : p_end;

    // B operand: column col supplies dims [8*grp, 8*grp + 8) and [32 + 8*grp, ...) of its head.
    bf16x8_t qf0 = {}, qf1 = {};
    if (live_col) {
      const uint16_t* qp = a.q + int64_t(b) * a.q_sb + int64_t(hq) * a.q_sh + 8 * grp;
      qf0 = as_bf16x8(ld16(qp));
      qf1 = as_bf16x8(ld16(qp + 32));
    }
    // This segment's kept logits: the wave's 8 heads of list entry c at lg + c * q_heads.
    // (KEEP only) A buffer resource over the wave's KV-head plane of the sequence's kept rows,
    // entries [0, lend): stores past it (lanes of groups 2/3, entries past lend, every entry when
    // lend = 0) are dropped by the buffer range check, so no store needs a branch.
    const int seq0 = a.indptr[b];
    __amdgpu_buffer_rsrc_t lrsrc = __builtin_amdgcn_make_buffer_rsrc(a.logits, 0, 0, BUFFER_RSRC_FLAGS);
    if (KEEP) {
      const int kept = __builtin_amdgcn_readfirstlane(a.lidx[load_index_dyn(a.rows, a.rows_dtype, b)]);
      const bool on = kept >= 0 && kept < a.lrows;
      const int lend = on ? (s1 - seq0 < a.lcap ? s1 - seq0 : a.lcap) : 0;
      // Uniform by construction; readfirstlane lets the compiler keep the descriptor in scalar
      // registers (it cannot prove the CSR bounds uniform).
      const uint64_t base = uint64_t(a.logits + (on ? (int64_t(kept) * a.q_heads + g * GROUP) * a.lcap : 0));
      const uint64_t sbase = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(base)))) |
                             uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(base >> 32)))) << 32;
      lrsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(sbase), 0,
                                                __builtin_amdgcn_readfirstlane(lend * GROUP * 4), BUFFER_RSRC_FLAGS);
    }
    float m_run = -INFINITY, l_run = 0.f;
    f32x4_t oacc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) oacc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // Slot of key i (BUFFER_NO_INDEX past the segment: its row loads read zeros from no
    // memory); every lane issues the index load, so every path issues the same loads.
    auto slot_at = [&](int i) -> int32_t {
      const int32_t s = int32_t(idx[i < s1 ? i : s1 - 1]);
      return i < s1 ? s : BUFFER_NO_INDEX;
    };
    auto issue_rows = [&](Tile& X) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        X.k[i] = buffer_load16_nt(krs, X.s[i], lane_bytes);
        X.v[i] = buffer_load16_nt(vrs, X.s[i], lane_bytes);
      }
    };

    auto compute = [&](int t, Tile& X) {
      const int tb = s0 + t * TILE;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        *reinterpret_cast<uint4*>(vt + (8 * i + krow) * LDS_ROW + 8 * piece) = X.v[i];
        *reinterpret_cast<uint4*>(kt + (8 * i + krow) * KROW + 8 * piece) = X.k[i];
      }
      __builtin_amdgcn_wave_barrier();
      // K in the MFMA layout: lane (col, grp) holds dims [8*grp, +8) and [32 + 8*grp, +8) of
      // key 16*st + col.
      uint4 kf[4][2];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        kf[st][0] = *reinterpret_cast<const uint4*>(kt + (16 * st + col) * KROW + 8 * grp);
        kf[st][1] = *reinterpret_cast<const uint4*>(kt + (16 * st + col) * KROW + 32 + 8 * grp);
      }
      // sc[st][r]: logit (unscaled) of key tb + 16*st + 4*grp + r against column col.
      f32x4_t sc[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
        acc = mfma16x16x32(as_bf16x8(kf[st][0]), qf0, acc);
        sc[st] = mfma16x16x32(as_bf16x8(kf[st][1]), qf1, acc);
      }
      if (KEEP) {
        // Kept logits: Q . K^T with the operands swapped, so a lane of groups 0/1 holds heads
        // 4*grp..4*grp+3 of key 16*st + col (the products the score flush forms from the queued
        // query) and stores them as one 16-byte piece of the key's 32-byte row in the wave's
        // KV-head plane: a store instruction writes 512 contiguous bytes. Every lane issues its
        // store (out of range where nothing is kept), so the compiler's load waits stay exact.
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          f32x4_t d = mfma16x16x32(qf0, as_bf16x8(kf[st][0]), f32x4_t{0.f, 0.f, 0.f, 0.f});
          d = mfma16x16x32(qf1, as_bf16x8(kf[st][1]), d);
          const int c = tb - seq0 + 16 * st + col;
          const int off = grp < 2 ? (c * GROUP + 4 * grp) * 4 : BUFFER_OUT_OF_RANGE;
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, d), lrsrc, off, 0, 0);
        }
      }
      if (tb + TILE > s1) {  // the segment's last tile: keys past its end take no mass
        const int lim = s1 - tb;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * st + 4 * grp + r >= lim) sc[st][r] = -INFINITY;
      }
      float tmax = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                         fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
      tmax = fmaxf(tmax, fmaxf(fmaxf(fmaxf(sc[2][0], sc[2][1]), fmaxf(sc[2][2], sc[2][3])),
                               fmaxf(fmaxf(sc[3][0], sc[3][1]), fmaxf(sc[3][2], sc[3][3]))));
      tmax = xor32_max(xor16_max(tmax)) * a.scale2;  // log2 units (scale > 0)
      // Lazy rescale: keep the reference unless some head's tile maximum exceeds it by more
      // than 2^8 (exact: O and l share the reference).
      if (__any(tmax > m_run + 8.f)) {
        const float m_new = fmaxf(m_run, tmax);
        const float corr = fast_exp2(m_run - m_new);
        m_run = m_new;
        l_run *= corr;
#pragma unroll
        for (int j = 0; j < 4; ++j) oacc[j] = oacc[j] * corr;
      }
      float psum = 0.f;
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[st][r] = fast_exp2(fmaf(sc[st][r], a.scale2, -m_run));
          psum += sc[st][r];
        }
      l_run += psum;
      // P^T operands: half 0 covers sub-tiles 0/1, half 1 sub-tiles 2/3; k-element e maps to
      // sub-tile 2*half + e/4, key 4*grp + e%4.
      uint4 pa, pb;
      pa.x = pack_bf16x2(sc[0][0], sc[0][1]);
      pa.y = pack_bf16x2(sc[0][2], sc[0][3]);
      pa.z = pack_bf16x2(sc[1][0], sc[1][1]);
      pa.w = pack_bf16x2(sc[1][2], sc[1][3]);
      pb.x = pack_bf16x2(sc[2][0], sc[2][1]);
      pb.y = pack_bf16x2(sc[2][2], sc[2][3]);
      pb.z = pack_bf16x2(sc[3][0], sc[3][1]);
      pb.w = pack_bf16x2(sc[3][2], sc[3][3]);
      __builtin_amdgcn_wave_barrier();
      // Lanes of group grp read the V^T fragments of keys 32*half + 16*h + 4*grp + e at dims
      // 16*j + 4*(lane%4) (ds_read_b64_tr_b16).
      const uint16_t* vr = vt + (4 * grp + ((lane & 15) >> 2)) * LDS_ROW + 4 * (lane & 3);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const s16x4_t a0 = ds_read_tr16(vr + 16 * j);
        const s16x4_t a1 = ds_read_tr16(vr + 16 * LDS_ROW + 16 * j);
        const s16x4_t b0 = ds_read_tr16(vr + 32 * LDS_ROW + 16 * j);
        const s16x4_t b1 = ds_read_tr16(vr + 48 * LDS_ROW + 16 * j);
        oacc[j] = mfma16x16x32(join_bf16x8(a0, a1), as_bf16x8(pa), oacc[j]);
        oacc[j] = mfma16x16x32(join_bf16x8(b0, b1), as_bf16x8(pb), oacc[j]);
      }
      __builtin_amdgcn_wave_barrier();
    };

    const int ntiles = (s1 - s0 + TILE - 1) / TILE;
    Tile A, B;
    int32_t s_ahead[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      A.s[i] = slot_at(s0 + 8 * i + krow);
      B.s[i] = slot_at(s0 + TILE + 8 * i + krow);
    }
    issue_rows(A);
    // Per step: slots two tiles ahead and rows one tile ahead are issued before the compute.
    // Past the segment the loads are issued with no index (the range check drops them) instead
    // of branching around them.
    auto step = [&](int t, Tile& X, Tile& Y) {
      const int tb = s0 + t * TILE;
#pragma unroll
      for (int i = 0; i < 8; ++i) s_ahead[i] = slot_at(tb + 2 * TILE + 8 * i + krow);
      issue_rows(Y);
      // Keep the loads above the compute: the scheduler would otherwise sink them below it
      // and expose their latency at the next step.
      __builtin_amdgcn_sched_barrier(0);
      compute(t, X);
#pragma unroll
      for (int i = 0; i < 8; ++i) X.s[i] = s_ahead[i];
    };
    // Both steps in every iteration, the odd last tile peeled: no path through the loop
    // skips a step's loads, so the compiler's wait counts stay exact.
    int t = 0;
    for (; t + 1 < ntiles; t += 2) {
      step(t, A, B);
      step(t + 1, B, A);
    }
    if (t < ntiles) step(t, A, B);

    // This segment's partial: O^T rows 4*grp + r of dim block j, column col; m and l.
    const float lt = xor32_sum(xor16_sum(l_run));
    if (live_col) {
      float* pp = a.part + ((slot0 + b) * a.q_heads + hq) * PART;
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4_t*>(pp + 16 * j + 4 * grp) = oacc[j];
      if (grp == 0) {
        pp[D] = m_run;
        pp[D + 1] = lt;
      }
    }
    p = s1;
  }
  count_steps(a, w, own_row, own_word);
}

// ---------------------------------------------------------------------------
// Merge of the partials, and the score queue
// ---------------------------------------------------------------------------
struct MergeArgs {
  const float* part;
  const int32_t* indptr;
  const void* sinks;
  int sinks_dtype;
  uint16_t* o;
  int64_t o_sb, o_sh;
  float* norm_out;  // [bs, q_heads]
  // Score queue (GSE_SCORE_QUEUE): for rows whose score mode is 1 or 2, entry n = qcount[row] - 1
  // (the fused kernel has counted the step) gets its query, normaliser and list length if n < cap (a
  // count above cap records dropped steps).
  const uint16_t* q;
  int64_t q_sb, q_sh;
  const int32_t* mode;
  const void* rows;
  int rows_dtype;
  uint16_t* qq;     // [rows, cap, q_heads, D]
  float* qnorm;     // [rows, cap, q_heads]
  int32_t* qlim;    // [rows, cap]
  int32_t* qcount;  // [rows]
  int cap;
  int bs, q_heads, nparts;  // nparts = P, the fused kernel's attention workgroup count
  bool whole_seq;           // its workgroups by sequence_shares
  // Sequences whose queue the fused kernel folded (score kinds 1 and 2): their step goes to
  // entry 0 and their count becomes 1, and their totals (the fused kernel's fold_buf / fold_hdr,
  // over the CSR list `indices`) are added to scores[g * ssg + slot * sss].
  const int32_t* fold_seq;
  int n_fold;
  const float* fold_buf;
  const int* fold_hdr;
  int fold_stride, kv_heads;
  int head_groups;  // merging grid rows (q_heads / HEADS); rows past them scatter the fold's totals
  const void* indices;
  int indices_dtype;
  float* scores;
  int64_t ssg, sss;
};

// The fold's totals added to the scores by the merge launch's scatter workgroups (grid rows
// y >= head_groups, beside the merging ones): of their T threads, thread t takes the fold
// sequences' list entries t, t + T, ... in order, one read-modify-write of a slot's kv_heads
// scores per entry (each (slot, head) has one total: the result equals one atomic add each). The
// fused kernel has finished, so these writes meet no attention stream.
GSE_DEVICE void fold_scatter(const MergeArgs& a) {
  const int T = gridDim.x * (gridDim.y - a.head_groups) * blockDim.x;
  int i = 0, base = 0, ext = a.fold_hdr[0];
  for (int e = ((blockIdx.y - a.head_groups) * gridDim.x + blockIdx.x) * blockDim.x + threadIdx.x;; e += T) {
    while (e >= base + ext) {
      base += ext;
      if (++i >= a.n_fold) return;
      ext = a.fold_hdr[i];
    }
    const int c = e - base;
    const int64_t slot = load_index_dyn(a.indices, a.indices_dtype, a.indptr[a.fold_seq[i]] + c);
    float* sp = a.scores + slot * a.sss;
    const float* tp = a.fold_buf + int64_t(i) * a.kv_heads * a.fold_stride + c;
    for (int g = 0; g < a.kv_heads; ++g) sp[g * a.ssg] += tp[int64_t(g) * a.fold_stride];
  }
}

// Grid (bs, q_heads / HEADS, plus MERGE_SCATTER_ROWS rows that run fold_scatter when the launch
// folded queues), 16 * HEADS * SPLIT threads: thread (head HEADS*y + t/16, dims [4*(t%16), +4))
// of partial group k = t / (16 * HEADS) merges every SPLIT-th batch of the sequence's partials
// of its head, group 0 starting from the sink:
//   o = sum_w 2^(m_w - M) o_w / (2^(sink - M) + sum_w 2^(m_w - M) l_w), M the maximum,
// MERGE_BATCH partials at a time with all their loads in flight together (a partial past
// the range is read again with weight 0), one rescale of the running sums per batch; with
// SPLIT > 1 (few sequences, each spread over many workgroups) the groups' (m, l, o) are then
// folded through LDS (SPLIT = 64: groups 8i fold groups 8i..8i+7, then group 0 folds those
// eight), so a sequence's partials cost ceil(count / (8 * SPLIT)) rounds of loads. Instances:
// <1, 8> for batches whose sequences span at most 8 workgroups, <8, 8> up to 64, <64, 1> past
// that (a single long sequence: one head per workgroup, 64 groups).
constexpr int MERGE_BATCH = 8;
constexpr int MERGE_SCATTER_ROWS = 8;  // grid rows of the merge launch that scatter the fold's totals
template <int SPLIT, int HEADS>
__global__ __launch_bounds__(16 * HEADS * SPLIT) void decode_merge_kernel(MergeArgs a) {
  constexpr int MERGE_THREADS = 16 * HEADS;
  __shared__ float red_m[SPLIT][MERGE_THREADS], red_l[SPLIT][MERGE_THREADS];
  __shared__ f32x4_t red_o[SPLIT][MERGE_THREADS];
  if (int(blockIdx.y) >= a.head_groups) {  // a scatter workgroup (launched only with folds)
    fold_scatter(a);
    return;
  }
  const int b = blockIdx.x;
  const int t = threadIdx.x % MERGE_THREADS;
  const int grp = threadIdx.x / MERGE_THREADS;
  const int h = blockIdx.y * HEADS + (t >> 4);
  const int j = t & 15;
  // Independent loads first: the queue slot (row -> mode, count) and the partial range
  // (indptr) are two short chains issued together.
  int64_t row = 0;
  int slot = 0;
  bool queue = false, folded = false;
  if (a.qq) {
    row = load_index_dyn(a.rows, a.rows_dtype, b);
    const int md = score_kind(a.mode[row]);
    slot = a.qcount[row] - 1;  // the fused kernel has counted the step
    queue = scoring_kind(md);
    bool listed = false;
    for (int i = 0; i < a.n_fold; ++i) listed |= a.fold_seq[i] == b;
    folded = listed && (md == 1 || md == 2);
    if (folded) slot = 0;
  }
  const bool live = h < a.q_heads;
  const int hh = live ? h : 0;
  const uint2 qv = *reinterpret_cast<const uint2*>(a.q + int64_t(b) * a.q_sb + int64_t(hh) * a.q_sh + 4 * j);
  const int start = a.indptr[b], end = a.indptr[b + 1];
  int wf = 1, wl = 0, slot0 = b;  // workgroup w's partial of this sequence is slot0 + w
  int C = 0;  // keys per workgroup of the even cut
  if (a.whole_seq) {
    const Share sh = sequence_shares(a.indptr, a.bs, a.nparts, threadIdx.x & 63);
    if (sh.even) {
      C = sh.chunk;
    } else {
      wf = __builtin_amdgcn_readlane(sh.before, b);
      wl = wf + __builtin_amdgcn_readlane(sh.mine, b) - 1;
      slot0 = 0;
    }
  } else if (end > start) {
    C = fused_chunk(a.indptr[a.bs], a.nparts);
  }
  if (C && end > start) {
    wf = start / C;
    wl = (end - 1) / C;
  }
  float mx = grp == 0 ? load_float_dyn(a.sinks, a.sinks_dtype, hh) * kLog2e : -INFINITY;
  float lsum = grp == 0 ? 1.f : 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int w0 = wf + grp * MERGE_BATCH; w0 <= wl; w0 += SPLIT * MERGE_BATCH) {
    float pm[MERGE_BATCH], pl[MERGE_BATCH];
    f32x4_t po[MERGE_BATCH];
#pragma unroll
    for (int k = 0; k < MERGE_BATCH; ++k) {
      const int w = w0 + k <= wl ? w0 + k : wl;
      const float* ps = a.part + ((int64_t(w) + slot0) * a.q_heads + hh) * PART;
      pm[k] = w0 + k <= wl ? ps[D] : -INFINITY;
      pl[k] = ps[D + 1];
      po[k] = *reinterpret_cast<const f32x4_t*>(ps + 4 * j);
    }
    float m_new = mx;
#pragma unroll
    for (int k = 0; k < MERGE_BATCH; ++k) m_new = fmaxf(m_new, pm[k]);
    const float so = fast_exp2(mx - m_new);  // 0 for a group still at -inf
    lsum *= so;
    acc = acc * so;
#pragma unroll
    for (int k = 0; k < MERGE_BATCH; ++k) {
      const float sk = fast_exp2(pm[k] - m_new);
      lsum += pl[k] * sk;
      acc += po[k] * sk;
    }
    mx = m_new;
  }
  // Folds groups first, first + step, ... (count of them) of LDS into this thread's (mx, lsum, acc).
  auto fold = [&](int first, int step, int count) {
    float m = -INFINITY;
    for (int k = 0; k < count; ++k) m = fmaxf(m, red_m[first + k * step][t]);
    lsum = 0.f;
    acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < count; ++k) {
      // 0 for a group at -inf (one that merged no partial), also when every group is
      const float sk = m == -INFINITY ? 0.f : fast_exp2(red_m[first + k * step][t] - m);
      lsum += red_l[first + k * step][t] * sk;
      acc += red_o[first + k * step][t] * sk;
    }
    mx = m;
  };
  if (SPLIT > 1) {
    red_m[grp][t] = mx;
    red_l[grp][t] = lsum;
    red_o[grp][t] = acc;
    __syncthreads();
    if (SPLIT > 8) {  // groups 8i fold eight each, then group 0 folds those
      if (grp % 8 == 0) {
        fold(grp, 1, 8);
        red_m[grp][t] = mx;
        red_l[grp][t] = lsum;
        red_o[grp][t] = acc;
      }
      __syncthreads();
      if (grp == 0) fold(0, 8, SPLIT / 8);  // group 0's sink keeps the maximum finite
    } else if (grp == 0) {
      fold(0, 1, SPLIT);
    }
  }
  if (live && grp == 0) {
    const float inv = 1.f / lsum;
    uint2 out;
    out.x = pack_bf16x2(acc[0] * inv, acc[1] * inv);
    out.y = pack_bf16x2(acc[2] * inv, acc[3] * inv);
    *reinterpret_cast<uint2*>(a.o + int64_t(b) * a.o_sb + int64_t(h) * a.o_sh + 4 * j) = out;
    const float norm = (mx + __log2f(lsum)) * kLn2;
    if (j == 0) a.norm_out[int64_t(b) * a.q_heads + h] = norm;
    if (queue && slot < a.cap) {
      const int64_t e = row * a.cap + slot;
      *reinterpret_cast<uint2*>(a.qq + (e * a.q_heads + h) * D + 4 * j) = qv;
      if (j == 0) a.qnorm[e * a.q_heads + h] = norm;
      if (threadIdx.x == 0 && blockIdx.y == 0) a.qlim[e] = end - start;
    }
  }
  if (folded && threadIdx.x == 0 && blockIdx.y == 0) a.qcount[row] = 1;  // the folded queue restarts
}

// ---------------------------------------------------------------------------
// Score of one query per sequence given its final normaliser
// ---------------------------------------------------------------------------
struct ScoreArgs {
  const uint16_t* q;
  int64_t q_sb, q_sh;
  const uint16_t* k;
  int64_t kv_ss, kv_sh;
  const int32_t* indptr;
  const void* indices;
  const float* norm;  // [bs, q_heads], natural log; null: from the split log-sum-exps below
  const int32_t* mode;
  const void* rows;
  int rows_dtype;
  float* scores;
  int64_t scores_sg, scores_ss;
  int kv_heads, q_heads, bs;
  float scale2;
  // An external kernel's split log-sum-exps (R:180-188): split i of sequence b covers keys
  // [i * per, +per), per = its length over num_splits[b], rounded up to min_kv.
  const float* lse;
  int64_t lse_sb, lse_sh;
  const int32_t* num_splits;
  const void* sinks;
  int sinks_dtype;
  int max_kv_splits, min_kv;
};

constexpr int SCORE_TILE = 64;  // keys per tile of decode_score_kernel: blocks of kind 4 lie within one
// Workgroups per CU: the two that fit at its registers (8 waves of 92). More of them wait for a
// second round: 29.0 us at 2, 31.9 at 4, 37.4 at 8 (8 lists, 115 MB), and 4 per CU in 64 registers
// 45.5 us.
constexpr int SCORE_WG_PER_CU = 2;

// Normaliser (natural log, sink included) of the wave's heads g*8 + lane/8 of sequence b, whose
// list holds len keys, from its split log-sum-exps: eight lanes per head.
GSE_DEVICE float norm_from_lse(const ScoreArgs& a, int b, int g, int len) {
  const int lane = threadIdx.x & 63;
  const int h = g * GROUP + (lane >> 3);
  const int splits = a.num_splits[b];
  const int64_t per = ((int64_t(len) + splits - 1) / splits + a.min_kv - 1) / a.min_kv * a.min_kv;
  const float* lse = a.lse + int64_t(b) * a.lse_sb + int64_t(h) * a.lse_sh;
  const float sink = load_float_dyn(a.sinks, a.sinks_dtype, h);
  auto at = [&](int i) { return i < a.max_kv_splits && i * per < len ? lse[i] : -INFINITY; };
  const float x0 = at(lane & 7), x1 = at((lane & 7) + 8);
  float m = fmaxf(sink, fmaxf(x0, x1));
  for (int i = (lane & 7) + 16; i < a.max_kv_splits; i += 8) m = fmaxf(m, at(i));
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) m = wave_max_xor(m, o);
  float s = expf(x0 - m) + expf(x1 - m);
  for (int i = (lane & 7) + 16; i < a.max_kv_splits; i += 8) s += expf(at(i) - m);
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) s = wave_sum_xor(s, o);
  return m + logf(s + expf(sink - m));
}

// Grid of P workgroups of 512 threads: the batch's lists, cut into 64-key tiles, are one range of
// tiles; workgroup w takes the w-th P-th of it (equal shares whatever the lengths; the host knows
// only an upper bound of them). Wave g = KV head g: per 16 keys, Sp = Q . K^T ([16 heads x 16 keys],
// heads 8-15 padding), so a lane holds 4 heads of one key: sum / max over heads is in-lane plus one
// lane swap. The waves' totals of a tile meet in LDS and thread (key, head) adds one to the score
// table: a key's heads are one 32-byte row there, read and written once instead of once per wave.
// Kind 4 (block counters): per key the maximum over the KV heads and per block the maximum over its
// keys (lane swaps: blocks of at most 64 entries are aligned lane groups of a wave), added to KV
// head 0's score of the block's first slot.
// Bound by HBM where a batch exceeds the 256 MB last-level cache: 32 lists, 1.1 GB: 375 -> 237 us with the
// clearing of the new slots (a kernel of its own for the normalisers, workgroups sized by the batch's
// longest possible list, a wave's share of a score row at a time), 4.6 TB/s. 8 lists of 4 to 18 thousand
// keys (115 MB): 52.8 -> 36.1 us among other batches (four in turn), 47.3 -> 29.1 us over the same one.
template <typename IdxT>
__global__ __launch_bounds__(512) void decode_score_kernel(ScoreArgs a) {
  __shared__ float totals[2][SCORE_TILE][MAX_KVH + 1];
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15;
  const int grp = lane >> 4;
  const bool live_wave = g < a.kv_heads;
  auto tiles_of = [&](int b) { return (a.indptr[b + 1] - a.indptr[b] + SCORE_TILE - 1) / SCORE_TILE; };
  // The batch's tiles (64 sequences at a time, a scan over the lanes), then this workgroup's first
  // sequence and the tiles before it.
  int tiles = 0;
  for (int b0 = 0; b0 < a.bs; b0 += kWave) {
    int n = b0 + lane < a.bs ? tiles_of(b0 + lane) : 0;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) n += __shfl_xor(n, o, kWave);
    tiles += n;
  }
  int t = int(int64_t(tiles) * blockIdx.x / gridDim.x);
  const int t_end = int(int64_t(tiles) * (blockIdx.x + 1) / gridDim.x);
  if (t >= t_end) return;
  int b = 0, before = 0;  // sequence b's first tile is `before`
  for (int b0 = 0;; b0 += kWave) {
    const int n = b0 + lane < a.bs ? tiles_of(b0 + lane) : 0;
    int upto = n;  // tiles of the sequences b0 .. b0 + lane
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int below = __shfl_up(upto, o, kWave);
      if (lane >= o) upto += below;
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64(before + upto > t);
    if (past) {  // t < tiles: some chunk of 64 sequences holds it
      const int l = __builtin_ctzll(past);
      b = b0 + l;
      before += __shfl(upto - n, l, kWave);
      break;
    }
    before += __shfl(upto, kWave - 1, kWave);
  }
  b = __builtin_amdgcn_readfirstlane(b);
  before = __builtin_amdgcn_readfirstlane(before);

  int parity = 0;
  for (; t < t_end; ++b) {
    const int n = tiles_of(b);
    const int t1 = min(t_end, before + n);  // this workgroup's tiles of sequence b: [t, t1)
    const int64_t row = load_index_dyn(a.rows, a.rows_dtype, b);
    const int word = a.mode[row];
    const int md = score_kind(word);
    const int base = a.indptr[b];
    const int full = a.indptr[b + 1] - base;
    const bool blocks = md == GSE_SCORE_KIND_BLOCK_STEP;
    // Keys the query scores.
    const int len = !scoring_kind(md) ? 0
                    : blocks          ? block_step_limit(full, score_delay(word), score_block_shift(word))
                                      : full - score_delay(word);
    const int first = (t - before) * SCORE_TILE;
    const int last = min((t1 - before) * SCORE_TILE, len);  // this workgroup's keys: [first, last)
    t = t1;
    before += n;
    if (first >= last) continue;
    const bool max_mode = md != 1;
    const IdxT* idx = static_cast<const IdxT*>(a.indices) + base;

    // A rows: heads g*8 + col (zero for col >= 8), dims [8*grp, +8) and [32 + 8*grp, +8).
    bf16x8_t qa0 = {}, qa1 = {};
    if (live_wave && col < GROUP) {
      const uint16_t* qp = a.q + int64_t(b) * a.q_sb + int64_t(g * GROUP + col) * a.q_sh + 8 * grp;
      qa0 = as_bf16x8(ld16(qp));
      qa1 = as_bf16x8(ld16(qp + 32));
    }
    // Normalisers of this lane's rows (heads 4*grp + r; rows 8-15 padding, probability 0).
    f32x4_t nrm = {INFINITY, INFINITY, INFINITY, INFINITY};
    if (live_wave && a.lse) {
      const float own = norm_from_lse(a, b, g, full) * kLog2e;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = __shfl(own, 8 * ((4 * grp + r) & 7), kWave);
        if (grp < 2) nrm[r] = x;
      }
    } else if (live_wave && grp < 2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) nrm[r] = a.norm[int64_t(b) * a.q_heads + g * GROUP + 4 * grp + r] * kLog2e;
    }
    const uint16_t* kbase = a.k + int64_t(live_wave ? g : 0) * a.kv_sh + 8 * grp;

    for (int t0 = first; t0 < last; t0 += SCORE_TILE, parity ^= 1) {
      // The tile's slot indices load together, then its K rows and old scores. A list holds each
      // slot once, so no two keys share a score.
      int32_t sl[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) sl[e] = int32_t(idx[min(t0 + 16 * e + col, last - 1)]);
      const int mine = threadIdx.x >> 3, h = threadIdx.x & 7;  // this thread's (key, KV head) of the tile
      const uint64_t my_slot = uint32_t(int32_t(idx[min(t0 + mine, last - 1)]));
      uint4 kl[4], kh[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint16_t* kp = kbase + uint64_t(uint32_t(sl[e])) * uint64_t(a.kv_ss);
        kl[e] = ld16(kp);
        kh[e] = ld16(kp + 32);
      }
      const bool adds = !blocks && h < a.kv_heads && t0 + mine < last;
      float* mp = a.scores + int64_t(h) * a.scores_sg + my_slot * a.scores_ss;
      const float old = adds ? *mp : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f32x4_t d = {0.f, 0.f, 0.f, 0.f};
        d = mfma16x16x32(qa0, as_bf16x8(kl[e]), d);
        d = mfma16x16x32(qa1, as_bf16x8(kh[e]), d);
        // Heads 0-3 (group 0) with heads 4-7 (group 1); groups 2, 3 carry padding (exactly 0). The
        // largest probability is 2^(largest exponent): max mode takes one exponential.
        float tot;
        if (max_mode) {
          const float y = fmaxf(fmaxf(fmaf(d[0], a.scale2, -nrm[0]), fmaf(d[1], a.scale2, -nrm[1])),
                                fmaxf(fmaf(d[2], a.scale2, -nrm[2]), fmaf(d[3], a.scale2, -nrm[3])));
          tot = fast_exp2(xor16_max(y));
        } else {
          const float u0 = fast_exp2(fmaf(d[0], a.scale2, -nrm[0]));
          const float u1 = fast_exp2(fmaf(d[1], a.scale2, -nrm[1]));
          const float u2 = fast_exp2(fmaf(d[2], a.scale2, -nrm[2]));
          const float u3 = fast_exp2(fmaf(d[3], a.scale2, -nrm[3]));
          tot = xor16_sum((u0 + u1) + (u2 + u3));
        }
        if (live_wave && grp == 0) totals[parity][16 * e + col][g] = tot;
      }
      // Two buffers: a wave writes this one again only past the next tile's barrier, which every
      // thread reaches after its reads here.
      __syncthreads();
      if (blocks) {
        if (g == 0) {
          const int shift = score_block_shift(word);
          // last - t0 is a multiple of the block, so a block's lanes are all live or all idle.
          const bool live = t0 + lane < last;
          float m = 0.f;
          if (live)
            for (int k = 0; k < a.kv_heads; ++k) m = fmaxf(m, totals[parity][lane][k]);
          for (int o = 1; o < (1 << shift); o <<= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
          if (live && (lane & ((1 << shift) - 1)) == 0)
            a.scores[uint64_t(uint32_t(int32_t(idx[t0 + lane]))) * a.scores_ss] += m;
        }
      } else if (adds) {
        *mp = old + totals[parity][mine][h];
      }
    }
  }
}

// gse_decode_noalloc's partials and normalisers: one copy per GPU, held until the process ends.
// In host code the name is a stand-in, not a device address: the library passes kernels the
// address hipGetSymbolAddress gives for the current device (noalloc_scratch).
static __device__ __align__(256) float scratch[GSE_DECODE_NOALLOC_SCRATCH_BYTES / sizeof(float)];

}  // namespace gse

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
#include <cstdio>
#include <mutex>

#include "host.hpp"

using namespace gse;

namespace {

// Workgroups of the fused kernel: one per compute unit of the current device.
int fused_workgroups() { return gse_device_cus(); }

int check_decode_shape(int q_heads, int kv_heads, int head_dim) {
  if (head_dim != D) return gse_fail(GSE_ESHAPE, "decode: head_dim must be 64");
  if (kv_heads < 1 || kv_heads > MAX_KVH || q_heads != GROUP * kv_heads)
    return gse_fail(GSE_ESHAPE, "decode: need q_heads == 8 * kv_heads and 1 <= kv_heads <= 8");
  return GSE_OK;
}

// One score-only pass over K; max_len bounds every sequence's length.
int score_pass(const ScoreArgs& s, int indices_dtype, int max_len, hipStream_t stream) {
  const int64_t tiles = int64_t(s.bs) * ((int64_t(std::max(max_len, 0)) + SCORE_TILE - 1) / SCORE_TILE);
  if (tiles <= 0) return GSE_OK;
  const int64_t blocks = std::min(tiles, SCORE_WG_PER_CU * int64_t(fused_workgroups()));
  const dim3 grid{static_cast<uint32_t>(blocks)}, block{FUSED_THREADS};
  if (indices_dtype == GSE_I64)
    hipLaunchKernelGGL(decode_score_kernel<int64_t>, grid, block, 0, stream, s);
  else
    hipLaunchKernelGGL(decode_score_kernel<int32_t>, grid, block, 0, stream, s);
  return gse_launch_check("decode_score");
}

}  // namespace

extern "C" int64_t gse_decode_workspace_bytes(int bs, int q_heads, int head_dim) {
  // Fused-kernel partials (one per workgroup-sequence segment: at most P + bs of them) and
  // the per-head normalisers.
  const int64_t parts = int64_t(fused_workgroups()) + bs;
  return parts * q_heads * (head_dim + 4) * int64_t(sizeof(float)) + int64_t(bs) * q_heads * 4;
}

extern "C" int64_t gse_decode_fold_bytes(int n_fold, int kv_heads, int max_len) {
  if (n_fold <= 0) return 0;
  // The extents (n_fold ints, 256-byte aligned), then the totals [n_fold, kv_heads, max_len].
  return (int64_t(n_fold) * 4 + 255) / 256 * 256 + int64_t(n_fold) * kv_heads * std::max(max_len, 1) * 4;
}

namespace {

// The decode launches over a workspace of at least gse_decode_workspace_bytes(bs, ...) bytes
// (the caller's, or the library's scratch); shapes and bs > 0 are checked by the caller.
int decode_run(const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* k_pool, const void* v_pool,
               int64_t kv_stride_s, int64_t kv_stride_h, const int32_t* kv_indptr, const void* kv_indices,
               int indices_dtype, const void* sinks, int sinks_dtype, const int32_t* mode_by_row, const void* rows,
               int rows_dtype, float* scores, int64_t scores_stride_g, int64_t scores_stride_s, void* o,
               int64_t o_stride_b, int64_t o_stride_h, float* norm_out, void* queue_q, float* queue_norm,
               int32_t* queue_lim, int32_t* queue_count, int queue_cap, int bs, int q_heads, int kv_heads,
               float sm_scale, int max_len, int score_mode, float* logits, const int32_t* logit_index,
               int logit_rows, int logit_cap, const int32_t* fold_seq, int n_fold, int fold_workgroups,
               void* workspace, gse_stream_t stream) {
  if (!q || !k_pool || !v_pool || !kv_indptr || !kv_indices || !sinks || !o)
    return gse_fail(GSE_EINVAL, "decode: null pointer");
  if (score_mode < GSE_SCORE_NONE || score_mode > GSE_SCORE_QUEUE) return gse_fail(GSE_EINVAL, "decode: bad score_mode");
  if (score_mode != GSE_SCORE_NONE && (!mode_by_row || !rows))
    return gse_fail(GSE_EINVAL, "decode: scoring needs mode_by_row and rows");
  if (score_mode == GSE_SCORE_EAGER && !scores) return gse_fail(GSE_EINVAL, "decode: eager scoring needs scores");
  if (score_mode == GSE_SCORE_QUEUE && (!queue_q || !queue_norm || !queue_lim || !queue_count || queue_cap < 1))
    return gse_fail(GSE_EINVAL, "decode: queue mode needs the queue buffers and queue_cap >= 1");
  if (logits && (!logit_index || !rows || logit_rows < 1 || logit_cap < 1))
    return gse_fail(GSE_EINVAL, "decode: kept logits need logit_index, rows, logit_rows >= 1 and logit_cap >= 1");
  if (logits && int64_t(logit_cap) * q_heads * 4 >= (int64_t(1) << 31))
    return gse_fail(GSE_EINVAL, "decode: kept logits of one row must stay below 2 GiB");
  if (n_fold < 0 || n_fold > bs) return gse_fail(GSE_EINVAL, "decode: n_fold must be in [0, bs]");
  if (n_fold > 0 && (score_mode != GSE_SCORE_QUEUE || !fold_seq || !scores))
    return gse_fail(GSE_EINVAL, "decode: folding queues needs queue mode, fold_seq and scores");
  if (n_fold > 0 && queue_cap > fl::MAX_QUEUE) return gse_fail(GSE_EINVAL, "decode: queue_cap above 64");
  if ((q_stride_h % 8) || (q_stride_b % 8) || (kv_stride_s % 8) || (kv_stride_h % 8) || (o_stride_b % 8) ||
      (o_stride_h % 8))
    return gse_fail(GSE_EINVAL, "decode: strides must be multiples of 8 elements (16-byte rows)");
  // The attention kernel reads slot rows as records of a structured buffer: a slot's kv_heads
  // head rows lie in one record of under 16 KiB (the [slots, kv_heads, 64] pool layout).
  if (kv_stride_s <= 0 || kv_stride_s * 2 >= (1 << 14) || kv_stride_h < 0 ||
      (int64_t(kv_heads - 1) * kv_stride_h + D) > kv_stride_s)
    return gse_fail(GSE_ESHAPE, "decode: each slot's K/V head rows must lie within one slot row of under 16 KiB "
                                "([slots, kv_heads, 64] pools)");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);

  // Fold workgroups: the caller's count, or FOLD_WORKGROUPS_PER_ROW per folded row up to a third
  // of the CUs; the attention workgroups take the rest (its partitions and partials are by its
  // own count).
  const int P_all = fused_workgroups();
  if (n_fold > 0 && (fold_workgroups < 0 || fold_workgroups > P_all / 2))
    return gse_fail(GSE_EINVAL, "decode: fold_workgroups must be in [0, CUs / 2]");
  const int F = n_fold <= 0 ? 0
                : fold_workgroups > 0 ? fold_workgroups
                                      : std::min(P_all / 3, FOLD_WORKGROUPS_PER_ROW * n_fold);
  // Attention workgroups: the rest of the CUs, but no more than one 64-key tile each of the batch's
  // at most bs * max_len keys (a small batch's launch is bound by each workgroup's load latency,
  // and every extra workgroup adds a partial to the merge).
  const int64_t tiles = (int64_t(bs) * std::max(max_len, 1) + TILE - 1) / TILE;
  int P = int(std::min<int64_t>(P_all - F, std::max<int64_t>(tiles, 1)));
  // By sequence every list's last tile counts, so that chunks of one tile fit. SHARE_MIN_WG workgroups
  // per sequence leave P - bs > 0 for its divisions.
  const bool whole_seq = bs > 1 && bs <= SHARE_MAX_BS && bs * SHARE_MIN_WG <= P;
  if (whole_seq) P = int(std::min<int64_t>(P_all - F, bs * ((int64_t(max_len) + TILE - 1) / TILE)));
  float* part = static_cast<float*>(workspace);
  float* norm_ws = part + (int64_t(P_all) + bs) * q_heads * PART;
  float* norm = norm_out ? norm_out : norm_ws;

  FusedArgs f = {};
  f.q = static_cast<const uint16_t*>(q);
  f.q_sb = q_stride_b;
  f.q_sh = q_stride_h;
  f.k = static_cast<const uint16_t*>(k_pool);
  f.v = static_cast<const uint16_t*>(v_pool);
  f.kv_ss = kv_stride_s;
  f.kv_sh = kv_stride_h;
  f.indptr = kv_indptr;
  f.indices = kv_indices;
  f.part = part;
  f.bs = bs;
  f.q_heads = q_heads;
  f.kv_heads = kv_heads;
  f.scale2 = sm_scale * kLog2e;
  f.rows = rows;
  f.rows_dtype = rows_dtype;
  if (logits) {
    f.logits = logits;
    f.lidx = logit_index;
    f.lrows = logit_rows;
    f.lcap = logit_cap;
  }
  f.P = P;
  if (score_mode == GSE_SCORE_QUEUE) {
    f.step_count = queue_count;
    f.step_mode = mode_by_row;
  }
  f.whole_seq = whole_seq;
  if (n_fold > 0) {
    f.fold_seq = fold_seq;
    f.n_fold = n_fold;
    f.mode = mode_by_row;
    f.scores = scores;
    f.ssg = scores_stride_g;
    f.sss = scores_stride_s;
    f.qq = static_cast<const uint16_t*>(queue_q);
    f.qnorm = queue_norm;
    f.qlim = queue_lim;
    f.qcount = queue_count;
    f.cap = queue_cap;
    // The fold region follows the partials and normalisers (gse_decode_fold_bytes).
    char* fold_ws = static_cast<char*>(workspace) + (gse_decode_workspace_bytes(bs, q_heads, D) + 255) / 256 * 256;
    f.fold_hdr = reinterpret_cast<int*>(fold_ws);
    f.fold_buf = reinterpret_cast<float*>(fold_ws + (int64_t(n_fold) * 4 + 255) / 256 * 256);
    f.fold_stride = std::max(max_len, 1);
  }
  const dim3 grid(P + F), block(FUSED_THREADS);
  // Kept logits take the kernel instance that has their MFMAs and stores; the other has none.
  if (indices_dtype == GSE_I64 && logits)
    hipLaunchKernelGGL((decode_fused_kernel<int64_t, true>), grid, block, 0, s, f);
  else if (indices_dtype == GSE_I64)
    hipLaunchKernelGGL((decode_fused_kernel<int64_t, false>), grid, block, 0, s, f);
  else if (logits)
    hipLaunchKernelGGL((decode_fused_kernel<int32_t, true>), grid, block, 0, s, f);
  else
    hipLaunchKernelGGL((decode_fused_kernel<int32_t, false>), grid, block, 0, s, f);
  int rc = gse_launch_check("decode_fused");
  if (rc) return rc;

  MergeArgs m = {};
  m.part = part;
  m.indptr = kv_indptr;
  m.sinks = sinks;
  m.sinks_dtype = sinks_dtype;
  m.o = static_cast<uint16_t*>(o);
  m.o_sb = o_stride_b;
  m.o_sh = o_stride_h;
  m.norm_out = norm;
  m.q = f.q;
  m.q_sb = q_stride_b;
  m.q_sh = q_stride_h;
  m.mode = mode_by_row;
  m.rows = rows;
  m.rows_dtype = rows_dtype;
  if (score_mode == GSE_SCORE_QUEUE) {
    m.qq = static_cast<uint16_t*>(queue_q);
    m.qnorm = queue_norm;
    m.qlim = queue_lim;
    m.qcount = queue_count;
    m.cap = queue_cap;
  }
  m.bs = bs;
  m.q_heads = q_heads;
  m.nparts = P;
  m.whole_seq = whole_seq;
  m.fold_seq = fold_seq;
  m.n_fold = n_fold;
  m.fold_buf = f.fold_buf;
  m.fold_hdr = f.fold_hdr;
  m.fold_stride = f.fold_stride;
  m.kv_heads = kv_heads;
  m.indices = kv_indices;
  m.indices_dtype = indices_dtype;
  m.scores = scores;
  m.ssg = scores_stride_g;
  m.sss = scores_stride_s;
  // By the average number of workgroups a sequence spans (P / bs); longer ones take more rounds.
  // With folds, MERGE_SCATTER_ROWS more grid rows add the fold's totals beside the merge.
  const uint32_t ub = static_cast<uint32_t>(bs);
  const unsigned extra = n_fold > 0 ? MERGE_SCATTER_ROWS : 0;
  if (int64_t(bs) * 8 >= P) {
    m.head_groups = q_heads / 8;
    hipLaunchKernelGGL((decode_merge_kernel<1, 8>), dim3(ub, unsigned(q_heads / 8) + extra), dim3(16 * 8), 0, s, m);
  } else if (int64_t(bs) * 64 >= P) {
    m.head_groups = q_heads / 8;
    hipLaunchKernelGGL((decode_merge_kernel<8, 8>), dim3(ub, unsigned(q_heads / 8) + extra), dim3(16 * 8 * 8), 0, s,
                       m);
  } else {
    m.head_groups = q_heads;
    hipLaunchKernelGGL((decode_merge_kernel<64, 1>), dim3(ub, unsigned(q_heads) + extra), dim3(16 * 64), 0, s, m);
  }
  if ((rc = gse_launch_check("decode_merge"))) return rc;

  if (score_mode == GSE_SCORE_EAGER) {
    // This step's scores need its final normaliser: a second, score-only pass over K.
    ScoreArgs sa = {f.q, q_stride_b, q_stride_h, f.k, kv_stride_s, kv_stride_h, kv_indptr, kv_indices, norm,
                    mode_by_row, rows, rows_dtype, scores, scores_stride_g, scores_stride_s, kv_heads, q_heads, bs,
                    sm_scale * kLog2e};
    if ((rc = score_pass(sa, indices_dtype, max_len, s))) return rc;
  }
  return GSE_OK;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch`, looked up once per device with it current.
int noalloc_scratch(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return gse_fail(GSE_ELAUNCH, "decode_noalloc: no current HIP device (or a device id >= 64)");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return gse_fail(GSE_ELAUNCH, "decode_noalloc: hipGetSymbolAddress of the scratch array failed");
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return GSE_OK;
}

}  // namespace

extern "C" int gse_decode(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                          const void* k_pool, const void* v_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                          const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
                          const void* sinks, int sinks_dtype, const int32_t* mode_by_row, const void* rows,
                          int rows_dtype, float* scores, int64_t scores_stride_g, int64_t scores_stride_s,
                          void* o, int64_t o_stride_b, int64_t o_stride_h, float* norm_out,
                          void* queue_q, float* queue_norm, int32_t* queue_lim, int32_t* queue_count, int queue_cap,
                          int bs, int q_heads, int kv_heads, int head_dim, float sm_scale, int max_len,
                          int score_mode, float* logits, const int32_t* logit_index, int logit_rows, int logit_cap,
                          const int32_t* fold_seq, int n_fold, int fold_workgroups, void* workspace,
                          int64_t workspace_bytes, gse_stream_t stream) {
  if (int rc = check_decode_shape(q_heads, kv_heads, head_dim)) return rc;
  if (bs < 0) return gse_fail(GSE_EINVAL, "decode: bs < 0");
  if (bs == 0) return GSE_OK;
  int64_t need = gse_decode_workspace_bytes(bs, q_heads, head_dim);
  if (n_fold > 0) need = (need + 255) / 256 * 256 + gse_decode_fold_bytes(n_fold, kv_heads, max_len);
  if (workspace_bytes < need) return gse_fail(GSE_EWORKSPACE, "decode: workspace too small");
  if (!workspace) return gse_fail(GSE_EINVAL, "decode: null workspace");
  return decode_run(q, q_stride_b, q_stride_h, k_pool, v_pool, kv_stride_s, kv_stride_h, kv_indptr, kv_indices,
                    indices_dtype, sinks, sinks_dtype, mode_by_row, rows, rows_dtype, scores, scores_stride_g,
                    scores_stride_s, o, o_stride_b, o_stride_h, norm_out, queue_q, queue_norm, queue_lim, queue_count,
                    queue_cap, bs, q_heads, kv_heads, sm_scale, max_len, score_mode, logits, logit_index, logit_rows,
                    logit_cap, fold_seq, n_fold, fold_workgroups, workspace, stream);
}

extern "C" int gse_decode_noalloc(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                                  const void* k_pool, const void* v_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                                  const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
                                  const void* sinks, int sinks_dtype, const int32_t* mode_by_row, const void* rows,
                                  int rows_dtype, float* scores, int64_t scores_stride_g, int64_t scores_stride_s,
                                  void* o, int64_t o_stride_b, int64_t o_stride_h, float* norm_out,
                                  void* queue_q, float* queue_norm, int32_t* queue_lim, int32_t* queue_count,
                                  int queue_cap, int bs, int q_heads, int kv_heads, int head_dim, float sm_scale,
                                  int max_len, int score_mode, float* logits, const int32_t* logit_index,
                                  int logit_rows, int logit_cap, const int32_t* fold_seq, int n_fold,
                                  int fold_workgroups, gse_stream_t stream) {
  if (int rc = check_decode_shape(q_heads, kv_heads, head_dim)) return rc;
  if (bs < 0) return gse_fail(GSE_EINVAL, "decode_noalloc: bs < 0");
  if (n_fold != 0) return gse_fail(GSE_EINVAL, "decode_noalloc: queue folds need gse_decode's workspace");
  if (bs == 0) return GSE_OK;
  const int64_t need = gse_decode_workspace_bytes(bs, q_heads, head_dim);
  if (need > int64_t(GSE_DECODE_NOALLOC_SCRATCH_BYTES)) {
    char msg[256];
    snprintf(msg, sizeof(msg),
             "decode_noalloc: bs=%d with %d query heads needs %lld bytes of scratch, more than the library's %lld "
             "(GSE_DECODE_NOALLOC_SCRATCH_BYTES); use gse_decode with a workspace",
             bs, q_heads, static_cast<long long>(need), static_cast<long long>(GSE_DECODE_NOALLOC_SCRATCH_BYTES));
    return gse_fail(GSE_EWORKSPACE, msg);
  }
  void* ws = nullptr;
  if (int rc = noalloc_scratch(&ws)) return rc;
  return decode_run(q, q_stride_b, q_stride_h, k_pool, v_pool, kv_stride_s, kv_stride_h, kv_indptr, kv_indices,
                    indices_dtype, sinks, sinks_dtype, mode_by_row, rows, rows_dtype, scores, scores_stride_g,
                    scores_stride_s, o, o_stride_b, o_stride_h, norm_out, queue_q, queue_norm, queue_lim, queue_count,
                    queue_cap, bs, q_heads, kv_heads, sm_scale, max_len, score_mode, logits, logit_index, logit_rows,
                    logit_cap, fold_seq, n_fold, fold_workgroups, ws, stream);
}

extern "C" int gse_decode_scores_from_lse(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                                          const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                                          const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
                                          const float* attn_lse, int64_t lse_stride_b, int64_t lse_stride_h,
                                          const int32_t* num_kv_splits, int max_kv_splits, int min_block_kv,
                                          const void* sinks, int sinks_dtype, const int32_t* mode_by_row,
                                          const void* rows, int rows_dtype, float* scores,
                                          int64_t scores_stride_g, int64_t scores_stride_s, int bs, int q_heads,
                                          int kv_heads, int head_dim, float sm_scale, int max_len, void*, int64_t,
                                          gse_stream_t stream) {
  if (int rc = check_decode_shape(q_heads, kv_heads, head_dim)) return rc;
  if (bs <= 0) return bs < 0 ? gse_fail(GSE_EINVAL, "scores_from_lse: bs < 0") : GSE_OK;
  if (max_kv_splits < 1 || min_block_kv < 1) return gse_fail(GSE_EINVAL, "scores_from_lse: split layout");
  if (!q || !k_pool || !kv_indptr || !kv_indices || !attn_lse || !num_kv_splits || !sinks || !mode_by_row || !rows ||
      !scores)
    return gse_fail(GSE_EINVAL, "scores_from_lse: null pointer");
  if ((q_stride_h % 8) || (q_stride_b % 8) || (kv_stride_s % 8) || (kv_stride_h % 8))
    return gse_fail(GSE_EINVAL, "scores_from_lse: strides must be multiples of 8 elements");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // The pass forms each sequence's normaliser itself.
  ScoreArgs sa = {static_cast<const uint16_t*>(q), q_stride_b, q_stride_h, static_cast<const uint16_t*>(k_pool),
                  kv_stride_s, kv_stride_h, kv_indptr, kv_indices, nullptr, mode_by_row, rows, rows_dtype, scores,
                  scores_stride_g, scores_stride_s, kv_heads, q_heads, bs, sm_scale * kLog2e, attn_lse, lse_stride_b,
                  lse_stride_h, num_kv_splits, sinks, sinks_dtype, max_kv_splits, min_block_kv};
  return score_pass(sa, indices_dtype, max_len, s);
}
