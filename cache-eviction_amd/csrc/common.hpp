// Shared device helpers for the gstar_evict HIP kernels (gfx950 / CDNA4).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/gstar_evict.h"

#define GSE_DEVICE __device__ __forceinline__

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// Wavefront size on CDNA is 64.
constexpr int kWave = 64;

// A score word (a row's mode_by_row entry, a prefill call's mode): the score kind in bits 0-3
// (1 sum, 2 max over a KV head's query heads, 4 block counters), log2 of the block size in
// bits 4-7 (kind 4) and the score delay from bit 8, in list entries.
// Blocks of kind 4 hold at most 64 entries (one wave's lanes); a larger shift scores nothing.
GSE_DEVICE int score_block_shift(int32_t word) { return (word >> 4) & 0xf; }
GSE_DEVICE int score_kind(int32_t word) {
  const int kind = word & 0xf;
  return kind == GSE_SCORE_KIND_BLOCK_STEP && score_block_shift(word) > 6 ? 0 : kind;
}
GSE_DEVICE int score_delay(int32_t word) { return word >> GSE_SCORE_DELAY_SHIFT; }
// Kinds that add scores (the others are attention only).
GSE_DEVICE bool scoring_kind(int kind) { return kind == 1 || kind == 2 || kind == GSE_SCORE_KIND_BLOCK_STEP; }
// Kind 4: of a list of `lim` entries (the query's own key last), the entries whose blocks a
// query credits: whole blocks of 2^shift aligned entries whose newest entry is at least
// `delay` entries older than the query.
GSE_DEVICE int block_step_limit(int lim, int delay, int shift) {
  const int n = lim - delay;
  return n > 0 ? (n >> shift) << shift : 0;
}

GSE_DEVICE float bf16_to_f32(uint16_t x) { return __uint_as_float(uint32_t(x) << 16); }

// Round-to-nearest-even float -> bf16 (NaN stays NaN).
GSE_DEVICE uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;

// Two floats to packed bf16 (round to nearest even): one v_cvt_pk_bf16_f32 on gfx950.
GSE_DEVICE uint32_t pack_bf16x2(float lo, float hi) {
  const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

GSE_DEVICE bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

// 16x16x32 bf16 MFMA, fp32 accumulate. Lane l supplies A[l%16][8*(l/16)+e] and
// B[8*(l/16)+e][l%16] for e = 0..7, and holds D[4*(l/16)+r][l%16] for r = 0..3.
GSE_DEVICE f32x4_t mfma16x16x32(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x, formed here: the compiler cannot move its computation past this point.
GSE_DEVICE float formed(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// fmaxf as one instruction: the compiler quiets operands it cannot trace to an arithmetic
// instruction (a lane swap's results) with a v_max each, which this instruction does itself.
GSE_DEVICE float vmax(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

GSE_DEVICE float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The wave's loaded registers are in use here: the compiler waits for exactly these loads.
GSE_DEVICE void landed(const uint4& x) { asm volatile("" ::"v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w)); }
GSE_DEVICE void landed(float x) { asm volatile("" ::"v"(x)); }
GSE_DEVICE void landed(const bf16x8_t& x) { landed(__builtin_bit_cast(uint4, x)); }

typedef __attribute__((ext_vector_type(4))) short s16x4_t;

// ds_read_b64_tr_b16: in each 16-lane group, source lane j supplies 4 consecutive
// 16-bit values at its address; lane i receives value (i % 4) of source lanes
// 4*e + i/4 for e = 0..3, i.e. one column of the 4 rows the group addressed.
GSE_DEVICE s16x4_t ds_read_tr16(const uint16_t* lds) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(lds));
}

GSE_DEVICE bf16x8_t join_bf16x8(s16x4_t lo, s16x4_t hi) {
  typedef __attribute__((ext_vector_type(8))) short s16x8_t;
  const s16x8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8_t, v);
}

// A pointer read from device memory (e.g. a per-layer pool table) is a generic pointer to the
// compiler; naming its global address space lets it issue global (not flat) loads and stores,
// whose waits it tracks per access.
template <typename T>
using global_ptr = __attribute__((address_space(1))) T*;

template <typename T>
GSE_DEVICE global_ptr<T> as_global(T* p) {
  return (global_ptr<T>)p;
}

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

// 16-byte global load / store through an address-space-1 pointer.
GSE_DEVICE uint4 gload16(const __attribute__((address_space(1))) void* p) {
  return __builtin_bit_cast(uint4, *(const __attribute__((address_space(1))) u32x4_t*)p);
}
GSE_DEVICE void gstore16(__attribute__((address_space(1))) void* p, uint4 v) {
  *(__attribute__((address_space(1))) u32x4_t*)p = __builtin_bit_cast(u32x4_t, v);
}

// Streaming forms (nontemporal: the line is not kept in the caches) for data that one kernel
// touches exactly once, such as rows that a relocation moves.
GSE_DEVICE uint4 gload16_nt(const __attribute__((address_space(1))) void* p) {
  return __builtin_bit_cast(uint4, __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4_t*)p));
}
GSE_DEVICE void gstore16_nt(__attribute__((address_space(1))) void* p, uint4 v) {
  __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, v), (__attribute__((address_space(1))) u32x4_t*)p);
}

// Buffer resources (word 3 of the descriptor as gfx9-family parts take it). The hardware's range
// check drops an access that is out of range (a load returns 0, a store writes nothing): with
// stride 0 (raw) an offset at or past num_records, with a stride (structured) an index at or past
// num_records. Code that must not touch memory for some lanes gives those lanes
// BUFFER_NO_INDEX and BUFFER_OUT_OF_RANGE, past both bounds.
constexpr int BUFFER_RSRC_FLAGS = 0x00020000;
constexpr int BUFFER_OUT_OF_RANGE = int(0x80000000u);
constexpr int BUFFER_NO_INDEX = int(0xFFFFFFFFu);
constexpr int BUFFER_NT = 2;  // cache policy: nontemporal

// 16 bytes at record `index`, byte `offset` of a structured buffer (the LLVM intrinsic; clang has
// builtins for the raw forms only).
__device__ u32x4_t struct_buffer_load_b128(__amdgpu_buffer_rsrc_t rsrc, int index, int offset, int soffset,
                                           int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v4i32");
__device__ void struct_buffer_store_b128(u32x4_t v, __amdgpu_buffer_rsrc_t rsrc, int index, int offset,
                                         int soffset, int aux) __asm("llvm.amdgcn.struct.ptr.buffer.store.v4i32");
GSE_DEVICE uint4 buffer_load16_nt(__amdgpu_buffer_rsrc_t rsrc, int index, int offset) {
  return __builtin_bit_cast(uint4, struct_buffer_load_b128(rsrc, index, offset, 0, BUFFER_NT));
}
GSE_DEVICE void buffer_store16_nt(uint4 v, __amdgpu_buffer_rsrc_t rsrc, int index, int offset) {
  struct_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), rsrc, index, offset, 0, BUFFER_NT);
}

// Structured-buffer resource over a K or V pool whose records are its slot rows (row_elems bf16,
// under 16 KiB): any int32 slot index addresses its row, and BUFFER_NO_INDEX reads zeros.
GSE_DEVICE __amdgpu_buffer_rsrc_t slot_rsrc(const uint16_t* pool, int64_t row_elems) {
  const uint64_t p = reinterpret_cast<uint64_t>(pool);
  // readfirstlane returns int: each half goes through uint32_t, or the low half's sign would fill
  // the high word.
  const uint64_t u = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(p >> 32)))) << 32 |
                     uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(p))));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(u), int16_t(row_elems * 2), INT32_MAX,
                                           BUFFER_RSRC_FLAGS);
}

// A value the compiler cannot see through: keeps a 32-bit product from being fused with a later
// add into a 64-bit multiply-add, whose unused high addend register the wait counting treats as
// read (it then waits for whatever load last wrote that register).
GSE_DEVICE uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <typename T>
GSE_DEVICE int64_t load_index(const void* p, int64_t i) {
  return int64_t(static_cast<const T*>(p)[i]);
}

GSE_DEVICE int64_t load_index_dyn(const void* p, int dtype, int64_t i) {
  return dtype == GSE_I64 ? static_cast<const int64_t*>(p)[i] : int64_t(static_cast<const int32_t*>(p)[i]);
}

GSE_DEVICE float load_float_dyn(const void* p, int dtype, int64_t i) {
  return dtype == GSE_BF16 ? bf16_to_f32(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}

GSE_DEVICE float wave_max_xor(float v, int mask) { return fmaxf(v, __shfl_xor(v, mask, kWave)); }
GSE_DEVICE float wave_sum_xor(float v, int mask) { return v + __shfl_xor(v, mask, kWave); }

// Value of lane l ^ 16 (row swap), without LDS: v_permlane16_swap on gfx950.
GSE_DEVICE float lane_xor16(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  // r[0] holds rows (0, 0, 2, 2) and r[1] rows (1, 1, 3, 3) of v: pick the other row of the pair.
  const int row = (threadIdx.x >> 4) & 1;
  return __uint_as_float(row ? r[0] : r[1]);
}

// Value of lane l ^ 32 (half swap), without LDS: v_permlane32_swap on gfx950.
GSE_DEVICE float lane_xor32(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  // r[0] holds halves (0, 0) and r[1] halves (1, 1) of v.
  const int half = (threadIdx.x >> 5) & 1;
  return __uint_as_float(half ? r[0] : r[1]);
}

// max / sum of v over lanes l and l ^ 16 (resp. l ^ 32): the swap returns both halves of
// each pair, so the symmetric reduction needs no lane-dependent select.
GSE_DEVICE float xor16_max(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
GSE_DEVICE float xor16_sum(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
GSE_DEVICE float xor32_max(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
GSE_DEVICE float xor32_sum(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
