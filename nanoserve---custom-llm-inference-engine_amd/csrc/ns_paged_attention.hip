// Paged attention for gfx950 (decode and chunked prefill).
//
// Follows nanoserve/kernels/paged_attention_triton.py:19-106 (per query token: online softmax over
// the sequence's KV blocks, GQA by h / NUM_KV_GROUPS, causal cut at the query's own KV position,
// zero output when no key is visible) and the launcher's index set-up (:109-131: sequence of each
// query token, its absolute KV position), re-designed for MI355X:
//
//  * One 256-thread workgroup per (query token, KV head, KV partition) computes every query head of
//    that KV head (G = num_heads_q / num_kv_heads of them), so each key and value row is read from
//    HBM once per query token instead of once per query head as the reference's per-(token, head)
//    programs do.  The 16-bit types take pa_decode_kernel (matrix core), float32 pa_partition_kernel
//    (vector arithmetic; the next two points are its).
//  * Lane layout per wave batch: 16 KV positions, 8 at a time, 8 lanes per position, each lane holding a
//    head_dim/8 slice (64 contiguous bytes at head_dim 128: four 16-byte loads; G = 8 at head_dim 128:
//    8 positions, 16 lanes each, 32 bytes a lane).  The slice's partial dot products are summed across
//    the position's lanes with ds_swizzle (no LDS traffic).
//  * Exact two-pass softmax inside a partition: scores (already in log2 units) go to LDS, one max
//    and one exp2 pass over LDS, then the value pass.
//  * Partitions of a long sequence (split-KV, sized on the host so that the grid holds >= 1024
//    workgroups) are merged by the last of the row's workgroups to arrive (max-rescaled sums); a
//    query that fits one partition is written directly.  One launch for the decode tokens of a call,
//    one for its prefill tiles.
//  * The sequence of a query token and its KV position are computed in the kernel (a search over
//    query_start_loc, 64 entries at a time), so a call needs no host copy of the batch layout.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include "ns_paged_attention.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kSub = 2;                 // KV positions per lane per batch
constexpr int kMaxPart = 1024;          // largest KV partition (LDS score buffer, block list)
constexpr int kMinPart = 64;
// partitions of a row merged through a table of their weights in LDS (one long row of few KV heads has
// hundreds): the loop that takes more reads three words per partition and output one after the other.
// one row of 17000 .. 65536 positions, 1 .. 3 KV heads (266 .. 1024 partitions, bf16, head_dim 128,
// G = 1 .. 8): 18-121 us with the table, 75-1145 by the loop
constexpr int kMaxMerge = 1024;
// workgroups a launch aims for before splitting stops: four per CU (the 128-dim 16-bit kernels hold three at once)
constexpr int kTargetGroups = 1024;
constexpr float kLog2e = 1.4426950408889634f;

thread_local char g_err[512];

int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
int fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return 1;
}

struct PaParams {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  const int32_t* bt;
  const int32_t* seq_lens;
  const int32_t* qsl;
  const int32_t* qlens;
  int32_t* status;
  float* ws_acc;    // (total_q, Hq, max_parts, D) unnormalised partition outputs
  float* ws_ml;     // (total_q, Hq, max_parts, 2) partition max (log2 units) and sum
  int32_t* counters;  // (total_q, Hkv) arrivals of split rows' partitions; zero between calls
                      // (a buffer of its own: any call shape leaves every counter at zero)
  int64_t sq_tok, sq_head, sk_blk, sk_tok, sk_head, sv_blk, sv_tok, sv_head, so_tok, so_head, sbt;
  int32_t num_seqs, hq, hkv, block_size, num_blocks, max_blocks_per_seq, part_tokens, max_parts;
  int32_t total_q;
  const int32_t* tokens;  // the query tokens the decode kernel takes (blockIdx.x indexes it), or NULL: all
  int32_t bs_shift;  // log2(block_size) when it is a power of two, else -1
  float scale_log2;  // scale * log2(e): scores in log2 units, exp2 for the softmax
};

// ---- element loads / stores -------------------------------------------------------------------

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int N> struct Int { static constexpr int value = N; };

struct Bf16 {};
struct F16 {};

template <typename T> struct Elem;
template <> struct Elem<float> { static constexpr int bytes = 4; };
template <> struct Elem<Bf16> { static constexpr int bytes = 2; };
template <> struct Elem<F16> { static constexpr int bytes = 2; };

// N consecutive floats (N a multiple of 4, 16-byte aligned)
template <int N>
__device__ __forceinline__ void load_floats(const void* base, int64_t elem_off, float (&x)[N]) {
  const u32x4* p = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(base) + elem_off);
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const u32x4 w = p[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[4 * i + j] = __uint_as_float(w[j]);
  }
}

template <typename T>
__device__ __forceinline__ void store_one(void* base, int64_t elem_off, float x) {
  if constexpr (Elem<T>::bytes == 4) {
    reinterpret_cast<float*>(base)[elem_off] = x;
  } else if constexpr (__is_same(T, Bf16)) {
    // round to nearest even; NaN stays a quiet NaN
    uint32_t u = __float_as_uint(x);
    uint16_t h;
    if ((u & 0x7FFFFFFFu) > 0x7F800000u) {
      h = (uint16_t)((u >> 16) | 0x40u);
    } else {
      u += 0x7FFFu + ((u >> 16) & 1u);
      h = (uint16_t)(u >> 16);
    }
    reinterpret_cast<uint16_t*>(base)[elem_off] = h;
  } else {
    reinterpret_cast<_Float16*>(base)[elem_off] = (_Float16)x;
  }
}

// ---- lane exchanges ---------------------------------------------------------------------------

// Sum over the 8 lanes of an aligned lane octet: ds_swizzle in bitmask mode (xor 1, 2, 4).
__device__ __forceinline__ float octet_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x041F));
  x += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x081F));
  x += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x101F));
  return x;
}

// Sum over the 16 lanes of an aligned group (the octet sum, then xor 8).
__device__ __forceinline__ float hex_sum(float x) {
  x = octet_sum(x);
  x += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x201F));
  return x;
}

// Sum over the lanes that share lane % L (xor L, 2L, ... 32).
template <int L>
__device__ __forceinline__ float slot_sum(float x) {
#pragma unroll
  for (int s = L; s < 64; s <<= 1) x += __shfl_xor(x, s);
  return x;
}

__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) x = fmaxf(x, __shfl_xor(x, s));
  return x;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) x += __shfl_xor(x, s);
  return x;
}

// Stores and loads of the partition partials at agent scope: the workgroups of one row run on
// different XCDs, whose L2s are not coherent with each other for plain accesses.
__device__ __forceinline__ void st_dev(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- batch layout -----------------------------------------------------------------------------

struct QueryPlace {
  int seq;
  int kv_len;  // visible KV positions: min(kv_pos + 1, seq_len), at least 0
};

// Sequence of query token qi: the largest s with query_start_loc[s] <= qi (empty sequences share
// their start with the next one, so the largest index is the one that owns qi), as the reference's
// repeat_interleave over query_lens (paged_attention_triton.py:109-112); its KV position
// seq_len - q_len + (qi - start) (:115-131), the causal and in-sequence cuts (:64-66).
// Searched by the whole wave, 64 entries at a time: one load for up to 64 sequences, two for up to
// 4096, where a binary search is a chain of log2 of them.
__device__ __forceinline__ QueryPlace place_query(const PaParams& p, int qi) {
  const int lane = threadIdx.x & 63;
  int lo = 0, len = p.num_seqs;
  for (;;) {
    const int stride = (len + 63) / 64;
    const int at = lane * stride;
    const int below = __popcll(__ballot(at < len && p.qsl[lo + (at < len ? at : 0)] <= qi));
    const int skip = (below > 0 ? below - 1 : 0) * stride;
    lo += skip;
    if (stride == 1) break;
    len = min(stride, len - skip);
  }
  const int seq_len = p.seq_lens[lo];
  const int kv_pos = seq_len - p.qlens[lo] + (qi - p.qsl[lo]);
  int kv_len = kv_pos + 1 < seq_len ? kv_pos + 1 : seq_len;
  if (kv_len < 0) kv_len = 0;
  return {lo, kv_len};
}

// ---- matrix core ------------------------------------------------------------------------------

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// The MFMA and the 16-bit type's conversions: pack2 rounds two floats to nearest even into one
// word (low half the first; v_cvt_pk_bf16_f32 for bfloat16), lo / hi widen a word's halves back.
//
// A weight 2^(score - m) enters the value product as a high and a low 16-bit part.  m follows a column's
// largest score: it moves when a score exceeds it by more than kLift + kGap (log2 units), then to kLift
// below that score, so that the largest weight lies in [2^kLift, 2^(kLift + kGap)].  bfloat16 has
// float32's exponents: both parts of every weight keep their bits, and m moves rarely.  float16 ends at
// 2^-24: the weights are lifted to just below its largest value, so that those far below a column's
// largest are not lost; where kLowScale is used the low part is a multiple larger too, and the sum of its
// products is divided by it.  A weight w relative to the largest then carries an absolute error of at
// most 2^-(25 + kLift) (2^-(36 + kLift) with kLowScale) besides the 2^-22 (bfloat16: 2^-17) relative one.
template <typename T> struct Mma;
template <> struct Mma<Bf16> {
  typedef bf16x8_t vec;
  static constexpr float kGap = 8.f, kLift = 0.f, kLowScale = 1.f;
  static __device__ __forceinline__ f32x4_t mma16(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4_t mma16(u32x2 a, u32x2 b, f32x4_t c) {   // k = 16
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b), c, 0,
                                                     0, 0);
  }
  static __device__ __forceinline__ f32x16_t mma(vec a, vec b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2_t));
  }
  static __device__ __forceinline__ float lo(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};
template <> struct Mma<F16> {
  typedef f16x8_t vec;
  static constexpr float kGap = 2.f, kLift = 13.f, kLowScale = 2048.f;
  static __device__ __forceinline__ f32x4_t mma16(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4_t mma16(u32x2 a, u32x2 b, f32x4_t c) {   // k = 16
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, a), __builtin_bit_cast(f16x4_t, b), c, 0, 0,
                                                 0);
  }
  static __device__ __forceinline__ f32x16_t mma(vec a, vec b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2_t));
  }
  static __device__ __forceinline__ float lo(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)w); }
  static __device__ __forceinline__ float hi(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  }
};

// ---- partition kernel ---------------------------------------------------------------------------

// The end of a partition: the sum over the waves of red(wave, head, dim), s_m and s_l the partition's
// maximum (log2 units) and sum of weights per head.  s_w: G * kMaxMerge floats of LDS, free once red
// has been read.  s_odd (or NULL): an LDS word, 0 so far; with a sum that is NaN, infinite or large enough
// to overflow in the merge, redo() makes red, s_m and s_l anew and they are stored again.
template <typename T, int D, int G, typename Red, typename Redo>
__device__ __forceinline__ void finish_partition(const PaParams& p, int qi, int kvh, int part, int n_parts, Red red,
                                                 float* s_m, float* s_l, float* s_w, int* s_odd, Redo redo) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool direct = n_parts == 1;
  auto store = [&]() -> bool {
    bool odd = false;
    for (int e = threadIdx.x; e < G * D; e += kThreads) {
      const int g = e / D, d = e % D;
      float o = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) o += red(w, g, d);
      odd |= !(fabsf(o) < 0x1p100f);
      const int h = kvh * G + g;
      if (direct) {
        const float l = s_l[g];
        store_one<T>(p.out, (int64_t)qi * p.so_tok + (int64_t)h * p.so_head + d, l > 0.f ? o / l : 0.f);
      } else if (p.ws_acc && part < p.max_parts) {
        const int64_t slot_idx = ((int64_t)qi * p.hq + h) * p.max_parts + part;
        st_dev(&p.ws_acc[slot_idx * D + d], o);
        if (d == 0) {
          st_dev(&p.ws_ml[slot_idx * 2], s_m[g]);
          st_dev(&p.ws_ml[slot_idx * 2 + 1], s_l[g]);
        }
      }
    }
    return odd;
  };
  const bool odd = store();
  if (s_odd != nullptr) {
    if (odd) *s_odd = 1;
    __syncthreads();
    if (__builtin_expect(*s_odd != 0, 0)) {
      redo();
      __syncthreads();
      store();
    }
  }
  if (direct || !p.ws_acc || part >= p.max_parts) return;

  // Split row: the last of its partitions to arrive merges them (max-rescaled sums, one pass)
  // and resets the row's counter. Every store above completes before the counter moves.
  const int arrivals = n_parts < p.max_parts ? n_parts : p.max_parts;
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int32_t* counter = p.counters + (int64_t)qi * p.hkv + kvh;
  // The partials went out through agent-scope atomic stores (served at the device coherence
  // point, past the per-XCD L2s) completed by the s_waitcnt above, and are read back through
  // agent-scope atomic loads, so the ticket needs no release / acquire fence (a buffer_wbl2 /
  // buffer_inv of the whole L2: 106 -> 128 us at 64 x 2048 decode).
  if (threadIdx.x == 0) s_last = atomicAdd(counter, 1) == arrivals - 1;
  __syncthreads();
  if (!s_last) return;
  if (threadIdx.x == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (arrivals <= kMaxMerge) {
    // weights w_i / L of the partitions into LDS (one wave per head, lanes over partitions), then
    // every output is an independent weighted sum of the partitions' unnormalised outputs
    for (int g = wave; g < G; g += kWaves) {
      const int64_t base = ((int64_t)qi * p.hq + kvh * G + g) * p.max_parts;
      float m = -INFINITY;
      for (int i = lane; i < arrivals; i += 64) m = fmaxf(m, ld_dev(&p.ws_ml[(base + i) * 2]));
      m = wave_max(m);
      float l = 0.f;
      for (int i = lane; i < arrivals; i += 64) {
        const float mi = ld_dev(&p.ws_ml[(base + i) * 2]);
        const float w = (m == -INFINITY || mi == -INFINITY) ? 0.f : exp2f(mi - m);
        s_w[g * kMaxMerge + i] = w;
        l = fmaf(w, ld_dev(&p.ws_ml[(base + i) * 2 + 1]), l);
      }
      l = wave_sum(l);
      if (lane == 0) s_l[g] = l;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < G * D; e += kThreads) {
      const int g = e / D, d = e % D;
      const int h = kvh * G + g;
      const int64_t base = ((int64_t)qi * p.hq + h) * p.max_parts;
      float o = 0.f;
      int i = 0;
      // so many partitions, their loads in flight together: 8, then 4, then one by one (1 x 65,536, 8 heads on 1
      // KV head: 284 us with 4 and one by one, 121 so; 8 x 300, five partitions: 10.6 both)
      auto add = [&](auto count) {
        float a[decltype(count)::value];
#pragma unroll
        for (int j = 0; j < decltype(count)::value; ++j) a[j] = ld_dev(&p.ws_acc[(base + i + j) * D + d]);
#pragma unroll
        for (int j = 0; j < decltype(count)::value; ++j) o = fmaf(s_w[g * kMaxMerge + i + j], a[j], o);
        i += decltype(count)::value;
      };
      while (i + 8 <= arrivals) add(Int<8>{});
      if (i + 4 <= arrivals) add(Int<4>{});
      while (i < arrivals) add(Int<1>{});
      const float l = s_l[g];
      store_one<T>(p.out, (int64_t)qi * p.so_tok + (int64_t)h * p.so_head + d, l > 0.f ? o / l : 0.f);
    }
    return;
  }
  // more partitions than the LDS weight table holds: one pass of max-rescaled sums per output
  for (int e = threadIdx.x; e < G * D; e += kThreads) {
    const int g = e / D, d = e % D;
    const int h = kvh * G + g;
    const int64_t base = ((int64_t)qi * p.hq + h) * p.max_parts;
    float m = -INFINITY, l = 0.f, o = 0.f;
    for (int i = 0; i < arrivals; ++i) {
      const float mi = ld_dev(&p.ws_ml[(base + i) * 2]);
      const float li = ld_dev(&p.ws_ml[(base + i) * 2 + 1]);
      const float ai = ld_dev(&p.ws_acc[(base + i) * D + d]);
      if (mi == -INFINITY) continue;  // a partition whose keys were all skipped
      if (mi > m) {
        const float r = m == -INFINITY ? 0.f : exp2f(m - mi);
        l *= r;
        o *= r;
        m = mi;
      }
      const float w = exp2f(mi - m);
      l = fmaf(w, li, l);
      o = fmaf(w, ai, o);
    }
    store_one<T>(p.out, (int64_t)qi * p.so_tok + (int64_t)h * p.so_head + d, l > 0.f ? o / l : 0.f);
  }
}

// float32: vector arithmetic, a partition's scores in LDS.
template <int D, int G>
__global__ __launch_bounds__(kThreads) void pa_partition_kernel(PaParams p) {
  // L lanes per KV position, DS dims each: 8 lanes, or 16 for eight heads of 128 dims (the query
  // slices and accumulators of eight heads would not fit the registers at 16 dims a lane)
  constexpr int L = (G == 8 && D == 128) ? 16 : 8;
  constexpr int DS = D / L;           // dims per lane
  constexpr int NSLOT = 64 / L;       // positions a wave covers per row of a batch
  constexpr int kBatch = NSLOT * kSub;  // KV positions per wave batch
  static_assert(G <= L, "the lane with dl == g stores head g's score");
  static_assert(kMaxMerge <= kMaxPart, "s_score becomes the merge's weight table");
  __shared__ float s_score[G * kMaxPart];
  __shared__ float s_red[kWaves * G * D];
  __shared__ float s_m[G], s_l[G];
  __shared__ int s_blk[kMaxPart + 2];  // physical block of each block-table entry the partition spans

  const int qi = p.tokens != nullptr ? p.tokens[blockIdx.x] : (int)blockIdx.x;
  const int kvh = blockIdx.y, part = blockIdx.z;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (qi < 0 || qi >= p.total_q) {   // a listed token outside the batch: flagged, nothing touched
    if (threadIdx.x == 0 && part == 0 && kvh == 0 && p.status) atomicOr(p.status, NS_PA_STATUS_BAD_TILE);
    return;
  }
  const int slot = lane / L;  // position within a row of the batch
  const int dl = lane % L;     // dim slice
  const QueryPlace qp = place_query(p, qi);
  const int n_parts = (qp.kv_len + p.part_tokens - 1) / p.part_tokens;

  if (part == 0 && n_parts > p.max_parts && threadIdx.x == 0 && p.status)
    atomicOr(p.status, NS_PA_STATUS_SEQ_TOO_LONG);
  if (part >= n_parts) {
    if (part == 0) {  // no visible key: zeros (the reference's l == 0 guard, :103-104)
      for (int i = threadIdx.x; i < G * D; i += kThreads)
        store_one<float>(p.out, (int64_t)qi * p.so_tok + (int64_t)(kvh * G + i / D) * p.so_head + i % D, 0.f);
    }
    return;
  }
  const int t0 = part * p.part_tokens;
  const int t1 = min(qp.kv_len, t0 + p.part_tokens);
  const int n = t1 - t0;
  const int32_t* bt_row = p.bt + (int64_t)qp.seq * p.sbt;

  // the partition's slice of the block table, validated once, into LDS
  const int bi0 = t0 / p.block_size;
  const int nbi = (t1 - 1) / p.block_size - bi0 + 1;
  for (int i = threadIdx.x; i < nbi; i += kThreads) {
    const int bi = bi0 + i;
    int blk = bi < p.max_blocks_per_seq ? bt_row[bi] : -1;
    if (blk < 0 || blk >= p.num_blocks) {
      blk = -1;
      if (p.status) atomicOr(p.status, NS_PA_STATUS_BAD_BLOCK);
    }
    s_blk[i] = blk;
  }

  // query slices, pre-scaled into log2 units
  float qv[G][DS];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    load_floats(p.q, (int64_t)qi * p.sq_tok + (int64_t)(kvh * G + g) * p.sq_head + dl * DS, qv[g]);
#pragma unroll
    for (int i = 0; i < DS; ++i) qv[g][i] *= p.scale_log2;
  }
  __syncthreads();

  // Position j of the partition for sub-row r of the batch starting at base; its physical block
  // from LDS (-1: past the partition or an invalid entry).
  auto block_of = [&](int j, int& off) -> int {
    if (j >= n) return -1;
    const int t = t0 + j;
    int bi;
    if (p.bs_shift >= 0) {  // the usual case (16): a shift and a mask instead of an integer division
      bi = t >> p.bs_shift;
      off = t & (p.block_size - 1);
    } else {
      bi = t / p.block_size;
      off = t - bi * p.block_size;
    }
    return s_blk[bi - bi0];
  };

  // pass 1: scores -> LDS. A wave takes batches of kBatch positions (wave w: batches w, w + 4, ...);
  // each lane requests its kSub rows of the batch before any arithmetic.
  for (int base = wave * kBatch; base < n; base += kWaves * kBatch) {
    float kx[kSub][DS];
    int blk[kSub];
#pragma unroll
    for (int r = 0; r < kSub; ++r) {
      int off = 0;
      blk[r] = block_of(base + r * NSLOT + slot, off);
      if (blk[r] >= 0)
        load_floats(p.k, (int64_t)blk[r] * p.sk_blk + (int64_t)off * p.sk_tok + (int64_t)kvh * p.sk_head + dl * DS,
                    kx[r]);
    }
#pragma unroll
    for (int r = 0; r < kSub; ++r) {
      const int j = base + r * NSLOT + slot;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float sc = 0.f;
#pragma unroll
        for (int i = 0; i < DS; ++i) sc = fmaf(qv[g][i], kx[r][i], sc);
        sc = L == 8 ? octet_sum(sc) : hex_sum(sc);
        if (dl == g && j < n) s_score[g * kMaxPart + j] = blk[r] >= 0 ? sc : -INFINITY;
      }
    }
  }
  // the wave's first value batch is requested before the softmax pass: the workgroups of a CU
  // reach that pass together, and the requests keep the memory pipe busy across it
  float vx[kSub][DS];
  int vblk[kSub];
  auto request_values = [&](int base) {
#pragma unroll
    for (int r = 0; r < kSub; ++r) {
      int off = 0;
      vblk[r] = block_of(base + r * NSLOT + slot, off);
      if (vblk[r] >= 0)
        load_floats(p.v, (int64_t)vblk[r] * p.sv_blk + (int64_t)off * p.sv_tok + (int64_t)kvh * p.sv_head + dl * DS,
                    vx[r]);
    }
  };
  request_values(wave * kBatch);
  __syncthreads();

  // pass 2: per-head max and exp2, in place (wave w takes heads w, w + 4)
  for (int g = wave; g < G; g += kWaves) {
    float m = -INFINITY;
    for (int j = lane; j < n; j += 64) m = fmaxf(m, s_score[g * kMaxPart + j]);
    m = wave_max(m);
    float l = 0.f;
    for (int j = lane; j < n; j += 64) {
      const float e = m == -INFINITY ? 0.f : exp2f(s_score[g * kMaxPart + j] - m);
      s_score[g * kMaxPart + j] = e;
      l += e;
    }
    l = wave_sum(l);
    if (lane == 0) {
      s_m[g] = m;
      s_l[g] = l;
    }
  }
  __syncthreads();

  // pass 3: probability-weighted values, the same batches
  float acc[G][DS];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < DS; ++i) acc[g][i] = 0.f;
  for (int base = wave * kBatch; base < n; base += kWaves * kBatch) {
    if (base != wave * kBatch) request_values(base);
#pragma unroll
    for (int r = 0; r < kSub; ++r) {
      if (vblk[r] < 0) continue;
      const int j = base + r * NSLOT + slot;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float w = s_score[g * kMaxPart + j];
#pragma unroll
        for (int i = 0; i < DS; ++i) acc[g][i] = fmaf(w, vx[r][i], acc[g][i]);
      }
    }
  }
  // sum the position slots of the wave, then the waves through LDS
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < DS; ++i) acc[g][i] = slot_sum<L>(acc[g][i]);
  if (slot == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < DS; ++i) s_red[(wave * G + g) * D + dl * DS + i] = acc[g][i];
  }
  __syncthreads();

  finish_partition<float, D, G>(p, qi, kvh, part, n_parts,
                            [&](int w, int g, int d) { return s_red[(w * G + g) * D + d]; }, s_m, s_l, s_score,
                            nullptr, []() {});
}

// A partition in float arithmetic throughout, as the float32 kernel computes it: what pa_decode_kernel
// falls back to when its sums are not finite, or near it.  The two 16-bit parts of a weight times an
// infinite value are NaN where the weight itself gives infinity (0 * inf for a low part of 0, inf - inf
// for a negative one), and its weights of up to 2^8 can overflow on values near bfloat16's largest.  One thread per
// score and per output, rows read element by element: a partition of 1024 positions takes some hundred
// microseconds, on such values alone.  Leaves the sums in s_buf as (wave, head, dim), all in wave 0.
template <typename T, int D, int G>
__device__ __forceinline__ void plain_partition(const PaParams& p, int qi, int kvh, int t0, int n, const int* s_blk,
                                                float* s_buf, float* s_m, float* s_l) {
  using M = Mma<T>;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bi0 = t0 / p.block_size;
  auto words = [](const void* base, int64_t elem) -> const uint32_t* {   // of a row, 16-byte aligned
    return reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint16_t*>(base) + elem);
  };
  for (int e = threadIdx.x; e < G * n; e += kThreads) {
    const int g = e / n, j = e - g * n;
    const int bi = (t0 + j) / p.block_size, off = t0 + j - bi * p.block_size;
    const int blk = s_blk[bi - bi0];
    float sc = -INFINITY;
    if (blk >= 0) {
      const uint32_t* q = words(p.q, (int64_t)qi * p.sq_tok + (int64_t)(kvh * G + g) * p.sq_head);
      const uint32_t* k = words(p.k, (int64_t)blk * p.sk_blk + (int64_t)off * p.sk_tok + (int64_t)kvh * p.sk_head);
      sc = 0.f;
      for (int i = 0; i < D / 2; ++i) {
        sc = fmaf(M::lo(q[i]) * p.scale_log2, M::lo(k[i]), sc);
        sc = fmaf(M::hi(q[i]) * p.scale_log2, M::hi(k[i]), sc);
      }
    }
    s_buf[g * kMaxPart + j] = sc;
  }
  __syncthreads();
  for (int g = wave; g < G; g += kWaves) {
    float m = -INFINITY, l = 0.f;
    for (int j = lane; j < n; j += 64) m = fmaxf(m, s_buf[g * kMaxPart + j]);
    m = wave_max(m);
    for (int j = lane; j < n; j += 64) {
      const float w = m == -INFINITY ? 0.f : exp2f(s_buf[g * kMaxPart + j] - m);
      s_buf[g * kMaxPart + j] = w;
      l += w;
    }
    l = wave_sum(l);
    if (lane == 0) {
      s_m[g] = m;
      s_l[g] = l;
    }
  }
  __syncthreads();
  constexpr int NE = (G * D + kThreads - 1) / kThreads;   // outputs per thread
  float o[NE];
#pragma unroll
  for (int r = 0; r < NE; ++r) {
    const int e = (int)threadIdx.x + r * kThreads;
    o[r] = 0.f;
    if (e >= G * D) continue;
    const int g = e / D, d = e % D;
    for (int j = 0; j < n; ++j) {
      const int bi = (t0 + j) / p.block_size, off = t0 + j - bi * p.block_size;
      const int blk = s_blk[bi - bi0];
      if (blk < 0) continue;
      const uint32_t w =
          words(p.v, (int64_t)blk * p.sv_blk + (int64_t)off * p.sv_tok + (int64_t)kvh * p.sv_head)[d >> 1];
      o[r] = fmaf(s_buf[g * kMaxPart + j], d & 1 ? M::hi(w) : M::lo(w), o[r]);
    }
  }
  __syncthreads();   // the weights are read
#pragma unroll
  for (int r = 0; r < NE; ++r) {
    const int e = (int)threadIdx.x + r * kThreads;
    if (e >= G * D) continue;
    s_buf[e] = o[r];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s_buf[w * G * D + e] = 0.f;
  }
}

// The 16-bit types' partition kernel: the same workgroups, partitions, partials and merge, with the
// products on the matrix core (v_mfma_f32_16x16x32, columns the G query heads padded to 16) and the
// softmax online per wave, so that the waves stream independently and meet once at the end.  The
// vector unit did about 165 instructions per 8 positions at G = 3 (the dot products, their lane sums,
// the widening) and the passes of all the workgroups of a launch fell together, so that the memory
// pipe idled across the softmax.
//   * A wave takes steps of 16 positions at 128 dims, 32 at 64 (8 KB of rows either way).  A load
//     instruction of a wave covers whole rows (4 of 128 dims, 8 of 64), so that every 128-byte line is
//     taken at one touch: loading the products' operand layout (16 rows by 64 bytes) directly was
//     slower with 128 KB in flight on a CU (64 x 2048 at G = 3: 114 us) than with half of it (105), as if
//     lines left the cache between their touches.  A step's loads are issued before the previous
//     step's arithmetic (8 KB a wave in flight) and go through the wave's own LDS rows.
//   * S^T: lane l holds head l % 16 at positions 16 b + 4 (l / 16) + i of row block b.  Its weights are
//     the B operand of O^T += V^T P^T as they are: a 16x16x16 product per 16 dims at 128 dims, k-slot i
//     of quarter l / 16 at position 4 (l / 16) + i; a 16x16x32 one at 64, whose k-slots 4 .. 7 are the
//     second row block's.  The V^T operand is read in that order by one transposing read (two at 64
//     dims) from the wave's own LDS rows.  P goes in as a high and a low 16-bit part (Mma);
//     float16's low parts are summed apart and scaled back (64 rows of up to 2048, 128 dims: 60.3 us
//     without, 61.5 with).
//   * LDS rows are unpadded; 16-byte chunk c of row r sits at c ^ swz(r), which spreads the 16 rows of a
//     write and the 8 rows of a transposing read over the 64 banks (the counters show 20 conflict
//     cycles left in a step, of some thousands).
// Bound by HBM.  Measured (bf16, 8 KV heads of 128 dims, blocks of 16; the vector form, then this):
// 8 x 8192 at G = 3: 60 -> 56 us; 64 x 2048: 108 -> 107 (5.0 TB/s); 256 x 512: 107 -> 98; G = 4, 64 x 2048:
// 141 -> 109; G = 8, 64 x 2048: 310 -> 109.  G = 1 gains least: 8 x 2048 20.2 -> 19.1, 64 x 2048 of 64 dims 57
// both (47 -> 50 where the last-level cache holds most of it).  At 128 dims three waves a SIMD (159 to 168
// registers of 168): four spill, and an earlier form took 63 us with them at 8 x 8192, 111 at 64 x 2048 and 63
// at 256 rows of up to 512, with two 61, 103 and 60, with three 58, 107 and 57.
// BW as in the prefill kernel: a row's address is a scalar plus a lane's fixed offset.
template <typename T, int D, int G, bool BW>
__global__ __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(D == 128 ? 3 : 4, D == 128 ? 3 : 4))) void pa_decode_kernel(PaParams p) {
  using M = Mma<T>;
  using vec = typename M::vec;
  constexpr int KS = D / 32;            // k-steps of S^T, and 16-byte chunks of a row per lane
  constexpr int DB = D / 16;            // 16-dim blocks of O^T
  constexpr int NB = D == 128 ? 1 : 2;  // 16-row blocks of a wave's step
  constexpr int kStep = 16 * NB;        // its positions
  constexpr uint32_t kAllOk = NB == 1 ? 0xffffu : 0xffffffffu;
  static_assert(G <= 16, "the heads are the 16 columns");
  __shared__ __align__(16) unsigned char s_kv[kWaves][2][kStep * D * 2];   // then the waves' outputs, then merge weights
  __shared__ float s_wm[kWaves][G], s_wl[kWaves][G];
  __shared__ int s_odd;   // a sum is not finite, or near it
  __shared__ float s_m[G], s_l[G];
  __shared__ int s_blk[kMaxPart + 2];   // physical block of each block-table entry the partition spans
  static_assert(sizeof(s_kv) >= (size_t)kWaves * G * D * 4 && sizeof(s_kv) >= (size_t)G * kMaxMerge * 4 &&
                    sizeof(s_kv) >= (size_t)G * kMaxPart * 4, "reuse");

  const int qi = p.tokens != nullptr ? p.tokens[blockIdx.x] : (int)blockIdx.x;
  const int kvh = blockIdx.y, part = blockIdx.z;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (qi < 0 || qi >= p.total_q) {   // a listed token outside the batch: flagged, nothing touched
    if (threadIdx.x == 0 && part == 0 && kvh == 0 && p.status) atomicOr(p.status, NS_PA_STATUS_BAD_TILE);
    return;
  }
  const QueryPlace qp = place_query(p, qi);
  const int n_parts = (qp.kv_len + p.part_tokens - 1) / p.part_tokens;
  if (part == 0 && n_parts > p.max_parts && threadIdx.x == 0 && p.status)
    atomicOr(p.status, NS_PA_STATUS_SEQ_TOO_LONG);
  if (part >= n_parts) {
    if (part == 0) {  // no visible key: zeros (the reference's l == 0 guard, :103-104)
      for (int i = threadIdx.x; i < G * D; i += kThreads)
        store_one<T>(p.out, (int64_t)qi * p.so_tok + (int64_t)(kvh * G + i / D) * p.so_head + i % D, 0.f);
    }
    return;
  }
  const int t0 = part * p.part_tokens;
  const int n = min(qp.kv_len, t0 + p.part_tokens) - t0;
  const int32_t* bt_row = p.bt + (int64_t)qp.seq * p.sbt;

  // the partition's slice of the block table, validated once, into LDS
  const int bi0 = t0 / p.block_size;
  const int nbi = (t0 + n - 1) / p.block_size - bi0 + 1;
  for (int i = threadIdx.x; i < nbi; i += kThreads) {
    const int bi = bi0 + i;
    int blk = bi < p.max_blocks_per_seq ? bt_row[bi] : -1;
    if (blk < 0 || blk >= p.num_blocks) {
      blk = -1;
      if (p.status) atomicOr(p.status, NS_PA_STATUS_BAD_BLOCK);
    }
    s_blk[i] = blk;
  }
  if (threadIdx.x == 0) s_odd = 0;

  const int c16 = lane & 15, q4 = lane >> 4;
  // Q^T operand: head c16 (zeros past G), dims 32 s + 8 q4 .. + 7
  vec qop[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    u32x4 x = {0u, 0u, 0u, 0u};
    if (c16 < G)
      x = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.q) + (int64_t)qi * p.sq_tok +
                                          (int64_t)(kvh * G + c16) * p.sq_head + 32 * s + 8 * q4);
    qop[s] = __builtin_bit_cast(vec, x);
  }
  __syncthreads();

  constexpr int LPR = D / 8;          // lanes (16-byte chunks) of a row
  constexpr int RPI = 64 / LPR;       // rows of a load instruction
  constexpr int NL = kStep / RPI;     // load instructions of each kind a step
  const int row0 = lane / LPR, ch = lane % LPR;
  const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)kvh * p.sk_head * 2;
  const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)kvh * p.sv_head * 2;
  const int sk_tok = (int)p.sk_tok, sv_tok = (int)p.sv_tok;
  const uint32_t koff = (uint32_t)(row0 * sk_tok) * 2u + 16u * ch, voff = (uint32_t)(row0 * sv_tok) * 2u + 16u * ch;
  auto swz = [](int r) -> int {
    return D == 128 ? ((r & 7) << 1) | ((r >> 3) & 1) : (((r >> 1) & 3) << 1) | ((r >> 3) & 1);
  };
  auto slot = [&](int r, int c) -> int { return r * (D * 2) + ((c ^ swz(r)) << 4); };
  unsigned char* sk = s_kv[wave][0];
  unsigned char* sv = s_kv[wave][1];

  u32x4 kreg[NL], vreg[NL];
  uint32_t ok = 0u;      // bit r: row r of the step in the registers is the sequence's
  int blk[NL], off[NL];
  auto place_rows = [&](int base) {
    ok = 0u;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      // the instruction's first row, past the end the last group again; or the lane's own row
      const int jr = base + RPI * i + (BW ? 0 : row0);
      const int t = t0 + min(jr, BW ? (n - 1) & -RPI : n - 1);
      int bi;
      if (BW || p.bs_shift >= 0) {
        bi = t >> p.bs_shift;
        off[i] = t & (p.block_size - 1);
      } else {
        bi = t / p.block_size;
        off[i] = t - bi * p.block_size;
      }
      blk[i] = s_blk[bi - bi0];
      if constexpr (BW) blk[i] = __builtin_amdgcn_readfirstlane(blk[i]);
      if constexpr (BW) {
        ok |= blk[i] >= 0 ? ((1u << RPI) - 1u) << (RPI * i) : 0u;
      } else {
        const uint64_t good = __ballot(blk[i] >= 0);
#pragma unroll
        for (int q = 0; q < RPI; ++q) ok |= (uint32_t)((good >> (q * LPR)) & 1ull) << (RPI * i + q);
      }
      if (blk[i] < 0) blk[i] = 0;   // block 0 stands in for an invalid one; its rows are not used
    }
    if (n - base < kStep) ok &= n > base ? (1u << (n - base)) - 1u : 0u;
  };
  auto load_k = [&]() {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      kreg[i] = *reinterpret_cast<const u32x4*>(
          BW ? kbase + ((uint64_t)(uint32_t)blk[i] * (uint32_t)p.sk_blk + (uint32_t)(off[i] * sk_tok)) * 2 + koff
             : kbase + ((int64_t)blk[i] * p.sk_blk + off[i] * sk_tok) * 2 + 16 * ch);
  };
  auto load_v = [&]() {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      vreg[i] = *reinterpret_cast<const u32x4*>(
          BW ? vbase + ((uint64_t)(uint32_t)blk[i] * (uint32_t)p.sv_blk + (uint32_t)(off[i] * sv_tok)) * 2 + voff
             : vbase + ((int64_t)blk[i] * p.sv_blk + off[i] * sv_tok) * 2 + 16 * ch);
  };
  auto store_rows = [&](unsigned char* dst, const u32x4 (&x)[NL]) {
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(dst + slot(RPI * i + row0, ch)) = x[i];
  };

  f32x4_t acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  // The transposing read: lane 16 q + i of a quarter addresses position 4 q + i / 4, dims 4 (i % 4) .. + 3
  // of the block, and receives positions 4 q .. + 3 of dim i.
  const int tr_row = 4 * q4 + (c16 >> 2);

  int base = __builtin_amdgcn_readfirstlane(wave) * kStep;
  if (base < n) {
    place_rows(base);
    load_k();
    __builtin_amdgcn_sched_barrier(0);   // keys first, as in the loop: the first wait is for them alone
    load_v();
    __builtin_amdgcn_sched_barrier(0);
  }
  // one step; `more`: the next step's rows are requested before the arithmetic, loads without a branch
  // around them, so that the wait for the older ones leaves them in flight
  auto step = [&](auto more) {
    const uint32_t okw = ok;
    store_rows(sk, kreg);
    if constexpr (decltype(more)::value != 0) {
      place_rows(base + kWaves * kStep);
      load_k();
      __builtin_amdgcn_sched_barrier(0);
    }
    if (okw != kAllOk) {   // weight 0 times a row not of this sequence must be 0
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (!((okw >> (RPI * i + row0)) & 1u)) vreg[i] = u32x4{0u, 0u, 0u, 0u};
    }
    store_rows(sv, vreg);
    if constexpr (decltype(more)::value != 0) load_v();
    __builtin_amdgcn_wave_barrier();   // the wave's own LDS rows: in order, no workgroup barrier
    // S^T = K Q^T
    f32x4_t st[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      st[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 x = *reinterpret_cast<const u32x4*>(sk + slot(16 * b + c16, 4 * s + q4));
        st[b] = M::mma16(__builtin_bit_cast(vec, x), qop[s], st[b]);
      }
    }

    // online softmax of head c16 over the step's positions, 4 NB of them in this lane
    float mt = -INFINITY;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = st[b][i] * p.scale_log2;
        if (okw != kAllOk && !((okw >> (16 * b + 4 * q4 + i)) & 1u)) x = -INFINITY;
        st[b][i] = x;
        mt = fmaxf(mt, x);
      }
    mt = fmaxf(mt, __shfl_xor(mt, 16));
    mt = fmaxf(mt, __shfl_xor(mt, 32));
    // the reference m moves only for a score well above it (Mma)
    const bool move = mt > m + (M::kLift + M::kGap);
    const float mn = move ? mt - M::kLift : m;
    const float msub = mn == -INFINITY ? 0.f : mn;
    if (__ballot(move) != 0ull) {
      const float alpha = move ? __builtin_amdgcn_exp2f(m - msub) : 1.f;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[db][i] *= alpha;
    }
    m = mn;
    uint32_t wh[2 * NB], wl[2 * NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i2 = 0; i2 < 2; ++i2) {
        const float p0 = __builtin_amdgcn_exp2f(st[b][2 * i2] - msub);
        const float p1 = __builtin_amdgcn_exp2f(st[b][2 * i2 + 1] - msub);
        l += p0 + p1;
        const uint32_t hi = M::pack2(p0, p1);
        wh[2 * b + i2] = hi;
        wl[2 * b + i2] = M::pack2((p0 - M::lo(hi)) * M::kLowScale, (p1 - M::hi(hi)) * M::kLowScale);
      }
    // the low parts' products, added to the sum, or by themselves and scaled back
    auto add_low = [&](auto a, auto w, f32x4_t& sum) {
      if constexpr (M::kLowScale == 1.f) {
        sum = M::mma16(a, w, sum);
      } else {
        const f32x4_t t = M::mma16(a, w, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = fmaf(t[i], 1.f / M::kLowScale, sum[i]);
      }
    };
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int c = 2 * db + ((c16 & 3) >> 1);
      const u32x2 a0 = __builtin_bit_cast(
          u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                     (__attribute__((address_space(3))) i16x4*)(sv + slot(tr_row, c) + 8 * (c16 & 1))));
      if constexpr (NB == 1) {
        acc[db] = M::mma16(a0, u32x2{wh[0], wh[1]}, acc[db]);
        add_low(a0, u32x2{wl[0], wl[1]}, acc[db]);
      } else {
        const u32x2 a1 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                       (__attribute__((address_space(3))) i16x4*)(sv + slot(16 + tr_row, c) + 8 * (c16 & 1))));
        const vec a = __builtin_bit_cast(vec, (u32x4{a0[0], a0[1], a1[0], a1[1]}));
        acc[db] = M::mma16(a, __builtin_bit_cast(vec, (u32x4{wh[0], wh[1], wh[2 * NB - 2], wh[2 * NB - 1]})), acc[db]);
        add_low(a, __builtin_bit_cast(vec, (u32x4{wl[0], wl[1], wl[2 * NB - 2], wl[2 * NB - 1]})), acc[db]);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };
  for (; base + kWaves * kStep < n; base += kWaves * kStep) step(Int<1>{});
  // the wave's last step requests none (it is one of one or two where partitions are 64 or 128 positions: 8 x 2048
  // at G = 1 20.0 us with its rows requested again, 19.1 without)
  if (base < n) step(Int<0>{});
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);

  // the waves' maxima and sums, then their outputs scaled to the common maximum
  if (q4 == 0 && c16 < G) {
    s_wm[wave][c16] = m;
    s_wl[wave][c16] = l;
  }
  __syncthreads();
  float* s_red = reinterpret_cast<float*>(&s_kv[0][0][0]);   // (wave, head, dim); every wave's value rows are read
  if (c16 < G) {
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, s_wm[w][c16]);
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mx);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) s_red[(wave * G + c16) * D + 16 * db + 4 * q4 + i] = acc[db][i] * f;
    if (wave == 0 && q4 == 0) {
      float L = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w)
        L = fmaf(s_wm[w][c16] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s_wm[w][c16] - mx), s_wl[w][c16], L);
      s_m[c16] = mx;
      s_l[c16] = L;
    }
  }
  __syncthreads();
  finish_partition<T, D, G>(p, qi, kvh, part, n_parts, [&](int w, int g, int d) { return s_red[(w * G + g) * D + d]; },
                            s_m, s_l, s_red, &s_odd,
                            [&]() { plain_partition<T, D, G>(p, qi, kvh, t0, n, s_blk, s_red, s_m, s_l); });
}

// ---- prefill kernel: query tiles on MFMA -------------------------------------------------------
//
// Sequences with several query tokens (chunked prefill) go by query tile: kPfCols = 128 query columns
// -- kPfCols / G tokens of one sequence times the G query heads of a KV head, column c = token
// (c / G), head (c % G) -- taken by a workgroup of four waves, 32 columns each, which walks a run of
// the sequence's positions 64 at a time.  Each step's key and value rows are read from memory once
// for the whole tile (all 256 threads load them into LDS, as rows), so each row is read once per
// 128 columns instead of once per query token.  On v_mfma_f32_32x32x16 (bf16 or f16 operands,
// float32 accumulation), per wave:
//   * S^T = K Q^T for the step's two 32-position row blocks: rows positions, columns the wave's
//     queries.  A lane holds one query column (lane % 32) of 16 positions per block, so the
//     online softmax of a column (max, exp2, sum) runs in the lane plus one exchange with
//     lane ^ 32;
//   * O^T += V^T P^T over the step's four 16-position k-steps, the probabilities taken straight
//     from the S^T layout as the B operand: k-slot i of the lanes of half h is position
//     16 s + 8 (i / 4) + 4 h + i % 4 of the step, and the V^T operand is read in that order from
//     the value rows by two transposing LDS reads.  P goes in as two 16-bit parts, hi = RN(p)
//     and lo = RN(p - hi), whose products with a value are exact in float32: bfloat16 carries p to
//     about 2^-17 relative, float16 to 2^-22 and 2^-38 of the column's largest weight (Mma; its low
//     parts summed apart, as in the decode kernel, took 5 to 9% more), where a single 16-bit P
//     would round each weight by up to 2^-9.  The parts of a weight times an infinite value are
//     NaN, also for a position of the step that the causal cut hides from the column.
// The scores are the float32 dot products times scale * log2(e) (folded into the exponent's fma)
// and exp2 replaces exp, as in the decode kernel.
//
// Work split: all steps of all (tile, KV head) pairs are shared evenly by up to 512 workgroups (two
// per CU, all resident), each taking a run of consecutive steps, so that they end together whatever
// the sequences' lengths and a tile is cut only where a run ends: at most two partials per
// workgroup, stored and merged in the lanes' accumulator layout (8 bytes a lane, 512 contiguous bytes a
// store).  Four 512-token chunks ending at 2048 .. 8192 positions (24 / 8 heads of 128 dims, bf16): 627 ->
// 257 us, 195 -> 475 TFLOP/s, against partitions of at most 1024 positions whose 64 KB of partials
// each went out and came back as scattered 4-byte accesses; 228 us, 535 TFLOP/s with scalar row
// addresses; three chunks of up to 417 tokens beside 29 decode rows (32 / 8 heads of 64 dims, f16):
// 89 -> 55 us for the call.
// Keys and values are double buffered in LDS (one barrier a step), the value rows at a pitch under
// which a transposing read's four rows hit different banks (the key rows' pitch left them 4-way
// conflicted), and the block table is read one step ahead of the rows instead of through LDS.

constexpr int kPfWaves = 4;
constexpr int kPfThreads = 64 * kPfWaves;
constexpr int kPfCols = 32 * kPfWaves;   // query columns of a tile (32 per wave)
constexpr int kPfPos = 64;               // positions per step (two 32-row blocks)
constexpr int kPfMaxPart = 1024;
constexpr int kPfMinPart = 256;
constexpr int kPfTargetGroups = 512;     // two four-wave workgroups per CU
constexpr int kPfMinSteps = 4;           // steps a workgroup takes at least when tiles are cut
static_assert(kPfCols == NS_PA_TILE_COLUMNS, "the header's tile width");

struct PfParams {
  const int32_t* tiles;   // (n_tiles, 3): sequence, first query token (flat index), token count
  float* ws_acc;          // (slots, kPfWaves, D / 2, 64 lanes) unnormalised outputs of cut tiles, as the lanes hold them
  float* ws_ml;           // (slots, kPfCols, 2) their max (log2 units) and sum
  int32_t* counters;      // (n_tiles, hkv) arrivals of a cut tile's segments; zero between calls
  int32_t n_tiles;
  int32_t grid;           // workgroups that share all steps evenly, or 0: one workgroup per (tile, KV head)
  int64_t cap;            // positions of a sequence the call takes (max_seq_len, rounded up to a partition)
  float scale_log2;       // |scale| * log2(e); 1 for a scale of 0
  uint32_t q_and, q_xor;  // applied to the query words: a negative scale flips their signs, a zero scale clears them
  int32_t out_vec;        // output rows 8-byte aligned: four elements a store
};

struct PfTile {
  int seq, t0, nq;
  int kv_pos0;   // the first token's KV position
  int lt;        // positions the last token sees, up to the call's capacity
  int steps;     // 64-position steps (at least 1), or 0: not a tile of this batch
  bool cut;      // the sequence is longer than the capacity
};

__device__ __forceinline__ PfTile pf_tile(const PaParams& p, const PfParams& f, int tile, int bq) {
  PfTile r;
  r.seq = f.tiles[3 * tile];
  r.t0 = f.tiles[3 * tile + 1];
  r.nq = f.tiles[3 * tile + 2];
  r.steps = 0;
  r.kv_pos0 = r.lt = 0;
  r.cut = false;
  // a tile must hold 1 .. bq consecutive query tokens of one sequence: anything else is flagged
  // and left alone (nothing is read or written out of bounds)
  if (r.seq < 0 || r.seq >= p.num_seqs || r.nq < 1 || r.nq > bq || r.t0 < 0) return r;
  const int q0 = p.qsl[r.seq], ql = p.qlens[r.seq];
  if (r.t0 < q0 || (int64_t)r.t0 + r.nq > (int64_t)q0 + ql || (int64_t)r.t0 + r.nq > p.total_q) return r;
  const int seq_len = p.seq_lens[r.seq];
  r.kv_pos0 = seq_len - ql + (r.t0 - q0);
  int lt = r.kv_pos0 + r.nq < seq_len ? r.kv_pos0 + r.nq : seq_len;
  if (lt < 0) lt = 0;
  r.cut = lt > f.cap;
  r.lt = r.cut ? (int)f.cap : lt;
  r.steps = r.lt > 0 ? (r.lt + kPfPos - 1) / kPfPos : 1;
  return r;
}

__device__ __forceinline__ void st_dev2(float* p, float a, float b) {
  const uint64_t w = (uint64_t)__float_as_uint(a) | ((uint64_t)__float_as_uint(b) << 32);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f32x2 ld_dev2(const float* p) {
  const uint64_t w = __hip_atomic_load(reinterpret_cast<uint64_t*>(const_cast<float*>(p)), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return f32x2{__uint_as_float((uint32_t)w), __uint_as_float((uint32_t)(w >> 32))};
}

// BW: the block size is a power of two and at least the consecutive positions one load instruction
// of a wave covers (4 at 128 dims, 8 at 64), so these never straddle two blocks: the block is the
// wave's, and a row's address a scalar address plus a lane's fixed offset instead of 64-bit products
// per lane (four 512-token chunks up to 8192 positions: 257 -> 228 us).
template <typename T, int D, int G, bool BW>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void pa_prefill_kernel(PaParams p,
                                                                                                        PfParams f) {
  using M = Mma<T>;
  using vec = typename M::vec;
  constexpr int BQ = kPfCols / G;                 // tokens per tile
  constexpr int KS = D / 16;                      // k-steps of S^T = K Q^T
  constexpr int DB = D / 32;                      // 32-dim blocks of O^T
  constexpr int CPP = D / 8;                      // 16-byte chunks of a key or value row
  constexpr int LPT = kPfPos * CPP / kPfThreads;  // chunks of each kind a thread loads per step
  // bytes per staged row: keys so that 16 rows' 16-byte reads hit the 64 banks once, values so
  // that the four rows of a transposing read do
  constexpr int PK = D * 2 + 16;
  constexpr int PV = D * 2 + 64;
  static_assert(LPT * kPfThreads == kPfPos * CPP, "the step's chunks split evenly over the threads");
  __shared__ __align__(16) unsigned char s_k[2][kPfPos * PK];
  __shared__ __align__(16) unsigned char s_v[2][kPfPos * PV];
  __shared__ int64_t s_wave[kPfWaves];
  __shared__ int s_place[2];   // the workgroup's first tile and its step in it
  __shared__ int s_bad;        // an invalid block met in this segment
  __shared__ int s_last;

  const int wave = threadIdx.x >> 6;
  const int n_tiles = f.n_tiles;

  // The workgroup's units: unit u of all hkv * S steps is step u % S of the tiles in order, KV
  // head u / S.  Each workgroup takes `per` consecutive units, so that all of them finish
  // together whatever the sequences' lengths; a tile cut between workgroups is merged by the
  // last of them to arrive.
  int64_t u0 = 0, u1 = 0, per = 1, S = 0;
  int w = 0, tile = 0, off = 0, kvh = 0;
  if (f.grid > 0) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int q = (n_tiles + kPfThreads - 1) / kPfThreads;   // tiles per thread, consecutive
    const int first = tid * q;
    int64_t mine = 0;
    for (int i = first; i < first + q && i < n_tiles; ++i) {
      const PfTile t = pf_tile(p, f, i, BQ);
      mine += t.steps;
      if (blockIdx.x == 0 && p.status) {
        if (t.steps == 0) atomicOr(p.status, NS_PA_STATUS_BAD_TILE);
        if (t.cut) atomicOr(p.status, NS_PA_STATUS_SEQ_TOO_LONG);
      }
    }
    int64_t pre = mine;
#pragma unroll
    for (int sh = 1; sh < 64; sh <<= 1) {
      const int64_t o = __shfl_up(pre, sh);
      if (lane >= sh) pre += o;
    }
    if (lane == 63) s_wave[wave] = pre;
    __syncthreads();
    for (int i = 0; i < kPfWaves; ++i) {
      if (i < wave) pre += s_wave[i];
      S += s_wave[i];
    }
    pre -= mine;
    const int64_t U = S * p.hkv;
    per = (U + f.grid - 1) / f.grid;
    if (per < kPfMinSteps) per = kPfMinSteps;
    // consecutive runs on one XCD: they read the same KV head's rows
    w = f.grid % 8 == 0 ? (int)(blockIdx.x % 8) * (f.grid / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    u0 = per * w;
    u1 = u0 + per < U ? u0 + per : U;
    if (u0 >= U) return;
    kvh = (int)(u0 / S);
    const int64_t rem = u0 - kvh * S;
    if (rem >= pre && rem < pre + mine) {
      int64_t at = rem - pre;
      int i = first;
      for (;; ++i) {   // the thread's steps hold `at`: one of its tiles does
        const int n = pf_tile(p, f, i, BQ).steps;
        if (at < n) break;
        at -= n;
      }
      s_place[0] = i;
      s_place[1] = (int)at;
    }
    __syncthreads();
    tile = s_place[0];
    off = s_place[1];
  } else {
    tile = blockIdx.x % n_tiles;
    kvh = blockIdx.x / n_tiles;
    const PfTile t = pf_tile(p, f, tile, BQ);
    if (threadIdx.x == 0 && kvh == 0 && p.status) {
      if (t.steps == 0) atomicOr(p.status, NS_PA_STATUS_BAD_TILE);
      if (t.cut) atomicOr(p.status, NS_PA_STATUS_SEQ_TOO_LONG);
    }
    if (t.steps == 0) return;
    u1 = t.steps;
  }

  // the host keeps token strides times block_size below 2^31, so a slot's offset is a 32-bit product
  const int sk_tok = (int)p.sk_tok, sv_tok = (int)p.sv_tok;
  constexpr int PW = 64 / CPP;   // positions of a wave's load instruction
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const float scale = f.scale_log2;

  for (int64_t u = u0; u < u1;) {
    if (tile == n_tiles) {
      tile = 0;
      ++kvh;
    }
    const PfTile t = pf_tile(p, f, tile, BQ);
    if (t.steps == 0) {   // not a tile of this batch: no units
      ++tile;
      continue;
    }
    // The lane's places and offsets.  At 128 dims they are made anew for each tile, from the lane's number (the
    // empty asm hides that it is the same each time): kept across the merge of a cut tile, whose loads in
    // flight take 64 registers, 11 to 15 of them spilled to scratch memory.
    int tid = threadIdx.x;
    if constexpr (D == 128) {
      uint32_t lanes = 0xffffffffu;
      asm volatile("" : "+s"(lanes));
      tid = 64 * wv + __builtin_amdgcn_mbcnt_hi(lanes, __builtin_amdgcn_mbcnt_lo(lanes, 0u));
    }
    const int lane = tid & 63, h = lane >> 5, c32 = lane & 31;
    // every chunk of the thread has dims 8 dc0 .. + 7 (kPfThreads is a multiple of CPP)
    const int dc0 = tid % CPP;
    const uint32_t koff = (uint32_t)(lane / CPP * sk_tok) * 2u + 16u * dc0;
    const uint32_t voff = (uint32_t)(lane / CPP * sv_tok) * 2u + 16u * dc0;
    // The transposing read (ds_read_b64_tr_b16): in each 16-lane group, lane j's four results are
    // element j % 4 of the 4-element rows that lanes 4 m + j / 4 address, m = 0..3.  So that lane L
    // receives positions 16 s + 4 h + m of dim 32 db + L % 32, lane L addresses position
    // 16 s + 4 (L / 32) + (L % 16) / 4, dims 32 db + 16 ((L / 16) % 2) + 4 (L % 4) .. + 3.
    const int tr_pos = 4 * (lane >> 5) + ((lane & 15) >> 2);
    const int tr_dim = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    // the lane's column: token tok, head hd
    const int c = wv * 32 + c32;
    const int tok = c / G, hd = c % G;
    const int take = (int)(u1 - u < t.steps - off ? u1 - u : t.steps - off);
    // visible positions of the lane's column (-1: a padding column, never written)
    int kvl = -1;
    if (c < BQ * G && tok < t.nq) {
      const int kl = t.kv_pos0 + tok + 1 < t.lt ? t.kv_pos0 + tok + 1 : t.lt;
      kvl = kl > 0 ? kl : 0;
    }
    const bool live = __ballot(kvl >= 0) != 0ull;   // a wave of padding columns only loads rows
    const int j0 = off * kPfPos;
    const int j1 = t.lt < j0 + take * kPfPos ? t.lt : j0 + take * kPfPos;
    const int kend = kvl < j1 ? kvl : j1;   // the column's positions below kend are visible here
    // the smallest kend of the wave's columns (padding columns aside): positions below it are
    // visible to every column of the wave
    int kend_w = kvl >= 0 ? kend : INT32_MAX;
#pragma unroll
    for (int sh = 1; sh < 64; sh <<= 1) kend_w = min(kend_w, __shfl_xor(kend_w, sh));
    const int32_t* bt_row = p.bt + (int64_t)t.seq * p.sbt;
    const char* kbase = reinterpret_cast<const char*>(p.k) + (int64_t)kvh * p.sk_head * 2;
    const char* vbase = reinterpret_cast<const char*>(p.v) + (int64_t)kvh * p.sv_head * 2;

    // Q^T operand: column c, dims 16 ks + 8 h .. + 7 (zeros for a padding column)
    vec qop[KS];
    {
      const int64_t qoff = (int64_t)(t.t0 + tok) * p.sq_tok + (int64_t)(kvh * G + hd) * p.sq_head;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        u32x4 x = {0u, 0u, 0u, 0u};
        if (kvl >= 0) x = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(p.q) + (qoff + 16 * ks + 8 * h) * 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = (x[i] & f.q_and) ^ f.q_xor;
        qop[ks] = __builtin_bit_cast(vec, x);
      }
    }

    // Position j's entry of the block table and its offset in the block; the table is read one
    // step ahead of the rows, the rows one step ahead of the products.  Chunk r of the thread is
    // position (tid + kPfThreads r) / CPP of a step.
    auto split = [&](int j, int& o) -> int {
      int bi;
      if (BW || p.bs_shift >= 0) { bi = j >> p.bs_shift; o = j & (p.block_size - 1); }
      else { bi = j / p.block_size; o = j - bi * p.block_size; }
      return bi;
    };
    u32x4 kreg[LPT], vreg[LPT];
    int blk[LPT];
    uint32_t bad_rows = 0u;   // bit r: chunk r's block is invalid
    // the first position of the wave's group for chunk r of the step at jt; past the segment, its last group
    auto group_of = [&](int jt, int r) -> int { return min(jt + wv * PW + kPfThreads / CPP * r, (j1 - 1) & -PW); };
    auto load_entries = [&](int jt) {   // -1: past the table
#pragma unroll
      for (int r = 0; r < LPT; ++r) {
        int o;
        const int bi = split(BW ? group_of(jt, r) : min(jt + (tid + kPfThreads * r) / CPP, j1 - 1), o);
        blk[r] = bi < p.max_blocks_per_seq ? bt_row[bi] : -1;
      }
    };
    auto load_rows = [&](int jt) {
      bad_rows = 0u;
#pragma unroll
      for (int r = 0; r < LPT; ++r) {
        int o;
        split(BW ? group_of(jt, r) : min(jt + (tid + kPfThreads * r) / CPP, j1 - 1), o);
        int b = BW ? __builtin_amdgcn_readfirstlane(blk[r]) : blk[r];
        // an invalid entry of the segment (past its end, its last one again): block 0 stands in, the
        // rows are not used
        const bool bad = (uint32_t)b >= (uint32_t)p.num_blocks;
        b = bad ? 0 : b;
        bad_rows |= bad ? 1u << r : 0u;
        if constexpr (BW) {   // block strides below 2^31: one 32 x 32 bit product each
          kreg[r] = *reinterpret_cast<const u32x4*>(
              kbase + ((uint64_t)(uint32_t)b * (uint32_t)p.sk_blk + (uint32_t)(o * sk_tok)) * 2 + koff);
          vreg[r] = *reinterpret_cast<const u32x4*>(
              vbase + ((uint64_t)(uint32_t)b * (uint32_t)p.sv_blk + (uint32_t)(o * sv_tok)) * 2 + voff);
        } else {
          kreg[r] = *reinterpret_cast<const u32x4*>(kbase + ((int64_t)b * p.sk_blk + o * sk_tok) * 2 + 16 * dc0);
          vreg[r] = *reinterpret_cast<const u32x4*>(vbase + ((int64_t)b * p.sv_blk + o * sv_tok) * 2 + 16 * dc0);
        }
      }
      if (bad_rows != 0u) {
        s_bad = 1;
        if (p.status) atomicOr(p.status, NS_PA_STATUS_BAD_BLOCK);
      }
    };
    auto store_rows = [&](int jt, int buf) {
      if (bad_rows != 0u || jt + kPfPos > j1) {   // weight 0 times a row not of this sequence must be 0
#pragma unroll
        for (int r = 0; r < LPT; ++r)
          if (((bad_rows >> r) & 1u) || jt + (tid + kPfThreads * r) / CPP >= j1) vreg[r] = u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int r = 0; r < LPT; ++r) {
        const int pos = (tid + kPfThreads * r) / CPP;
        *reinterpret_cast<u32x4*>(s_k[buf] + pos * PK + dc0 * 16) = kreg[r];
        *reinterpret_cast<u32x4*>(s_v[buf] + pos * PV + dc0 * 16) = vreg[r];
      }
    };

    f32x16_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;
    float m = -INFINITY, l = 0.f;

    if (t.lt > 0) {
      if (tid == 0) s_bad = 0;
      __syncthreads();   // the flag is cleared, and an earlier segment's last step is read
      load_entries(j0);
      load_rows(j0);
      load_entries(j0 + kPfPos);
      store_rows(j0, 0);
      __syncthreads();
    }
    int buf = 0;
    for (int jt = j0; jt < j1; jt += kPfPos, buf ^= 1) {
      // the next step's rows and the table entries of the one after it, in flight across this
      // step's products and softmax
      const bool more = jt + kPfPos < j1;
      if (more) {
        load_rows(jt + kPfPos);
        load_entries(jt + 2 * kPfPos);
      }
      if (live) {
        const unsigned char* kt = s_k[buf] + c32 * PK + 16 * h;
        const unsigned char* vt = s_v[buf] + tr_pos * PV + tr_dim * 2;
        // S^T = K Q^T for the step's two 32-position row blocks (two independent MFMA chains)
        f32x16_t st[2];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int e = 0; e < 16; ++e) st[rb][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
          for (int rb = 0; rb < 2; ++rb) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(kt + 32 * rb * PK + 32 * ks);
            st[rb] = M::mma(__builtin_bit_cast(vec, x), qop[ks], st[rb]);
          }
        }
        // the online softmax of the lane's column over the step's 64 positions (element e of block
        // rb: position 32 rb + 8 (e / 4) + 4 h + e % 4; the other half in lane ^ 32)
        const bool bad = s_bad != 0;
        if (jt + kPfPos > kend_w || bad) {   // a position of the step hidden from a column
#pragma unroll
          for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int r = 32 * rb + 8 * (e >> 2) + 4 * h + (e & 3);
              st[rb][e] = jt + r < kend ? st[rb][e] : -INFINITY;
            }
          if (bad) {   // look the step's blocks up again
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const int j = jt + 32 * rb + 8 * (e >> 2) + 4 * h + (e & 3);
                int o;
                const int bi = split(j < j1 ? j : j1 - 1, o);
                const int b = bi < p.max_blocks_per_seq ? bt_row[bi] : -1;
                if (b < 0 || b >= p.num_blocks) st[rb][e] = -INFINITY;
              }
          }
        }
        float mt = -INFINITY;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int e = 0; e < 16; ++e) mt = fmaxf(mt, st[rb][e]);
        mt = fmaxf(mt, __shfl_xor(mt, 32)) * scale;
        // The column's reference m moves only for a score well above it (Mma): the accumulators are
        // rescaled rarely.  exp2 by v_exp_f32 (a weight below 2^-126 flushes to zero); -inf scores weigh 0,
        // and a column with no score yet subtracts 0.
        const bool move = mt > m + (M::kLift + M::kGap);
        const float mn = move ? mt - M::kLift : m;
        const float msub = mn == -INFINITY ? 0.f : mn;
        const float alpha = move ? __builtin_amdgcn_exp2f(m - msub) : 1.f;
        m = mn;
        if (__ballot(move) != 0ull) {   // a column's reference moved: rescale
          l *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[db][e] *= alpha;
        }
        // per 16-position k-step s: P as the hi / lo B operands, then O^T += V^T P^T with the V^T
        // operand of dim 32 db + c32 (k-slot i of half h at position 16 s + 8 (i / 4) + 4 h + i % 4)
        // read from the value rows by two transposing reads (k-slots 0-3, then 4-7)
        float ls = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          u32x4 wh, wl;
#pragma unroll
          for (int i2 = 0; i2 < 4; ++i2) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(st[s >> 1][8 * (s & 1) + 2 * i2], scale, -msub));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(st[s >> 1][8 * (s & 1) + 2 * i2 + 1], scale, -msub));
            ls += p0 + p1;
            wh[i2] = M::pack2(p0, p1);
            wl[i2] = M::pack2(p0 - M::lo(wh[i2]), p1 - M::hi(wh[i2]));
          }
          const vec phi = __builtin_bit_cast(vec, wh), plo = __builtin_bit_cast(vec, wl);
#pragma unroll
          for (int db = 0; db < DB; ++db) {
            const unsigned char* src = vt + 16 * s * PV + 64 * db;
            const u32x2 lo4 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                            (__attribute__((address_space(3))) i16x4*)(src)));
            const u32x2 hi4 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                            (__attribute__((address_space(3))) i16x4*)(src + 8 * PV)));
            const u32x4 x = {lo4[0], lo4[1], hi4[0], hi4[1]};
            const vec a = __builtin_bit_cast(vec, x);
            acc[db] = M::mma(a, phi, acc[db]);
            acc[db] = M::mma(a, plo, acc[db]);
          }
        }
        l += ls;   // this half's positions; the other half's sum is in lane ^ 32
      }
      if (more) store_rows(jt + kPfPos, buf ^ 1);
      __syncthreads();   // the next step staged, this one read
    }
    l += __shfl_xor(l, 32);

    // O^T layout: lane, element e -> column c, dim 32 db + 8 (e / 4) + 4 h + e % 4
    const int64_t obase = (int64_t)(t.t0 + tok) * p.so_tok + (int64_t)(kvh * G + hd) * p.so_head + 4 * h;
    auto write_out = [&](const f32x16_t (&o)[DB], float sum) {
      if (kvl < 0) return;
      const float inv = sum > 0.f ? 1.f / sum : 0.f;   // no visible key: zeros (the reference's l == 0 guard)
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = sum > 0.f ? o[db][4 * e4 + i] * inv : 0.f;
          const int64_t d = obase + 32 * db + 8 * e4;
          if (f.out_vec) {
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.out) + d) =
                u32x2{M::pack2(x[0], x[1]), M::pack2(x[2], x[3])};
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) store_one<T>(p.out, d + i, x[i]);
          }
        }
    };
    if (take == t.steps) {
      write_out(acc, l);
    } else {
      // A cut tile: this segment's partials to its slot (agent-scope stores: the segments' workgroups
      // run on different XCDs).  Workgroup i's slot for a tile begun by an earlier workgroup is i; for
      // a tile it begins and does not finish, grid + (i or the (tile, KV head), whichever are fewer).
      const int th = kvh * n_tiles + tile;
      const int64_t us = u - off;   // the tile's first unit
      const int wa = (int)(us / per), wb = (int)((us + t.steps - 1) / per);
      const int begin_slot = f.grid + (f.grid <= n_tiles * p.hkv ? wa : th);
      constexpr int SW = D / 2 * 64;   // floats of a slot per wave
      const int mine = w == wa ? begin_slot : w;
      if (live) {
        float* dst = f.ws_acc + ((int64_t)mine * kPfWaves + wv) * SW + 2 * lane;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int e = 0; e < 16; e += 2) st_dev2(dst + (db * 16 + e) * 64, acc[db][e], acc[db][e + 1]);
        if (h == 0) st_dev2(f.ws_ml + ((int64_t)mine * kPfCols + c) * 2, m, l);
      }
      // the last segment to arrive merges (the partials crossed through agent-scope atomic stores
      // completed by the s_waitcnt, read back through agent-scope loads)
      const int arrivals = wb - wa + 1;
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      int32_t* counter = f.counters + th;
      if (tid == 0) s_last = atomicAdd(counter, 1) == arrivals - 1;
      __syncthreads();
      if (s_last) {
        if (tid == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (live) {
          float mx = -INFINITY;
          for (int i = wa; i <= wb; ++i)
            mx = fmaxf(mx, ld_dev2(f.ws_ml + ((int64_t)(i == wa ? begin_slot : i) * kPfCols + c) * 2)[0]);
          float L = 0.f;
#pragma unroll
          for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;
          for (int i = wa; i <= wb; ++i) {
            const int64_t slot = __builtin_amdgcn_readfirstlane(i == wa ? begin_slot : i);
            const float* src = f.ws_acc + (slot * kPfWaves + wv) * SW + 2 * lane;
            const f32x2 ml = ld_dev2(f.ws_ml + (slot * kPfCols + c) * 2);
            f32x2 a[D / 4];   // all of a segment's loads issued before the first is used
#pragma unroll
            for (int e = 0; e < D / 4; ++e) a[e] = ld_dev2(src + e * 128);
            // a segment whose keys were all skipped (m = -inf) weighs 0
            const float wt = ml[0] == -INFINITY ? 0.f : exp2f(ml[0] - mx);
            L = fmaf(wt, ml[1], L);
#pragma unroll
            for (int e = 0; e < D / 4; ++e) {
              acc[e / 8][2 * (e % 8)] = fmaf(wt, a[e][0], acc[e / 8][2 * (e % 8)]);
              acc[e / 8][2 * (e % 8) + 1] = fmaf(wt, a[e][1], acc[e / 8][2 * (e % 8) + 1]);
            }
          }
          write_out(acc, L);
        }
      }
    }
    u += take;
    off = 0;
    ++tile;
  }
}

// ---- host side ---------------------------------------------------------------------------------

int pf_part_tokens_for(int32_t n_tiles, int32_t hkv, int32_t max_seq_len) {
  int part = kPfMaxPart;
  while (part > kPfMinPart) {
    const int64_t parts = ((int64_t)max_seq_len + part - 1) / part;
    if ((int64_t)n_tiles * hkv * parts >= kPfTargetGroups) break;
    part >>= 1;
  }
  return part;
}

// Workgroups that share the steps of the prefill tiles, or 0 for one workgroup per (tile, KV head):
// tiles are cut when the longest could be (max_seq_len above the partition length above, which
// shrinks while there are fewer than 512 of them).  512 workgroups are all resident at once, so
// equal shares end together.  Fewer, so that the slots they need stay within the partials' room
// of one slot per (tile, KV head, partition).  With few tiles that costs nothing throughout: one tile of
// 16 tokens, 24 / 8 heads of 128 dims, with this grid, and with one workgroup per (tile, KV head,
// partition) and the room it needs: 300 positions 18.0 and 22.7 us, 512 24.2 and 19.4, 600 21.5 and
// 23.8, 700 28.2 and 24.9, 1100 28.1 and 25.7 (a workgroup per partition of 256, before: 30.7 to 40.7).
int pf_grid_for(int32_t n_tiles, int32_t hkv, int32_t max_seq_len) {
  if (n_tiles <= 0) return 0;
  const int part = pf_part_tokens_for(n_tiles, hkv, max_seq_len);
  const int64_t parts = ((int64_t)max_seq_len + part - 1) / part;
  if (parts <= 1) return 0;
  const int64_t th = (int64_t)n_tiles * hkv;
  return (int)(th * (parts - 1) < kPfTargetGroups ? th * (parts - 1) : kPfTargetGroups);
}

// Bytes of the prefill tiles' partials (0 when no tile is cut): a slot per workgroup for a tile
// begun by another, and one per workgroup or (tile, KV head), whichever are fewer, for a tile begun
// and not finished.
uint64_t pf_workspace_bytes(int32_t n_tiles, int32_t hkv, int32_t head_dim, int32_t max_seq_len) {
  const int64_t grid = pf_grid_for(n_tiles, hkv, max_seq_len);
  if (grid == 0) return 0;
  const int64_t th = (int64_t)n_tiles * hkv;
  return (uint64_t)(grid + (grid < th ? grid : th)) * kPfCols * (head_dim + 2) * sizeof(float);
}

int part_tokens_for(int32_t total_q, int32_t hkv, int32_t max_seq_len) {
  int part = kMaxPart;
  while (part > kMinPart) {
    const int64_t parts = ((int64_t)max_seq_len + part - 1) / part;
    if ((int64_t)total_q * hkv * parts >= kTargetGroups) break;
    part >>= 1;
  }
  return part;
}

int check_sizes(int32_t total_q, int32_t hq, int32_t hkv, int32_t head_dim, int32_t max_seq_len) {
  if (total_q < 0) return fail("total_q must be >= 0 (got %d)", total_q);
  if (hq <= 0 || hkv <= 0 || hq % hkv != 0)
    return fail("num_heads_q (%d) must be a positive multiple of num_kv_heads (%d)", hq, hkv);
  const int g = hq / hkv;
  if (g != 1 && g != 2 && g != 3 && g != 4 && g != 8)
    return fail("query heads per KV head must be 1, 2, 3, 4 or 8 (got %d)", g);
  if (head_dim != 64 && head_dim != 128) return fail("head_dim must be 64 or 128 (got %d)", head_dim);
  if (max_seq_len < 0) return fail("max_seq_len must be >= 0 (got %d)", max_seq_len);
  if (hkv > 65535 || hq > 65535) return fail("too many heads (grid y is at most 65535)");
  return 0;
}

// Bytes of the per-token kernel's partials: total_q query slots (the kernel indexes them by query
// token), the partition length sized for the n_tokens workgroups along x.
uint64_t workspace_bytes(int32_t total_q, int32_t hq, int32_t hkv, int32_t head_dim, int32_t max_seq_len,
                         int32_t n_tokens) {
  const int part = part_tokens_for(n_tokens, hkv, max_seq_len);
  const int64_t max_parts = ((int64_t)max_seq_len + part - 1) / part;
  if (max_parts <= 1) return 0;
  return (uint64_t)total_q * hq * max_parts * (head_dim + 2) * sizeof(float);
}
uint64_t workspace_bytes(int32_t total_q, int32_t hq, int32_t hkv, int32_t head_dim, int32_t max_seq_len) {
  return workspace_bytes(total_q, hq, hkv, head_dim, max_seq_len, total_q);
}

// n_tokens decode workgroups along x (p.tokens or the first n_tokens tokens); the prefill tiles
// when f.tiles is set (16-bit types only)
template <typename T, int D, int G>
void launch(const PaParams& p, const PfParams& f, int n_tokens, int n_tiles, hipStream_t stream) {
  const dim3 grid(n_tokens, p.hkv, p.max_parts > 0 ? p.max_parts : 1);
  if constexpr (Elem<T>::bytes == 4) {
    if (n_tokens > 0) hipLaunchKernelGGL((pa_partition_kernel<D, G>), grid, dim3(kThreads), 0, stream, p);
  } else {
    // scalar row addresses: power-of-two blocks that hold a wave's load, block strides in 32 bits
    const bool by_wave = p.bs_shift >= 0 && p.block_size >= 512 / D && p.sk_blk >= 0 && p.sv_blk >= 0 &&
                         p.sk_blk < INT32_MAX && p.sv_blk < INT32_MAX;
    const dim3 tiles((unsigned)(f.grid > 0 ? f.grid : n_tiles * p.hkv));
    if (n_tokens > 0) {
      if (by_wave) hipLaunchKernelGGL((pa_decode_kernel<T, D, G, true>), grid, dim3(kThreads), 0, stream, p);
      else hipLaunchKernelGGL((pa_decode_kernel<T, D, G, false>), grid, dim3(kThreads), 0, stream, p);
    }
    if (n_tiles > 0) {
      if (by_wave) hipLaunchKernelGGL((pa_prefill_kernel<T, D, G, true>), tiles, dim3(kPfThreads), 0, stream, p, f);
      else hipLaunchKernelGGL((pa_prefill_kernel<T, D, G, false>), tiles, dim3(kPfThreads), 0, stream, p, f);
    }
  }
}

template <typename T, int D>
void launch_g(const PaParams& p, const PfParams& f, int n_tokens, int n_tiles, int g, hipStream_t stream) {
  switch (g) {
    case 1: launch<T, D, 1>(p, f, n_tokens, n_tiles, stream); break;
    case 2: launch<T, D, 2>(p, f, n_tokens, n_tiles, stream); break;
    case 3: launch<T, D, 3>(p, f, n_tokens, n_tiles, stream); break;
    case 4: launch<T, D, 4>(p, f, n_tokens, n_tiles, stream); break;
    default: launch<T, D, 8>(p, f, n_tokens, n_tiles, stream); break;
  }
}

template <typename T>
void launch_d(const PaParams& p, const PfParams& f, int n_tokens, int n_tiles, int d, int g, hipStream_t stream) {
  if (d == 64) launch_g<T, 64>(p, f, n_tokens, n_tiles, g, stream);
  else launch_g<T, 128>(p, f, n_tokens, n_tiles, g, stream);
}

}  // namespace

extern "C" {

int ns_pa_abi_version(void) { return NS_PA_ABI_VERSION; }

const char* ns_pa_last_error(void) { return g_err; }

int ns_paged_attention_workspace_bytes(int32_t total_q, int32_t num_heads_q, int32_t num_kv_heads,
                                       int32_t head_dim, int32_t max_seq_len, uint64_t* bytes) {
  if (!bytes) return fail("bytes is NULL");
  if (check_sizes(total_q, num_heads_q, num_kv_heads, head_dim, max_seq_len)) return 1;
  *bytes = workspace_bytes(total_q, num_heads_q, num_kv_heads, head_dim, max_seq_len);
  return 0;
}

int ns_paged_attention_call_workspace(const ns_paged_attn_args* a, uint64_t* bytes, uint64_t* counters) {
  if (!a || !bytes || !counters) return fail("a pointer argument is NULL");
  if (check_sizes(a->total_q, a->num_heads_q, a->num_kv_heads, a->head_dim, a->max_seq_len)) return 1;
  if (a->n_decode_tokens < 0 || a->n_prefill_tiles < 0) return fail("token and tile counts must be >= 0");
  const int32_t n_tokens = a->decode_tokens ? a->n_decode_tokens : a->total_q;
  const uint64_t dec =
      workspace_bytes(a->total_q, a->num_heads_q, a->num_kv_heads, a->head_dim, a->max_seq_len, n_tokens);
  const int32_t tiles = a->prefill_tiles ? a->n_prefill_tiles : 0;
  *bytes = dec + pf_workspace_bytes(tiles, a->num_kv_heads, a->head_dim, a->max_seq_len);
  *counters = (uint64_t)a->total_q * a->num_kv_heads + (uint64_t)tiles * a->num_kv_heads;
  return 0;
}

int ns_paged_attention(const ns_paged_attn_args* a, hipStream_t stream) {
  if (!a) return fail("args is NULL");
  if (check_sizes(a->total_q, a->num_heads_q, a->num_kv_heads, a->head_dim, a->max_seq_len)) return 1;
  if (a->dtype != NS_PA_DTYPE_F32 && a->dtype != NS_PA_DTYPE_BF16 && a->dtype != NS_PA_DTYPE_F16)
    return fail("dtype must be NS_PA_DTYPE_F32, _BF16 or _F16 (got %d)", a->dtype);
  if (a->total_q == 0) return 0;
  if (a->num_seqs <= 0) return fail("num_seqs must be > 0 when total_q > 0 (got %d)", a->num_seqs);
  if (a->block_size <= 0) return fail("block_size must be > 0 (got %d)", a->block_size);
  if (a->num_blocks <= 0) return fail("num_blocks must be > 0 (got %d)", a->num_blocks);
  if (!a->query || !a->k_cache || !a->v_cache || !a->out || !a->block_tables || !a->seq_lens ||
      !a->query_start_loc || !a->query_lens)
    return fail("a tensor pointer is NULL");
  const int esz = a->dtype == NS_PA_DTYPE_F32 ? 4 : 2;
  // 16-byte vector loads of each lane's head_dim/8 slice: rows and strides 16-byte aligned
  const int64_t strides[] = {a->stride_q_token, a->stride_q_head, a->stride_k_block, a->stride_k_token,
                             a->stride_k_head, a->stride_v_block, a->stride_v_token, a->stride_v_head};
  for (int64_t s : strides)
    if ((s * esz) % 16 != 0) return fail("query/cache strides must be multiples of 16 bytes");
  if (((uintptr_t)a->query | (uintptr_t)a->k_cache | (uintptr_t)a->v_cache) % 16 != 0)
    return fail("query and cache pointers must be 16-byte aligned");
  if (a->stride_bt_seq < 0) return fail("stride_bt_seq must be >= 0");
  if (a->stride_k_token < 0 || a->stride_v_token < 0 ||
      (int64_t)a->block_size * (a->stride_k_token > a->stride_v_token ? a->stride_k_token : a->stride_v_token) >=
          ((int64_t)1 << 31))
    return fail("token strides times block_size must lie in [0, 2^31)");
  if (a->max_blocks_per_seq < 0) return fail("max_blocks_per_seq must be >= 0");
  // the prefill tiles (16-bit types) and the token list of the per-token kernel
  if (a->n_decode_tokens < 0 || a->n_prefill_tiles < 0) return fail("token and tile counts must be >= 0");
  if (a->prefill_tiles && a->dtype == NS_PA_DTYPE_F32)
    return fail("prefill tiles take bfloat16 or float16 (float32 queries go through the per-token kernel)");
  if (a->prefill_tiles && !a->decode_tokens)
    return fail("a call with prefill tiles lists its other query tokens in decode_tokens");
  const int32_t n_tiles = a->prefill_tiles ? a->n_prefill_tiles : 0;
  const int32_t n_tokens = a->decode_tokens ? a->n_decode_tokens : a->total_q;
  const uint64_t need =
      workspace_bytes(a->total_q, a->num_heads_q, a->num_kv_heads, a->head_dim, a->max_seq_len, n_tokens);
  if (need > 0 && !a->counters) return fail("a call with split rows needs the zero-filled counters buffer");
  const int part = part_tokens_for(n_tokens, a->num_kv_heads, a->max_seq_len);
  const int64_t max_parts = ((int64_t)a->max_seq_len + part - 1) / part;
  if (max_parts > 65535) return fail("max_seq_len too large");
  const uint64_t pf_need = pf_workspace_bytes(n_tiles, a->num_kv_heads, a->head_dim, a->max_seq_len);
  if (need + pf_need > 0 && (!a->workspace || a->workspace_bytes < need + pf_need))
    return fail("workspace of %llu bytes needed (got %llu)", (unsigned long long)(need + pf_need),
                (unsigned long long)a->workspace_bytes);
  if (pf_need > 0 && !a->counters) return fail("a call with split tiles needs the zero-filled counters buffer");
  const int pf_part = pf_part_tokens_for(n_tiles, a->num_kv_heads, a->max_seq_len);
  const int64_t pf_max_parts = ((int64_t)a->max_seq_len + pf_part - 1) / pf_part;
  if (pf_max_parts > 65535) return fail("max_seq_len too large");

  PaParams p;
  p.q = a->query;
  p.k = a->k_cache;
  p.v = a->v_cache;
  p.out = a->out;
  p.bt = a->block_tables;
  p.seq_lens = a->seq_lens;
  p.qsl = a->query_start_loc;
  p.qlens = a->query_lens;
  p.status = a->status;
  // no room of its own (the workspace may still be there for the tiles): a row longer than max_seq_len
  // allows is flagged and leaves no partials
  p.ws_acc = need ? reinterpret_cast<float*>(a->workspace) : nullptr;
  p.ws_ml = need ? p.ws_acc + (uint64_t)a->total_q * a->num_heads_q * max_parts * a->head_dim : nullptr;
  p.counters = a->counters;
  p.sq_tok = a->stride_q_token;
  p.sq_head = a->stride_q_head;
  p.sk_blk = a->stride_k_block;
  p.sk_tok = a->stride_k_token;
  p.sk_head = a->stride_k_head;
  p.sv_blk = a->stride_v_block;
  p.sv_tok = a->stride_v_token;
  p.sv_head = a->stride_v_head;
  p.so_tok = a->stride_o_token;
  p.so_head = a->stride_o_head;
  p.sbt = a->stride_bt_seq;
  p.num_seqs = a->num_seqs;
  p.hq = a->num_heads_q;
  p.hkv = a->num_kv_heads;
  p.block_size = a->block_size;
  p.bs_shift = -1;
  if ((a->block_size & (a->block_size - 1)) == 0)
    for (int sh = 0; sh < 31; ++sh)
      if ((1 << sh) == a->block_size) p.bs_shift = sh;
  p.num_blocks = a->num_blocks;
  p.max_blocks_per_seq = a->max_blocks_per_seq;
  p.part_tokens = part;
  p.max_parts = (int32_t)max_parts;
  p.scale_log2 = a->scale * kLog2e;
  p.total_q = a->total_q;
  p.tokens = a->decode_tokens;

  PfParams f;
  f.tiles = a->prefill_tiles;
  char* ws = reinterpret_cast<char*>(a->workspace);
  f.grid = pf_grid_for(n_tiles, a->num_kv_heads, a->max_seq_len);
  if (((uintptr_t)a->workspace + need) % 8 != 0) f.grid = 0;   // the partials go in 8-byte pieces
  f.n_tiles = n_tiles;
  f.ws_acc = pf_need ? reinterpret_cast<float*>(ws + need) : nullptr;
  f.ws_ml = pf_need ? f.ws_acc + pf_need / sizeof(float) / (a->head_dim + 2) * a->head_dim : nullptr;
  f.counters = a->counters ? a->counters + (int64_t)a->total_q * a->num_kv_heads : nullptr;
  f.cap = (pf_max_parts > 0 ? pf_max_parts : 1) * pf_part;
  f.scale_log2 = a->scale == 0.f ? 1.f : fabsf(a->scale) * kLog2e;
  f.q_and = a->scale == 0.f ? 0u : 0xffffffffu;
  f.q_xor = a->scale < 0.f ? 0x80008000u : 0u;
  f.out_vec = (uintptr_t)a->out % 8 == 0 && a->stride_o_token % 4 == 0 && a->stride_o_head % 4 == 0;

  const int g = a->num_heads_q / a->num_kv_heads;
  switch (a->dtype) {
    case NS_PA_DTYPE_F32: launch_d<float>(p, f, n_tokens, 0, a->head_dim, g, stream); break;
    case NS_PA_DTYPE_BF16: launch_d<Bf16>(p, f, n_tokens, n_tiles, a->head_dim, g, stream); break;
    default: launch_d<F16>(p, f, n_tokens, n_tiles, a->head_dim, g, stream); break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail("kernel launch failed: %s", hipGetErrorString(e));
  return 0;
}

}  // extern "C"
