// attn_exact.hip -- ATTN_QK -> causal SOFTMAX -> ATTN_KQV in the reference's
// own operation order (src/ops_cpu.cpp:304-410), bit for bit:
//
//   S_i  = sum_d K[d, kvh, i] * Q[d, h, j]     d ascending, product and sum
//                                              each rounded (no fused multiply-add)
//   v_i  = S_i * scale;  m = max_i v_i         i < a = min(n_past + j + 1, n_kv)
//   e_i  = expf(v_i - m)                       the host C library's expf (libm_ref.h)
//   sum  = sum_i e_i                           i ascending
//   P_i  = e_i * (1 / sum)
//   O[o] = sum_t V[o, kvh, t] * P_t            t ascending (masked t add +-0, skipped)
//
// The order leaves two chains of a dependent additions per row (8.4 cycles
// each: 3.5 ns), the sum of the exponentials and an output element's sum;
// everything else is independent and is taken off them. Short rows run one
// workgroup per row with all its K, then V rows in LDS
// (attn_exact_staged_kernel); few longer rows (a decode step) one workgroup
// per row that shortens the chains (attn_exact_row_kernel); many (a prompt) one
// row per wave, whose workgroups share the K and V tiles and fill the chip
// (attn_exact_tile_kernel); of many rows too long for those, some run one row
// per wave on its own (attn_exact_wave_kernel).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_common.h"
#include "kernels.h"

#define MI_LIBM_HD __host__ __device__
#include "libm_ref.h"

namespace mi {

static __constant__ uint64_t kExpfTab[32] = MI_EXPF_TABLE;

namespace {
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// 16 bytes per lane from each lane's address into LDS at lds + 16 * lane
// (kept out of templates: the host pass drops a kernel template whose body
// names the builtin directly).
__device__ __forceinline__ void dma16_from(const char* p, lds_t* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// s + p[0] + p[1] + ... + p[n - 1] (n a multiple of 16, p 16-byte aligned), one
// rounded addition each, in order; chunk c + 1 of 16 terms is read from LDS
// between chunk c's additions (a dependent addition takes 8.4 cycles and
// issues in 4.6, so the reads cost the chain nothing). Reads up to 16 floats
// past n (never added).
__device__ __forceinline__ float exact_sum(const lds_t* p, int n, float s) {
#pragma clang fp contract(off)
  f32x4_t x[4], y[4];
  auto get = [&](f32x4_t (&b)[4], int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) b[u] = lds_load<f32x4_t>(p + 64 * c + 16 * u);
  };
  auto add = [&](const f32x4_t (&b)[4], f32x4_t (&next)[4], int c) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s = s + b[u].x;
      next[u] = lds_load<f32x4_t>(p + 64 * c + 16 * u);
      s = s + b[u].y;
      s = s + b[u].z;
      s = s + b[u].w;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);  // an addition
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a read
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int nch = n >> 4;
  get(x, 0);
  int c = 0;
  for (; c + 1 < nch; c += 2) {
    add(x, y, c + 1);
    add(y, x, c + 2);
  }
  if (c < nch) add(x, y, c);
  return s;
}

// acc + p[0] + p[S] + ... + p[(n - 1) S] (p in LDS, S floats apart), in order,
// read two chunks of 16 ahead (a column of 64 lanes is 256 bytes a term: its
// reads are further away than one chunk's additions). Reads rows up to the
// next multiple of 16 past n (never added).
template <int S>
__device__ __forceinline__ float exact_column(const lds_t* p, int n, float acc) {
#pragma clang fp contract(off)
  float x[3][16];
  auto get = [&](float (&b)[16], int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 16; ++u) b[u] = lds_load<float>(p + 4 * S * (16 * c + u));
  };
  auto add = [&](const float (&b)[16], float (&next)[16], int c) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      acc = acc + b[u];
      next[u] = lds_load<float>(p + 4 * S * (16 * c + u));
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);  // an addition
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a read
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int nch = n >> 4, last = (n - 1) >> 4;  // whole chunks; the last chunk
  get(x[0], 0);
  get(x[1], min(1, last));
  int c = 0;
  for (; c + 2 < nch; c += 3) {
    add(x[0], x[2], c + 2);
    add(x[1], x[0], min(c + 3, last));
    add(x[2], x[1], min(c + 4, last));
  }
  if (c < nch) {
    add(x[0], x[2], min(c + 2, last));
    if (c + 1 < nch) add(x[1], x[0], min(c + 3, last));
  }
  for (int t = 16 * nch; t < n; ++t) acc = acc + lds_load<float>(p + 4 * S * t);
  return acc;
}

// Output element o (its lane's, in aligned groups of 32 lanes) of row (j, h).
__device__ __forceinline__ void store_out(const ExactAttn& p, int j, int h, int o, float v) {
  if (p.blocks) {
    float d;
    const int q = q8_lane_quant(v, d);
    const int e = h * p.head_dim + o;
    char* const blk = p.out + (int64_t)j * p.o_s2 + 36 * (e / 32);
    if ((e & 31) == 0) gstore<float>(blk, d);
    gstore<signed char>(blk + 4 + (e & 31), (signed char)q);
  } else {
    gstore<float>(p.out + h * p.o_s1 + (int64_t)j * p.o_s2 + 4 * o, v);
  }
}

// Rows row0 .. row0 + n - 1 of one KV head (past `last`: row `last` again) into
// LDS, n * D / 4 a multiple of 64, by NW waves of which this is the w-th: whole
// 1 KB requests; 16-byte slots XOR-swizzled by row if SW, so that one row per
// lane reads free of bank conflicts. A wave's requests are NW / 4 x 64 / D x 16
// rows apart: an address is the one before plus a constant (a computed one
// cost 20 instructions a request), but for the slot where the swizzle does not
// repeat.
template <int D, int NW, bool SW>
__device__ __forceinline__ void rows_to_lds(lds_t* dst, const char* base, int64_t s2, int row0, int n, int last,
                                            int w, int lane) {
  constexpr int PPR = D / 4;  // 16-byte pieces per row
  constexpr int STEP = kWave * NW / PPR;
  const int slot = lane % PPR;
  int r = (kWave * w + lane) / PPR;
  int col = 16 * (SW ? slot ^ swz<PPR>(r) : slot);
  auto next = [&]() __attribute__((always_inline)) {
    r += STEP;
    if (SW && STEP % 16 != 0) col = 16 * (slot ^ swz<PPR>(r));
  };
  if (row0 + n - 1 <= last) {
    const char* p = base + (int64_t)(row0 + r) * s2;
    for (int i0 = kWave * w; i0 < n * PPR; i0 += kWave * NW) {
      dma16_from(p + col, dst + 16 * i0);
      p += STEP * s2;
      next();
    }
  } else {
    for (int i0 = kWave * w; i0 < n * PPR; i0 += kWave * NW) {
      dma16_from(base + (int64_t)min(row0 + r, last) * s2 + col, dst + 16 * i0);
      next();
    }
  }
}

// A workgroup past the rows: its share of what the next launches read, pieces
// of its own XCD (the same workgroup number modulo 8).
template <int T>
__device__ __forceinline__ void warm_up(const ExactAttnWarm& p) {
  const int n_rows = p.n_tokens * p.n_head;
  const int xcd = blockIdx.x % 8, first = (n_rows + 7 - xcd) / 8, per_xcd = ((int)gridDim.x + 7 - xcd) / 8 - first;
  for (int w = 0, c = blockIdx.x / 8 - first; w < kMaxWarmUps; ++w) {
    const int n = (p.warm[w].n + 7 - xcd) / 8;  // pieces of this XCD
    for (; c < n; c += per_xcd)
      warm_lines(p.warm[w].p + (int64_t)(xcd + 8 * c) * p.warm[w].bytes, p.warm[w].bytes, threadIdx.x, T);
    c -= n;
  }
}
}  // namespace

// ---------------------------------------------------------------------------
// One workgroup of 4 waves per (token, head), for short rows: all K rows come
// into LDS and the threads form one key's score each from there; then three
// waves bring the V rows over the K rows while wave 0 forms the maximum, the
// exponentials and their ordered sum; then each output element's lane runs its
// ordered V sum from LDS. Fewer barriers than the kernel below and nothing to
// divide, which is what short rows take their time for (a launch takes 3.4 us
// with 16 keys, where the row kernel takes 5.3), at the price of LDS for a
// whole row's V and of the sums' whole chains (7 ns a key and chain).
constexpr int kStagedThreads = 256;
constexpr int kStagedWaves = kStagedThreads / kWave;

// The V rows (whole 1 KB requests) and the probabilities have 16 entries of
// room past n_kv: the ordered sums read the chunk past the last whole one too.
__host__ __device__ inline int staged_v_bytes(int n_kv, int d) { return ((n_kv + 16) * d * 4 + 1023) & ~1023; }
__host__ __device__ inline int staged_prob_bytes(int n_kv) { return 4 * (((n_kv + 15) & ~15) + 16); }
inline int staged_lds_bytes(int n_kv, int d) { return staged_v_bytes(n_kv, d) + staged_prob_bytes(n_kv) + 256 + 32; }

// acc + v[0] * p[0] + v[D] * p[1] + ... + v[(n - 1) D] * p[n - 1], each
// product and sum rounded (v: one output element's column of V rows D floats
// apart; 16 rows and probabilities readable past n). The products do not
// depend on the running sum: chunk c + 1's 16 are formed between chunk c's
// additions, so each addition waits only for the one before it, not for a
// multiplication issued just before it. (The same products, added in the
// same order: the same bits.)
template <int D>
__device__ __forceinline__ float exact_dot(const lds_t* v, const lds_t* p, int n) {
#pragma clang fp contract(off)
  float acc = 0.0f;
  float va[16], vb[16];
  f32x4_t pa[4], pb[4];
  float ra[16], rb[16];  // products
  auto get = [&](float (&vv)[16], f32x4_t (&pp)[4], int c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 16; ++u) vv[u] = lds_load<float>(v + 4 * D * (16 * c + u));
#pragma unroll
    for (int u = 0; u < 4; ++u) pp[u] = lds_load<f32x4_t>(p + 64 * c + 16 * u);
  };
  auto prod = [&](float (&r)[16], const float (&vv)[16], const f32x4_t (&pp)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r[4 * u] = vv[4 * u] * pp[u].x;
      r[4 * u + 1] = vv[4 * u + 1] * pp[u].y;
      r[4 * u + 2] = vv[4 * u + 2] * pp[u].z;
      r[4 * u + 3] = vv[4 * u + 3] * pp[u].w;
    }
  };
  // chunk r's additions, chunk (vv, pp)'s products into rn between them
  auto add_prod = [&](const float (&r)[16], float (&rn)[16], const float (&vv)[16], const f32x4_t (&pp)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      acc = acc + r[4 * u];
      rn[4 * u] = vv[4 * u] * pp[u].x;
      acc = acc + r[4 * u + 1];
      rn[4 * u + 1] = vv[4 * u + 1] * pp[u].y;
      acc = acc + r[4 * u + 2];
      rn[4 * u + 2] = vv[4 * u + 2] * pp[u].z;
      acc = acc + r[4 * u + 3];
      rn[4 * u + 3] = vv[4 * u + 3] * pp[u].w;
    }
  };
  auto add = [&](const float (&r)[16]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 16; ++t) acc = acc + r[t];
  };
  const int nch = n >> 4;
  if (nch > 0) {
    get(va, pa, 0);
    prod(ra, va, pa);
    if (nch > 1) get(vb, pb, 1);
    int c = 0;
    // ra: chunk c's products; vb, pb: chunk c + 1's values
    for (; c + 2 < nch; c += 2) {
      get(va, pa, c + 2);
      __builtin_amdgcn_sched_barrier(0);
      add_prod(ra, rb, vb, pb);
      get(vb, pb, c + 3);  // (c + 3 <= nch: at most the chunk past the last whole one)
      __builtin_amdgcn_sched_barrier(0);
      add_prod(rb, ra, va, pa);
    }
    if (c + 1 < nch) {
      add_prod(ra, rb, vb, pb);
      add(rb);
    } else {
      add(ra);
    }
  }
  for (int t = 16 * nch; t < n; ++t) acc = acc + lds_load<float>(v + 4 * D * t) * lds_load<float>(p + 4 * t);
  return acc;
}

template <int D, typename P>
__global__ __launch_bounds__(kStagedThreads) void attn_exact_staged_kernel(const P p) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) char ex_lds[];
  lds_t* const lds = (lds_t*)ex_lds;
  constexpr int PPR = D / 4;               // 16-byte pieces per row
  constexpr int kWhole = kWave / PPR;      // rows per request
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  // every parameter in one round of scalar loads, not one where each is first used
  asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.q_s1), "s"(p.q_s2), "s"(p.k_s1), "s"(p.k_s2), "s"(p.v_s1),
               "s"(p.v_s2), "s"(p.n_head), "s"(p.n_rep), "s"(p.n_past), "s"(p.n_tokens), "s"(p.scale), "s"(p.out),
               "s"(p.o_s1), "s"(p.o_s2), "s"(p.blocks));
  if constexpr (std::is_same<P, ExactAttnWarm>::value)
    if ((int)blockIdx.x >= p.n_tokens * p.n_head) {
      warm_up<kStagedThreads>(p);
      return;
    }
  const int h = blockIdx.x % p.n_head;
  const int j = p.n_tokens - 1 - blockIdx.x / p.n_head;  // the longest rows first
  const int kvh = h / p.n_rep;
  const int a = p.n_past + j + 1, n_kv = p.n_past + p.n_tokens;
  lds_t* const rows = lds;  // K, later V
  lds_t* const prob = lds + staged_v_bytes(n_kv, D);
  lds_t* const tab = prob + staged_prob_bytes(n_kv);
  lds_t* const red = tab + 256;
  const uint64_t te = kExpfTab[lane & 31];  // requested first: loads complete in order
  const int n_req = (a + kWhole - 1) & ~(kWhole - 1);  // rows requested
  rows_to_lds<D, kStagedWaves, true>(rows, p.k + kvh * p.k_s1, p.k_s2, 0, n_req, a - 1, wv, lane);
  // the query meanwhile (a uniform address: scalar loads)
  const char* q = p.q + h * p.q_s1 + (int64_t)j * p.q_s2;
  f32x4_t qv[PPR];
#pragma unroll
  for (int u = 0; u < PPR; ++u) qv[u] = *(const __attribute__((address_space(4))) f32x4_t*)(q + 16 * u);
  wait_vmem<0>();  // this wave's K requests have landed
  wg_barrier();
  // one key's score per thread, d ascending, product and sum each rounded
  float mx = -INFINITY;
  for (int i = tid; i < a; i += kStagedThreads) {
    const lds_t* const rowp = rows + i * (4 * D);
    // the D products first (independent), then their sum in order
    float pr[D];
#pragma unroll
    for (int u = 0; u < PPR; ++u) {
      const f32x4_t kv = lds_load<f32x4_t>(rowp + 16 * (u ^ swz<PPR>(i)));
      pr[4 * u] = kv.x * qv[u].x;
      pr[4 * u + 1] = kv.y * qv[u].y;
      pr[4 * u + 2] = kv.z * qv[u].z;
      pr[4 * u + 3] = kv.w * qv[u].w;
    }
    float acc = 0.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) acc = acc + pr[d];
    const float v = acc * p.scale;
    lds_store<float>(prob + 4 * i, v);
    mx = v > mx ? v : mx;
  }
  mx = wave_max_dpp(mx);  // (never NaN; the sign of a zero maximum changes no exponential)
  if (tid < 32) lds_store<uint64_t>(tab + 8 * tid, te);
  if (lane == 0) lds_store<float>(red + 4 * wv, mx);
  wg_barrier();  // the scores are in LDS and every K row has been read
  if (wv > 0) {
    rows_to_lds<D, kStagedWaves - 1, false>(rows, p.v + kvh * p.v_s1, p.v_s2, 0, n_req, a - 1, wv - 1, lane);
    wait_vmem<0>();  // this wave's V requests have landed
  } else {
    mx = lds_load<float>(red);
#pragma unroll
    for (int w = 1; w < kStagedWaves; ++w) {
      const float o = lds_load<float>(red + 4 * w);
      mx = o > mx ? o : mx;
    }
    // zeros past the keys, up to a whole chunk: they leave the sum unchanged
    const int n_pad = (a + 15) & ~15;
    for (int i = lane; i < n_pad; i += kWave) {
      const float x = lds_load<float>(prob + 4 * i) - mx;
      lds_store<float>(prob + 4 * i,
                       i < a ? expf_ref(x, (const __attribute__((address_space(3))) uint64_t*)tab) : 0.0f);
    }
    wave_lds_fence();
    const float sum = exact_sum(prob, n_pad, 0.0f);
    if (lane == 0) lds_store<float>(red + 16, (float)(1.0 / (double)sum));  // the correctly rounded 1.0f / sum
  }
  wg_barrier();  // the V rows and 1 / sum
  const float inv = lds_load<float>(red + 16);
  for (int i = tid; i < a; i += kStagedThreads) lds_store<float>(prob + 4 * i, lds_load<float>(prob + 4 * i) * inv);
  wg_barrier();
  if (tid < D) store_out(p, j, h, tid, exact_dot<D>(rows + 4 * tid, prob, a));
}

// ---------------------------------------------------------------------------
// One workgroup per (token, head), for longer rows.
//
// Scores: K rows come through two LDS buffers, one key per thread. The sum of
// the exponentials is cut into 8 segments, one per wave, run from 64 candidate
// start values each (as ordered_sum_lds_8waves states), so the chain is an
// eighth as long. The output elements' chains are bare additions in one wave
// (two at D = 128): four other waves form the products P_t V[t] into LDS, a
// chunk ahead.
//
// Measured (14 / 2 heads, D 64, us per launch; before: the staged kernel up to
// 512 keys, a wave of its own per row beyond): n_kv 301 9.6 -> 8.6, 1001 38.5 ->
// 17.4, 1501 75.4 -> 24.5, 8001 391 -> 122. At 1501 the output chains take 10.5
// (7 ns a key, 4.2 of them the addition itself), the scores 6.7 (LDS-direct
// requests bring about 55 GB/s into a CU, and a row has one CU), the
// exponentials and their sum 2.7.
constexpr int kRowThreads = 512;
constexpr int kRowWaves = kRowThreads / kWave;
constexpr int kRowLoaders = 4;          // waves that form the products
constexpr int kRowWork = 256 + 64 + 64 + kRowWaves * kWave * 4;  // expf's table, maxima, segment sums, ends
constexpr int kLdsMax = 160 * 1024;

// floats of the probabilities: 8 segments of whole 16s, 16 readable past them
__host__ __device__ inline int row_segment(int n) { return ((n + 7) / 8 + 15) & ~15; }
__host__ __device__ inline int row_prob_bytes(int n) { return 4 * (8 * row_segment(n) + 16); }
inline int row_lds_bytes(int n, int buf) { return row_prob_bytes(n) + kRowWork + 2 * buf; }
static_assert(4 * (kExactMaxKeys + 16) + kRowWork + 2 * 14 * 1024 <= kLdsMax, "the longest row fits");

// BUF: bytes of a buffer of K rows (two, whole requests of every wave), later
// of CK rows of products.
template <int D, int BUF, int CK, typename P>
__global__ __launch_bounds__(kRowThreads) void attn_exact_row_kernel(const P p) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) char ex_lds[];
  lds_t* const lds = (lds_t*)ex_lds;
  constexpr int PPR = D / 4;
  constexpr int KB = BUF / (4 * D);                       // keys per buffer
  constexpr int kReq = BUF / (1024 * kRowWaves);          // requests per wave and buffer, at least
  static_assert(BUF % 1024 == 0 && kReq > 0 && KB <= kRowThreads, "whole requests, a key per thread");
  static_assert(CK % 16 == 0 && 4 * CK * D <= BUF, "whole chunks of products in a buffer");
  constexpr int NV = CK * PPR / (kRowLoaders * kWave);    // pieces of V per loader thread and buffer
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  // every parameter in one round of scalar loads, not one where each is first used
  asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.q_s1), "s"(p.q_s2), "s"(p.k_s1), "s"(p.k_s2), "s"(p.v_s1),
               "s"(p.v_s2), "s"(p.n_head), "s"(p.n_rep), "s"(p.n_past), "s"(p.n_tokens), "s"(p.scale));
  if constexpr (std::is_same<P, ExactAttnWarm>::value)
    if ((int)blockIdx.x >= p.n_tokens * p.n_head) {
      warm_up<kRowThreads>(p);
      return;
    }
  const int h = blockIdx.x % p.n_head;
  const int j = p.n_tokens - 1 - blockIdx.x / p.n_head;  // the longest rows first
  const int kvh = h / p.n_rep;
  const int a = p.n_past + j + 1;
  const int L = row_segment(a);
  lds_t* const prob = lds;
  lds_t* const tab = lds + row_prob_bytes(p.n_past + p.n_tokens);
  lds_t* const red = tab + 256;
  lds_t* const segsum = red + 64;
  lds_t* const ends = segsum + 64;
  lds_t* const buf = tab + kRowWork;
  const char* const kbase = p.k + kvh * p.k_s1;
  const char* const vbase = p.v + kvh * p.v_s1;
  const uint64_t te = kExpfTab[lane & 31];
  const float* q = reinterpret_cast<const float*>(p.q + h * p.q_s1 + (int64_t)j * p.q_s2);
  f32x4_t qv[PPR];
#pragma unroll
  for (int u = 0; u < PPR; ++u) qv[u] = gload<f32x4_t>(q + 4 * u);
  auto request = [&](int k0, int s, int n) __attribute__((always_inline)) {
    rows_to_lds<D, kRowWaves, true>(buf + s * BUF, kbase, p.k_s2, k0, n, a - 1, wv, lane);
  };
  // one key's score, d ascending, product and sum each rounded
  float mx = -INFINITY;
  auto score = [&](int key, const lds_t* rowp, int row) __attribute__((always_inline)) {
    float acc = 0.0f;
    // 64 products first (they do not depend on one another), then their sum
#pragma unroll
    for (int u0 = 0; u0 < PPR; u0 += 16) {
      f32x4_t pr[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const f32x4_t kv = lds_load<f32x4_t>(rowp + 16 * ((u0 + u) ^ swz<PPR>(row)));
        pr[u] = f32x4_t{kv.x * qv[u0 + u].x, kv.y * qv[u0 + u].y, kv.z * qv[u0 + u].z, kv.w * qv[u0 + u].w};
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        acc = acc + pr[u].x;
        acc = acc + pr[u].y;
        acc = acc + pr[u].z;
        acc = acc + pr[u].w;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const float v = acc * p.scale;
    lds_store<float>(prob + 4 * key, v);
    mx = v > mx ? v : mx;
  };
  if (2 * KB <= kRowThreads && a <= 2 * KB) {
    // both buffers at once, a key per thread (whole requests of 1 KB)
    constexpr int kWhole = kWave / PPR;  // rows per request
    const int n = (a + kWhole - 1) & ~(kWhole - 1);
    request(0, 0, min(n, KB));
    if (n > KB) request(KB, 1, n - KB);
    // V is asked for only after the scores: a dword of each of its 128-byte
    // lines now, so that they are in L2 by then. The wait below counts these
    // loads as the wave's latest: the fence keeps them behind the requests
    // (and the wait, which clobbers memory too, keeps them before it).
    asm volatile("" ::: "memory");
    constexpr int kLines = D / 32, kTouch = (2 * KB * kLines + kRowThreads - 1) / kRowThreads;
    unsigned vt[kTouch];
#pragma unroll
    for (int u = 0; u < kTouch; ++u) {
      const int i = min(tid + u * kRowThreads, a * kLines - 1);
      vt[u] = gload<unsigned>(vbase + (int64_t)(i / kLines) * p.v_s2 + 128 * (i % kLines));
    }
    wait_vmem<kTouch>();  // the K rows
    wg_barrier();
    // (the buffers are adjacent; a row's slots are swizzled by its place in its own)
    if (tid < a) score(tid, buf + tid * (4 * D), tid < KB ? tid : tid - KB);
#pragma unroll
    for (int u = 0; u < kTouch; ++u) asm volatile("" ::"v"(vt[u]));
  } else {
    request(0, 0, KB);
    request(KB, 1, KB);  // (past the row: its last key, never used)
    for (int k0 = 0, s = 0; k0 < a; k0 += KB, s ^= 1) {
      wait_vmem<kReq>();  // this wave's requests for the buffer (and the query) have landed
      wg_barrier();       // and everyone's
      if (tid < KB && k0 + tid < a) score(k0 + tid, buf + s * BUF + tid * (4 * D), tid);
      if (k0 + KB < a) {
        wg_barrier();  // the buffer has been read
        request(k0 + 2 * KB, s, KB);
      }
    }
    // the last requests are past the row, but they are writes all the same:
    // the products overwrite their buffers
    wait_vmem<0>();
  }
  if (tid < 32) lds_store<uint64_t>(tab + 8 * tid, te);
  // the first V rows meanwhile, in the loaders' registers, two buffers ahead
  // (waves 2, 3, 6 and 7: not on the SIMDs of the chains' waves 0 and 1)
  const bool loader = (wv & 2) != 0;
  const int lt = ((wv >> 2) * 2 + (wv & 1)) * kWave + lane;
  f32x4_t vr[2][NV];
  auto load_v = [&](f32x4_t (&x)[NV], int t0) __attribute__((always_inline)) {
    constexpr int STEP = kRowLoaders * kWave / PPR;  // rows between a thread's pieces
    const int r = t0 + lt / PPR;
    if (t0 + CK <= a) {
      const char* v = vbase + (int64_t)r * p.v_s2 + 16 * (lt % PPR);
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        x[u] = gload<f32x4_t>(v);
        v += STEP * p.v_s2;
      }
    } else {
#pragma unroll
      for (int u = 0; u < NV; ++u)
        x[u] = gload<f32x4_t>(vbase + (int64_t)min(r + u * STEP, a - 1) * p.v_s2 + 16 * (lt % PPR));
    }
  };
  if (loader) {
    load_v(vr[0], 0);
    load_v(vr[1], CK);
  }
  mx = wave_max_dpp(mx);  // (never NaN; the sign of a zero maximum changes no exponential)
  if (lane == 0) lds_store<float>(red + 4 * wv, mx);
  wg_barrier();  // the scores and the waves' maxima
  mx = lds_load<float>(red);
#pragma unroll
  for (int w = 1; w < kRowWaves; ++w) {
    const float o = lds_load<float>(red + 4 * w);
    mx = o > mx ? o : mx;
  }
  // each wave its segment's exponentials, and their sum in double, which
  // places the candidates
  lds_t* const seg = prob + 4 * L * wv;
  double qs = 0.0;
  for (int i = lane; i < L; i += kWave) {
    const float x = lds_load<float>(seg + 4 * i) - mx;
    const float e = L * wv + i < a ? expf_ref(x, (const __attribute__((address_space(3))) uint64_t*)tab) : 0.0f;
    lds_store<float>(seg + 4 * i, e);
    qs += (double)e;
  }
  qs = wave_sum_f64(qs);
  if (lane == 0) lds_store<double>(segsum + 8 * wv, qs);
  wg_barrier();
  int base[kRowWaves];
  double pre = 0.0;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) {
    const int gb = __builtin_bit_cast(int, (float)pre);
    base[w] = gb > 32 ? gb - 32 : 0;
    pre += lds_load<double>(segsum + 8 * w);
  }
  int my_base = base[0];
#pragma unroll
  for (int w = 1; w < kRowWaves; ++w) my_base = wv == w ? base[w] : my_base;
  lds_store<float>(ends + 4 * (kWave * wv + lane), exact_sum(seg, L, __builtin_bit_cast(float, my_base + lane)));
  wg_barrier();
  float e[kRowWaves], sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) e[w] = lds_load<float>(ends + 4 * (kWave * w + lane));
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) {
    const int c = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, sum) - base[w]);
    if (c >= 0 && c < kWave)
      sum = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, e[w]), c));
    else
      sum = exact_sum(prob + 4 * L * w, L, sum);
  }
  const float inv = (float)(1.0 / (double)sum);  // the correctly rounded 1.0f / sum
  // products by the loaders, chains by the first waves, a buffer apart
  if (tid < D) __builtin_amdgcn_s_setprio(3);
  float acc = 0.0f;
  auto chunk = [&](int t0, f32x4_t (&x)[NV], lds_t* b) __attribute__((always_inline)) {
    if (loader) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int i = u * kRowLoaders * kWave + lt, row = i / PPR;
        const float pt = lds_load<float>(prob + 4 * min(t0 + row, a - 1)) * inv;
        lds_store<f32x4_t>(b + 16 * i, f32x4_t{x[u].x * pt, x[u].y * pt, x[u].z * pt, x[u].w * pt});
      }
      load_v(x, t0 + 2 * CK);
    }
    wg_barrier();
    if (tid < D) acc = exact_column<D>(b + 4 * tid, min(CK, a - t0), acc);
  };
  for (int t0 = 0; t0 < a; t0 += 2 * CK) {
    chunk(t0, vr[0], buf);
    if (t0 + CK < a) chunk(t0 + CK, vr[1], buf + BUF);
  }
  if (tid < D) store_out(p, j, h, tid, acc);
}

// ---------------------------------------------------------------------------
// Many rows: the T n_rep rows (token, head) of one KV head, one per wave, W
// waves per workgroup. Tiles of 64 keys come through two LDS buffers, first all
// of K, then all of V, each request a tile ahead. Per tile a wave forms its
// row's scores with one key per lane (the query is uniform: scalar loads),
// later the row's sums with one output element per lane (two at D = 128); in
// between, the ordered sum of the exponentials. (Two rows a wave, sharing its
// reads: 128 tokens 10.1 us, with one 7.4, 384 tokens 23.8 and 19.7.)
//
// The vector units and LDS reads bound it: two vector instructions per product
// (the order forbids the fused one), 4 D per (row, key) in all, and every
// operand of them read from LDS or through scalar loads. Measured (14 / 2
// heads, D 64, us; before: a workgroup with its own copy of K and V per row):
// 128 tokens 10.9 -> 7.4, 384 tokens 123.8 -> 19.7.
constexpr int kTileKeys = 64;
// floats per row of scores: whole tiles, plus 4 so that the waves' rows start
// in different banks (and 16 readable past the last)
__host__ __device__ inline int tile_row_floats(int n) { return ((n + 63) & ~63) + 4; }
template <int D, int W>
constexpr int tile_lds_bytes(int n) {
  return 2 * kTileKeys * D * 4 + 256 + 4 * W * tile_row_floats(n) + 64;
}

template <int D, int W>
__global__ __launch_bounds__(W* kWave) void attn_exact_tile_kernel(const ExactAttn p, int n_tiles) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) char ex_lds[];
  lds_t* const lds = (lds_t*)ex_lds;
  constexpr int PPR = D / 4, kBuf = kTileKeys * D * 4, ND = D / kWave;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int n_hkv = p.n_head / p.n_rep;
  const int kvh = blockIdx.x % n_hkv;
  const int n_rows = p.n_tokens * p.n_rep;
  const int tile = n_tiles - 1 - blockIdx.x / n_hkv;  // the longest rows first
  const int np = tile_row_floats(p.n_past + p.n_tokens);
  lds_t* const tab = lds + 2 * kBuf;
  lds_t* const sc = tab + 256 + 4 * np * wv;  // this wave's scores
  const char* const kbase = p.k + kvh * p.k_s1;
  const char* const vbase = p.v + kvh * p.v_s1;
  // the wave's row (past the last: the last again, not stored) and its keys
  const int r = min(tile * W + wv, n_rows - 1), j = r / p.n_rep, h = kvh * p.n_rep + (r - j * p.n_rep);
  const int a = p.n_past + j + 1;
  const char* const q = p.q + h * p.q_s1 + (int64_t)j * p.q_s2;
  const int a_wg = p.n_past + min((tile + 1) * W - 1, n_rows - 1) / p.n_rep + 1;
  const int nt = (a_wg + kTileKeys - 1) / kTileKeys;
  const uint64_t te = kExpfTab[lane & 31];
  if (tid < 32) lds_store<uint64_t>(tab + 8 * tid, te);
  auto request = [&](int s) __attribute__((always_inline)) {
    lds_t* const b = lds + (s & 1) * kBuf;
    if (s < nt)
      rows_to_lds<D, W, true>(b, kbase, p.k_s2, s * kTileKeys, kTileKeys, a_wg - 1, wv, lane);
    else
      rows_to_lds<D, W, false>(b, vbase, p.v_s2, (s - nt) * kTileKeys, kTileKeys, a_wg - 1, wv, lane);
  };
  request(0);
  float mx = -INFINITY;
  for (int s = 0; s < nt; ++s) {
    wait_vmem<0>();
    wg_barrier();  // tile s has landed, and everyone has left the other buffer
    request(s + 1);
    const int k0 = s * kTileKeys;
    if (k0 >= a) continue;
    const lds_t* const rowp = lds + (s & 1) * kBuf + lane * (4 * D);
    float acc = 0.0f;
#pragma unroll
    for (int u0 = 0; u0 < PPR; u0 += 4) {
      f32x4_t kv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) kv[u] = lds_load<f32x4_t>(rowp + 16 * ((u0 + u) ^ swz<PPR>(lane)));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // uniform address: a scalar load
        const f32x4_t qv = *(const __attribute__((address_space(4))) f32x4_t*)(q + 16 * (u0 + u));
        acc = acc + kv[u].x * qv.x;
        acc = acc + kv[u].y * qv.y;
        acc = acc + kv[u].z * qv.z;
        acc = acc + kv[u].w * qv.w;
      }
    }
    const float v = acc * p.scale;
    lds_store<float>(sc + 4 * (k0 + lane), v);
    mx = k0 + lane < a && v > mx ? v : mx;
  }
  // exponentials, zeros past the row's keys (they leave its sum unchanged)
  const int n_pad = (a + 15) & ~15;
  mx = wave_max_dpp(mx);  // (never NaN; the sign of a zero maximum changes no exponential)
  for (int t = lane; t < n_pad; t += kWave) {
    const float x = lds_load<float>(sc + 4 * t) - mx;
    lds_store<float>(sc + 4 * t, t < a ? expf_ref(x, (const __attribute__((address_space(3))) uint64_t*)tab) : 0.0f);
  }
  wave_lds_fence();
  const float sum = exact_sum(sc, n_pad, 0.0f);
  const float inv = (float)(1.0 / (double)sum);  // the correctly rounded 1.0f / sum
  for (int t = lane; t < n_pad; t += kWave) lds_store<float>(sc + 4 * t, lds_load<float>(sc + 4 * t) * inv);
  wave_lds_fence();
  float acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = 0.0f;
  for (int s = 0; s < nt; ++s) {
    wait_vmem<0>();
    wg_barrier();
    if (s + 1 < nt) request(nt + s + 1);
    const int k0 = s * kTileKeys;
    const lds_t* const vb = lds + ((nt + s) & 1) * kBuf + 4 * lane;
    const lds_t* const pb = sc + 4 * k0;
    // the row's keys of the tile, 4 at a time, then the others one by one
    const int n1 = min(a - k0, kTileKeys), n4 = max(n1, 0) >> 2;
#pragma unroll 4
    for (int t4 = 0; t4 < n4; ++t4) {
      float v[4][ND];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int d = 0; d < ND; ++d) v[t][d] = lds_load<float>(vb + (4 * t4 + t) * (4 * D) + 4 * kWave * d);
      const f32x4_t pr = lds_load<f32x4_t>(pb + 16 * t4);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int d = 0; d < ND; ++d) acc[d] = acc[d] + v[t][d] * pr[t];
    }
    for (int t = 4 * n4; t < n1; ++t) {
      const float pt = lds_load<float>(pb + 4 * t);
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[d] = acc[d] + lds_load<float>(vb + t * (4 * D) + 4 * kWave * d) * pt;
    }
  }
  if (tile * W + wv < n_rows) {
#pragma unroll
    for (int d = 0; d < ND; ++d) store_out(p, j, h, kWave * d + lane, acc[d]);
  }
}

// ---------------------------------------------------------------------------
// One wave per (token, head), its probabilities alone in LDS: lanes split the
// keys, then the output elements, straight from memory. Slow for one row (its
// chains wait for every read), but a CU holds as many rows as its LDS has room
// for: see long_form.
__global__ __launch_bounds__(kWave) void attn_exact_wave_kernel(const ExactAttn p) {
#pragma clang fp contract(off)
  extern __shared__ float prob[];
  __shared__ float s_inv;
  const int lane = threadIdx.x;
  const int h = blockIdx.x % p.n_head;
  const int j = blockIdx.x / p.n_head;
  const int kvh = h / p.n_rep;
  const int D = p.head_dim;
  const int a = min(p.n_past + j + 1, p.n_past + p.n_tokens);
  const float* q = reinterpret_cast<const float*>(p.q + h * p.q_s1 + (int64_t)j * p.q_s2);
  float mx = -INFINITY;
  for (int i = lane; i < a; i += kWave) {
    const float* kr = reinterpret_cast<const float*>(p.k + kvh * p.k_s1 + (int64_t)i * p.k_s2);
    float acc = 0.0f;
#pragma unroll 16  // (the row's loads in flight together)
    for (int d = 0; d < D; d += 4) {
      const float4 kv = *reinterpret_cast<const float4*>(kr + d);
      const float4 qv = *reinterpret_cast<const float4*>(q + d);
      acc = acc + kv.x * qv.x;
      acc = acc + kv.y * qv.y;
      acc = acc + kv.z * qv.z;
      acc = acc + kv.w * qv.w;
    }
    const float v = acc * p.scale;
    prob[i] = v;
    mx = v > mx ? v : mx;
  }
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const float o = __shfl_xor(mx, off);
    mx = o > mx ? o : mx;
  }
  for (int i = lane; i < a; i += kWave) prob[i] = expf_ref(prob[i] - mx, kExpfTab);
  __syncthreads();
  if (lane == 0) {
    float sum = 0.0f;
    for (int i = 0; i < a; ++i) sum = sum + prob[i];
    s_inv = (float)(1.0 / (double)sum);  // the correctly rounded 1.0f / sum
  }
  __syncthreads();
  const float inv = s_inv;
  for (int i = lane; i < a; i += kWave) prob[i] = prob[i] * inv;
  __syncthreads();
  const char* vbase = p.v + kvh * p.v_s1;
  for (int o = lane; o < D; o += kWave) {
    float acc = 0.0f;
#pragma unroll 16  // (16 keys' loads in flight ahead of the ordered additions)
    for (int t = 0; t < a; ++t)
      acc = acc + *reinterpret_cast<const float*>(vbase + (int64_t)t * p.v_s2 + 4 * o) * prob[t];
    store_out(p, j, h, o, acc);
  }
}


// Workgroups past the rows: what is to be warmed up gets the idle CUs, two
// pieces each.
static int side_workgroups(const ExactAttn&, int) { return 0; }
static int side_workgroups(const ExactAttnWarm& p, int n_cu) {
  int64_t pieces = 0;
  for (const WarmUp& w : p.warm) pieces += w.n;
  return (int)std::min<int64_t>(std::max(n_cu - p.n_tokens * p.n_head, 0) & ~7, (pieces + 15) / 16 * 8);
}

template <int D, typename P>
static hipError_t launch_staged(const P& p, int n_cu, hipStream_t stream) {
  const auto fn = &attn_exact_staged_kernel<D, P>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
  if (attr != hipSuccess) return attr;
  const int rows = p.n_tokens * p.n_head;
  hipLaunchKernelGGL(fn, dim3((unsigned)(rows + side_workgroups(p, n_cu))), dim3(kStagedThreads),
                     (unsigned)staged_lds_bytes(p.n_past + p.n_tokens, D), stream, p);
  return hipGetLastError();
}

template <int D, int BUF, int CK, typename P>
static hipError_t launch_row(const P& p, int n_cu, hipStream_t stream) {
  const auto fn = &attn_exact_row_kernel<D, BUF, CK, P>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
  if (attr != hipSuccess) return attr;
  const int rows = p.n_tokens * p.n_head;
  hipLaunchKernelGGL(fn, dim3((unsigned)(rows + side_workgroups(p, n_cu))), dim3(kRowThreads),
                     (unsigned)row_lds_bytes(p.n_past + p.n_tokens, BUF), stream, p);
  return hipGetLastError();
}
template <int D, typename P>
static hipError_t launch_row(const P& p, int n_cu, hipStream_t stream) {
  // the largest buffers that fit beside the probabilities; short rows start
  // their chains after half as many products
  const int n_kv = p.n_past + p.n_tokens;
  if (n_kv <= 512) return launch_row<D, 64 * 1024, 4096 / D>(p, n_cu, stream);
  if (row_lds_bytes(n_kv, 64 * 1024) <= kLdsMax) return launch_row<D, 64 * 1024, 8192 / D>(p, n_cu, stream);
  if (row_lds_bytes(n_kv, 32 * 1024) <= kLdsMax) return launch_row<D, 32 * 1024, 8192 / D>(p, n_cu, stream);
  // (28 heads of 128, us a launch: 24001 keys 1523, with buffers of 8 KB 2690;
  // 32001 keys 2040, 3590. From 32129 keys on the buffers are of 14 KB.)
  if (row_lds_bytes(n_kv, 16 * 1024) <= kLdsMax) return launch_row<D, 16 * 1024, 4096 / D>(p, n_cu, stream);
  return launch_row<D, 14 * 1024, D == 64 ? 48 : 16>(p, n_cu, stream);
}

template <int D, int W>
static hipError_t launch_tile(const ExactAttn& p, hipStream_t stream) {
  static const hipError_t attr = hipFuncSetAttribute((const void*)&attn_exact_tile_kernel<D, W>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax);
  if (attr != hipSuccess) return attr;
  const int n_tiles = (p.n_tokens * p.n_rep + W - 1) / W;
  const unsigned lds = (unsigned)tile_lds_bytes<D, W>(p.n_past + p.n_tokens);
  hipLaunchKernelGGL((attn_exact_tile_kernel<D, W>), dim3((unsigned)(n_tiles * (p.n_head / p.n_rep))),
                     dim3(W * kWave), lds, stream, p, n_tiles);
  return hipGetLastError();
}

static hipError_t launch_wave(const ExactAttn& p, hipStream_t stream) {
  static const hipError_t attr = hipFuncSetAttribute((const void*)&attn_exact_wave_kernel,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kExactMaxKeys * 4);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(attn_exact_wave_kernel, dim3((unsigned)(p.n_tokens * p.n_head)), dim3(kWave),
                     4 * (unsigned)(p.n_past + p.n_tokens), stream, p);
  return hipGetLastError();
}

// Rows whose scores do not fit in LDS eight to a workgroup (about 4000 keys of
// 64 elements, 3000 of 128), more than there are CUs: the row kernel runs one a
// CU, tiles of 4 rows run 4 (to 8128 keys, 6080), the wave kernel as many as
// LDS has room for, each the slower the more they are. What a round of each
// takes, in ns a key, measured on launches of 20 to 128 tokens x 14 heads of 64
// and 28 of 128 after 3200 to 16000 keys, which it says the faster form of. us,
// row / tile / wave: 14 heads of 64, 20 tokens after 4300 113 / 163 / 196, 100
// (wave) 324 / 319 / 307, 128 (tile) 399 / 328 / 364; 28 of 128, 40 after 4300
// (tile) 593 / 484 / 533, after 7600 (wave) 1341 / - / 935, after 8200 (row)
// 1446 / - / 1717.
enum class LongForm { kRow, kTile, kWave };
template <int D>
static LongForm long_form(int n_kv, int64_t rows, int n_cu) {
  const int64_t per_cu = kLdsMax / (4 * n_kv), whole = rows / (n_cu * per_cu);
  const double rest = (double)(rows - whole * n_cu * per_cu) / n_cu;
  auto rounds = [](int64_t n, int64_t at_once) { return (double)((n + at_once - 1) / at_once); };
  auto wave_round = [](double at_once) { return D == 64 ? 40 + 6 * at_once : 77 + 10 * at_once; };
  const bool whole_buffers = row_lds_bytes(n_kv, 64 * 1024) <= kLdsMax;
  const double row = rounds(rows, n_cu) * (D == 64 ? (whole_buffers ? 14 : 15) : (whole_buffers ? 28.5 : 36));
  const double wave = whole * wave_round((double)per_cu) + (rest > 0 ? wave_round(rest) : 0);
  const double tile = tile_lds_bytes<D, 4>(n_kv) <= kLdsMax ? rounds(rows, 4 * n_cu) * (D == 64 ? 38 : 57) : row + 1;
  if (row <= tile && row <= wave) return LongForm::kRow;
  return tile <= wave ? LongForm::kTile : LongForm::kWave;
}

// Short rows: as many as run at once (LDS, and 5 or 3 waves' registers per
// SIMD) and, where every row has a CU, up to the length at which the row kernel
// overtakes. us, staged against row or tile: 1 row x 14 heads of 64, n_kv 16
// 3.4 / 5.3, 128 4.9 / 6.3, 256 6.8 / 7.7, 301 8.7 / 8.5; 28 heads of 128, 257
// 10.3 / 14.4 (301 no longer fits). Heads of 64, 19 rows after 256 8.6 / 13.4,
// 64 after 40 5.8 / 7.2, 96 after 40 (more than run at once) 9.4 / 8.8; of 128,
// 24 after 0 5.2 / 5.8, 32 after 0 7.8 / 6.0.
template <int D>
static bool staged_form(int n_kv, int64_t rows, int n_cu) {
  const int per_cu = kLdsMax / staged_lds_bytes(n_kv, D);
  if (rows <= n_cu) return D == 64 ? n_kv <= 256 : per_cu > 0;
  return rows <= (int64_t)n_cu * std::min(per_cu, D == 64 ? 4 : 3);
}

template <int D>
static hipError_t launch(const ExactAttn& p, int n_cu, hipStream_t stream) {
  const int n_kv = p.n_past + p.n_tokens;
  const int64_t rows = (int64_t)p.n_tokens * p.n_head;
  if (staged_form<D>(n_kv, rows, n_cu)) return launch_staged<D>(p, n_cu, stream);
  // Rows that get a CU each take a workgroup each (14 rows of 1501 keys: 24.5
  // us, 57 in tiles); more share tiles (128 tokens x 14 heads: 7.4 us, 41 a row
  // per workgroup).
  if (rows <= n_cu) return launch_row<D>(p, n_cu, stream);
  if (tile_lds_bytes<D, 8>(n_kv) <= kLdsMax) return launch_tile<D, 8>(p, stream);
  switch (long_form<D>(n_kv, rows, n_cu)) {
    case LongForm::kTile:
      return launch_tile<D, 4>(p, stream);
    case LongForm::kWave:
      return launch_wave(p, stream);
    default:
      return launch_row<D>(p, n_cu, stream);
  }
}

template <int D>
static hipError_t launch(const ExactAttnWarm& p, int n_cu, hipStream_t stream) {
  const int64_t rows = (int64_t)p.n_tokens * p.n_head;
  if (rows > n_cu) return launch<D>(static_cast<const ExactAttn&>(p), n_cu, stream);  // (no CU is idle)
  return staged_form<D>(p.n_past + p.n_tokens, rows, n_cu) ? launch_staged<D>(p, n_cu, stream)
                                                          : launch_row<D>(p, n_cu, stream);
}

hipError_t launch_attn_exact(const ExactAttn& p, int n_cu, hipStream_t stream) {
  n_cu = n_cu > 0 ? n_cu : 256;
  return p.head_dim == 64 ? launch<64>(p, n_cu, stream) : launch<128>(p, n_cu, stream);
}
hipError_t launch_attn_exact_warm(const ExactAttnWarm& p, int n_cu, hipStream_t stream) {
  n_cu = n_cu > 0 ? n_cu : 256;
  return p.head_dim == 64 ? launch<64>(p, n_cu, stream) : launch<128>(p, n_cu, stream);
}

}  // namespace mi
