// mul_mat_cols.hip -- MI_OP_MUL_MAT with Q8_0 weights for several activation
// columns (a prompt's tokens), on the matrix cores, bit for bit the engine's
// dot product (mul_mat.hip states its order): accumulator l (0..7) of an
// output takes fma(float(int8 dot of bytes 4l..4l+3 of the block), w.d * a.d,
// acc_l) block by block, then ((a0 + a4) + (a1 + a5)) + ((a2 + a6) + (a3 + a7)).
//
// The accumulator chains are what the order asks for: one float multiply-add
// per 4 products, so k n m / 4 of them, on the vector units. Everything else
// is taken off those units. A dot of 4 int8 is exact in f16 products summed
// in float (at most 2^16), so v_mfma_f32_16x16x4_4b_f16, four independent
// 16 x 16 products with K = 4, gives float(dot) of 4 byte groups of 256
// outputs at once, with no integer dot and no conversion per output; the
// scale products w.d * a.d (one rounded float product, plus zero) come from
// v_mfma_f32_16x16x1_4b_f32, 4 blocks at once. What is left beside the
// multiply-adds is the int8 -> f16 conversion of the operands, once per
// workgroup on their way into LDS.
//
// Measured (MI355X, us, the product alone in launches back to back; before: one
// wave per 8 rows with integer dots, weight rows in LDS, 8 columns at a time):
// 4864 x 896 with 512 columns 532 -> 35, 9728 x 896 with 128 163 -> 19.5, 896 x
// 4864 with 128 542 -> 15.6, with 37 161 -> 13.2, with 8 36 -> 13.1; 896 x 896
// with 128 129 -> 5.8, with 8 (the streaming form) 15.1 -> 5.1. 512 columns take
// 14 us of multiply-adds at one per 4 cycles and SIMD; issue slots (conversions,
// products, LDS) fill the rest: a lone wave issues an instruction every 5 cycles
// or so.
#include <algorithm>
#include <type_traits>

#include "attn_common.h"
#include "kernels.h"

namespace mi {
namespace {

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
// bytes of a weight block (34 bytes, 2-byte aligned) and of an activation
// block (36 bytes, 4-byte aligned)
typedef unsigned u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u32_a2 __attribute__((aligned(2)));

// f(0), f(1), .. f(N - 1) with the index a compile-time constant (so that
// arrays indexed by it stay in registers).
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

constexpr int kKB = 4;  // 32-element blocks per stage

// Four int8 as f16, exactly: v + 128 as the low mantissa bits of 1024.0, then
// minus 1152.
__device__ __forceinline__ f16x4_t i8_to_f16(unsigned x) {
  const unsigned y = x ^ 0x80808080u;
  const unsigned lo = __builtin_amdgcn_perm(0x64646464u, y, 0x04010400u);
  const unsigned hi = __builtin_amdgcn_perm(0x64646464u, y, 0x04030402u);
  const f16x2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
  const f16x2_t a = __builtin_bit_cast(f16x2_t, lo) - bias, b = __builtin_bit_cast(f16x2_t, hi) - bias;
  return f16x4_t{a.x, a.y, b.x, b.y};
}

// (kept out of templates: the host pass drops a kernel template whose body
// names the builtin directly)
// Four 16 x 16 products at once, K = 4 each: register 4 b + r of lane (c, g) =
// (lane % 16, lane / 16) is the dot of the 4 values that lane (4g + r, b)
// holds in a with the 4 that lane (c, b) holds in b.
__device__ __forceinline__ f32x16_t dot4_tiles(f16x4_t a, f16x4_t b) {
  const f32x16_t zero = {};
  return __builtin_amdgcn_mfma_f32_16x16x4f16(a, b, zero, 0, 0, 0);
}
// the same with K = 1: the (rounded) products of two scales
__device__ __forceinline__ f32x16_t scale_tiles(float a, float b) {
  const f32x16_t zero = {};
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 0, 0, 0);
}

// The multiply-adds of one sub-tile and stage: acc[l][r] is the chain of the
// wave's l-th accumulator (of 4 NQ) of (column 4g + r, row c). Each product is
// issued before the multiply-adds of the one before it.
template <int NQ>
__device__ __forceinline__ void stage_fma(float (&acc)[4 * NQ][4], const f16x4_t (&a)[kKB][NQ],
                                          const f16x4_t (&b)[kKB][NQ], float sa, float sb) {
  const f32x16_t d = scale_tiles(sa, sb);
  f32x16_t t[2];
  t[0] = dot4_tiles(a[0][0], b[0][0]);
  static_for<kKB * NQ>([&](auto n_) __attribute__((always_inline)) {
    constexpr int n = n_, m = n + 1 < kKB * NQ ? n + 1 : n;
    if constexpr (m != n) t[m & 1] = dot4_tiles(a[m / NQ][m % NQ], b[m / NQ][m % NQ]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float& s = acc[(v / 4) * NQ + n % NQ][v % 4];
      s = __builtin_fmaf(t[n & 1][v], d[4 * (n / NQ) + v % 4], s);
    }
    __builtin_amdgcn_sched_barrier(0);
  });
  // (the sums exist here: otherwise they are moved into the next stage, with
  // every product they need)
#pragma unroll
  for (int l = 0; l < 4 * NQ; ++l) asm volatile("" : "+v"(acc[l][0]), "+v"(acc[l][1]), "+v"(acc[l][2]), "+v"(acc[l][3]));
}

// (row, 4 columns from col): one lane's finished outputs. Lane c has row `row`,
// lane c ^ 1 the other row of its RoPE pair (stored rows 2j and 2j + 1).
__device__ __forceinline__ void store_cols(const Q8MulMat& p, int64_t row, int64_t col, const float (&out)[4]) {
#pragma clang fp contract(off)
  const bool live = row < p.n;
  float v[4];
  const char* const ad = p.add + row * p.add_nb0;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = p.add && live && col + r < p.m ? out[r] + gload<float>(ad + (col + r) * p.add_nb1) : out[r];
  char* d;
  int64_t step;
  if (p.rope_on) {
    const RopeEpi& re = p.rope;
    const int r0 = (int)row, qk_rows = re.n_q + re.n_kv, h = r0 / re.hd, w = r0 - h * re.hd;
    float other[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) other[r] = dpp_mov<0xB1>(v[r]);  // quad_perm [1,0,3,2]
    if (!live) return;
    const bool odd = w & 1;
    if (r0 < qk_rows) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (col + r < p.m) {
          const f32x2_t cs = gload<f32x2_t>(re.cs + 2 * ((re.pos + col + r) * (re.hd / 2) + w / 2));
          const float c = cs.x, s = cs.y;
          const float x0 = odd ? other[r] : v[r], x1 = odd ? v[r] : other[r];
          v[r] = odd ? x0 * s + x1 * c : x0 * c - x1 * s;
        }
    }
    const int e = r0 < qk_rows ? (w >> 1) + odd * (re.hd / 2) : w;
    if (r0 < re.n_q) {
      d = reinterpret_cast<char*>(re.q_out + h * re.hd + e);
      step = 4 * re.q_ld;
    } else {
      d = (r0 < qk_rows ? re.k_row + (h - re.n_q / re.hd) * re.c_s1 : re.v_row + (h - qk_rows / re.hd) * re.c_s1) + 4 * e;
      step = re.c_s2;
    }
  } else {
    if (!live) return;
    d = p.dst + q8_unperm_row(row, p.perm_hd, p.perm_rows) * p.dst_nb0;
    step = p.dst_nb1;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (col + r < p.m) gstore<float>(d + (col + r) * step, v[r]);
}

}  // namespace

// A workgroup computes 16 WI NI columns x 16 WJ NJ rows: WI x WJ waves (LS = 2:
// pairs of waves, each with half of an output's accumulators), NI x NJ
// sub-tiles of 16 x 16 per wave. A stage of 4 blocks goes from memory through
// registers (PD stages ahead) into LDS, converted to f16 on the way, in the
// order of the products' operands: lane (c, g) of block b reads its 16 bytes
// at kBlkB b + kGrpB g + 16 c, conflict-free for the reads and for the staging
// writes. With PW = 0 the multiplying waves stage; otherwise PW waves of their
// own do nothing else, which shortens the stage of a launch too small to fill
// the chip (896 x 4864 with 8 columns 17.9 -> 13.8 us) and costs a full one.
constexpr int kGrpB = 16 * 16 + 16, kBlkB = 4 * kGrpB;
constexpr int kSubB = kKB * kBlkB;  // the operands of 16 columns or rows
template <int WI, int WJ, int NI, int NJ, int LS, int PW>
struct TileShape {
  static constexpr int kC = WI * WJ * LS;                  // waves that multiply
  static constexpr int kT = (kC + PW) * kWave;
  static constexpr int kTS = (PW ? PW : kC) * kWave;       // threads that stage
  static constexpr int kIS = WI * NI, kJS = WJ * NJ;       // sub-tiles
  static constexpr int kM = 16 * kIS, kN = 16 * kJS;
  static constexpr int kScale = (kIS + kJS) * kSubB;       // [sub-tile][block][row] floats
  static constexpr int kBuf = kScale + (kIS + kJS) * 16 * kKB * 4;
};
template <int WI, int WJ, int NI, int NJ, int LS, int PD, int OCC, int PW>
__global__ __launch_bounds__((WI * WJ * LS + PW) * kWave, OCC) void mul_mat_q8_0_tile_kernel(const Q8MulMat p, int n_jt,
                                                                                   int n_it) {
#pragma clang fp contract(off)
  typedef TileShape<WI, WJ, NI, NJ, LS, PW> S;
  constexpr int T = S::kTS, NQ = 2 / LS;
  extern __shared__ __attribute__((aligned(16))) char tile_lds[];
  lds_t* const lds = (lds_t*)tile_lds;
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int ls = wv % LS, wj = (wv / LS) % WJ, wi = wv / (LS * WJ);
  // the column tiles of one row tile run on one XCD one after another, so
  // that the weight rows are read from HBM once and then from its L2
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const int jt = xcd + 8 * (slot / n_it), it = slot % n_it;
  if (jt >= n_jt) return;
  const int64_t row0 = (int64_t)jt * S::kN, col0 = (int64_t)it * S::kM;
  const int nblk = (int)(p.k / 32), n_st = (nblk + kKB - 1) / kKB;
  const int c = lane & 15, g = lane >> 4;
  // Stage st starts at block min(4 st, nblk - 4): the last one's blocks that
  // the stage before had already get zero scales, so that they add +-0.0 (a
  // sum is never -0.0); so do the missing blocks of a row of fewer than 4.
  // Rows, columns and blocks past the end re-read the last one.
  const int n_again = n_st * kKB - nblk;
  // Staging units over the tile's columns, then its rows: 16 bytes (half a
  // block), and one block's scale (the dword it is in)
  constexpr int R = S::kM + S::kN;
  constexpr int NU = (R * 2 * kKB + T - 1) / T, NV = (R * kKB + T - 1) / T;
  constexpr bool kWholeU = R * 2 * kKB % T == 0, kWholeV = R * kKB % T == 0;
  struct Src {
    const char* p;
    unsigned blk;  // bytes of a block
    int at;        // where it goes in a buffer, -1: nowhere
  } su[NU], sv[NV];
  auto source = [&](int r, int block) __attribute__((always_inline)) {
    const bool w = r >= S::kM;
    block = min(block, nblk - 1);
    const int64_t i = w ? min<int64_t>(row0 + r - S::kM, p.n - 1) : min<int64_t>(col0 + r, p.m - 1);
    Src x;
    x.p = w ? p.w + i * p.w_nb1 + 34 * block : p.a + i * p.a_nb1 + 36 * block;
    x.blk = w ? 34 : 36;
    return x;
  };
  const int stager = (int)threadIdx.x - (PW ? S::kC * kWave : 0);
  const int vb = stager & (kKB - 1);
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int id = max(u * T + stager, 0), r = min(id / (2 * kKB), R - 1), h = id % (2 * kKB);
    su[u] = source(r, h / 2);
    su[u].p += su[u].blk - 32 + 16 * (h & 1);
    su[u].at = !kWholeU && id >= R * 2 * kKB ? -1
                                             : (r / 16) * kSubB + (h / 2) * kBlkB + (h & 1) * 2 * kGrpB + (r % 16) * 16;
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {
    const int id = max(u * T + stager, 0), r = min(id / kKB, R - 1);
    sv[u] = source(r, vb);
    sv[u].at = !kWholeV && id >= R * kKB ? -1 : S::kScale + 4 * ((r / 16) * 64 + vb * 16 + r % 16);
  }
  struct Regs {
    u32x4_t q[NU];
    unsigned s[NV];
  } regs[PD];
  int at = 0;  // the block the sources point to
  // the stages are loaded in order; past the last one nothing moves on
  auto load = [&](Regs& x, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; ++u) x.q[u] = gload<u32x4_a2>(su[u].p);
#pragma unroll
    for (int u = 0; u < NV; ++u) x.s[u] = gload<u32_a2>(sv[u].p);
    const int next = max(min((st + 1) * kKB, nblk - kKB), 0);
#pragma unroll
    for (int u = 0; u < NU; ++u) su[u].p += (next - at) * su[u].blk;
#pragma unroll
    for (int u = 0; u < NV; ++u) sv[u].p += (next - at) * sv[u].blk;
    at = next;
  };
  auto stage = [&](const Regs& x, int buf, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (!kWholeU && u == NU - 1 && su[u].at < 0) continue;
      lds_t* const d = lds + buf + su[u].at;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const f16x4_t s = i8_to_f16(x.q[u][2 * v]), t = i8_to_f16(x.q[u][2 * v + 1]);
        lds_store<f16x8_t>(d + v * kGrpB, f16x8_t{s.x, s.y, s.z, s.w, t.x, t.y, t.z, t.w});
      }
    }
    const bool zero = st == n_st - 1 && (n_st > 1 ? vb < n_again : vb >= nblk);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      if (!kWholeV && u == NV - 1 && sv[u].at < 0) continue;
      const float s = sv[u].blk == 36 ? __builtin_bit_cast(float, x.s[u])
                                      : (float)__builtin_bit_cast(_Float16, (unsigned short)x.s[u]);
      lds_store<float>(lds + buf + sv[u].at, zero ? 0.0f : s);
    }
  };
  float acc[NI][NJ][4 * NQ][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int l = 0; l < 4 * NQ; ++l)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][l][r] = 0.0f;
  auto read = [&](f16x4_t (&f)[kKB][NQ], float& s, int buf, int sub) __attribute__((always_inline)) {
    const lds_t* const q = lds + buf + sub * kSubB + g * kGrpB + c * 16;
    s = lds_load<float>(lds + buf + S::kScale + 4 * (sub * 64 + lane));
#pragma unroll
    for (int b = 0; b < kKB; ++b) {
      if constexpr (LS == 1) {
        const f16x8_t v = lds_load<f16x8_t>(q + b * kBlkB);
        f[b][0] = f16x4_t{v[0], v[1], v[2], v[3]};
        f[b][1] = f16x4_t{v[4], v[5], v[6], v[7]};
      } else {
        f[b][0] = lds_load<f16x4_t>(q + b * kBlkB + 8 * ls);
      }
    }
  };
  // One stage, from buffer st % 2, while stage st + 1 goes into the other
  // one, which every wave has left at the barrier before.
  auto step = [&](int st, auto u_, auto loads_, auto multiplies_) __attribute__((always_inline)) {
    constexpr int u = u_, buf = (u & 1) * S::kBuf;
    if constexpr (loads_) load(regs[u % PD], st + PD);
    if constexpr (multiplies_) {
      f16x4_t fw[NJ][kKB][NQ];
      float sw[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) read(fw[j], sw[j], buf, S::kIS + wj * NJ + j);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        f16x4_t fa[kKB][NQ];
        float sa;
        read(fa, sa, buf, wi * NI + i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) stage_fma<NQ>(acc[i][j], fa, fw[j], sa, sw[j]);
      }
    }
    if constexpr (loads_) stage(regs[(u + 1) % PD], S::kBuf - buf, st + 1);
    wg_barrier();
  };
  constexpr int U = PD > 2 ? PD : 2;
  static_assert(U % PD == 0 && U % 2 == 0, "the loop's unrolling covers the register sets and the buffers");
  auto stages = [&](auto loads, auto multiplies) __attribute__((always_inline)) {
    const int n_whole = n_st / U * U;
    for (int st = 0; st < n_whole; st += U)
      static_for<U>([&](auto u) __attribute__((always_inline)) { step(st + u, u, loads, multiplies); });
    static_for<U - 1>([&](auto u) __attribute__((always_inline)) {
      if (n_whole + u < n_st) step(n_whole + u, u, loads, multiplies);
    });
  };
  const std::true_type yes;
  const std::false_type no;
  if (PW == 0 || wv >= S::kC) {
    static_for<PD>([&](auto u) __attribute__((always_inline)) { load(regs[u], u); });
    stage(regs[0], 0, 0);
  }
  wg_barrier();
  if constexpr (PW == 0) {
    stages(yes, yes);
  } else if (wv >= S::kC) {
    stages(yes, no);
    if constexpr (LS == 2) {
#pragma unroll
      for (int x = 0; x < NI * NJ; ++x) wg_barrier();  // the halves' exchange below
    }
    return;
  } else {
    stages(no, yes);
  }
  // ((a0 + a4) + (a1 + a5)) + ((a2 + a6) + (a3 + a7)): accumulator 2b + q is
  // acc[2b + q], or acc[b] of wave ls = q
  float out[NI][NJ][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const auto& a = acc[i][j];
      if constexpr (LS == 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[i][j][r] = ((a[0][r] + a[4][r]) + (a[1][r] + a[5][r])) + ((a[2][r] + a[6][r]) + (a[3][r] + a[7][r]));
      } else {
        lds_t* const x = lds + 4 * ((((wi * WJ + wj) * NI + i) * NJ + j) * 8 * kWave + lane);
        float t0[4], t1[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          t0[r] = a[0][r] + a[2][r];
          t1[r] = a[1][r] + a[3][r];
          if (ls) {
            lds_store<float>(x + 8 * kWave * r, t0[r]);
            lds_store<float>(x + 8 * kWave * r + 4 * kWave, t1[r]);
          }
        }
        wg_barrier();
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[i][j][r] = (t0[r] + lds_load<float>(x + 8 * kWave * r)) + (t1[r] + lds_load<float>(x + 8 * kWave * r + 4 * kWave));
      }
    }
  if (LS == 2 && ls) return;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      store_cols(p, row0 + 16 * (wj * NJ + j) + c, col0 + 16 * (wi * NI + i) + 4 * g, out[i][j]);
}

template <int WI, int WJ, int NI, int NJ, int LS, int PD, int OCC, int PW>
static hipError_t launch_tile(Q8MulMat p, hipStream_t stream) {
  typedef TileShape<WI, WJ, NI, NJ, LS, PW> S;
  static_assert(LS == 1 || 2 * S::kBuf >= WI * WJ * NI * NJ * 8 * kWave * 4, "room for the halves' exchange");
  const auto fn = &mul_mat_q8_0_tile_kernel<WI, WJ, NI, NJ, LS, PD, OCC, PW>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * S::kBuf);
  if (attr != hipSuccess) return attr;
  // one launch, unless rows or columns are too many for one grid
  const int64_t most = INT32_MAX / S::kT;  // workgroups of a launch
  const int64_t n_step = most / 8 * 8 * S::kN, n = p.n, m = p.m;
  if (n > n_step && (p.rope_on || p.perm_hd)) return hipErrorInvalidValue;  // (their rows are not dealt in parts)
  const Q8MulMat whole = p;
  for (int64_t r0 = 0; r0 < n; r0 += n_step) {
    p.n = std::min(n_step, n - r0);
    const int64_t n_jt = (p.n + S::kN - 1) / S::kN, per_it = (n_jt + 7) / 8 * 8;
    const int64_t m_step = most / per_it * S::kM;
    for (int64_t c0 = 0; c0 < m; c0 += m_step) {
      p.m = std::min(m_step, m - c0);
      p.w = whole.w + r0 * p.w_nb1;
      p.a = whole.a + c0 * p.a_nb1;
      p.dst = whole.dst + r0 * p.dst_nb0 + c0 * p.dst_nb1;
      if (p.add) p.add = whole.add + r0 * p.add_nb0 + c0 * p.add_nb1;
      p.rope.pos = whole.rope.pos + (int32_t)c0;
      p.rope.q_out = whole.rope.q_out + c0 * p.rope.q_ld;
      p.rope.k_row = whole.rope.k_row + c0 * p.rope.c_s2;
      p.rope.v_row = whole.rope.v_row + c0 * p.rope.c_s2;
      const int64_t n_it = (p.m + S::kM - 1) / S::kM;
      hipLaunchKernelGGL(fn, dim3((unsigned)(per_it * n_it)), dim3(S::kT), 2 * S::kBuf, stream, p, (int)n_jt, (int)n_it);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

// Which tile: as large as still gives about a workgroup per CU, since a
// launch that does not fill the chip is bound by the time of one workgroup's
// stages (896 x 4864 with 37 columns: 14.4 us in 168 tiles of 16 x 16, 16.1 in
// 112 of 32 x 16, 25.7 in 56 of 32 x 32; with 128: 17.2 in 224 of 32 x 16, 20.7
// in 448 of 16 x 16). At most 16 columns that do fill it take 16-column tiles
// (151936 x 896 with 8: 45 us, 66 in tiles of 32).
hipError_t launch_mul_mat_q8_0_cols(const Q8MulMat& p, int n_cu, hipStream_t stream) {
  const int64_t cu = n_cu > 0 ? n_cu : 256;
  const int64_t j16 = (p.n + 15) / 16, i16 = (p.m + 15) / 16, i32 = (p.m + 31) / 32;
  if (j16 * i16 <= cu) return launch_tile<1, 1, 1, 1, 2, 4, 2, 4>(p, stream);
  if (p.m <= 16) return launch_tile<1, 2, 1, 1, 2, 2, 3, 0>(p, stream);
  if (j16 * i32 <= cu) return launch_tile<2, 1, 1, 1, 2, 4, 2, 6>(p, stream);
  return launch_tile<2, 2, 1, 1, 1, 2, 3, 0>(p, stream);
}

}  // namespace mi
