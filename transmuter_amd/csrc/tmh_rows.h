// MatMulNBits for up to 64 rows of A, any float types (lib/transmuter/ops/quantized.ex:30-46): the
// decode and small-batch products that the f16 decode GEMV (tmh_gemv.h) does not take.
//
// A workgroup of NW wavefronts covers TN 16-column tiles and 16*MT rows of A; its wavefronts take
// the chunks of K in turn (the next chunk's weights in flight while one is computed) and add
// their sums through LDS. Weights are the MFMAs' first operand, so a lane ends with 4 consecutive
// columns of one row of Y.
//
// These calls are bound by latency and by each CU's path to the L2: a workgroup reads its weights
// once (HBM) and 16*MT rows of A (L2), and every workgroup reads all of K of its rows. So the A
// fragments are loaded in the natural order of k (an MFMA step covers 32 consecutive values of k,
// 64 or 128 contiguous bytes of each row per load) rather than in the order the packed layout
// holds the weights in (a lane's k-group is 32 consecutive values, four MFMA steps): the lanes
// trade their weight words instead, a 4 x 4 transposition over the wavefront's four rows of
// lanes in four permlane swaps per chunk, and their scales and zero points in three.
//
// Operand paths (OP):
//  ROW_F16   f16 A and weights: exact f16 weights (q - zero) * scale (unpack_step);
//  ROW_BF16  bf16 A and weights: (q - zero) * scale formed in f32 and rounded once to bf16, as the
//            reference's bf16 dequantization rounds it (a scale of 2^117 and more overflows on the way,
//            natural_values: rows_again forms the sums of such weights);
//  ROW_INT   f32 A and f32 weights of blocks of 32 and more: q - zero is a whole number of at most
//            8 bits and so exact in bf16, a value of A is the exact sum of three bf16 parts, and a
//            step's 32 products sit in one block, whose f32 scale multiplies the step's f32 sums:
//            three MFMAs and four FMAs a lane per step, with f32 products throughout. (A step's sum
//            before its scale can pass f32's range, from |a| near 4e34 with 8 bits and 7e35 with 4
//            on: it comes out infinite or NaN then, and rows_again forms the sums again.);
//  ROW_GEN   every other combination (mixed types, float zero points, f32 weights in blocks of 16 or
//            of 2 bits): the weights dequantize in f32 as the reference does in their type, and
//            three bf16 parts of each factor (exact) meet in all nine products, so that none is
//            rounded. (The parts are cut, so what the three smallest products add always has the
//            product's own sign: left out, up to 2^-23 of each product would be missing from every sum.)
// f16 and bf16 weights with float zero points take ROW_GEN too.
#pragma once

#include "tmh_device.h"
#include "tmh_internal.h"

namespace tmh {

enum : int { ROW_F16 = 0, ROW_BF16 = 1, ROW_INT = 2, ROW_GEN = 3 };

constexpr int64_t kRowsMax = 4032;  // rows of A of one launch: 12 bits of its shape, in sets of 64

typedef __bf16 rows_bf16x8_t __attribute__((ext_vector_type(8)));

// Eight f32 values as the sum of three bf16 parts each: the top 8 bits of the significand, the next
// 8 and the last 8 (cut, not rounded: every part is exact, and no part of a finite value
// overflows; below 2^-110 the last bits fall under bf16's own range). An infinity leaves a NaN
// behind: the sums it enters are formed again (rows_again).
__device__ __forceinline__ void split3(const float (&a)[8], uint4_t (&part)[3]) {
  float rest[8];
  uint32_t top[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    top[j] = __builtin_bit_cast(uint32_t, a[j]);
    rest[j] = a[j] - __builtin_bit_cast(float, top[j] & 0xFFFF0000u);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t m0 = __builtin_bit_cast(uint32_t, rest[2 * j]), m1 = __builtin_bit_cast(uint32_t, rest[2 * j + 1]);
    const float l0 = rest[2 * j] - __builtin_bit_cast(float, m0 & 0xFFFF0000u);
    const float l1 = rest[2 * j + 1] - __builtin_bit_cast(float, m1 & 0xFFFF0000u);
    part[0][j] = __builtin_amdgcn_perm(top[2 * j + 1], top[2 * j], 0x07060302u);
    part[1][j] = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
    part[2][j] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, l1), __builtin_bit_cast(uint32_t, l0), 0x07060302u);
  }
}

__device__ __forceinline__ float4_t mma_bf16(const uint4_t& b, const uint4_t& a, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rows_bf16x8_t, b), __builtin_bit_cast(rows_bf16x8_t, a),
                                                 c, 0, 0, 0);
}

__device__ __forceinline__ float round_rt(float x, int dt) {
  return dt == DT_F16 ? round_to<DT_F16>(x) : (dt == DT_BF16 ? round_to<DT_BF16>(x) : x);
}

// Four consecutive outputs at element `at` (columns n.., those below N) in any float type: the dot
// type's rounding, then the columns' bias (its bits b); in one store where Y is aligned (vec). Out of line: the
// uniform branches over the types cost the common stores nothing.
__device__ __noinline__ void rows_store_any(float4_t v, void* Y, uint32_t types, uint4_t b, int64_t at, uint32_t n,
                                            uint32_t N, bool vec) {
  const int y_dt = types & 0xFFu, dot_dt = (types >> 8) & 0xFFu, b_dt = (types >> 16) & 0xFFu;
  if (dot_dt == DT_F16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = round_to<DT_F16>(v[e]);
  } else if (dot_dt == DT_BF16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = round_to<DT_BF16>(v[e]);
  }
  if (b_dt) {
    float4_t f = __builtin_bit_cast(float4_t, b);  // whole vector: hipcc 7.2 miscompiled element casts
    if (b_dt != DT_F32) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        f[e] = b_dt == DT_F16 ? f16_bits_to_f32(static_cast<uint16_t>(b[e])) : bf16_bits_to_f32(static_cast<uint16_t>(b[e]));
    }
    v += f;
  }
  if (y_dt == DT_F32) {
    float* y = static_cast<float*>(Y) + at;
    if (vec && n + 4 <= N) {
      *reinterpret_cast<float4_t*>(y) = v;
    } else {
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e)
        if (n + e < N) y[e] = v[e];
    }
    return;
  }
  uint16_t h[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = y_dt == DT_F16 ? f32_to_f16_bits(v[e]) : f32_to_bf16_bits(v[e]);
  uint16_t* y = static_cast<uint16_t*>(Y) + at;
  if (vec && n + 4 <= N) {
    *reinterpret_cast<uint2*>(y) = make_uint2(h[0] | (static_cast<uint32_t>(h[1]) << 16), h[2] | (static_cast<uint32_t>(h[3]) << 16));
  } else {
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e)
      if (n + e < N) y[e] = h[e];
  }
}

// (q - z) * s of eight values as the reference dequantizes them in the weights' type: one uniform branch
// over the type, not two a value.
__device__ __forceinline__ void dequantize8(float (&q)[8], float z, float s, int w_dt) {
  if (w_dt == DT_F32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = (q[e] - z) * s;
  } else if (w_dt == DT_F16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = round_to<DT_F16>(round_to<DT_F16>(q[e] - z) * s);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = round_to<DT_BF16>(round_to<DT_BF16>(q[e] - z) * s);
  }
}

// Four consecutive columns' sums v of one row, over the chunks c0, c0 + step, ..., with those that are
// infinite or NaN formed again, one f32 FMA per product as k_matmul_general forms them: where the parts
// of a factor may be at fault (0 times an infinity's other part, a block's sum past f32's range ahead of
// its scale, a weight whose scale lies at the end of its type). Not where A's row holds a NaN, which no
// other sum would change, nor (scales_only) where no scale is that large. Out of line: inside the kernel
// its code spread the rest apart (bf16 M = 8 1024 -> 4096 3.52 us, 3.45 out of line). us of a call whose A
// holds a NaN / an infinity / neither: f32 M = 16 1024 -> 4096 6.2 / 31.9 / 5.1 (k_matmul_general 55), bf16
// M = 8 6.7 / 6.7 / 3.4.
template <int BITS>
__device__ __noinline__ float4_t rows_again(float4_t v, const uint4_t* qt, const void* sc, const uint8_t* zp, const void* A,
                                            int a_dt, int w_dt, uint32_t zk, uint32_t tile, uint32_t col, uint32_t a_at,
                                            uint32_t nch, uint32_t nbc, uint32_t bsc_shift, uint32_t K, uint32_t c0,
                                            uint32_t step, bool scales_only) {
  constexpr uint32_t CW = 512 / BITS, GW = CW / 4, STEPS = GW / 8;
  if (v[0] * 0.f + v[1] * 0.f + v[2] * 0.f + v[3] * 0.f == 0.f) return v;
  if (scales_only) {
    uint32_t most = 0;  // the largest bf16 scale's magnitude, in the upper half
    for (uint32_t c = c0; c < nch; c += step)
#pragma unroll 2
      for (uint32_t b = 0; b < nbc; ++b) {
        const uint2 s4 = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(sc) + ((tile * nch + c) * nbc + b) * 16 + col);
        most = max(max(most, max((s4.x << 16) & 0x7FFF0000u, s4.x & 0x7FFF0000u)),
                   max((s4.y << 16) & 0x7FFF0000u, s4.y & 0x7FFF0000u));
      }
    const bool large = most >= 0x7A000000u;  // 2^117
    if (!large) return v;
  }
  // Eight values of A from k on: 16-byte loads, as gemv_rows_ok has A aligned and K a multiple of 8.
  auto load8 = [&](uint32_t k, float (&a)[8]) {
    if (a_dt == DT_F32) {
      const auto* p = reinterpret_cast<const float4_t*>(static_cast<const float*>(A) + a_at + k);
      const float4_t x = p[0], y = p[1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = x[j];
        a[4 + j] = y[j];
      }
    } else {
      const uint4_t x = *reinterpret_cast<const uint4_t*>(static_cast<const uint16_t*>(A) + a_at + k);
      const uint32_t h[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const auto u = static_cast<uint16_t>(h[j / 2] >> (16 * (j % 2)));
        a[j] = a_dt == DT_F16 ? f16_bits_to_f32(u) : bf16_bits_to_f32(u);
      }
    }
  };
  bool nan = false;
#pragma unroll 1
  for (uint32_t c = c0; c < nch; c += step) {
    const uint32_t end = min(c * CW + CW, K);
#pragma unroll 2
    for (uint32_t k = c * CW; k < end; k += 8) {
      float a[8];
      load8(k, a);
#pragma unroll
      for (int j = 0; j < 8; ++j) nan |= a[j] != a[j];
    }
  }
  if (nan) return v;
  float4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (uint32_t c = c0; c < nch; c += step)
#pragma unroll 1
    for (uint32_t kge = 0; kge < 16; ++kge) {  // a k-group of a column: its parameters' loads in one go
      const uint32_t kg = kge >> 2, e = kge & 3, k0 = c * CW + kg * GW;
      const uint4_t w = qt[(tile * nch + c) * 64 + kg * 16 + col + e];
      float s[STEPS], z[STEPS], x = 0.f;
#pragma unroll
      for (uint32_t i = 0; i < STEPS; ++i) {
        const uint32_t at = ((tile * nch + c) * nbc + ((kg * GW + 8 * i) >> bsc_shift)) * 16 + col + e;
        s[i] = load_float_rt(sc, w_dt, at);
        z[i] = zk == TMH_ZP_FLOAT ? reinterpret_cast<const float*>(zp)[at]
               : zk == TMH_ZP_PACKED ? static_cast<float>(zp_field<BITS>(zp[zp_byte<BITS>(at)], zp_shift<BITS>(col + e)))
                                     : static_cast<float>(1 << (BITS - 1));
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) x = f == static_cast<int>(e) ? sum[f] : x;
#pragma unroll
      for (uint32_t i = 0; i < STEPS; ++i) {
        if (k0 + 8 * i >= K) break;
        float a[8], q[8];
        load8(k0 + 8 * i, a);
        natural_values<BITS>(w, static_cast<int>(i), 1.f, 0.f, q);
        dequantize8(q, z[i], s[i], w_dt);
#pragma unroll
        for (int j = 0; j < 8; ++j) x = fmaf(q[j], a[j], x);
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) sum[f] = f == static_cast<int>(e) ? x : sum[f];
    }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] * 0.f == 0.f ? v[e] : sum[e];
  return v;
}

// types = the type of Y | the dot's << 8 | the bias's << 16 (0: none) | A's << 24 (ROW_GEN); kinds =
// the zero point kind | the weights' type << 8 (ROW_GEN). shape = M (up to
// kRowsMax) | nbc << 12 | the shift of a block's k in its chunk << 20 | the eights of the last chunk past K << 24
// | a bias << 31.
// The leading arguments are preloaded into SGPRs at wave launch.
template <int BITS, int OP, bool SPLIT, int MT, int TN, int NW>
__global__ __launch_bounds__(64 * NW) void k_gemv_rows(
    const uint4_t* __restrict__ qt, const void* __restrict__ sc, const uint8_t* __restrict__ zp,
    const void* __restrict__ A, uint32_t nch, uint32_t ntiles, uint32_t lda, uint32_t shape, void* __restrict__ Y,
    int64_t ldy, uint32_t N, uint32_t types, uint32_t kinds, const void* __restrict__ bias) {
  constexpr int CW = 512 / BITS;
  constexpr int GW = CW / 4;
  constexpr int STEPS = GW / 8;
  constexpr bool NAT = BITS != 2 && OP != ROW_GEN;  // natural order of k
  constexpr bool F32A = OP == ROW_INT || OP == ROW_GEN;
  constexpr int AL = F32A ? 2 : 1;                  // 16-byte loads of A per step
  constexpr int NJ = SPLIT ? STEPS : 1;             // parameter entries a lane loads per chunk
  // A of the next chunk held in registers too, where they hold it without spilling.
  constexpr bool PREFETCH_A = STEPS * AL * MT <= (F32A && NW == 16 ? 4 : 8);
  static_assert(OP != ROW_INT || (!SPLIT && NAT), "one block per step");
  static_assert(NW * MT * TN <= 128, "the partial sums must fit the LDS");
  extern __shared__ float4_t rows_red[];
  const uint32_t M = shape & 0xFFFu, nbc = (shape >> 12) & 0xFFu, bsc_shift = (shape >> 20) & 0xFu;
  const uint32_t K = nch * CW - ((shape >> 24) & 0x7Fu) * 8;
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const uint32_t t0 = blockIdx.x * TN, m0 = blockIdx.y * 16 * MT;
  const uint32_t n_params = ntiles * nch * nbc * 16;
  const bool a_f32 = OP == ROW_INT || (OP == ROW_GEN && (types >> 24) == DT_F32);
  const uint32_t a_size = a_f32 ? 4 : 2;
  // Without zero points zp is null; ROW_GEN's kinds, which tells float ones, is no preloaded argument,
  // and waiting for it ahead of the first loads would cost every launch of the other paths.
  const uint32_t zk = OP == ROW_GEN ? kinds & 0xFFu : zp ? TMH_ZP_PACKED : TMH_ZP_NONE;
  const bool s_f32 = OP == ROW_INT || (OP == ROW_GEN && ((kinds >> 8) & 0xFFu) == DT_F32);
  const auto q_rsrc = buffer_rsrc(qt, ntiles * nch * 1024);
  const auto s_rsrc = buffer_rsrc(sc, n_params * (s_f32 ? 4 : 2));
  // (Without zero points the resource is empty and its loads read zeros, not used.)
  const auto z_rsrc = buffer_rsrc(zp, zk == TMH_ZP_NONE ? 0u : zk == TMH_ZP_FLOAT ? n_params * 4 : zp_byte<BITS>(n_params));
  const uint32_t zsh = zp_shift<BITS>(r);
  const auto a_rsrc = buffer_rsrc(A, M * lda * a_size);
  uint32_t a_row[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) a_row[mt] = m0 + mt * 16 + r < M ? (m0 + mt * 16 + r) * lda * a_size : 0x80000000u;
  auto k_of = [&](int i) -> uint32_t { return NAT ? 32 * i + 8 * g : g * GW + 8 * i; };  // first k of step i in the chunk

  struct Weights {
    uint4_t w[TN];
    uint32_t s[TN][NJ], z[TN][NJ];
    float4_t sq[OP == ROW_INT ? TN : 1][OP == ROW_INT ? STEPS : 1];  // ROW_INT: scales of the lane's 4 columns
  };
  struct Rows {
    uint4_t a[MT][STEPS][AL];
  };
  auto load_w = [&](uint32_t c, Weights& st) {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const uint32_t tc = (t0 + tn) * nch + c;  // tiles past the last read zeros
      st.w[tn] = __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, ((t0 + tn) * nch * 64 + lane) * 16, c * 1024, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint32_t e = (tc * nbc + ((SPLIT ? k_of(j) : static_cast<uint32_t>(g * GW)) >> bsc_shift)) * 16 + r;
        if constexpr (OP == ROW_GEN) {
          if (s_f32) st.s[tn][j] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc, e * 4, 0, 0);
          else st.s[tn][j] = __builtin_amdgcn_raw_buffer_load_b16(s_rsrc, e * 2, 0, 0);
          if (zk == TMH_ZP_FLOAT) st.z[tn][j] = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc, e * 4, 0, 0);
          else st.z[tn][j] = __builtin_amdgcn_raw_buffer_load_b8(z_rsrc, zp_byte<BITS>(e), 0, 0);
        } else {
          if constexpr (OP != ROW_INT) st.s[tn][j] = __builtin_amdgcn_raw_buffer_load_b16(s_rsrc, e * 2, 0, 0);
          st.z[tn][j] = __builtin_amdgcn_raw_buffer_load_b8(z_rsrc, zp_byte<BITS>(e), 0, 0);
        }
      }
      if constexpr (OP == ROW_INT) {
#pragma unroll
        for (int i = 0; i < STEPS; ++i)
          st.sq[tn][i] = __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(
              s_rsrc, ((tc * nbc + ((32 * i) >> bsc_shift)) * 16 + 4 * g) * 4, 0, 0));
      }
    }
  };
  auto load_a = [&](uint32_t c, Rows& st) {
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const uint32_t k = c * CW + k_of(i);  // K is a multiple of 8: the step lies wholly in or past K
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint32_t off = k < K ? a_row[mt] + k * a_size : 0x80000000u;
        st.a[mt][i][0] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off, 0, 0);
        if constexpr (AL == 2) {
          if (a_f32) st.a[mt][i][1] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off, 16, 0);
        }
      }
    }
  };
  float4_t acc[MT][TN];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[mt][tn] = float4_t{0.f, 0.f, 0.f, 0.f};

  auto zero_of = [&](uint32_t raw) -> uint32_t { return zk == TMH_ZP_NONE ? 1u << (BITS - 1) : zp_field<BITS>(raw, zsh); };
  auto compute = [&](const Weights& st, const Rows& rows) {
    uint4_t wn[TN];
    uint32_t par[TN][STEPS];  // scale | zero << 16 (ROW_INT: the zero) of the lane's weights in each step
    if constexpr (OP != ROW_GEN) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        if constexpr (NAT) wn[tn] = natural_words<BITS>(st.w[tn]);
        else wn[tn] = st.w[tn];
        uint32_t own[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint32_t z = zero_of(st.z[tn][j]);
          if constexpr (OP == ROW_INT) own[j] = z;
          else own[j] = (st.s[tn][j] & 0xFFFFu) | (z << 16);
        }
        if constexpr (NAT && !SPLIT) {
          natural_params<BITS>(own[0], par[tn]);
        } else {
#pragma unroll
          for (int i = 0; i < STEPS; ++i) par[tn][i] = own[SPLIT ? i : 0];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      if constexpr (OP == ROW_F16 || OP == ROW_BF16) {
        uint4_t b[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const uint32_t s = par[tn][i] & 0xFFFFu, z = par[tn][i] >> 16;
          if constexpr (OP == ROW_F16) {
            const uint32_t zz = 0x6400u + z;
            b[tn] = __builtin_bit_cast(uint4_t, unpack_step<BITS>(wn[tn], i, __builtin_bit_cast(half2_t, zz | (zz << 16)),
                                                                  __builtin_bit_cast(half2_t, s | (s << 16))));
          } else {
            const float sf = __builtin_bit_cast(float, s << 16), zf = static_cast<float>(z);
            float q[8];
            natural_values<BITS>(wn[tn], i, sf, zf, q);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[tn][j] = pack_bf16_rne(q[2 * j], q[2 * j + 1]);
          }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) {
            if constexpr (OP == ROW_F16)
              acc[mt][tn] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, b[tn]),
                                                                   __builtin_bit_cast(half8_t, rows.a[mt][i][0]),
                                                                   acc[mt][tn], 0, 0, 0);
            else acc[mt][tn] = mma_bf16(b[tn], rows.a[mt][i][0], acc[mt][tn]);
          }
      } else if constexpr (OP == ROW_INT) {
        uint4_t b[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const float zf = static_cast<float>(par[tn][i]);
          float q[8];
          natural_values<BITS>(wn[tn], i, 1.f, zf, q);
#pragma unroll
          for (int j = 0; j < 4; ++j) b[tn][j] = pack_bf16_rne(q[2 * j], q[2 * j + 1]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const float4_t x = __builtin_bit_cast(float4_t, rows.a[mt][i][0]), y = __builtin_bit_cast(float4_t, rows.a[mt][i][1]);
          const float av[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          uint4_t part[3];
          split3(av, part);
#pragma unroll
          for (int tn = 0; tn < TN; ++tn) {
            float4_t sum = mma_bf16(b[tn], part[2], float4_t{0.f, 0.f, 0.f, 0.f});
            sum = mma_bf16(b[tn], part[1], sum);
            sum = mma_bf16(b[tn], part[0], sum);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[mt][tn][e] = fmaf(st.sq[tn][i][e], sum[e], acc[mt][tn][e]);
          }
        }
      } else {
        const int w_dt = static_cast<int>((kinds >> 8) & 0xFFu), a_dt = static_cast<int>(types >> 24);
        uint4_t ap[MT][3];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float av[8];
          if (a_f32) {
            const float4_t x = __builtin_bit_cast(float4_t, rows.a[mt][i][0]), y = __builtin_bit_cast(float4_t, rows.a[mt][i][1]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              av[e] = x[e];
              av[4 + e] = y[e];
            }
          } else if (a_dt == DT_F16) {
            const half8_t x = __builtin_bit_cast(half8_t, rows.a[mt][i][0]);
#pragma unroll
            for (int e = 0; e < 8; ++e) av[e] = static_cast<float>(x[e]);
          } else {
            const rows_bf16x8_t x = __builtin_bit_cast(rows_bf16x8_t, rows.a[mt][i][0]);
#pragma unroll
            for (int e = 0; e < 8; ++e) av[e] = static_cast<float>(x[e]);
          }
          split3(av, ap[mt]);
        }
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
          const uint32_t sraw = st.s[tn][i], zraw = st.z[tn][i];
          const float s = s_f32 ? __builtin_bit_cast(float, sraw)
                                : (w_dt == DT_F16 ? f16_bits_to_f32(static_cast<uint16_t>(sraw))
                                                  : bf16_bits_to_f32(static_cast<uint16_t>(sraw)));
          const float z = zk == TMH_ZP_FLOAT ? __builtin_bit_cast(float, zraw) : static_cast<float>(zero_of(zraw));
          float q[8];
          natural_values<BITS>(st.w[tn], i, 1.f, 0.f, q);  // q itself: a float zero point is subtracted as it is
          dequantize8(q, z, s, w_dt);
          uint4_t wp[3];
          split3(q, wp);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            float4_t sum = mma_bf16(wp[2], ap[mt][2], float4_t{0.f, 0.f, 0.f, 0.f});
            sum = mma_bf16(wp[2], ap[mt][1], sum);
            sum = mma_bf16(wp[1], ap[mt][2], sum);
            sum = mma_bf16(wp[2], ap[mt][0], sum);
            sum = mma_bf16(wp[1], ap[mt][1], sum);
            sum = mma_bf16(wp[0], ap[mt][2], sum);
            sum = mma_bf16(wp[1], ap[mt][0], sum);
            sum = mma_bf16(wp[0], ap[mt][1], sum);
            sum = mma_bf16(wp[0], ap[mt][0], sum);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[mt][tn][e] += sum[e];
          }
        }
      }
    }
  };
  // The bias (its bits; zeros past N) of the columns of the tile this wavefront stores: on its way while
  // the sums meet in LDS (fetched ahead of each store instead, an f32 bias cost f16 calls of few rows 5
  // to 10%).
  auto load_bias = [&](uint32_t tn) -> uint4_t {
    uint4_t b = {0u, 0u, 0u, 0u};
    if (!(shape >> 31)) return b;  // (types, no preloaded argument, is not waited for here)
    const uint32_t b_dt = (types >> 16) & 0xFFu, n = (t0 + tn) * 16 + 4 * g;
    if (b_dt == DT_F32) {
      const auto b_rsrc = buffer_rsrc(bias, N * 4);
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) b[e] = __builtin_amdgcn_raw_buffer_load_b32(b_rsrc, (n + e) * 4, 0, 0);
    } else {
      const auto b_rsrc = buffer_rsrc(bias, N * 2);
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) b[e] = __builtin_amdgcn_raw_buffer_load_b16(b_rsrc, (n + e) * 2, 0, 0);
    }
    return b;
  };
  if (wave < nch) {
    // Two register sets used in turn: a copy between them would wait for the loads in flight.
    Weights wa, wb;
    Rows ra, rb;
    load_w(wave, wa);
    load_a(wave, ra);
    for (uint32_t c = wave;;) {
      const bool second = c + NW < nch;
      if (second) {
        load_w(c + NW, wb);
        if constexpr (PREFETCH_A) load_a(c + NW, rb);
      }
      compute(wa, ra);
      if (!second) break;
      if constexpr (!PREFETCH_A) load_a(c + NW, ra);
      const bool third = c + 2 * NW < nch;
      if (third) {
        load_w(c + 2 * NW, wa);
        if constexpr (PREFETCH_A) load_a(c + 2 * NW, ra);
      }
      if constexpr (PREFETCH_A) compute(wb, rb);
      else compute(wb, ra);
      if (!third) break;
      c += 2 * NW;
      if constexpr (!PREFETCH_A) load_a(c, ra);
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) rows_red[(wave * MT * TN + mt * TN + tn) * 64 + lane] = acc[mt][tn];
  if constexpr (OP == ROW_INT || OP == ROW_GEN) {
    float odd = 0.f;  // NaN where a sum is infinite or NaN, else 0
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int e = 0; e < 4; ++e) odd = fmaf(acc[mt][tn][e], 0.f, odd);
    if (__builtin_expect(__any(odd != 0.f), 0)) {
#pragma unroll 1
      for (int p = 0; p < MT * TN; ++p) {
        const uint32_t m = m0 + p / TN * 16 + r, tile = t0 + p % TN;
        float4_t* const mine = rows_red + (wave * MT * TN + p) * 64 + lane;
        if (m < M && tile < ntiles)
          *mine = rows_again<BITS>(*mine, qt, sc, zp, A, types >> 24, (kinds >> 8) & 0xFFu, kinds & 0xFFu, tile, 4 * g, m * lda,
                                   nch, nbc, bsc_shift, K, wave, NW, false);
      }
    }
  }
  uint4_t b0 = {0u, 0u, 0u, 0u};
  if (wave < MT * TN) b0 = load_bias(wave % TN);
  __syncthreads();
  constexpr uint32_t kOwn = OP == ROW_F16 ? DT_F16 : OP == ROW_BF16 ? DT_BF16 : DT_F32;
  const bool plain = (types & 0xFFFFFFu) == (kOwn | (kOwn << 8)) && ldy % 4 == 0 &&
                     (reinterpret_cast<uintptr_t>(Y) & (F32A ? 15 : 7)) == 0;
#pragma unroll
  for (int p0 = 0; p0 < MT * TN; p0 += NW) {
    const int p = p0 + static_cast<int>(wave);
    if (p >= MT * TN) return;
    const int mt = p / TN, tn = p % TN;
    const uint32_t m = m0 + mt * 16 + r, n = (t0 + tn) * 16 + 4 * g;
    if (m >= M || n >= N) continue;
    float4_t part[NW];
#pragma unroll
    for (int w2 = 0; w2 < NW; ++w2) part[w2] = rows_red[(w2 * MT * TN + p) * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);  // every partial sum is read before the first is added
    float4_t v = part[0];
#pragma unroll
    for (int w2 = 1; w2 < NW; ++w2) v += part[w2];
    const int64_t at = static_cast<int64_t>(m) * ldy + n;
    if (plain && n + 4 <= N) {  // Y in the operands' own type, no bias
      if constexpr (OP == ROW_F16) {
        const half2_t lo = {static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1])};
        const half2_t hi = {static_cast<_Float16>(v[2]), static_cast<_Float16>(v[3])};
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(Y) + at) =
            make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
      } else if constexpr (OP == ROW_BF16) {
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(Y) + at) =
            make_uint2(pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3]));
      } else {
        *reinterpret_cast<float4_t*>(static_cast<float*>(Y) + at) = v;
      }
    } else {
      rows_store_any(v, Y, types, p0 == 0 ? b0 : load_bias(tn), at, n, N,
                     ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(Y) & ((types & 0xFFu) == DT_F32 ? 15 : 7)) == 0);
    }
    // bf16 weights fail at the largest scales alone: looked for behind the store, over all of K (ahead of
    // the sums' meeting the search cost every bf16 call up to 2.5%).
    if constexpr (OP == ROW_BF16) {
      if (__builtin_expect(v[0] * 0.f + v[1] * 0.f + v[2] * 0.f + v[3] * 0.f != 0.f, 0))
        rows_store_any(rows_again<BITS>(v, qt, sc, zp, A, DT_BF16, DT_BF16, kinds & 0xFFu, t0 + tn, 4 * g, m * lda, nch, nbc,
                                        bsc_shift, K, 0, 1, true),
                       Y, types, p0 == 0 ? b0 : load_bias(tn), at, n, N, false);
    }
  }
}

}  // namespace tmh
