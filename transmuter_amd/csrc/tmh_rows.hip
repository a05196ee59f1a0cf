// Launch plan of k_gemv_rows (tmh_rows.h): MatMulNBits with up to 64 rows of A
// (lib/transmuter/ops/quantized.ex:30-46).
#include <algorithm>

#include "tmh_rows.h"

namespace tmh {
namespace {

struct RowsArgs {
  const uint4_t* qt;
  const void* sc;
  const uint8_t* zp;
  const void* a;
  uint32_t nch, ntiles, lda, shape;
  void* y;
  int64_t ldy;
  uint32_t n, types, kinds;
  const void* bias;
};

struct RowsPlan {
  int mt, tn, nw;
};

template <int BITS, int OP, bool SPLIT, int MT, int TN, int NW>
void go_rows(const RowsArgs& d, int64_t M, hipStream_t s) {
  constexpr int kLds = NW * MT * TN * 1024;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemv_rows<BITS, OP, SPLIT, MT, TN, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  (void)attr;
  const dim3 grid((d.ntiles + TN - 1) / TN, static_cast<unsigned>((M + 16 * MT - 1) / (16 * MT)));
  k_gemv_rows<BITS, OP, SPLIT, MT, TN, NW><<<grid, 64 * NW, kLds, s>>>(d.qt, d.sc, d.zp, d.a, d.nch, d.ntiles, d.lda,
                                                                       d.shape, d.y, d.ldy, d.n, d.types, d.kinds, d.bias);
}

// The shapes plan_rows() chooses from, per operand path.
template <int BITS, int OP, bool SPLIT>
void launch_op(const RowsArgs& d, int64_t M, const RowsPlan& p, hipStream_t s) {
#define TMH_ROWS(MT_, TN_, NW_) \
  if (p.mt == MT_ && p.tn == TN_ && p.nw == NW_) return go_rows<BITS, OP, SPLIT, MT_, TN_, NW_>(d, M, s)
  if constexpr (OP != ROW_GEN) {
    TMH_ROWS(1, 2, 8);
    TMH_ROWS(2, 2, 8);
    if constexpr (BITS == 2 && SPLIT) {
      TMH_ROWS(1, 1, 4);
      TMH_ROWS(2, 2, 2);
    } else {
      TMH_ROWS(1, 2, 4);
    }
    if constexpr (BITS != 2 && SPLIT) TMH_ROWS(2, 2, 4);
    if constexpr (BITS != 2 && !SPLIT) {
      TMH_ROWS(1, 1, 16);
      if constexpr (OP != ROW_INT) {
        TMH_ROWS(1, 2, 16);
        TMH_ROWS(2, 2, 4);
        TMH_ROWS(2, 4, 8);
      }
    }
  }
  go_rows<BITS, OP, SPLIT, 1, 1, 8>(d, M, s);
#undef TMH_ROWS
}

// Rows of A, tiles and wavefronts per workgroup. Every workgroup reads its rows of A whole, through
// its CU's path to the L2, and unpacks (ROW_INT: splits A) once for all its tiles: so the grid
// should give each CU one workgroup and no more, of the fewest rows. Measured in graph replays
// (us per call, q4 block 32; mt,tn,nw):
//  - up to one workgroup a CU: 16 rows, one tile, as many wavefronts as the chunks fill (f16
//    3072->1024, M = 32: 1,1,16 5.4, 2,1,16 8.1, 1,2,16 5.9; bf16 2048->1024, M = 8: 1,1,16 3.8,
//    1,1,8 4.1);
//  - up to two: two tiles share the rows (f16 1024->4096, M = 32: 1,2,8 3.8, 1,1,8 4.6; 4096->4096,
//    M = 32: 1,2,16 7.6, 1,2,8 7.7, 1,1,16 11.3; f32 1024->6144, M = 16: 1,2,8 5.8, 1,1,8 8.3);
//  - up to four, eight: two sets of 16 rows share the unpacking too, then four tiles (bf16
//    1024->6144, M = 32: 2,2,8 5.0, 1,2,8 5.1, 1,1,8 6.5; f16 1024->6144, M = 64: 2,4,8 5.9, 1,2,8
//    6.6, 2,2,8 7.9);
//  - beyond, the workgroups come in rounds: four wavefronts with more chunks each keep their loads
//    going (bf16 1024->151936, M = 12: 1,2,4 27.4, 1,2,8 34.1; f32 2048->22016, M = 12: 1,2,4 20.4,
//    1,2,8 25.2; f16 2048->22016, M = 24: 2,2,4 14.8, 1,2,8 16.5, 2,4,8 16.7).
// 8 bits lie the same way (of 35 sizes none has a shape over 6% faster). 2-bit weights and parameters that
// change within a lane's group hold more registers per tile: two tiles at most, and with few chunks of K
// fewer wavefronts, as idle ones keep other workgroups off the CU:
//  - 2 bits (f16): M = 64 512->16000 1,2,4 8.4, 1,2,8 15.7, 2,2,8 10.4; 1024->6144 5.8, 8.5, 9.7; 2048->8192
//    12.1, 15.1, 27.4; one set of rows and eight chunks 1,2,8 5.0, 1,2,4 5.3. With 17 or 18 rows the second
//    set is nearly free (bf16 M = 17 2048->8192 2,2,8 7.6, 1,2,4 8.4);
//  - 2 bits in blocks of 16 or 32: M = 64 512->16000 2,2,2 10.0, 1,1,4 12.9, 1,2,8 20.8; 1024->6144 1,1,4 9.1,
//    2,2,2 10.0, 1,2,8 10.7; 2048->8192 1,2,8 17.8, 1,1,4 21.5, 2,2,2 31.9; up to four workgroups a CU M = 32
//    768->5000 2,2,8 5.5, 2,2,2 6.1;
//  - 4 bits in blocks of 16: M = 64 512->16000 2,2,4 8.4, 2,2,8 12.4, 1,2,4 10.2; 2048->8192 11.9, 13.7, 14.0;
//    M = 20 512->16000 4.8, 6.5, 6.4; 2048->8192 7.0, 6.8, 7.9; M = 8 512->16000 1,2,4 4.4, 1,2,8 5.3, six
//    chunks 4.2, 4.0.
RowsPlan plan_rows(int op, int bits, bool split, int64_t M, int64_t ntiles, int64_t nch, int cus) {
  const int64_t r = (M + 15) / 16, work = ntiles * r;
  const int nw = nch > 8 ? 16 : 8;
  const bool wide_regs = bits == 2 || split;
  if (op == ROW_GEN) return {1, 1, 8};
  if (work <= cus) return {1, 1, wide_regs ? 8 : nw};
  if (wide_regs) {
    const bool few = nch < (bits == 2 ? 8 : 5), barely = r == 2 && M <= 18;
    if (r == 1 || work <= 2 * cus) return {1, 2, few && !(bits == 2 && split) ? 4 : 8};
    if (bits == 2 && split) {
      if (barely || (few && work <= 4 * cus)) return {2, 2, 8};
      return nch <= 3 ? RowsPlan{2, 2, 2} : few ? RowsPlan{1, 1, 4} : RowsPlan{1, 2, 8};
    }
    if (bits == 2) return barely ? RowsPlan{2, 2, 8} : RowsPlan{1, 2, 4};
    return {2, 2, r == 2 && !few ? 8 : 4};
  }
  if (op == ROW_INT) {
    if (work <= 2 * cus) return {1, 2, 8};
    if (r > 1 && work <= 4 * cus) return {2, 2, 8};
    return {1, 2, 4};
  }
  if (work <= 2 * cus) return {1, 2, nw};
  if (r == 1) return {1, 2, ntiles >= 8 * cus ? 4 : 8};
  if (work <= 4 * cus) return {2, 2, 8};
  if (work <= 8 * cus) return {2, 4, 8};
  return {2, 2, 4};
}

// The operand path of a call's types, or -1 where the kernel does not apply to them.
int rows_op(const tmh_weight* w, int a_dtype) {
  if (w->zp_kind != TMH_ZP_FLOAT) {
    if (a_dtype == TMH_F16 && w->wdtype == TMH_F16) return ROW_F16;
    if (a_dtype == TMH_BF16 && w->wdtype == TMH_BF16) return ROW_BF16;
    if (a_dtype == TMH_F32 && w->wdtype == TMH_F32 && w->bits != 2 && w->block_size >= 32) return ROW_INT;
  }
  return ROW_GEN;
}

}  // namespace

bool gemv_rows_ok(const tmh_weight* w, const void* a, int a_dtype, int64_t M, int64_t lda) {
  const int64_t a_size = dtype_size(a_dtype), limit = int64_t(1) << 31;
  const int64_t pad = (w->nchunks * chunk_weights(w->bits) - w->K) / 4;
  return M >= 1 && M <= 64 && reinterpret_cast<uintptr_t>(a) % 16 == 0 && lda * a_size % 16 == 0 && w->K % 8 == 0 &&
         M * lda * a_size < limit && (w->ntiles + 4) * w->nchunks * 1024 < limit &&
         (w->ntiles + 4) * w->nchunks * w->nbc * 16 * 4 < limit && w->N < limit && pad < 256 && w->nbc < 256;
}

namespace {

void launch_rows(const tmh_weight* w, const void* a, int a_dtype, int64_t M, int64_t lda, const void* bias, int bias_dtype,
                 void* y, int y_dtype, int dot_dtype, int64_t ldy, hipStream_t s, int num_cus) {
  const int cw = chunk_weights(w->bits);
  int shift = 0;
  while ((1 << shift) < std::min(w->block_size, cw)) ++shift;
  const int op = rows_op(w, a_dtype);
  const bool split = w->block_size < cw / 4;  // a lane's k-group spans several blocks
  const uint32_t pad = static_cast<uint32_t>((w->nchunks * cw - w->K) / 4);
  const RowsArgs d{reinterpret_cast<const uint4_t*>(w->d_q), w->d_scale, static_cast<const uint8_t*>(w->d_zero), a,
                   static_cast<uint32_t>(w->nchunks), static_cast<uint32_t>(w->ntiles), static_cast<uint32_t>(lda),
                   static_cast<uint32_t>(M) | (static_cast<uint32_t>(w->nbc) << 12) | (static_cast<uint32_t>(shift) << 20) | (pad / 2 << 24) |
                       (bias ? 1u << 31 : 0u),
                   y, ldy, static_cast<uint32_t>(w->N),
                   static_cast<uint32_t>(y_dtype) | (static_cast<uint32_t>(dot_dtype) << 8) |
                       (static_cast<uint32_t>(bias ? bias_dtype : 0) << 16) | (static_cast<uint32_t>(a_dtype) << 24),
                   static_cast<uint32_t>(w->zp_kind) | (static_cast<uint32_t>(w->wdtype) << 8), bias};
  const RowsPlan p = plan_rows(op, w->bits, split, M, w->ntiles, w->nchunks, num_cus > 0 ? num_cus : 256);
#define TMH_ROWS_BITS(B)                                                          \
  switch (op) {                                                                   \
    case ROW_F16:                                                                 \
      if (split) launch_op<B, ROW_F16, true>(d, M, p, s);                         \
      else launch_op<B, ROW_F16, false>(d, M, p, s);                              \
      break;                                                                      \
    case ROW_BF16:                                                                \
      if (split) launch_op<B, ROW_BF16, true>(d, M, p, s);                        \
      else launch_op<B, ROW_BF16, false>(d, M, p, s);                             \
      break;                                                                      \
    case ROW_INT:                                                                 \
      if constexpr (B != 2) launch_op<B, ROW_INT, false>(d, M, p, s);             \
      break;                                                                      \
    default: launch_op<B, ROW_GEN, true>(d, M, p, s);                             \
  }
  switch (w->bits) {
    case 2: TMH_ROWS_BITS(2) break;
    case 4: TMH_ROWS_BITS(4) break;
    default: TMH_ROWS_BITS(8)
  }
#undef TMH_ROWS_BITS
}

}  // namespace

// As many rows a launch as its shape and 32-bit offsets over A take: a launch for every 64 rows would
// leave the chip idle where N is small (bf16 in blocks of 16, us: 16384 x 64 -> 64 k_matmul_general 218,
// a launch for every 64 rows 516, this 14.1; 1024 x 2048 -> 2048 2390, 93, 37).
void launch_gemv_rows(const tmh_weight* w, const void* a, int a_dtype, int64_t M, int64_t lda, const void* bias,
                      int bias_dtype, void* y, int y_dtype, int dot_dtype, int64_t ldy, hipStream_t s, int num_cus) {
  const int64_t a_size = dtype_size(a_dtype), fit = ((int64_t(1) << 31) - 1) / (lda * a_size) / 64 * 64;
  const int64_t most = std::max<int64_t>(64, std::min(kRowsMax, fit));  // (gemv_rows_ok: M or 64 rows fit)
  for (int64_t m = 0; m < M; m += most)
    launch_rows(w, static_cast<const uint8_t*>(a) + m * lda * a_size, a_dtype, std::min(most, M - m), lda, bias, bias_dtype,
                static_cast<uint8_t*>(y) + m * ldy * dtype_size(y_dtype), y_dtype, dot_dtype, ldy, s, num_cus);
}

}  // namespace tmh
