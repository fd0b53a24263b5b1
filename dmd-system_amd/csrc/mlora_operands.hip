// Adapter operands of one call, all matrices in one launch: the bf16 hi part (and lo part, for
// fp32 masters used at fp32-class precision: hi = bf16(v), lo = bf16(v - hi)) of every lora_a /
// lora_b, zero-padded and at any place of a stacked matrix, and their transposes (A_aᵀ [K, r], the
// NT form of dX's LoRA term).
//
// The matrices are small (a few hundred KB), so launches and not bytes set the time: one torch
// op per matrix and step took 2.5-5 us of GPU time each (10 launches and 27 us for one rank-128
// master pair forward, 16 for a transposing backward of 16 adapters) and ~8 us of host time. One
// workgroup moves a 64x64 tile with 16-byte accesses (element by element where the pointers or
// pitches do not allow them), all of its loads in flight at once; the transpose goes through LDS.
#include "mlora_common.h"
#include "mlora_host.h"

namespace mlora {

constexpr int kOperandItems = 64;  // matrices per launch (the table travels in the kernel arguments)

struct OperandItem {
  const void *src;          // [rows, cols], pitch lds (elements)
  uint16_t *hi, *lo, *t;    // hi / lo [prows, pcols] (pitch ldo); t [pcols, prows] (pitch ldt); any may be null
  int32_t lds, ldo, ldt;
  int32_t rows, cols, prows, pcols;
  int32_t vec;  // every pointer and pitch allows 16-byte accesses
};

struct OperandArgs {
  int32_t n;
  int32_t src_f32;
  int32_t tile_start[kOperandItems + 1];
  OperandItem item[kOperandItems];
};

__global__ __launch_bounds__(256) void operands_kernel(const OperandArgs args) {
  __shared__ uint16_t tile[64][72];  // 16-byte chunks of a row stay aligned
  const int bid = blockIdx.x;
  int lo = 0, hi = args.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (args.tile_start[mid] <= bid) lo = mid; else hi = mid - 1;
  }
  const OperandItem it = args.item[lo];
  const int tc = (it.pcols + 63) / 64, local = bid - args.tile_start[lo];
  const int r0 = local / tc * 64, c0 = local % tc * 64;
  // thread: 8 columns of rows q and q + 32 of the tile
  const int c8 = 8 * (threadIdx.x & 7), q = threadIdx.x >> 3;
  float v[2][8];  // both rows' loads in flight together
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = r0 + q + 32 * i, c = c0 + c8;
    const int64_t e = (int64_t)r * it.lds + c;
    const bool whole = it.vec && r < it.rows && c + 8 <= it.cols;
    if (args.src_f32) {
      const MLORA_GLOBAL float *p = gp(static_cast<const float *>(it.src)) + e;
      if (whole) {
        const f32x4 x0 = *(const MLORA_GLOBAL f32x4 *)p, x1 = *(const MLORA_GLOBAL f32x4 *)(p + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = x0[j], v[i][4 + j] = x1[j];
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = r < it.rows && c + j < it.cols ? p[j] : 0.f;
      }
    } else {
      const MLORA_GLOBAL uint16_t *p = gp(static_cast<const uint16_t *>(it.src)) + e;
      if (whole) {
        const u32x4 u = *(const MLORA_GLOBAL u32x4 *)p;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = bf16_to_f32((uint16_t)(j % 2 ? u[j / 2] >> 16 : u[j / 2] & 0xffff));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = r < it.rows && c + j < it.cols ? bf16_to_f32(p[j]) : 0.f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int rl = q + 32 * i, r = r0 + rl, c = c0 + c8;
    u32x4 h, l;
    split_hi_lo(v[i], h, l);
    // (a bf16 source keeps its bits: the conversion of its own value is exact, not-a-numbers aside)
    *(MLORA_LDS u32x4 *)((MLORA_LDS uint16_t *)&tile[rl][c8]) = h;
    if (r >= it.prows) continue;
    const int64_t o = (int64_t)r * it.ldo + c;
    if (it.vec && c + 8 <= it.pcols) {
      if (it.hi != nullptr) *(MLORA_GLOBAL u32x4 *)(it.hi + o) = h;
      if (it.lo != nullptr) *(MLORA_GLOBAL u32x4 *)(it.lo + o) = l;
    } else {
      for (int j = 0; j < 8 && c + j < it.pcols; ++j) {
        const int sh = 16 * (j % 2);
        if (it.hi != nullptr) it.hi[o + j] = (uint16_t)(word_of(h, j / 2) >> sh);
        if (it.lo != nullptr) it.lo[o + j] = (uint16_t)(word_of(l, j / 2) >> sh);
      }
    }
  }
  if (it.t == nullptr) return;  // uniform
  __syncthreads();
  // thread: 8 rows (r8 ..) of tile columns q and q + 32, one 16-byte run of t
  const int r8 = c8;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int cl = q + 32 * i, c = c0 + cl, r = r0 + r8;
    if (c >= it.pcols || r >= it.prows) continue;
    uint16_t w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = tile[r8 + j][cl];
    uint16_t *d = it.t + (int64_t)c * it.ldt + r;
    if (it.vec && r + 8 <= it.prows) {
      *(MLORA_GLOBAL u32x4 *)d = u32x4{w[0] | (uint32_t)w[1] << 16, w[2] | (uint32_t)w[3] << 16,
                                       w[4] | (uint32_t)w[5] << 16, w[6] | (uint32_t)w[7] << 16};
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (r + j < it.prows) d[j] = w[j];
    }
  }
}

}  // namespace mlora

using namespace mlora;

extern "C" int mlora_prepare_operands(const void *const *src, int src_dtype, const int64_t *src_ld,
                                      const int64_t *rows, const int64_t *cols, const int64_t *padded_rows,
                                      const int64_t *padded_cols, void *const *hi, void *const *lo,
                                      const int64_t *out_ld, void *const *t, const int64_t *t_ld, int32_t n,
                                      void *stream) {
  if (n < 0) return MLORA_ERR_INVALID;
  if (src_dtype != MLORA_F32 && src_dtype != MLORA_BF16) return MLORA_ERR_UNSUPPORTED;
  if (n == 0) return MLORA_OK;
  if (src == nullptr || src_ld == nullptr || rows == nullptr || cols == nullptr || padded_rows == nullptr ||
      padded_cols == nullptr || hi == nullptr || lo == nullptr || out_ld == nullptr || t == nullptr || t_ld == nullptr)
    return MLORA_ERR_INVALID;
  for (int32_t i = 0; i < n; ++i) {
    const int64_t r = rows[i], c = cols[i], pr = padded_rows[i], pc = padded_cols[i];
    if (r < 0 || c < 0 || pr < r || pc < c) return MLORA_ERR_INVALID;
    if (pr > INT32_MAX - 64 || pc > INT32_MAX - 64) return MLORA_ERR_LIMIT;
    if (r > 0 && c > 0 && (src[i] == nullptr || src_ld[i] < c)) return MLORA_ERR_INVALID;
    if ((hi[i] != nullptr || lo[i] != nullptr) && out_ld[i] < pc) return MLORA_ERR_INVALID;
    if (t[i] != nullptr && t_ld[i] < pr) return MLORA_ERR_INVALID;
    if (src_ld[i] > INT32_MAX || out_ld[i] > INT32_MAX || t_ld[i] > INT32_MAX) return MLORA_ERR_LIMIT;
  }
  for (int32_t i0 = 0; i0 < n; i0 += kOperandItems) {
    OperandArgs a{};
    a.src_f32 = src_dtype == MLORA_F32;
    int64_t tiles = 0;
    for (int32_t i = i0; i < n && i < i0 + kOperandItems; ++i) {
      if (hi[i] == nullptr && lo[i] == nullptr && t[i] == nullptr) continue;
      const int64_t m = ((padded_rows[i] + 63) / 64) * ((padded_cols[i] + 63) / 64);
      if (m == 0) continue;
      const bool vec = aligned16(src[i]) && aligned16(hi[i]) && aligned16(lo[i]) && aligned16(t[i]) &&
                       src_ld[i] % 8 == 0 && out_ld[i] % 8 == 0 && t_ld[i] % 8 == 0;
      a.tile_start[a.n] = (int32_t)tiles;
      a.item[a.n++] = OperandItem{src[i], static_cast<uint16_t *>(hi[i]), static_cast<uint16_t *>(lo[i]),
                                  static_cast<uint16_t *>(t[i]), (int32_t)src_ld[i], (int32_t)out_ld[i],
                                  (int32_t)t_ld[i], (int32_t)rows[i], (int32_t)cols[i], (int32_t)padded_rows[i],
                                  (int32_t)padded_cols[i], vec ? 1 : 0};
      tiles += m;
      if (tiles > INT32_MAX) return MLORA_ERR_LIMIT;
    }
    if (a.n == 0) continue;
    a.tile_start[a.n] = (int32_t)tiles;
    hipLaunchKernelGGL(operands_kernel, dim3((unsigned)tiles), dim3(256), 0, static_cast<hipStream_t>(stream), a);
    const int st = launch_status();
    if (st) return st;
  }
  return MLORA_OK;
}
