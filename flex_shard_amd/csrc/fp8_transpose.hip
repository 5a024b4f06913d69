// Operand preparation for the backward products of the blockwise FP8 linear:
// both need an operand whose contraction index is contiguous in memory.
//
//   fp8_transpose_kernel       dst[c][r] = src[r][c] for a byte matrix (the
//                              gathered weight, read along its output index
//                              by the input-gradient product)
//   act_quant_128x1_t_kernel   quantizes every run of 128 consecutive ROWS of
//                              a column of a bf16 matrix and writes the bytes
//                              transposed, q[c][r]; serves both operands of
//                              the weight-gradient product (contraction over
//                              tokens)
//   backward_operands_kernel   both of one layer's backward in one launch: the
//                              output gradient's tiles, then the weight's
//   bias_gradient_kernel       adds up the column sums that the quantizer left
//                              per 128 tokens
//
// The first three work on 128 x 128 tiles through LDS: rows go in as they are read
// (16-byte global loads along the source rows), and come out along the
// source columns as 16-byte runs of 16 source rows each.
#include "common.hpp"

namespace fsh {
namespace {

constexpr int kTileDim = 128;
constexpr int kTransposeThreads = 256;
// LDS pitch of a tile row in bytes: 33 dwords, so that the sixteen rows a
// lane gathers from and the eight row groups of a wave spread over the banks.
constexpr int kTilePitch = 132;

// Writes the transposed tile held in LDS (`tile[r * kTilePitch + c]`, r = tile
// row = destination column) to dst rows [c0, c0 + 128) x columns [r0, r0 + 128).
// Destination columns up to ld_dst are written (the caller zero-fills the tile
// rows past the source), destination rows past dst_rows are skipped.
__device__ __forceinline__ void store_tile_transposed(const uint8_t* tile, uint8_t* dst, int64_t c0, int64_t r0,
                                                      int64_t dst_rows, int64_t ld_dst, int tid) {
  const int rchunk = tid & 7;  // destination bytes [16 rchunk, +16) of the row
#pragma unroll
  for (int pass = 0; pass < kTileDim / 32; ++pass) {
    const int c = pass * 32 + (tid >> 3);
    uint32_t w[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t v = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b)
        v |= static_cast<uint32_t>(tile[(16 * rchunk + 4 * d + b) * kTilePitch + c]) << (8 * b);
      w[d] = v;
    }
    const int64_t row = c0 + c, col = r0 + 16 * rchunk;
    if (row < dst_rows && col < ld_dst)  // ld_dst is a multiple of 16
      *reinterpret_cast<u32x4*>(dst + row * ld_dst + col) = u32x4{w[0], w[1], w[2], w[3]};
  }
}

struct TransposeParams {
  const uint8_t* src;
  uint8_t* dst;
  int64_t rows, cols, ld_src, ld_dst;
  int32_t tiles_c;
};

__device__ __forceinline__ void transpose_tile(const TransposeParams& p, uint8_t* tile, uint32_t id) {
  const int tid = threadIdx.x;
  const int64_t r0 = static_cast<int64_t>(id / p.tiles_c) * kTileDim;
  const int64_t c0 = static_cast<int64_t>(id % p.tiles_c) * kTileDim;
  const int chunk = tid & 7;
  u32x4 v[4];
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int64_t row = r0 + pass * 32 + (tid >> 3), col = c0 + chunk * 16;
    v[pass] = u32x4{0, 0, 0, 0};
    if (row < p.rows && col < p.cols) {  // cols is a multiple of 16
      v[pass] = load_stream_u32x4(p.src + row * p.ld_src + col);
    }
  }
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    uint32_t* dst = reinterpret_cast<uint32_t*>(tile + (pass * 32 + (tid >> 3)) * kTilePitch + chunk * 16);
    dst[0] = v[pass].x; dst[1] = v[pass].y; dst[2] = v[pass].z; dst[3] = v[pass].w;
  }
  __syncthreads();
  store_tile_transposed(tile, p.dst, c0, r0, p.cols, p.ld_dst, tid);
}

__global__ __launch_bounds__(kTransposeThreads) void fp8_transpose_kernel(const TransposeParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t tile[kTileDim * kTilePitch];
  transpose_tile(p, tile, blockIdx.x);
}

struct ActQuantTParams {
  const uint8_t* x;
  uint8_t* q;      // [cols][ldq]
  float* scales;   // [ldq / 128][cols]
  int64_t rows, cols, ldx, ldq;
  int32_t tiles_c;
  float eps;
  // the row-run outputs of the dual kernel: q_row [rows][ldq_row], scales_row [ldq_row / 128][rows]
  uint8_t* q_row;
  float* scales_row;
  int64_t ldq_row;
  float* column_sums;  // [ldq / 128][cols] sums over each run of 128 rows, or null
};

template <bool kAlsoRowRuns>
struct ActQuantTShared {
  __attribute__((aligned(16))) uint8_t tile[kTileDim * kTilePitch];  // first the threads' column sums
  __attribute__((aligned(16))) uint16_t col_max[16 * kTileDim];
  __attribute__((aligned(16))) float col_scale[kTileDim];
  float row_recip[kAlsoRowRuns ? kTileDim : 1];
};
static_assert(16 * kTileDim * 4 <= kTileDim * kTilePitch, "the column sums fit the tile's LDS");

// Thread t loads columns [8 (t & 15), +8) of tile rows (t >> 4) + 16 k, k = 0..7.
// kAlsoRowRuns: the same tile also leaves quantized in runs of 128 along its
// rows (the arithmetic and the outputs of act_quant_1x128_kernel), so an
// operand needed in both forms is read once.  A tile row's 128 columns lie in
// one row of 16 lanes, whose maximum takes four DPP steps.
// column_sums: the tile is in registers, so its column sums (the bias gradient
// is the sum of the output gradient over the tokens) cost eight additions per
// element row and 8 KB through LDS instead of a pass of its own over the
// matrix (14.6 us at 1000 x 5120, and 4 us for a fill that the pass needed).
template <bool kAlsoRowRuns>
__device__ __forceinline__ void quantize_tile_transposed(const ActQuantTParams& p, ActQuantTShared<kAlsoRowRuns>& shared, uint32_t id) {
  uint8_t* const tile = shared.tile;
  uint16_t* const col_max = shared.col_max;
  float* const col_scale = shared.col_scale;
  float* const row_recip = shared.row_recip;
  float* const col_sum = reinterpret_cast<float*>(shared.tile);
  const int tid = threadIdx.x;
  const int cg = tid & 15, rl = tid >> 4;
  const int64_t rb = id / p.tiles_c;
  const int64_t r0 = rb * kTileDim, c0 = static_cast<int64_t>(id % p.tiles_c) * kTileDim;
  const int64_t col = c0 + cg * 8;

  u32x4 v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int64_t row = r0 + rl + 16 * k;
    v[k] = u32x4{0, 0, 0, 0};
    if (row < p.rows && col < p.cols) v[k] = load_stream_u32x4(p.x + (row * p.ldx + col) * 2);  // cols % 8 == 0
  }
  if (kAlsoRowRuns) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t row = r0 + rl + 16 * k;
      uint32_t mr = pk_max_u16(v[k].x & 0x7FFF7FFFu, v[k].y & 0x7FFF7FFFu);
      mr = pk_max_u16(mr, v[k].z & 0x7FFF7FFFu);
      mr = pk_max_u16(mr, v[k].w & 0x7FFF7FFFu);
      const uint32_t lo = mr & 0xFFFFu, hi = mr >> 16;
      mr = row16_max_u32(lo > hi ? lo : hi);
      float scale, recip;
      tile_scale(bf16_bits_to_f32(mr), p.eps, scale, recip);
      if (cg == 0) row_recip[rl + 16 * k] = recip;
      if (row < p.rows && col < p.ldq_row) {  // columns past `cols` hold zeros: the pad of the last run
        const uint32_t d[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        uint32_t w[2] = {0, 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e0 = u32_as_f32(d[j] << 16) * scale;
          const float e1 = u32_as_f32(d[j] & 0xFFFF0000u) * scale;
          w[j >> 1] = cvt2_fp8(e0, e1, w[j >> 1], (j & 1) != 0);
        }
        store_stream_u32x2(p.q_row + row * p.ldq_row + col, w[0], w[1]);
      }
    }
  }
  // Largest magnitude (bf16 bit pattern) of the thread's eight rows, per column.
  uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    m[0] = pk_max_u16(m[0], v[k].x & 0x7FFF7FFFu);
    m[1] = pk_max_u16(m[1], v[k].y & 0x7FFF7FFFu);
    m[2] = pk_max_u16(m[2], v[k].z & 0x7FFF7FFFu);
    m[3] = pk_max_u16(m[3], v[k].w & 0x7FFF7FFFu);
  }
  *reinterpret_cast<u32x4*>(col_max + rl * kTileDim + cg * 8) = u32x4{m[0], m[1], m[2], m[3]};
  if (p.column_sums) {
    f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;  // (rows past the matrix were loaded as zero)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      lo.x += u32_as_f32(v[k].x << 16); lo.y += u32_as_f32(v[k].x & 0xFFFF0000u);
      lo.z += u32_as_f32(v[k].y << 16); lo.w += u32_as_f32(v[k].y & 0xFFFF0000u);
      hi.x += u32_as_f32(v[k].z << 16); hi.y += u32_as_f32(v[k].z & 0xFFFF0000u);
      hi.z += u32_as_f32(v[k].w << 16); hi.w += u32_as_f32(v[k].w & 0xFFFF0000u);
    }
    *reinterpret_cast<f32x4*>(col_sum + rl * kTileDim + cg * 8) = lo;
    *reinterpret_cast<f32x4*>(col_sum + rl * kTileDim + cg * 8 + 4) = hi;
  }
  __syncthreads();
  if (tid < kTileDim) {
    uint32_t best = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t candidate = col_max[r * kTileDim + tid];
      best = candidate > best ? candidate : best;
    }
    float scale, recip;
    tile_scale(bf16_bits_to_f32(best), p.eps, scale, recip);
    col_scale[tid] = scale;
    if (c0 + tid < p.cols) p.scales[rb * p.cols + c0 + tid] = recip;
    // (row_recip was filled before the first barrier above)
    if (kAlsoRowRuns && r0 + tid < p.rows) p.scales_row[(c0 / kTileDim) * p.rows + r0 + tid] = row_recip[tid];
  } else if (p.column_sums) {  // the other half of the threads
    const int c = tid - kTileDim;
    float sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) sum += col_sum[r * kTileDim + c];
    if (c0 + c < p.cols) p.column_sums[rb * p.cols + c0 + c] = sum;
  }
  __syncthreads();
  const f32x4 s_lo = *reinterpret_cast<const f32x4*>(col_scale + cg * 8);
  const f32x4 s_hi = *reinterpret_cast<const f32x4*>(col_scale + cg * 8 + 4);
  const float s[8] = {s_lo.x, s_lo.y, s_lo.z, s_lo.w, s_hi.x, s_hi.y, s_hi.z, s_hi.w};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t d[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float e0 = u32_as_f32(d[j] << 16) * s[2 * j];
      const float e1 = u32_as_f32(d[j] & 0xFFFF0000u) * s[2 * j + 1];
      w[j >> 1] = cvt2_fp8(e0, e1, w[j >> 1], (j & 1) != 0);
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(tile + (rl + 16 * k) * kTilePitch + cg * 8);
    dst[0] = w[0];
    dst[1] = w[1];
  }
  __syncthreads();
  store_tile_transposed(tile, p.q, c0, r0, p.cols, p.ldq, tid);
}

template <bool kAlsoRowRuns>
__global__ __launch_bounds__(kTransposeThreads) void act_quant_128x1_t_kernel(const ActQuantTParams p) {
  __shared__ ActQuantTShared<kAlsoRowRuns> shared;
  quantize_tile_transposed(p, shared, blockIdx.x);
}

// One launch for what the two backward products of a layer read: workgroups
// [0, quant_tiles) quantize the output gradient in both forms, the others
// transpose the weight's bytes.  Neither fills the chip for long at a few
// thousand tokens; together they share one start and one end.
__global__ __launch_bounds__(kTransposeThreads) void backward_operands_kernel(const ActQuantTParams quant, const TransposeParams transpose,
                                                                              uint32_t quant_tiles) {
  __shared__ ActQuantTShared<true> shared;
  if (blockIdx.x < quant_tiles)
    quantize_tile_transposed(quant, shared, blockIdx.x);
  else
    transpose_tile(transpose, shared.tile, blockIdx.x - quant_tiles);
}

// out[c] = bf16(sum over runs of sums[run][c]).  64 columns per workgroup,
// four quarters of the runs side by side.
__global__ __launch_bounds__(256) void bias_gradient_kernel(const float* sums, uint16_t* out, int64_t runs, int64_t cols) {
  __shared__ float part[4][64];
  const int lane = threadIdx.x & 63, quarter = threadIdx.x >> 6;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  float sum = 0.0f;
  if (c < cols) {
#pragma unroll 8
    for (int64_t r = quarter; r < runs; r += 4) sum += sums[r * cols + c];
  }
  part[quarter][lane] = sum;
  __syncthreads();
  if (quarter == 0 && c < cols) out[c] = static_cast<uint16_t>(f32_to_bf16_bits(part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane]));
}

float floor_for(int32_t eps_mode) {
  const float eps32 = 1e-12f;
  uint32_t bits;
  memcpy(&bits, &eps32, 4);
  bits = (bits + 0x7FFFu + ((bits >> 16) & 1u)) & 0xFFFF0000u;
  float eps_bf16;
  memcpy(&eps_bf16, &bits, 4);
  return eps_mode == FSH_EPS_FP32 ? eps32 : eps_bf16;
}


int transpose_params(TransposeParams& p, int64_t& tiles, const void* src_dev, int64_t rows, int64_t cols, int64_t ld_src,
                     void* dst_dev, int64_t ld_dst, const char* who) {
  if (!src_dev || !dst_dev) return fail(FSH_EINVAL, "%s: null pointer", who);
  if (ld_src < cols || ld_dst < rows)
    return fail(FSH_EINVAL, "%s: ld_src %lld < cols %lld or ld_dst %lld < rows %lld", who, (long long)ld_src, (long long)cols,
                (long long)ld_dst, (long long)rows);
  if (cols % 16 || ld_src % 16 || ld_dst % 16 || !aligned(src_dev, 16) || !aligned(dst_dev, 16))
    return fail(FSH_ENOTSUP, "%s: cols and both leading dimensions must be multiples of 16, pointers 16-byte aligned", who);
  if (ld_dst > ceil_div(rows, (int64_t)kTileDim) * kTileDim)
    return fail(FSH_ENOTSUP, "%s: ld_dst %lld exceeds rows %lld rounded up to 128 (only that much is zero-filled)", who,
                (long long)ld_dst, (long long)rows);
  p.src = static_cast<const uint8_t*>(src_dev);
  p.dst = static_cast<uint8_t*>(dst_dev);
  p.rows = rows; p.cols = cols; p.ld_src = ld_src; p.ld_dst = ld_dst;
  const int64_t tiles_c = ceil_div(cols, (int64_t)kTileDim);
  tiles = ceil_div(rows, (int64_t)kTileDim) * tiles_c;
  if (tiles > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "%s: too many tiles", who);
  p.tiles_c = static_cast<int32_t>(tiles_c);
  return FSH_OK;
}

// q_row_dev null: the token-run form alone.
int act_quant_params(ActQuantTParams& p, int64_t& tiles, const void* x_dev, int64_t rows, int64_t cols, int64_t ldx,
                     void* q_row_dev, int64_t ldq_row, float* scales_row_dev, void* q_col_dev, int64_t ldq_col,
                     float* scales_col_dev, float* column_sums_dev, int32_t eps_mode, const char* who) {
  if (eps_mode != FSH_EPS_INPUT_DTYPE && eps_mode != FSH_EPS_FP32) return fail(FSH_EINVAL, "%s: unknown eps_mode %d", who, eps_mode);
  const int64_t padded_rows = ceil_div(rows, (int64_t)kTileDim) * kTileDim;
  const int64_t padded_cols = ceil_div(cols, (int64_t)kTileDim) * kTileDim;
  if (ldx < cols || ldq_col != padded_rows || (q_row_dev && ldq_row != padded_cols))
    return fail(FSH_EINVAL,
                "%s: ldx %lld < cols %lld, or an output's leading dimension (%lld, %lld) is not its length rounded up to 128 (%lld, %lld)",
                who, (long long)ldx, (long long)cols, (long long)ldq_col, (long long)ldq_row, (long long)padded_rows,
                (long long)padded_cols);
  if (cols % 8 || ldx % 8 || !aligned(x_dev, 16) || !aligned(q_col_dev, 16) || !aligned(q_row_dev, 8) ||
      !aligned(scales_row_dev, 4) || !aligned(scales_col_dev, 4) || !aligned(column_sums_dev, 4))
    return fail(FSH_ENOTSUP, "%s: cols and ldx must be multiples of 8, x and the transposed bytes 16-byte and the row bytes 8-byte aligned", who);
  p.x = static_cast<const uint8_t*>(x_dev);
  p.q = static_cast<uint8_t*>(q_col_dev);
  p.scales = scales_col_dev;
  p.rows = rows; p.cols = cols; p.ldx = ldx; p.ldq = ldq_col;
  p.eps = floor_for(eps_mode);
  p.q_row = static_cast<uint8_t*>(q_row_dev);
  p.scales_row = scales_row_dev;
  p.ldq_row = ldq_row;
  p.column_sums = column_sums_dev;
  const int64_t tiles_c = padded_cols / kTileDim;
  tiles = (padded_rows / kTileDim) * tiles_c;
  if (tiles > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "%s: too many tiles", who);
  p.tiles_c = static_cast<int32_t>(tiles_c);
  return FSH_OK;
}

// Where the operands of a backward lie in its scratch memory (every part a
// multiple of 128 bytes): the output gradient in runs along its rows, its
// token-run form, the weight's transposed bytes, the column sums.
struct BackwardScratch {
  int64_t tokens_padded, cols_padded, q_row, scales_row, q_col, scales_col, weight_t, sums, nbytes;
};
BackwardScratch backward_scratch(int64_t tokens, int64_t cols, int64_t in_cols, bool grad_x, bool grad_w, bool grad_bias) {
  BackwardScratch s;
  auto round = [](int64_t n) { return ceil_div(n, (int64_t)128) * 128; };
  s.tokens_padded = round(tokens);
  s.cols_padded = round(cols);
  int64_t at = 0;
  auto take = [&](bool wanted, int64_t nbytes) {
    const int64_t mine = at;
    if (wanted) at += round(nbytes);
    return mine;
  };
  s.q_row = take(grad_x, tokens * s.cols_padded);
  s.scales_row = take(grad_x, s.cols_padded / 128 * tokens * 4);
  s.q_col = take(grad_w, cols * s.tokens_padded);
  s.scales_col = take(grad_w, s.tokens_padded / 128 * cols * 4);
  s.weight_t = take(grad_x, in_cols * s.cols_padded);
  s.sums = take(grad_bias, s.tokens_padded / 128 * cols * 4);
  s.nbytes = at;
  return s;
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_fp8_transpose(const void* src_dev, int64_t rows, int64_t cols, int64_t ld_src, void* dst_dev,
                              int64_t ld_dst, void* stream) {
  using namespace fsh;
  if (rows < 0 || cols < 0) return fail(FSH_EINVAL, "fsh_fp8_transpose: negative shape");
  if (rows == 0 || cols == 0) return FSH_OK;
  TransposeParams p;
  int64_t tiles = 0;
  if (int rc = transpose_params(p, tiles, src_dev, rows, cols, ld_src, dst_dev, ld_dst, "fsh_fp8_transpose")) return rc;
  hipLaunchKernelGGL(fp8_transpose_kernel, dim3(static_cast<uint32_t>(tiles)), dim3(kTransposeThreads), 0,
                     static_cast<hipStream_t>(stream), p);
  return check_launch("fp8_transpose_kernel");
}

FSH_API int fsh_act_quant_128x1_transposed(const void* x_dev, int64_t rows, int64_t cols, int64_t ldx, void* q_dev,
                                           int64_t ldq, float* scales_dev, int32_t eps_mode, void* stream) {
  using namespace fsh;
  if (rows < 0 || cols < 0) return fail(FSH_EINVAL, "fsh_act_quant_128x1_transposed: negative shape");
  if (rows == 0 || cols == 0) return FSH_OK;
  if (!x_dev || !q_dev || !scales_dev) return fail(FSH_EINVAL, "fsh_act_quant_128x1_transposed: null pointer");
  ActQuantTParams p;
  int64_t tiles = 0;
  if (int rc = act_quant_params(p, tiles, x_dev, rows, cols, ldx, nullptr, 0, nullptr, q_dev, ldq, scales_dev, nullptr,
                                eps_mode, "fsh_act_quant_128x1_transposed"))
    return rc;
  hipLaunchKernelGGL(act_quant_128x1_t_kernel<false>, dim3(static_cast<uint32_t>(tiles)), dim3(kTransposeThreads), 0,
                     static_cast<hipStream_t>(stream), p);
  return check_launch("act_quant_128x1_t_kernel");
}

FSH_API int fsh_act_quant_both(const void* x_dev, int64_t rows, int64_t cols, int64_t ldx, void* q_row_dev,
                               int64_t ldq_row, float* scales_row_dev, void* q_col_dev, int64_t ldq_col,
                               float* scales_col_dev, int32_t eps_mode, void* stream) {
  using namespace fsh;
  if (rows < 0 || cols < 0) return fail(FSH_EINVAL, "fsh_act_quant_both: negative shape");
  if (rows == 0 || cols == 0) return FSH_OK;
  if (!x_dev || !q_row_dev || !scales_row_dev || !q_col_dev || !scales_col_dev)
    return fail(FSH_EINVAL, "fsh_act_quant_both: null pointer");
  ActQuantTParams p;
  int64_t tiles = 0;
  if (int rc = act_quant_params(p, tiles, x_dev, rows, cols, ldx, q_row_dev, ldq_row, scales_row_dev, q_col_dev, ldq_col,
                                scales_col_dev, nullptr, eps_mode, "fsh_act_quant_both"))
    return rc;
  hipLaunchKernelGGL(act_quant_128x1_t_kernel<true>, dim3(static_cast<uint32_t>(tiles)), dim3(kTransposeThreads), 0,
                     static_cast<hipStream_t>(stream), p);
  return check_launch("act_quant_128x1_t_kernel<true>");
}

FSH_API int64_t fsh_fp8_linear_backward_scratch_bytes(int64_t tokens, int64_t out_cols, int64_t in_cols, int32_t grad_x,
                                                      int32_t grad_w, int32_t grad_bias) {
  using namespace fsh;
  if (tokens < 0 || out_cols < 0 || in_cols < 0) return 0;
  return backward_scratch(tokens, out_cols, in_cols, grad_x != 0, grad_w != 0, grad_bias != 0).nbytes;
}

FSH_API int fsh_fp8_linear_backward(const void* grad_dev, int64_t tokens, int64_t out_cols, int64_t ldg, const void* wq_dev,
                                    int64_t out_dim, int64_t in_cols, int64_t in_dim, int64_t ldwq, const float* ws_dev,
                                    int64_t ws_cols, const void* x_runs_dev, const float* x_runs_scales_dev, int64_t x_cols,
                                    void* grad_x_dev, void* grad_w_dev, void* grad_bias_dev, void* scratch_dev,
                                    int64_t scratch_nbytes, void* stream) {
  using namespace fsh;
  const char* who = "fsh_fp8_linear_backward";
  if (tokens < 0 || out_cols <= 0 || in_dim <= 0 || out_dim <= 0) return fail(FSH_EINVAL, "%s: empty or negative shape", who);
  if (tokens == 0 && grad_w_dev) return fail(FSH_ENOTSUP, "%s: a weight gradient needs tokens", who);
  if (tokens == 0) return FSH_OK;
  if (!grad_dev || !scratch_dev) return fail(FSH_EINVAL, "%s: null pointer", who);
  if (grad_bias_dev && !grad_w_dev) return fail(FSH_ENOTSUP, "%s: the bias gradient comes with the weight gradient", who);
  if (out_cols < out_dim || in_cols < in_dim) return fail(FSH_EINVAL, "%s: fewer columns than the layer has", who);
  const BackwardScratch at = backward_scratch(tokens, out_cols, in_cols, grad_x_dev, grad_w_dev, grad_bias_dev);
  if (scratch_nbytes < at.nbytes || !aligned(scratch_dev, 128))
    return fail(FSH_EINVAL, "%s: scratch of %lld bytes, %lld needed, 128-byte aligned", who, (long long)scratch_nbytes, (long long)at.nbytes);
  if (grad_x_dev && ceil_div(out_dim, (int64_t)128) * 128 != at.cols_padded)
    return fail(FSH_EINVAL, "%s: %lld gradient columns for %lld outputs", who, (long long)out_cols, (long long)out_dim);
  uint8_t* scratch = static_cast<uint8_t*>(scratch_dev);
  float* const scales_row = reinterpret_cast<float*>(scratch + at.scales_row);
  float* const scales_col = reinterpret_cast<float*>(scratch + at.scales_col);
  float* const sums = grad_bias_dev ? reinterpret_cast<float*>(scratch + at.sums) : nullptr;

  TransposeParams transpose;
  ActQuantTParams quant;
  int64_t transpose_tiles = 0, quant_tiles = 0;
  if (grad_x_dev)
    if (int rc = transpose_params(transpose, transpose_tiles, wq_dev, out_dim, in_cols, ldwq, scratch + at.weight_t,
                                  at.cols_padded, who))
      return rc;
  if (grad_w_dev)
    if (int rc = act_quant_params(quant, quant_tiles, grad_dev, tokens, out_cols, ldg, grad_x_dev ? scratch + at.q_row : nullptr,
                                  at.cols_padded, grad_x_dev ? scales_row : nullptr, scratch + at.q_col, at.tokens_padded,
                                  scales_col, sums, FSH_EPS_FP32, who))
      return rc;
  if (transpose_tiles + quant_tiles > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "%s: too many tiles", who);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (grad_x_dev && grad_w_dev) {
    hipLaunchKernelGGL(backward_operands_kernel, dim3(static_cast<uint32_t>(quant_tiles + transpose_tiles)), dim3(kTransposeThreads),
                       0, s, quant, transpose, static_cast<uint32_t>(quant_tiles));
    if (int rc = check_launch("backward_operands_kernel")) return rc;
  } else if (grad_w_dev) {
    hipLaunchKernelGGL(act_quant_128x1_t_kernel<false>, dim3(static_cast<uint32_t>(quant_tiles)), dim3(kTransposeThreads), 0, s, quant);
    if (int rc = check_launch("act_quant_128x1_t_kernel")) return rc;
  } else if (grad_x_dev) {
    if (int rc = fsh_act_quant_1x128(grad_dev, tokens, out_cols, ldg, scratch + at.q_row, at.cols_padded, scales_row, FSH_EPS_FP32, stream))
      return rc;
    hipLaunchKernelGGL(fp8_transpose_kernel, dim3(static_cast<uint32_t>(transpose_tiles)), dim3(kTransposeThreads), 0, s, transpose);
    if (int rc = check_launch("fp8_transpose_kernel")) return rc;
  }
  if (grad_x_dev)
    if (int rc = fsh_fp8_gemm_1x128_128x128_dgrad(scratch + at.q_row, scales_row, scratch + at.weight_t, ws_dev, grad_x_dev, tokens,
                                                  in_dim, at.cols_padded, at.cols_padded, at.cols_padded, in_dim, ws_cols, stream))
      return rc;
  if (grad_w_dev)
    if (int rc = fsh_fp8_gemm_1x128_128x1(scratch + at.q_col, scales_col, x_runs_dev, x_runs_scales_dev, grad_w_dev, out_cols, x_cols,
                                          at.tokens_padded, at.tokens_padded, at.tokens_padded, x_cols, stream))
      return rc;
  if (grad_bias_dev) {
    hipLaunchKernelGGL(bias_gradient_kernel, dim3(static_cast<uint32_t>(ceil_div(out_cols, (int64_t)64))), dim3(256), 0, s, sums,
                       static_cast<uint16_t*>(grad_bias_dev), at.tokens_padded / 128, out_cols);
    if (int rc = check_launch("bias_gradient_kernel")) return rc;
  }
  return FSH_OK;
}
