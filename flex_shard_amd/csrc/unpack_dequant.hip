// Unpack of gathered rank rows: byte compaction into the parameter-ordered
// buffer fused with blockwise dequantization to bf16 (or fp32), one pass over
// the FP8 bytes.
//
// A chunk is one contiguous run of bytes, and so are its compact bytes and its
// dequantized values.  For block = 128 its T tiles' worth of workgroups split
// that run into T consecutive pieces: eight FP8 bytes per thread and pass (one
// 8-byte load, one 8-byte store into the compact buffer, four v_cvt_pk_f32_fp8
// + multiplies by the tile's reciprocal scale, one 16-byte bf16 store), each
// access contiguous across the wave whatever the width, the dequantized stores
// whole memory lines.  Only the wider output's alignment is arranged; FP8
// bytes at odd offsets (an odd width; rank rows inside a mixed bucket) go out
// unaligned, which global memory instructions may be.  Bound by memory.  Other
// block sizes and widths below eight take an element-wise path.
#include "common.hpp"

namespace fsh {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float load_f32_any(const uint8_t* p) {
  if ((reinterpret_cast<uintptr_t>(p) & 3) == 0) return *reinterpret_cast<const float*>(p);
  uint32_t u = static_cast<uint32_t>(p[0]) | (static_cast<uint32_t>(p[1]) << 8) |
               (static_cast<uint32_t>(p[2]) << 16) | (static_cast<uint32_t>(p[3]) << 24);
  return u32_as_f32(u);
}

__device__ __forceinline__ void store_f32_any(uint8_t* p, float f) {
  if ((reinterpret_cast<uintptr_t>(p) & 3) == 0) {
    *reinterpret_cast<float*>(p) = f;
    return;
  }
  const uint32_t u = f32_as_u32(f);
  p[0] = static_cast<uint8_t>(u);
  p[1] = static_cast<uint8_t>(u >> 8);
  p[2] = static_cast<uint8_t>(u >> 16);
  p[3] = static_cast<uint8_t>(u >> 24);
}

// Four FP8 bytes of `w` -> four floats times `s`.
__device__ __forceinline__ void dequant4(uint32_t w, float s, float* out) {
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w), false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(w), true);
  out[0] = lo.x * s;
  out[1] = lo.y * s;
  out[2] = hi.x * s;
  out[3] = hi.y * s;
}

// `kAligned`: FP8 bytes of every group of eight on 8-byte boundaries, and the
// compact bytes of a piece from a memory line's start: they stream.  Pieces of
// lines stay in the caches until the rest of the line is there.
template <typename V, bool kAligned>
__device__ __forceinline__ V load_group(const uint8_t* p) {
  // A plain load: with the nontemporal hint this kernel, three quarters of
  // whose traffic are stores, measured 13 % slower on rows from HBM and
  // 25 % slower on rows still in the last-level cache (where a gather
  // has just written them).
  if (kAligned) return *reinterpret_cast<const V*>(p);
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
}
template <bool kAligned>
__device__ __forceinline__ void store_group(uint8_t* p, const u32x2& v) {
  if (kAligned)
    store_stream_u32x2(p, v.x, v.y);
  else
    __builtin_memcpy(p, &v, sizeof(v));
}
template <int DQ>
__device__ __forceinline__ void store_value(uint8_t* dq, int64_t idx, float f) {
  if (DQ == FSH_DT_BF16)
    reinterpret_cast<uint16_t*>(dq)[idx] = static_cast<uint16_t>(f32_to_bf16_bits(f));
  else if (DQ == FSH_DT_F16)
    reinterpret_cast<uint16_t*>(dq)[idx] = static_cast<uint16_t>(f32_to_f16_bits(f));
  else
    reinterpret_cast<float*>(dq)[idx] = f;
}

// a / b of a >= 0 and b > 0 that are the same in every lane (a 64-bit division
// is a few hundred cycles ahead of a workgroup's first load).
__device__ __forceinline__ int64_t divide(int64_t a, int64_t b) {
  if (((a | b) >> 32) == 0) return static_cast<uint32_t>(a) / static_cast<uint32_t>(b);
  return a / b;
}

// Eight dequantized values to dq[idx ..], 16-byte aligned.  fp32 ones are two
// stores of every other 16 bytes: plain, so that the caches put them together
// (59 M values to fp32, just gathered: 130 us with the streaming hint, 57 without).
template <int DQ>
__device__ __forceinline__ void store_values8(uint8_t* dq, uint32_t idx, const float (&f)[8]) {
  if (DQ == FSH_DT_F32) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<u32x4*>(dq + idx * 4 + 16 * j) = u32x4{f32_as_u32(f[4 * j]), f32_as_u32(f[4 * j + 1]),
                                                               f32_as_u32(f[4 * j + 2]), f32_as_u32(f[4 * j + 3])};
    return;
  }
  u32x4 o;
  if (DQ == FSH_DT_BF16) {
    o = pack8_bf16(f);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = f32_to_f16_bits(f[2 * j]) | (f32_to_f16_bits(f[2 * j + 1]) << 16);
  }
  store_stream_u32x4(dq + idx * 2, o);
}

// Piece t of `tiles` of a chunk.  `scales`: the chunk's table [rows / 128][in_dim / 128].
// With a tile's own 128 rows per workgroup, memory lines were written in pieces
// wherever the width is no multiple of 128, and completed by workgroups on
// other XCDs.  All loads of a piece go out ahead of its first store and without
// a branch between them, and nothing that waits for memory (the ends of a run
// that are no whole group, the scale's own copy) comes before them.  Four
// passes' FP8 bytes go ahead of the four scales, whose addresses take a
// division.  Us with a tile per workgroup / a branch per load / here, rows from
// HBM and (just gathered, in the last-level cache):
//   218 M layer on eight ranks      169 / 163 / 149     (168 / 159 / 148)
//   67 M of 4096 on one             57 / 56 / 49        (44 / 46 / 44)
//   33 M of 4104 on three           61 / 36 / 29        (57 / 30 / 25)
//   16.8 M of 4096 on one           18.3 / 16.7 / 15.7  (15.1 / 16.0 / 15.1)
//   8.4 M of 4096 on one            10.7 / 11.0 / 10.3  (10.2 / 11.1 / 10.3)
//   2.1 M of 4096 on one            8.2 / 10.3 / 8.3    (8.9 / 10.1 / 8.8)
//   59 M of 4096 to fp32            100 / 118 / 88      (110 / 125 / 61)
// Byte and scale loads in turn: up to 10 % longer from 17 M on down, the layer 148;
// all bytes ahead of all scales: the layer 152.  A tile per workgroup is nowhere
// ahead by more than the 1 % that runs differ by: no second form.
template <int DQ, bool kAligned>
__device__ __forceinline__ void unpack_piece(const uint8_t* src, uint8_t* cq, uint8_t* dq, const uint8_t* scales, int64_t rows,
                                             int64_t in_dim, int64_t tiles_c, int64_t t, int64_t tiles, int64_t lead, int tid) {
  constexpr int kElem = DQ == FSH_DT_F32 ? 4 : 2, kPasses = 8;
  const int64_t n = rows * in_dim;
  const bool scales_aligned = (reinterpret_cast<uintptr_t>(scales) & 3) == 0;  // (the same for the whole launch)
  const auto scale_at = [&](int64_t row, uint32_t col) {
    const uint8_t* p = scales + 4 * ((row >> 7) * tiles_c + (col >> 7));
    return scales_aligned ? *reinterpret_cast<const float*>(p) : load_f32_any(p);
  };
  lead = lead < n ? lead : n;
  const int64_t groups = (n - lead) / 8, per = (divide(groups + tiles - 1, tiles) + 15) / 16 * 16;
  const int64_t first = t * per, end = first + per < groups ? first + per : groups;  // per <= 2048: a tile has 16384 elements at most
  const int64_t idx0 = lead + 8 * first, row0 = divide(idx0, in_dim);
  const uint32_t width = static_cast<uint32_t>(in_dim), col0 = static_cast<uint32_t>(idx0 - row0 * in_dim);
  const bool splits = (width & 7) != 0 || (col0 & 7) != 0;  // groups that reach into the next tile or row
  const uint32_t count = first < end ? static_cast<uint32_t>(end - first) : 0;
  const uint8_t* run = src + idx0;
  uint8_t* run_cq = cq ? cq + idx0 : nullptr;
  uint8_t* run_dq = dq ? dq + idx0 * kElem : nullptr;
  u32x2 vin[kPasses];
  uint32_t cols[kPasses], belows[kPasses];
  float scale[kPasses];
  if (count > 0) {
    // (groups past the piece's end: its last one again)
    const auto group_of = [&](int k) { return min(static_cast<uint32_t>(k * kThreads + tid), count - 1); };
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int k = 4 * half; k < 4 * half + 4; ++k) vin[k] = load_group<u32x2, kAligned>(run + 8 * group_of(k));
      if (dq) {
#pragma unroll
        for (int k = 4 * half; k < 4 * half + 4; ++k) {
          const uint32_t c = col0 + 8 * group_of(k);
          belows[k] = c / width;
          cols[k] = c - belows[k] * width;
          scale[k] = scale_at(row0 + belows[k], cols[k]);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kPasses; ++k) {
    const uint32_t g = k * kThreads + tid;
    if (g >= count) break;
    if (cq) store_group<kAligned>(run_cq + 8 * g, vin[k]);
    if (!dq) continue;
    float f[8];
    if (!splits) {
      dequant4(vin[k].x, scale[k], f);
      dequant4(vin[k].y, scale[k], f + 4);
    } else {
      dequant4(vin[k].x, 1.0f, f);
      dequant4(vin[k].y, 1.0f, f + 4);
      // Of the group, `cut` elements belong to the first tile; what follows may
      // cross one more edge (a column block's, then the row's).
      const uint32_t in_row = width - cols[k], in_tile = 128 - (cols[k] & 127);
      const uint32_t cut = in_row < in_tile ? in_row : in_tile;
      float s1 = scale[k], s2 = scale[k];
      uint32_t cut2 = 8;
      if (cut < 8) {
        const int64_t row = row0 + belows[k];
        s1 = cut == in_row ? scale_at(row + 1, 0) : scale_at(row, cols[k] + cut);
        if (cut < in_row && in_row < 8) {
          cut2 = in_row;
          s2 = scale_at(row + 1, 0);
        }
      }
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) f[j] *= j < cut ? scale[k] : j < cut2 ? s1 : s2;
    }
    store_values8<DQ>(run_dq, 8 * g, f);
  }
  const int64_t edge = t == 0 && tid < lead ? tid : t == tiles - 1 && lead + 8 * groups + tid < n ? lead + 8 * groups + tid : -1;
  if (edge >= 0) {  // (fewer than 128 elements in front, than eight behind; a chunk of one piece has both ends)
    for (int64_t idx = edge; idx >= 0;) {
      const uint8_t b = src[idx];
      if (cq) cq[idx] = b;
      const int64_t row = idx / in_dim;
      if (dq) store_value<DQ>(dq, idx, __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(b), 0) * scale_at(row, static_cast<uint32_t>(idx - row * in_dim)));
      const int64_t last = lead + 8 * groups + tid;
      idx = idx < lead && t == tiles - 1 && last < n ? last : -1;
    }
  }
}

template <int DQ>  // FSH_DT_BF16, FSH_DT_F32 or FSH_DT_F16
__global__ __launch_bounds__(kThreads) void unpack_dequant_kernel(
    const uint8_t* __restrict__ rows, const fsh_unpack_chunk* __restrict__ chunks,
    const int64_t* __restrict__ tile_starts, int nchunks, uint8_t* __restrict__ compact,
    uint8_t* __restrict__ dequant, int block) {
  const int64_t bid = blockIdx.x;
  // Largest c with tile_starts[c] <= bid.  Up to 64 chunks are resolved in one
  // memory round trip (a lane per chunk and a ballot) instead of a dependent
  // chain of binary-search probes; tile_starts is ascending, so the count of
  // entries <= bid is the index plus one.
  int lo = 0;
  if (nchunks <= 64) {
    const int l = threadIdx.x & 63;
    const bool below = l < nchunks && tile_starts[l] <= bid;
    lo = __builtin_popcountll(__ballot(below)) - 1;
  } else {
    int hi = nchunks - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (tile_starts[mid] <= bid)
        lo = mid;
      else
        hi = mid - 1;
    }
  }
  const fsh_unpack_chunk ch = chunks[lo];
  const int64_t tiles_c = (ch.in_dim + block - 1) / block;
  const int64_t t = bid - tile_starts[lo];
  const int tid = threadIdx.x;
  constexpr int kElem = DQ == FSH_DT_F32 ? 4 : 2;

  const uint8_t* scales = rows + ch.src_scale_offset;
  const float scale = load_f32_any(scales + 4 * t);

  const uint8_t* src = rows + ch.src_qdata_offset;
  uint8_t* cq = compact ? compact + ch.dst_qdata_offset : nullptr;
  uint8_t* dq = dequant ? dequant + ch.dst_dequant_offset * kElem : nullptr;
  if (block == 128 && ch.in_dim >= 8 && ch.in_dim < (1LL << 31)) {
    // The pieces start `lead` elements in, where the wider output's memory lines do.
    const int64_t lead = dq ? (-reinterpret_cast<uintptr_t>(dq) & 255) / kElem : (-reinterpret_cast<uintptr_t>(cq) & 127);
    const bool on_lines = (cq == nullptr || ((reinterpret_cast<uintptr_t>(cq) + lead) & 127) == 0) &&
                          ((reinterpret_cast<uintptr_t>(src) + lead) & 7) == 0;
    const int64_t tiles = ((ch.rows + 127) / 128) * tiles_c;
    if (on_lines)
      unpack_piece<DQ, true>(src, cq, dq, scales, ch.rows, ch.in_dim, tiles_c, t, tiles, lead, tid);
    else
      unpack_piece<DQ, false>(src, cq, dq, scales, ch.rows, ch.in_dim, tiles_c, t, tiles, lead, tid);
    if (compact != nullptr && tid == 0) store_f32_any(compact + ch.dst_scale_offset + 4 * t, scale);
    return;
  }

  // Element-wise path.
  if (compact != nullptr && tid == 0) store_f32_any(compact + ch.dst_scale_offset + 4 * t, scale);
  const int64_t tr = t / tiles_c, tc = t - tr * tiles_c;
  const int64_t row0 = tr * block, col0 = tc * block;
  const int64_t nrows = (ch.rows - row0) < block ? (ch.rows - row0) : block;
  const int64_t ncols = (ch.in_dim - col0) < block ? (ch.in_dim - col0) : block;
  for (int64_t i = tid; i < nrows * ncols; i += kThreads) {
    const int64_t idx = (row0 + i / ncols) * ch.in_dim + col0 + i % ncols;
    const uint8_t b = src[idx];
    if (cq) cq[idx] = b;
    if (dq) {
      store_value<DQ>(dq, idx, __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(b), 0) * scale);
    }
  }
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_unpack_dequant(const void* rows_dev, const fsh_unpack_chunk* chunks_dev,
                               const int64_t* tile_starts_dev, int32_t nchunks, int64_t total_tiles,
                               void* compact_dev, void* dequant_dev, int32_t dequant_dtype,
                               int32_t block, void* stream) {
  using namespace fsh;
  if (nchunks < 0 || total_tiles < 0) return fail(FSH_EINVAL, "fsh_unpack_dequant: negative size");
  if (block <= 0) return fail(FSH_EINVAL, "fsh_unpack_dequant: block must be positive, got %d", block);
  if (nchunks == 0 || total_tiles == 0) return FSH_OK;
  if (!rows_dev || !chunks_dev || !tile_starts_dev) return fail(FSH_EINVAL, "fsh_unpack_dequant: null pointer");
  if (!compact_dev && !dequant_dev) return fail(FSH_EINVAL, "fsh_unpack_dequant: nothing to write");
  if (dequant_dtype != FSH_DT_BF16 && dequant_dtype != FSH_DT_F32 && dequant_dtype != FSH_DT_F16)
    return fail(FSH_EINVAL, "fsh_unpack_dequant: unsupported dequant dtype %d", dequant_dtype);
  if (dequant_dev && !aligned(dequant_dev, dequant_dtype == FSH_DT_F32 ? 4 : 2))
    return fail(FSH_EINVAL, "fsh_unpack_dequant: dequant buffer misaligned for its dtype");
  if (total_tiles > 0x7FFFFFFFLL)
    return fail(FSH_ENOTSUP, "fsh_unpack_dequant: %lld tiles exceed the grid limit", (long long)total_tiles);
  const dim3 g(static_cast<uint32_t>(total_tiles)), b(kThreads);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dequant_dtype == FSH_DT_BF16)
    hipLaunchKernelGGL((unpack_dequant_kernel<FSH_DT_BF16>), g, b, 0, s, static_cast<const uint8_t*>(rows_dev),
                       chunks_dev, tile_starts_dev, nchunks, static_cast<uint8_t*>(compact_dev),
                       static_cast<uint8_t*>(dequant_dev), block);
  else if (dequant_dtype == FSH_DT_F16)
    hipLaunchKernelGGL((unpack_dequant_kernel<FSH_DT_F16>), g, b, 0, s, static_cast<const uint8_t*>(rows_dev),
                       chunks_dev, tile_starts_dev, nchunks, static_cast<uint8_t*>(compact_dev),
                       static_cast<uint8_t*>(dequant_dev), block);
  else
    hipLaunchKernelGGL((unpack_dequant_kernel<FSH_DT_F32>), g, b, 0, s, static_cast<const uint8_t*>(rows_dev),
                       chunks_dev, tile_starts_dev, nchunks, static_cast<uint8_t*>(compact_dev),
                       static_cast<uint8_t*>(dequant_dev), block);
  return check_launch("fsh_unpack_dequant");
}
