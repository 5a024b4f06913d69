// Segment copy / zero / cast-pack over device descriptor tables.
//
// Each kernel takes the same three (or four) int64 device arrays the Triton
// kernels they replace take.  The grid is (segment, slice): a slice is
// kSliceBytes of one segment, copied by 256 threads with the widest vector the
// relative alignment of source and destination allows (16-byte in the common
// case, falling back to 8/4/2/1-byte units, so rank rows at odd byte offsets
// work too).
#include "common.hpp"

namespace fsh {
namespace {

constexpr int kThreads = 256;
constexpr int64_t kSliceBytes = 16384;  // 4 x 16 B per thread

__global__ __launch_bounds__(kThreads) void copy_segments_kernel(
    const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, const int64_t* __restrict__ src_offsets,
    const int64_t* __restrict__ numels, const int64_t* __restrict__ dst_offsets, int64_t slices_per_segment,
    int64_t unit) {
  const int64_t seg = blockIdx.x / slices_per_segment;
  const int64_t slice = blockIdx.x - seg * slices_per_segment;
  const int64_t nbytes = numels[seg] * unit;
  const int64_t begin = slice * kSliceBytes;
  if (begin >= nbytes) return;
  const int64_t len = (nbytes - begin) < kSliceBytes ? (nbytes - begin) : kSliceBytes;
  copy_bytes(src + src_offsets[seg] * unit + begin, dst + dst_offsets[seg] * unit + begin, len, threadIdx.x,
             kThreads);
}

// Segments of several separately allocated source rows, whose addresses come
// with the launch: the tables then depend on the layout alone, and new rows
// need neither an upload nor a table of their own.
struct RowPointers {
  const uint8_t* row[FSH_MAX_COPY_ROWS];
};
__global__ __launch_bounds__(kThreads) void copy_row_segments_kernel(const RowPointers rows, uint8_t* __restrict__ dst,
                                                                    const int64_t* __restrict__ table, int64_t nsegments,
                                                                    int64_t slices_per_segment) {
  const int64_t seg = blockIdx.x / slices_per_segment;
  const int64_t slice = blockIdx.x - seg * slices_per_segment;
  const int64_t nbytes = table[2 * nsegments + seg];
  const int64_t begin = slice * kSliceBytes;
  if (begin >= nbytes) return;
  const int64_t len = (nbytes - begin) < kSliceBytes ? (nbytes - begin) : kSliceBytes;
  copy_bytes(rows.row[table[seg]] + table[nsegments + seg] + begin, dst + table[3 * nsegments + seg] + begin, len,
             threadIdx.x, kThreads);
}

__global__ __launch_bounds__(kThreads) void zero_segments_kernel(uint8_t* __restrict__ dst,
                                                                const int64_t* __restrict__ numels,
                                                                const int64_t* __restrict__ dst_offsets,
                                                                int64_t slices_per_segment, int64_t unit) {
  const int64_t seg = blockIdx.x / slices_per_segment;
  const int64_t slice = blockIdx.x - seg * slices_per_segment;
  const int64_t nbytes = numels[seg] * unit;
  const int64_t begin = slice * kSliceBytes;
  if (begin >= nbytes) return;
  const int64_t len = (nbytes - begin) < kSliceBytes ? (nbytes - begin) : kSliceBytes;
  zero_bytes(dst + dst_offsets[seg] * unit + begin, len, threadIdx.x, kThreads);
}

// A casting slice: four accesses per thread, all requested before the first is
// stored, each contiguous across the wave with 16 bytes of fp32 per lane.
// Bound by memory and, with small slices, by the chain of table loads at a
// block's start: a layer's rank share (27 M elements) fp32 -> bf16 38 us with
// one access per thread, 28 with two, 27 with four or eight, against 34 with
// eight elements per thread in two 16-byte accesses 32 bytes apart; 12 M
// elements bf16 -> fp32 20.5 / 15.5 / 15.8 / 19.1 against 17.7 us.
constexpr int kCastUnroll = 4;
// Elements of one block.  A launch whose thread count would pass 32 bits takes
// larger slices.
template <typename SRC, typename DST>
constexpr int64_t kPackSliceElems = sizeof(SRC) == sizeof(DST) ? 2048 : kCastUnroll * 4 * kThreads;

template <typename SRC, typename DST>
__device__ __forceinline__ DST cast_elem(SRC v);
template <>
__device__ __forceinline__ float cast_elem<float, float>(float v) { return v; }
template <>
__device__ __forceinline__ uint16_t cast_elem<uint16_t, uint16_t>(uint16_t v) { return v; }
template <>
__device__ __forceinline__ float cast_elem<uint16_t, float>(uint16_t v) { return bf16_bits_to_f32(v); }
template <>
__device__ __forceinline__ uint16_t cast_elem<float, uint16_t>(float v) {
  return static_cast<uint16_t>(f32_to_bf16_bits(v));
}

// Four consecutive elements, 16 bytes of fp32 or 8 of bf16, as loaded and
// cast to the other type.
struct Bf16To32 {
  typedef u32x2 Raw;
  static __device__ __forceinline__ Raw load(const uint16_t* src) { return load_stream_u32x2(src); }
  static __device__ __forceinline__ void store(float* dst, const Raw v) {
    *reinterpret_cast<f32x4*>(dst) = f32x4{u32_as_f32(v.x << 16), u32_as_f32(v.x & 0xFFFF0000u), u32_as_f32(v.y << 16),
                                           u32_as_f32(v.y & 0xFFFF0000u)};
  }
};
struct F32ToBf16 {
  typedef f32x4 Raw;
  static __device__ __forceinline__ Raw load(const float* src) { return load_stream_f32x4(src); }
  static __device__ __forceinline__ void store(uint16_t* dst, const Raw v) {
    *reinterpret_cast<u32x2*>(dst) = u32x2{f32_to_bf16_bits(v.x) | (f32_to_bf16_bits(v.y) << 16),
                                           f32_to_bf16_bits(v.z) | (f32_to_bf16_bits(v.w) << 16)};
  }
};
__device__ __forceinline__ Bf16To32 caster(const uint16_t*, float*) { return {}; }
__device__ __forceinline__ F32ToBf16 caster(const float*, uint16_t*) { return {}; }

// Multi-input gather with cast.  A negative tensor index marks a zero-fill
// segment.  Same-dtype segments move as bytes with the widest legal vector;
// casting segments convert four elements per access where both sides allow it.
template <typename SRC, typename DST>
__global__ __launch_bounds__(kThreads) void pack_segments_kernel(
    const int64_t* __restrict__ input_ptrs, const int64_t* __restrict__ tensor_indices,
    const int64_t* __restrict__ src_offsets, const int64_t* __restrict__ numels,
    const int64_t* __restrict__ dst_offsets, DST* __restrict__ out, uint32_t slices_per_segment,
    int64_t slice_elems) {
  const uint32_t seg = blockIdx.x / slices_per_segment;
  const int64_t begin = static_cast<int64_t>(blockIdx.x - seg * slices_per_segment) * slice_elems;
  // (asked for together: what follows waits for them once)
  const int64_t n = numels[seg], ti = tensor_indices[seg], src_offset = src_offsets[seg], dst_offset = dst_offsets[seg];
  if (begin >= n) return;
  const int64_t len = (n - begin) < slice_elems ? (n - begin) : slice_elems;
  DST* dst = out + dst_offset + begin;
  if (ti < 0) {
    zero_bytes(reinterpret_cast<uint8_t*>(dst), len * static_cast<int64_t>(sizeof(DST)), threadIdx.x, kThreads);
    return;
  }
  const SRC* src = reinterpret_cast<const SRC*>(static_cast<uintptr_t>(input_ptrs[ti])) + src_offset + begin;
  if constexpr (sizeof(SRC) == sizeof(DST)) {
    copy_bytes(reinterpret_cast<const uint8_t*>(src), reinterpret_cast<uint8_t*>(dst),
               len * static_cast<int64_t>(sizeof(DST)), threadIdx.x, kThreads);
  } else {
    // Four elements per thread and access when the fp32 side starts on a
    // 16-byte boundary and the bf16 side on an 8-byte one; the rest, and
    // slices that do not, go element by element.
    typedef decltype(caster(src, dst)) Cast;
    constexpr int64_t kStep = 4 * kThreads;
    int64_t done = 0;
    if (reinterpret_cast<uintptr_t>(src) % (4 * sizeof(SRC)) == 0 && reinterpret_cast<uintptr_t>(dst) % (4 * sizeof(DST)) == 0) {
      const int64_t i = 4 * static_cast<int64_t>(threadIdx.x);
      for (; done + kCastUnroll * kStep <= len; done += kCastUnroll * kStep) {
        typename Cast::Raw raw[kCastUnroll];
#pragma unroll
        for (int u = 0; u < kCastUnroll; ++u) raw[u] = Cast::load(src + done + u * kStep + i);
#pragma unroll
        for (int u = 0; u < kCastUnroll; ++u) Cast::store(dst + done + u * kStep + i, raw[u]);
      }
      for (; done + kStep <= len; done += kStep) Cast::store(dst + done + i, Cast::load(src + done + i));
    }
    for (int64_t i = done + threadIdx.x; i < len; i += kThreads) dst[i] = cast_elem<SRC, DST>(src[i]);
  }
}

int check_unit(const char* who, int32_t unit) {
  if (unit != 1 && unit != 2 && unit != 4 && unit != 8 && unit != 16)
    return fail(FSH_EINVAL, "%s: unit_nbytes must be 1, 2, 4, 8 or 16, got %d", who, unit);
  return FSH_OK;
}

}  // namespace
}  // namespace fsh

FSH_API int fsh_copy_segments(const void* src_dev, void* dst_dev, const int64_t* src_offsets_dev,
                              const int64_t* numels_dev, const int64_t* dst_offsets_dev,
                              int64_t nsegments, int64_t max_segment_numel, int32_t unit_nbytes,
                              void* stream) {
  using namespace fsh;
  if (int rc = check_unit("fsh_copy_segments", unit_nbytes)) return rc;
  if (nsegments < 0 || max_segment_numel < 0) return fail(FSH_EINVAL, "fsh_copy_segments: negative size");
  if (nsegments == 0 || max_segment_numel == 0) return FSH_OK;
  if (!src_dev || !dst_dev || !src_offsets_dev || !numels_dev || !dst_offsets_dev)
    return fail(FSH_EINVAL, "fsh_copy_segments: null pointer");
  if (!aligned(src_dev, unit_nbytes) || !aligned(dst_dev, unit_nbytes))
    return fail(FSH_EINVAL, "fsh_copy_segments: base pointers must be aligned to unit_nbytes=%d", unit_nbytes);
  const int64_t slices = ceil_div(max_segment_numel * unit_nbytes, kSliceBytes);
  const int64_t grid = nsegments * slices;
  if (grid > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "fsh_copy_segments: %lld workgroups exceed the grid limit", (long long)grid);
  hipLaunchKernelGGL(copy_segments_kernel, dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(src_dev),
                     static_cast<uint8_t*>(dst_dev), src_offsets_dev, numels_dev, dst_offsets_dev, slices,
                     static_cast<int64_t>(unit_nbytes));
  return check_launch("fsh_copy_segments");
}

FSH_API int fsh_copy_row_segments(const void* const* rows, int32_t nrows, void* dst_dev, const int64_t* table_dev,
                                  int64_t nsegments, int64_t max_segment_nbytes, void* stream) {
  using namespace fsh;
  if (nsegments < 0 || max_segment_nbytes < 0 || nrows < 0) return fail(FSH_EINVAL, "fsh_copy_row_segments: negative size");
  if (nsegments == 0 || max_segment_nbytes == 0) return FSH_OK;
  if (nrows == 0 || nrows > FSH_MAX_COPY_ROWS)
    return fail(FSH_EINVAL, "fsh_copy_row_segments: %d rows, not 1 to %d", nrows, FSH_MAX_COPY_ROWS);
  if (!rows || !dst_dev || !table_dev) return fail(FSH_EINVAL, "fsh_copy_row_segments: null pointer");
  RowPointers p;
  for (int i = 0; i < FSH_MAX_COPY_ROWS; ++i) {
    p.row[i] = static_cast<const uint8_t*>(rows[i < nrows ? i : nrows - 1]);
    if (!p.row[i]) return fail(FSH_EINVAL, "fsh_copy_row_segments: row %d is null", i);
  }
  const int64_t slices = ceil_div(max_segment_nbytes, kSliceBytes);
  const int64_t grid = nsegments * slices;
  if (grid > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "fsh_copy_row_segments: %lld workgroups exceed the grid limit", (long long)grid);
  hipLaunchKernelGGL(copy_row_segments_kernel, dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), p, static_cast<uint8_t*>(dst_dev), table_dev, nsegments, slices);
  return check_launch("fsh_copy_row_segments");
}

FSH_API int fsh_zero_segments(void* dst_dev, const int64_t* numels_dev, const int64_t* dst_offsets_dev,
                              int64_t nsegments, int64_t max_segment_numel, int32_t unit_nbytes,
                              void* stream) {
  using namespace fsh;
  if (int rc = check_unit("fsh_zero_segments", unit_nbytes)) return rc;
  if (nsegments < 0 || max_segment_numel < 0) return fail(FSH_EINVAL, "fsh_zero_segments: negative size");
  if (nsegments == 0 || max_segment_numel == 0) return FSH_OK;
  if (!dst_dev || !numels_dev || !dst_offsets_dev) return fail(FSH_EINVAL, "fsh_zero_segments: null pointer");
  if (!aligned(dst_dev, unit_nbytes))
    return fail(FSH_EINVAL, "fsh_zero_segments: base pointer must be aligned to unit_nbytes=%d", unit_nbytes);
  const int64_t slices = ceil_div(max_segment_numel * unit_nbytes, kSliceBytes);
  const int64_t grid = nsegments * slices;
  if (grid > 0x7FFFFFFFLL) return fail(FSH_ENOTSUP, "fsh_zero_segments: %lld workgroups exceed the grid limit", (long long)grid);
  hipLaunchKernelGGL(zero_segments_kernel, dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<uint8_t*>(dst_dev), numels_dev,
                     dst_offsets_dev, slices, static_cast<int64_t>(unit_nbytes));
  return check_launch("fsh_zero_segments");
}

FSH_API int fsh_pack_segments(const int64_t* input_ptrs_dev, const int64_t* tensor_indices_dev,
                              const int64_t* src_offsets_dev, const int64_t* numels_dev,
                              const int64_t* dst_offsets_dev, int64_t nsegments,
                              int64_t max_segment_numel, int32_t src_dtype, int32_t dst_dtype,
                              void* dst_dev, void* stream) {
  using namespace fsh;
  if (nsegments < 0 || max_segment_numel < 0) return fail(FSH_EINVAL, "fsh_pack_segments: negative size");
  if (nsegments == 0 || max_segment_numel == 0) return FSH_OK;
  if (!input_ptrs_dev || !tensor_indices_dev || !src_offsets_dev || !numels_dev || !dst_offsets_dev || !dst_dev)
    return fail(FSH_EINVAL, "fsh_pack_segments: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto launch = [&](auto src_tag, auto dst_tag) -> int {
    using SRC = decltype(src_tag);
    using DST = decltype(dst_tag);
    int64_t elems = kPackSliceElems<SRC, DST>;
    while (nsegments * ceil_div(max_segment_numel, elems) >= (1 << 24) && elems < max_segment_numel) elems *= 2;
    const int64_t slices = ceil_div(max_segment_numel, elems), grid = nsegments * slices;
    if (grid > 0x7FFFFFFFLL)
      return fail(FSH_ENOTSUP, "fsh_pack_segments: %lld workgroups exceed the grid limit", (long long)grid);
    hipLaunchKernelGGL((pack_segments_kernel<SRC, DST>), dim3(static_cast<uint32_t>(grid)), dim3(kThreads), 0, s, input_ptrs_dev,
                       tensor_indices_dev, src_offsets_dev, numels_dev, dst_offsets_dev, static_cast<DST*>(dst_dev),
                       static_cast<uint32_t>(slices), elems);
    return check_launch("fsh_pack_segments");
  };
  if (src_dtype == FSH_DT_F32 && dst_dtype == FSH_DT_BF16) return launch(float{}, uint16_t{});
  if (src_dtype == FSH_DT_BF16 && dst_dtype == FSH_DT_F32) return launch(uint16_t{}, float{});
  if (src_dtype == FSH_DT_F32 && dst_dtype == FSH_DT_F32) return launch(float{}, float{});
  if (src_dtype == FSH_DT_BF16 && dst_dtype == FSH_DT_BF16) return launch(uint16_t{}, uint16_t{});
  return fail(FSH_EINVAL, "fsh_pack_segments: unsupported dtype pair (%d -> %d)", src_dtype, dst_dtype);
}
