// Elementwise launches around the Newton-Schulz products, one launch for all
// shape groups of a call: momentum + sums of squares, sums of squares alone,
// Frobenius normalization, update.
//
// All are HBM-bound streams.  A launch of its own per group left the chip
// idle between and inside them: 64 blocks for one 14336 x 4096 fp32 matrix
// took 477 us (2.2 TB/s), and the three launches for each of four groups of
// small matrices 8-16 us each.  The blocks of all groups now share a launch,
// a block owns 8192 elements (four 16-byte vectors per thread, all requested
// before the first is used), and a matrix gets as many blocks as it has such
// slices.
#pragma once
#include "mfma_tiles.hpp"
#include "muon_elementwise.hpp"

namespace fsh {
namespace {

constexpr int kNormThreads = 256;
constexpr int kMaxMuonGroups = FSH_MAX_NS_PROBLEMS;
constexpr int64_t kSliceVectors = 1024;  // 8-element vectors per block and slice
constexpr int64_t kMaxSlices = 2048;     // per matrix: one block adds up all partial sums (see kNormSlices)

// Slices (and partial sums of squares) of a matrix of `vectors` 8-element
// vectors; a matter of the matrix alone, so that the order of the additions is
// the same in every launch it takes part in.
inline int64_t slices_of(int64_t vectors) {
  const int64_t n = ceil_div(vectors, kSliceVectors);
  return n < 1 ? 1 : (n > kMaxSlices ? kMaxSlices : n);
}

// s plus the squares of the eight bf16 values of v, added one after the
// other in element order.
__device__ __forceinline__ float add_squares8(float s, const u32x4 v) {
  const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float lo = u32_as_f32(d[j] << 16), hi = u32_as_f32(d[j] & 0xFFFF0000u);
    s += lo * lo;
    s += hi * hi;
  }
  return s;
}
// The workgroup's total in a fixed order: lanes by the wave reduction, then
// the four waves as (0 + 1) + (2 + 3).  All threads call it and get it.
__device__ __forceinline__ float block_sum(float s, float* lds) {
  s = wave_sum_f32(s);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
  __syncthreads();
  return (lds[0] + lds[1]) + (lds[2] + lds[3]);
}

// A group's matrices: separate allocations (address tables) and their slots in
// the contiguous batch buffer, [rows, cols] rounded up to multiples of 8.
struct MuonGroupDev {
  const int64_t* param_ptrs;     // device tables [batch]
  const int64_t* momentum_ptrs;
  const int64_t* grad_ptrs;
  uint16_t* batch;               // [batch, vectors * 8]
  float* partial;                // [batch, slices]
  int64_t vectors;               // 8-element vectors of a (padded) matrix
  int64_t rows, cols;            // of the separate matrices
  int64_t row_vectors;           // vectors per padded row
  int32_t slices;                // blocks per matrix
  int32_t first_block;           // INT32_MAX past the last group
  int32_t f32;                   // masters are fp32
  int32_t padded;                // rows or cols are not multiples of 8
  float neg_lr, dir_scale;
};
struct MuonLaunch {
  MuonGroupDev group[kMaxMuonGroups];
  float one_minus_mu, mu, decay;
  int32_t nesterov;
};

template <typename Launch>
__device__ __forceinline__ int group_of_block(const Launch& launch) {
  int w = 0;
#pragma unroll
  for (int i = 1; i < kMaxMuonGroups; ++i) w += static_cast<int>(blockIdx.x) >= launch.group[i].first_block ? 1 : 0;
  return uniform_i32(w);
}

// Eight elements of a separately allocated matrix as floats and back: the
// whole vector g of a matrix whose rows are whole vectors, or the part of it
// inside an odd matrix (zero outside).  A vector that lies inside an odd matrix
// as a whole is accessed as one, unaligned, which global memory instructions
// may be; only a row's last, partial one goes element by element (31 M elements
// 5576 x 5573: momentum 146 us element by element, 80 here; update 95 / 53).
template <bool kF32, bool kPadded>
struct MasterVector {
  const MuonGroupDev& q;
  __device__ __forceinline__ void locate(int64_t g, int64_t* at, int* n) const {
    // (a 64-bit division takes longer than the rest of a vector's work)
    const int64_t row = q.vectors <= UINT32_MAX ? static_cast<uint32_t>(g) / static_cast<uint32_t>(q.row_vectors) : g / q.row_vectors;
    const int64_t col = (g - row * q.row_vectors) * 8;
    *at = row * q.cols + col;
    const int64_t left = row < q.rows ? q.cols - col : 0;
    *n = static_cast<int>(left < 0 ? 0 : (left > 8 ? 8 : left));
  }
  __device__ __forceinline__ void load(const void* base, int64_t g, float (&f)[8]) const {
    if (!kPadded) {
      if (kF32) load8_f32(static_cast<const float*>(base) + g * 8, f);
      else unpack8(load_stream_u32x4(static_cast<const uint16_t*>(base) + g * 8), f);
      return;
    }
    int64_t at;
    int n;
    locate(g, &at, &n);
    if (n == 8) {
      if (kF32) {
        __builtin_memcpy(f, static_cast<const float*>(base) + at, sizeof(f));
      } else {
        u32x4 v;
        __builtin_memcpy(&v, static_cast<const uint16_t*>(base) + at, sizeof(v));
        unpack8(v, f);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      f[j] = j >= n ? 0.0f : kF32 ? static_cast<const float*>(base)[at + j] : bf16_bits_to_f32(static_cast<const uint16_t*>(base)[at + j]);
  }
  // `bits`: the bf16 bits of a bf16 master (f unused), f: the values of an fp32 one
  __device__ __forceinline__ void store(void* base, int64_t g, const float (&f)[8], const uint32_t (&bits)[8]) const {
    if (!kPadded) {
      if (kF32) store8_f32(static_cast<float*>(base) + g * 8, f);
      else store_stream_u32x4(static_cast<uint16_t*>(base) + g * 8, pack8(bits));
      return;
    }
    int64_t at;
    int n;
    locate(g, &at, &n);
    if (n == 8) {
      if (kF32) {
        __builtin_memcpy(static_cast<float*>(base) + at, f, sizeof(f));
      } else {
        const u32x4 v = pack8(bits);
        __builtin_memcpy(static_cast<uint16_t*>(base) + at, &v, sizeof(v));
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < n) {
        if (kF32) static_cast<float*>(base)[at + j] = f[j];
        else static_cast<uint16_t*>(base)[at + j] = static_cast<uint16_t>(bits[j]);
      }
  }
};

// The momentum step of one slice, fused with the sum of squares of its output:
//   m = lerp(m, g, 1 - mu);  u = nesterov ? lerp(g, m, mu) : m
// (each rounded to the master's dtype; u rounded to bf16 into the batch
// buffer).  The squares are added vector by vector in walk order, as
// sumsq_groups_kernel adds them.
template <bool kF32, bool kPadded>
__device__ __forceinline__ float muon_prepare_slice(const MuonLaunch& launch, const MuonGroupDev& q, int64_t matrix,
                                                    int64_t begin, int64_t end) {
  void* mom = reinterpret_cast<void*>(uniform_i64(q.momentum_ptrs[matrix]));
  const void* grad = reinterpret_cast<const void*>(uniform_i64(q.grad_ptrs[matrix]));
  uint16_t* out = q.batch + matrix * q.vectors * 8;
  const MasterVector<kF32, kPadded> master{q};
  constexpr int kUnroll = kF32 || kPadded ? 2 : 4;  // (four odd vectors would cost the whole launch occupancy)
  float s = 0.0f;
  if constexpr (kF32 && !kPadded) {
    // fp32 accesses contiguous across the wave: lane l takes the four-element
    // chunks l and 64 + l of its 64 vectors.  (Vector by vector, a lane's two
    // 16-byte accesses lie 32 bytes apart and each asks for half of every line:
    // 101 M elements 281 us that way, 269 here, 253 with streaming stores.)  The rounded results then
    // change lanes, so that lane l has vector l: the sums of squares keep their
    // order.
    const int lane = threadIdx.x & 63;
    const int64_t chunks = 2 * end;
    float* moms = static_cast<float*>(mom);
    const float* grads = static_cast<const float*>(grad);
    for (int64_t w0 = begin + threadIdx.x - lane; w0 < end; w0 += kUnroll * kNormThreads) {  // (the same in the whole wave)
      f32x4 mv[kUnroll][2], gv[kUnroll][2];
#pragma unroll
      for (int k = 0; k < kUnroll; ++k)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int64_t c = 2 * (w0 + k * kNormThreads) + 64 * h + lane;
          mv[k][h] = gv[k][h] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (c < chunks) {
            mv[k][h] = load_stream_f32x4(moms + c * 4);
            gv[k][h] = load_stream_f32x4(grads + c * 4);
          }
        }
#pragma unroll
      for (int k = 0; k < kUnroll; ++k) {
        u32x2 words[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int64_t c = 2 * (w0 + k * kNormThreads) + 64 * h + lane;
          uint32_t ob[4];
          float mo[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            muon_prepare_one_f32(mv[k][h][j], gv[k][h][j], launch.one_minus_mu, launch.mu, launch.nesterov, &mo[j], &ob[j]);
          words[h] = u32x2{ob[0] | (ob[1] << 16), ob[2] | (ob[3] << 16)};
          if (c < chunks) __builtin_nontemporal_store(f32x4{mo[0], mo[1], mo[2], mo[3]}, reinterpret_cast<f32x4*>(moms + c * 4));
        }
        u32x4 u;
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int from = ((2 * lane + part) & 63) * 4;
            const int first = __builtin_amdgcn_ds_bpermute(from, static_cast<int>(words[0][j]));
            const int second = __builtin_amdgcn_ds_bpermute(from, static_cast<int>(words[1][j]));
            u[2 * part + j] = static_cast<uint32_t>(lane < 32 ? first : second);
          }
        const int64_t g = w0 + k * kNormThreads + lane;
        if (g < end) {
          store_stream_u32x4(out + g * 8, u);
          s = add_squares8(s, u);
        }
      }
    }
    return s;
  }
  for (int64_t g0 = begin + threadIdx.x; g0 < end; g0 += kUnroll * kNormThreads) {
    float mv[kUnroll][8], gv[kUnroll][8];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const int64_t g = g0 + k * kNormThreads;
      if (g < end) {
        master.load(mom, g, mv[k]);
        master.load(grad, g, gv[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const int64_t g = g0 + k * kNormThreads;
      if (g < end) {
        uint32_t mb[8], ob[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (kF32)
            muon_prepare_one_f32(mv[k][j], gv[k][j], launch.one_minus_mu, launch.mu, launch.nesterov, &mv[k][j], &ob[j]);
          else
            muon_prepare_one(mv[k][j], gv[k][j], launch.one_minus_mu, launch.mu, launch.nesterov, &mb[j], &ob[j]);
        }
        master.store(mom, g, mv[k], mb);
        const u32x4 u = pack8(ob);
        store_stream_u32x4(out + g * 8, u);
        s = add_squares8(s, u);
      }
    }
  }
  return s;
}

__global__ __launch_bounds__(kNormThreads) void muon_prepare_groups_kernel(const MuonLaunch launch) {
  __shared__ float lds[kNormThreads / 64];
  const MuonGroupDev& q = launch.group[group_of_block(launch)];
  const int64_t block = static_cast<int64_t>(blockIdx.x) - q.first_block;
  const int64_t matrix = block / q.slices, slice = block - matrix * q.slices;
  const int64_t per = ceil_div(q.vectors, static_cast<int64_t>(q.slices));
  const int64_t begin = slice * per, end = begin + per < q.vectors ? begin + per : q.vectors;
  float s;
  if (q.padded)
    s = q.f32 ? muon_prepare_slice<true, true>(launch, q, matrix, begin, end)
              : muon_prepare_slice<false, true>(launch, q, matrix, begin, end);
  else
    s = q.f32 ? muon_prepare_slice<true, false>(launch, q, matrix, begin, end)
              : muon_prepare_slice<false, false>(launch, q, matrix, begin, end);
  s = block_sum(s, lds);
  if (threadIdx.x == 0) q.partial[block] = s;
}

// partial[b][j] = sum of squares of slice j of matrix b of the batch buffers, in fp32.
__global__ __launch_bounds__(kNormThreads) void sumsq_groups_kernel(const MuonLaunch launch) {
  __shared__ float lds[kNormThreads / 64];
  const MuonGroupDev& q = launch.group[group_of_block(launch)];
  const int64_t block = static_cast<int64_t>(blockIdx.x) - q.first_block;
  const int64_t matrix = block / q.slices, slice = block - matrix * q.slices;
  const int64_t per = ceil_div(q.vectors, static_cast<int64_t>(q.slices));
  const int64_t begin = slice * per, end = begin + per < q.vectors ? begin + per : q.vectors;
  const uint16_t* m = q.batch + matrix * q.vectors * 8;
  constexpr int kUnroll = 4;
  float s = 0.0f;
  for (int64_t g0 = begin + threadIdx.x; g0 < end; g0 += kUnroll * kNormThreads) {
    u32x4 v[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
      if (g0 + k * kNormThreads < end) v[k] = load_stream_u32x4(m + (g0 + k * kNormThreads) * 8);
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
      if (g0 + k * kNormThreads < end) s = add_squares8(s, v[k]);
  }
  s = block_sum(s, lds);
  if (threadIdx.x == 0) q.partial[block] = s;
}

// The update: parameter b takes the direction in slot b of the batch buffer,
//   p = p * decay;  p = p + neg_lr * d   (d first scaled if the scale is not 1)
// with a rounding to bf16 after each step on bf16 masters, in fp32 on fp32 ones.
template <bool kF32, bool kPadded>
__device__ __forceinline__ void muon_apply_slice(const MuonLaunch& launch, const MuonGroupDev& q, int64_t matrix,
                                                 int64_t begin, int64_t end) {
  void* param = reinterpret_cast<void*>(uniform_i64(q.param_ptrs[matrix]));
  const uint16_t* dir = q.batch + matrix * q.vectors * 8;
  const MasterVector<kF32, kPadded> master{q};
  constexpr int kUnroll = kF32 || kPadded ? 2 : 4;  // (four odd vectors would cost the whole launch occupancy)
  if (kF32 && !kPadded) {
    // Every element is on its own, so fp32 masters go in chunks of four: one
    // 16-byte access contiguous across the wave.  Eight per lane are two of
    // them 32 bytes apart, each asking for half of every line (101 M
    // parameters: 178 us that way, 158 us here, 6.4 TB/s).
    constexpr int kChunks = 4;
    float* out = static_cast<float*>(param);
    for (int64_t c0 = 2 * begin + threadIdx.x; c0 < 2 * end; c0 += kChunks * kNormThreads) {
      f32x4 p[kChunks];
      u32x2 d[kChunks];
#pragma unroll
      for (int k = 0; k < kChunks; ++k)
        if (c0 + k * kNormThreads < 2 * end) {
          p[k] = load_stream_f32x4(out + (c0 + k * kNormThreads) * 4);
          d[k] = load_stream_u32x2(dir + (c0 + k * kNormThreads) * 4);
        }
#pragma unroll
      for (int k = 0; k < kChunks; ++k)
        if (c0 + k * kNormThreads < 2 * end) {
          const auto apply = [&](float value, uint32_t bits) {
            return muon_apply_one_f32(value, u32_as_f32(bits), launch.decay, q.neg_lr, q.dir_scale);
          };
          *reinterpret_cast<f32x4*>(out + (c0 + k * kNormThreads) * 4) =
              f32x4{apply(p[k].x, d[k].x << 16), apply(p[k].y, d[k].x & 0xFFFF0000u), apply(p[k].z, d[k].y << 16),
                    apply(p[k].w, d[k].y & 0xFFFF0000u)};
        }
    }
    return;
  }
  for (int64_t g0 = begin + threadIdx.x; g0 < end; g0 += kUnroll * kNormThreads) {
    float pv[kUnroll][8];
    u32x4 draw[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const int64_t g = g0 + k * kNormThreads;
      if (g < end) {
        master.load(param, g, pv[k]);
        draw[k] = load_stream_u32x4(dir + g * 8);
      }
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const int64_t g = g0 + k * kNormThreads;
      if (g < end) {
        float dv[8];
        uint32_t pb[8];
        unpack8(draw[k], dv);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (kF32)
            pv[k][j] = muon_apply_one_f32(pv[k][j], dv[j], launch.decay, q.neg_lr, q.dir_scale);
          else
            pb[j] = muon_apply_one(pv[k][j], dv[j], launch.decay, q.neg_lr, q.dir_scale);
        }
        master.store(param, g, pv[k], pb);
      }
    }
  }
}

__global__ __launch_bounds__(kNormThreads) void muon_apply_groups_kernel(const MuonLaunch launch) {
  const MuonGroupDev& q = launch.group[group_of_block(launch)];
  const int64_t block = static_cast<int64_t>(blockIdx.x) - q.first_block;
  const int64_t matrix = block / q.slices, slice = block - matrix * q.slices;
  const int64_t per = ceil_div(q.vectors, static_cast<int64_t>(q.slices));
  const int64_t begin = slice * per, end = begin + per < q.vectors ? begin + per : q.vectors;
  if (q.padded) {
    if (q.f32) muon_apply_slice<true, true>(launch, q, matrix, begin, end);
    else muon_apply_slice<false, true>(launch, q, matrix, begin, end);
  } else {
    if (q.f32) muon_apply_slice<true, false>(launch, q, matrix, begin, end);
    else muon_apply_slice<false, false>(launch, q, matrix, begin, end);
  }
}

// A matrix's norm from its partial sums: bf16(sqrt(sum)) floored at eps.
__device__ __forceinline__ float norm_of_partials(const float* partial, int slices, float eps, float* lds) {
  float total = 0.0f;
  for (int j = threadIdx.x; j < slices; j += kNormThreads) total += partial[j];
  total = block_sum(total, lds);
  const float norm = bf16_bits_to_f32(f32_to_bf16_bits(sqrtf(total)));
  return norm < eps ? eps : norm;
}

// The partials of a 7168 x 2048 matrix (7 KB) are as much to read as a block
// of the normalization has data, ahead of its first store: from more than
// kNormSlices slices on a launch of its own adds them up and leaves the norm in
// place of the matrix's first partial (48 such and square matrices: 468 us in
// one launch, 5 + 292 us in two with the cheaper division below).
// Fewer are added up by every block, which costs less than the 5 us launch (20
// matrices of at most 288 slices: 33.5 us in one launch, 4.8 + 30.5 in two).
constexpr int kNormSlices = 512;
constexpr int kNormTile = 64;
constexpr int kNormPitch = kNormTile + 2;  // u16 per LDS row
struct NormalizeGroup {
  const uint16_t* in;
  uint16_t* out_same;
  uint16_t* out_t;
  float* partial;        // [batch, slices]
  int64_t rows, cols;
  int32_t tiles, tiles_c;  // blocks per matrix; 64 x 64 tiles per row of tiles (transposing groups)
  int32_t slices;
  int32_t first_block;   // INT32_MAX past the last group
  int32_t first_matrix;  // of all groups of the launch
};
struct NormalizeLaunch {
  NormalizeGroup group[kMaxMuonGroups];
  float eps_bf16;
  int32_t norms_ready;  // norm_groups_kernel ran
};
__global__ __launch_bounds__(kNormThreads) void norm_groups_kernel(const NormalizeLaunch launch) {
  __shared__ float lds[kNormThreads / 64];
  int w = 0;
#pragma unroll
  for (int i = 1; i < kMaxMuonGroups; ++i) w += static_cast<int>(blockIdx.x) >= launch.group[i].first_matrix ? 1 : 0;
  const NormalizeGroup& p = launch.group[uniform_i32(w)];
  float* partial = p.partial + (static_cast<int64_t>(blockIdx.x) - p.first_matrix) * p.slices;
  const float norm = norm_of_partials(partial, p.slices, launch.eps_bf16, lds);  // all are read behind its barrier
  if (threadIdx.x == 0) partial[0] = norm;
}

// bf16(x / norm), the bits of the correctly rounded fp32 quotient rounded to
// bf16, for eight bf16 values: x times the reciprocal with one residual
// correction (Markstein).  Eight IEEE divisions and software roundings per
// vector (22 operations a value) had the vector ALU as busy as the memory.  x
// and norm have eight significant bits, so a quotient that is not a tie of the
// bf16 rounding is 2^-17 away from one, and a tie is met exactly; 2^64 keeps
// the residuals of small x out of the subnormals.  The residual of a negative
// zero is a positive one: the sign of x, which is the quotient's, is put back.
// Norms outside [2^-60, 2^60], where the scaled values could leave the range,
// and infinite or NaN ones divide.
struct Normalizer {
  float norm, recip;
  bool divide;  // the same for the whole workgroup
  __device__ __forceinline__ explicit Normalizer(float norm_of_matrix) {
    norm = u32_as_f32(static_cast<uint32_t>(uniform_i32(static_cast<int>(f32_as_u32(norm_of_matrix)))));
    divide = !(norm >= 0x1p-60f && norm <= 0x1p60f);
    recip = 1.0f / norm;
  }
  __device__ __forceinline__ float quotient(float x) const {
    const float scaled = x * 0x1p64f, q = scaled * recip;
    return __builtin_fmaf(__builtin_fmaf(-q, norm, scaled), recip, q) * 0x1p-64f;
  }
  __device__ __forceinline__ u32x4 operator()(const u32x4& v) const {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    uint32_t out[4];
    if (divide) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        out[j] = f32_to_bf16_bits(u32_as_f32(d[j] << 16) / norm) | (f32_to_bf16_bits(u32_as_f32(d[j] & 0xFFFF0000u) / norm) << 16);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        out[j] = pack_bf16x2(quotient(u32_as_f32(d[j] << 16)), quotient(u32_as_f32(d[j] & 0xFFFF0000u))) | (d[j] & 0x80008000u);
    }
    return u32x4{out[0], out[1], out[2], out[3]};
  }
};

// Divides matrix b of `in` ([rows, cols]) by its norm as bf16 tensor ops would
// (fp32 division, bf16 result) and writes it to `out_same` ([rows, cols]) and
// `out_t` ([cols, rows]); either may be null.  Bound by memory.
// Without a transposed output a block takes 1024 consecutive 8-element vectors,
// four per thread, requested together.  With one it owns a 64 x 64 tile:
// 16-byte loads and stores of 8 elements along the rows, and the tile goes
// through LDS and leaves as 16-byte stores of 8 elements along the columns.
// rows and cols are multiples of 8, so an 8-element group is whole or absent.
__global__ __launch_bounds__(kNormThreads) void normalize_groups_kernel(const NormalizeLaunch launch) {
  __shared__ uint16_t tile[kNormTile * kNormPitch];
  __shared__ float lds[kNormThreads / 64];
  const NormalizeGroup& p = launch.group[group_of_block(launch)];
  const int64_t rows = p.rows, cols = p.cols;
  const uint32_t block = blockIdx.x - static_cast<uint32_t>(p.first_block);
  const uint32_t b = block / static_cast<uint32_t>(p.tiles), t = block - b * static_cast<uint32_t>(p.tiles);
  const uint16_t* m = p.in + b * rows * cols;
  const float* partial = p.partial + static_cast<int64_t>(b) * p.slices;
  const auto norm_of_matrix = [&]() {
    return launch.norms_ready ? *partial : norm_of_partials(partial, p.slices, launch.eps_bf16, lds);
  };
  uint16_t* o = p.out_same ? p.out_same + b * rows * cols : nullptr;
  if (p.out_t == nullptr) {  // the same for the whole workgroup
    const int64_t vectors = rows * cols / 8, g0 = t * kSliceVectors + threadIdx.x;
    constexpr int kUnroll = static_cast<int>(kSliceVectors / kNormThreads);
    u32x4 v[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
      if (g0 + k * kNormThreads < vectors) v[k] = load_stream_u32x4(m + (g0 + k * kNormThreads) * 8);
    const Normalizer normalized(norm_of_matrix());
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
      if (g0 + k * kNormThreads < vectors) store_stream_u32x4(o + (g0 + k * kNormThreads) * 8, normalized(v[k]));
    return;
  }
  const uint32_t tile_r = t / static_cast<uint32_t>(p.tiles_c), tile_c = t - tile_r * static_cast<uint32_t>(p.tiles_c);
  const int64_t r0 = static_cast<int64_t>(tile_r) * kNormTile, c0 = static_cast<int64_t>(tile_c) * kNormTile;
  const int q = threadIdx.x & 7, line = threadIdx.x >> 3;  // 8 groups of 8 elements per line, 32 lines per pass
  u32x4 v[2];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int64_t r = r0 + line + 32 * pass, c = c0 + 8 * q;
    if (r < rows && c < cols) v[pass] = load_stream_u32x4(m + r * cols + c);
  }
  const Normalizer normalized(norm_of_matrix());
  uint16_t* ot = p.out_t + b * rows * cols;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int lr = line + 32 * pass;
    const int64_t r = r0 + lr, c = c0 + 8 * q;
    if (r < rows && c < cols) {
      const u32x4 n = normalized(v[pass]);
      if (o != nullptr) store_stream_u32x4(o + r * cols + c, n);
      const uint32_t d[4] = {n.x, n.y, n.z, n.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(&tile[lr * kNormPitch + 8 * q + 2 * j]) = d[j];
    }
  }
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int lc = line + 32 * pass;  // tile column = row of the transposed output
    const int64_t c = c0 + lc, r = r0 + 8 * q;
    if (c < cols && r < rows) {
      uint32_t bits[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) bits[j] = tile[(8 * q + j) * kNormPitch + lc];
      store_stream_u32x4(ot + c * rows + r, pack8(bits));
    }
  }
}

}  // namespace
}  // namespace fsh
