// fp32 products of the GatedDelta kernels on the fp32 matrix instructions, over matrices
// held in LDS as rows of odd stride, and the unit lower triangular inverse of a chunk.
#pragma once

#include "common.h"

namespace motif {

__device__ __forceinline__ f32x16 mfma32_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Row of accumulator register r of a 32x32 tile for lane half h: 8 (r / 4) + 4 h + r % 4.
__device__ __forceinline__ int acc_row32(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// NP products over STEPS k-steps of two in one loop, operands from LDS: op(p, s, a, b) reads
// product p's operands of step s for this lane.  The operands of a block of steps are read while
// the block before it runs on the matrix cores (the scheduling barriers keep them there: left to
// itself the compiler reads each operand right in front of its use, and with the one or two waves
// per SIMD that the LDS planes leave, every step then waits out an LDS round trip).
template <int STEPS, int NP, typename OP>
__device__ __forceinline__ void mm_pipe(f32x16 (&acc)[NP], OP op) {
  constexpr int U = NP == 1 ? 4 : 2;  // steps per block: at most 15 reads in flight
  static_assert(STEPS % U == 0, "whole blocks");
  float a[2][U][NP], b[2][U][NP];
  auto read = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int p = 0; p < NP; ++p) op(p, s0 + u, a[buf][u][p], b[buf][u][p]);
  };
  read(0, 0);
#pragma unroll
  for (int blk = 0; blk < STEPS / U; ++blk) {
    if (blk + 1 < STEPS / U) read((blk + 1) & 1, (blk + 1) * U);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int p = 0; p < NP; ++p) acc[p] = mfma32_f32(a[blk & 1][u][p], b[blk & 1][u][p], acc[p]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The same with a rolled loop, for kernels whose accumulators leave no room for a fully unrolled
// body's addresses: STEPS k-steps in blocks of U, two blocks per iteration.
template <int STEPS, int NP, typename OP>
__device__ __forceinline__ void mm_loop(f32x16 (&acc)[NP], OP op) {
  constexpr int U = NP == 1 ? 4 : 2;
  static_assert(STEPS % (2 * U) == 0, "whole block pairs");
  float a[2][U][NP], b[2][U][NP];
  auto read = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int p = 0; p < NP; ++p) op(p, s0 + u, a[buf][u][p], b[buf][u][p]);
  };
  auto mul = [&](int buf) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int p = 0; p < NP; ++p) acc[p] = mfma32_f32(a[buf][u][p], b[buf][u][p], acc[p]);
    __builtin_amdgcn_sched_barrier(0);
  };
  read(0, 0);
#pragma unroll 1
  for (int s = 0; s < STEPS; s += 2 * U) {
    read(1, s + U);
    mul(0);
    read(0, s + 2 * U < STEPS ? s + 2 * U : 0);  // (the last iteration's repeat is not used)
    mul(1);
  }
}

// A chunk's 64 rows of COLS elements of type T (the first `cols` of them valid) in registers, four
// per piece, by NT threads: every load of a workgroup's matrices is issued before the first LDS
// store.  Rows past len repeat the last valid one and are zeroed by put.  VEC: rows start on
// four-element boundaries.  Offsets from the (uniform) first row are 32-bit: st below kTileMaxStride.
constexpr int64_t kTileMaxStride = int64_t(1) << 23;
template <typename T, int COLS, int NT>
struct TileRows {
  static constexpr int q4 = COLS / 4, n = 64 * q4 / NT;
  static_assert(64 * q4 % NT == 0, "whole pieces per thread");
  typedef T vec4 __attribute__((ext_vector_type(4)));
  vec4 x[n];
  template <bool VEC = true>
  __device__ __forceinline__ void fetch(const T *src, int64_t st, int len, int cols) {
    const char *base = reinterpret_cast<const char *>(src);
#pragma unroll
    for (int j = 0; j < n; ++j) {
      const int e = threadIdx.x + NT * j, r = e / q4, c = 4 * (e - r * q4);
      const uint32_t off = (static_cast<uint32_t>(min(r, len - 1)) * static_cast<uint32_t>(st) + min(c, cols - 4)) * sizeof(T);
      if (VEC) {
        x[j] = *reinterpret_cast<const vec4 *>(base + off);
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) x[j][t] = *reinterpret_cast<const T *>(base + off + t * sizeof(T));
      }
    }
  }
  template <typename F>
  __device__ __forceinline__ void put(float *dst, int ld, int len, int cols, F scale) const {
#pragma unroll
    for (int j = 0; j < n; ++j) {
      const int e = threadIdx.x + NT * j, r = e / q4, c = 4 * (e - r * q4);
      const bool ok = r < len && c < cols;
      const float s = scale(r);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const T v = x[j][t];
        dst[r * ld + c + t] = ok ? ld_val(v) * s : 0.f;
      }
    }
  }
  __device__ __forceinline__ void put(float *dst, int ld, int len, int cols) const {
    put(dst, ld, len, cols, [](int) { return 1.f; });
  }
  __device__ __forceinline__ static float ld_val(T v) { return motif::ld(&v); }
};

// 64 rows of COLS elements at row stride st >= COLS, as TileRows, through a range-checked buffer
// over the first len rows: rows past them read zeros, so staging needs no clamps or selects (code
// that a workgroup runs once is bound by its own fetch).
template <typename T, int COLS, int NT>
struct BufRows {
  static constexpr int q4 = COLS / 4, n = 64 * q4 / NT;
  static_assert(64 * q4 % NT == 0 && NT % q4 == 0, "whole pieces per thread, one column per thread");
  uint4 x[n];
  __device__ __forceinline__ void fetch(const T *src, int64_t st, int len) {
    const buf_t buf = make_buf(src, static_cast<uint32_t>(((len - 1) * st + COLS) * sizeof(T)));
    const uint32_t r = threadIdx.x / q4, c = 4 * (threadIdx.x % q4), step = static_cast<uint32_t>(NT / q4 * st * sizeof(T));
    uint32_t off = (r * static_cast<uint32_t>(st) + c) * sizeof(T);
#pragma unroll
    for (int j = 0; j < n; ++j, off += step) {
      if constexpr (sizeof(T) == 4) {
        x[j] = buf_ld16(buf, off);
      } else {
        const uint2 u = buf_ld8(buf, off);
        x[j] = uint4{u.x << 16, u.x & 0xffff0000u, u.y << 16, u.y & 0xffff0000u};
      }
    }
  }
  __device__ __forceinline__ void put(float *dst, int ld) const {
    float *p = dst + threadIdx.x / q4 * ld + 4 * (threadIdx.x % q4);
#pragma unroll
    for (int j = 0; j < n; ++j) {
      const uint32_t w[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
      for (int t = 0; t < 4; ++t) p[j * (NT / q4) * ld + t] = __uint_as_float(w[t]);
    }
  }
};

// The entries of a 64-row vector at this lane's accumulator rows first + 8 (r / 4) + 4 h + r % 4.
__device__ __forceinline__ void acc_rows(float (&x)[16], const float *v, int first) {
  const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 u = *reinterpret_cast<const f32x4 *>(v + first + 8 * q + 4 * h);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[4 * q + t] = u[t];
  }
}

// T = (I - A)^{-1} of a strictly lower triangular 64 x 64 A, both in LDS with row stride
// LD, by a workgroup of at least 256 threads (every thread calls it; it starts and ends
// behind a barrier of its own).  16 x 16 diagonal blocks by substitution (one wave each),
// then T_ab = T_aa (A_ab T_bb) for the blocks (1, 0) and (3, 2) (a 16-term dot per
// element) and for the lower left 32 x 32 block (four waves, a 16 x 16 tile each, on
// v_mfma_f32_16x16x4_f32).  A is kept; xs is 32 * 33 floats of scratch.  Of T the diagonal
// 32 x 32 blocks (zeros above the diagonal included) and the lower left block are
// written; the upper right block is not.
template <int LD>
__device__ __forceinline__ void invert_unit_lower64(const float *sA, float *sT, float *xs) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nt = blockDim.x;
  __syncthreads();
  if (w < 4 && lane < 16) {
    const int b = w, c = lane;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = i == c ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) s = fmaf(sA[(16 * b + i) * LD + 16 * b + j], x[j], s);
      x[i] = s;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sT[(16 * b + i) * LD + 16 * b + c] = x[i];
  } else if (w < 4 && lane >= 32 && lane < 48 && !(w & 1)) {  // zeros of the blocks (0, 1) and (2, 3)
#pragma unroll
    for (int i = 0; i < 16; ++i) sT[(16 * w + i) * LD + 16 * w + 16 + (lane - 32)] = 0.f;
  }
  __syncthreads();
  for (int e = tid; e < 512; e += nt) {
    const int bj = 2 * (e >> 8), rr = (e >> 4) & 15, cc = e & 15, bi = bj + 1;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s = fmaf(sA[(16 * bi + rr) * LD + 16 * bj + k], sT[(16 * bj + k) * LD + 16 * bj + cc], s);
    xs[e] = s;
  }
  __syncthreads();
  for (int e = tid; e < 512; e += nt) {
    const int bj = 2 * (e >> 8), rr = (e >> 4) & 15, cc = e & 15, bi = bj + 1;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) s = fmaf(sT[(16 * bi + rr) * LD + 16 * bi + k], xs[((e >> 8) << 8) + (k << 4) + cc], s);
    sT[(16 * bi + rr) * LD + 16 * bj + cc] = s;
  }
  __syncthreads();
  const int ln = lane & 15, g = lane >> 4, ti = 16 * (w >> 1), tj = 16 * (w & 1);
  if (w < 4) {  // X = A[32:, :32] T[:32, :32]
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < 32; k0 += 4)
      x = mfma16_f32(sA[(32 + ti + ln) * LD + k0 + g], sT[(k0 + g) * LD + tj + ln], x);
#pragma unroll
    for (int r = 0; r < 4; ++r) xs[(ti + 4 * g + r) * 33 + tj + ln] = x[r];
  }
  __syncthreads();
  if (w < 4) {  // T[32:, :32] = T[32:, 32:] X
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < 32; k0 += 4)
      t = mfma16_f32(sT[(32 + ti + ln) * LD + 32 + k0 + g], xs[(k0 + g) * 33 + tj + ln], t);
#pragma unroll
    for (int r = 0; r < 4; ++r) sT[(32 + ti + 4 * g + r) * LD + tj + ln] = t[r];
  }
  __syncthreads();
}

}  // namespace motif
