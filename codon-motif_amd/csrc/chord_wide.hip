// Chord attention prefill in fp32 arithmetic on the matrix instructions (gfx950): fp32, fp16 and
// bf16 inputs at head dims 16, 32, 64 and 128 (bf16 at 64 has its own kernel, chord.hip).
//
// A workgroup is NW waves over the same 32 queries of one head; wave w takes the 32-key tiles
// w, w + NW, ... and the partial softmaxes meet in LDS at the end, so the longest row's chain is
// ceil(S / 32 / NW) tiles and short prompts still fill the chip.  The waves share no keys, so
// nothing is staged: K and V come from global memory (L2) straight into the operand registers.
//   S^T = K Q^T    lane l: key l % 32 of the tile against query l % 32.  fp32 inputs take
//                  v_mfma_f32_32x32x2_f32 in D / 8 chains of eight features, two side by
//                  side, summed pairwise (the lane half h holds features 8 j + 4 h + 0..3, so
//                  both operands are 16-byte pieces of a row); 16-bit inputs take 32x32x16,
//                  whose products are exact and whose sums are fp32.
//   O^T += V^T P^T on v_mfma_f32_32x32x2_f32 for every type: P stays fp32, straight from the
//                  score accumulators (register r of half h is key 8 (r / 4) + 4 h + r % 4), V
//                  converts to fp32 exactly.  Row m of output tile t is feature VD m + t
//                  (VD = D / 32), so a lane's V piece of a key is VD consecutive features.
// This tile's V is requested before S^T, the next tile's K when S^T is done.  K has the softmax and
// the whole O product to arrive in (D / 2 MFMAs of 64 cycles: 2048 cycles at D = 64).  V has the
// score product and the softmax: D / 2 MFMAs of 64 cycles for fp32, but only D / 16 of 32 cycles
// (128 at D = 64) for 16-bit inputs.  The distance bias of a tile depends on 63 distances: each
// lane evaluates one into a wave-private LDS window.
// Bound: per 32 x 32 scores at D = 64, 64 fp32 MFMAs of 64 cycles (32 and four of 32 cycles for
// 16-bit inputs), where the query blocks fill the chip: the matrix pipe is busy 58% of the time at
// 4096 tokens, fp32.  At 1023 tokens (28%; fp16 21%) the 384 workgroups, one per CU, are a round
// and a half, and the longest rows' chain of tiles sets its length.  Kernel time under the tracer, 12 heads, 3 kv heads, in
// us (and of the vector kernel that served these shapes, with its bias table's launch): fp32 1023
// tokens 34.5 (151), 4096 tokens 325 (1355), 3 tokens over 4096 82 (101); fp16 1023 tokens 22 (148);
// bf16 D = 128 1000 tokens 36 (381).  Error against 64 bits, fp32: 3.7e-7 (4.1e-7).
#include <algorithm>

#include "capi_internal.h"
#include "chord_internal.h"
#include "common.h"
#include "gdn_tiles.h"

namespace motif {

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;

// features held per lane for one row: D / 2 (the two lane halves share a row)
template <typename T, int D> struct RowOp;  // a K or Q row operand of the score product
template <int D> struct RowOp<float, D> {
  f32x4 x[D / 8];
  __device__ __forceinline__ void load(buf_t r, uint32_t off, int h) {
#pragma unroll
    for (int j = 0; j < D / 8; ++j) x[j] = __builtin_bit_cast(f32x4, buf_ld16(r, off + 32 * j + 16 * h));
  }
};
template <typename T, int D> struct RowOp {
  uint4 x[D / 16];
  __device__ __forceinline__ void load(buf_t r, uint32_t off, int h) {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) x[j] = buf_ld16(r, off + 32 * j + 16 * h);
  }
};
// fp32: eight features per chain, the D / 8 chains summed pairwise (a chain over the whole row
// would collect 1.5 times the rounding)
template <int D, int J0, int NJ> __device__ __forceinline__ f32x16 score_f32(const RowOp<float, D> &k, const RowOp<float, D> &q) {
  if constexpr (NJ == 1) {
    f32x16 c = {};
#pragma unroll
    for (int t = 0; t < 4; ++t) c = mfma32_f32(k.x[J0][t], q.x[J0][t], c);
    return c;
  } else if constexpr (NJ == 2) {  // two chains side by side
    f32x16 c0 = {}, c1 = {};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      c0 = mfma32_f32(k.x[J0][t], q.x[J0][t], c0);
      c1 = mfma32_f32(k.x[J0 + 1][t], q.x[J0 + 1][t], c1);
    }
    return c0 + c1;
  } else {
    const f32x16 lo = score_f32<D, J0, NJ / 2>(k, q);
    return lo + score_f32<D, J0 + NJ / 2, NJ / 2>(k, q);
  }
}
// The score products of a tile: fp32 as two half-row sums (their sum would be rounded at the size
// of a whole score, and a score is scaled by up to log2(e) ln(n) before the exponential).
template <int D> __device__ __forceinline__ void score(const RowOp<float, D> &k, const RowOp<float, D> &q, f32x16 (&s)[2]) {
  s[0] = score_f32<D, 0, D / 16>(k, q);
  s[1] = score_f32<D, D / 16, D / 16>(k, q);
}
template <int D> __device__ __forceinline__ void score(const RowOp<bf16_t, D> &k, const RowOp<bf16_t, D> &q, f32x16 (&s)[1]) {
  f32x16 c = {};
#pragma unroll
  for (int j = 0; j < D / 16; ++j)
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, k.x[j]), __builtin_bit_cast(bf16x8, q.x[j]), c, 0, 0, 0);
  s[0] = c;
}
template <int D> __device__ __forceinline__ void score(const RowOp<f16_t, D> &k, const RowOp<f16_t, D> &q, f32x16 (&s)[1]) {
  f32x16 c = {};
#pragma unroll
  for (int j = 0; j < D / 16; ++j)
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, k.x[j]), __builtin_bit_cast(f16x8, q.x[j]), c, 0, 0, 0);
  s[0] = c;
}

// N consecutive elements of type T at byte offset off, as loaded
template <typename T, int N> struct Piece {
  static constexpr int kBytes = N * static_cast<int>(sizeof(T)), kW = kBytes > 4 ? kBytes / 4 : 1;
  uint32_t w[kW];
  __device__ __forceinline__ void load(buf_t r, uint32_t off) {
    if constexpr (kBytes == 2) {
      w[0] = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
    } else if constexpr (kBytes == 4) {
      w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    } else if constexpr (kBytes == 8) {
      const uint2 u = buf_ld8(r, off);
      w[0] = u.x; w[1] = u.y;
    } else {
      static_assert(kBytes == 16, "a piece is 2 to 16 bytes");
      const uint4 u = buf_ld16(r, off);
      w[0] = u.x; w[1] = u.y; w[2] = u.z; w[3] = u.w;
    }
  }
  __device__ __forceinline__ float get(int e) const {
    if constexpr (sizeof(T) == 4) return __uint_as_float(w[e]);
    const uint16_t b = static_cast<uint16_t>(w[e >> 1] >> (16 * (e & 1)));
    if constexpr (__is_same(T, bf16_t)) return bf16_to_f32(b);
    else return static_cast<float>(__builtin_bit_cast(f16_t, b));
  }
};

template <typename T, int D, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4)))
chord_wide_kernel(ChordArgs a) {
  constexpr int VD = D >= 32 ? D / 32 : 1;  // output tiles, and features of a V piece
  constexpr int ES = sizeof(T), NS = ES == 4 ? 2 : 1;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, h = lane >> 5;
  // (the heads vary fastest, the latest -- longest -- query blocks first)
  const int head = blockIdx.x, qb = gridDim.y - 1 - blockIdx.y, b = blockIdx.z;
  const int kvh = head / (a.H / a.Hkv);
  const int q0 = 32 * qb, my_q = q0 + i, q_abs = a.q_start + my_q;
  const int kv_end = min(a.S, a.q_start + min(a.L, q0 + 32));  // keys any query of the block sees
  const int ntiles = (kv_end + 31) / 32;

  const T *kp = static_cast<const T *>(a.k) + b * a.k_sb + kvh * a.k_sh;
  const T *vp = static_cast<const T *>(a.v) + b * a.v_sb + kvh * a.v_sh;
  // the buffer of tile t: its rows below kv_end (rows past it read zeros)
  auto tile_buf = [&](const T *p, int64_t st, int t) {
    const int rows = min(32, kv_end - 32 * t);
    return make_buf(p + int64_t(32 * t) * st, rows > 0 ? static_cast<uint32_t>(((rows - 1) * st + D) * ES) : 0u);
  };
  const uint32_t koff = static_cast<uint32_t>(i * a.k_st) * ES;
  const uint32_t voff = static_cast<uint32_t>(4 * h * a.v_st + VD * (D < 32 ? i & (D - 1) : i)) * ES;
  const uint32_t vrow = static_cast<uint32_t>(a.v_st) * ES;

  RowOp<T, D> q, k;
  {
    const T *qp = static_cast<const T *>(a.q) + b * a.q_sb + head * a.q_sh + int64_t(q0) * a.q_st;
    const int rows = min(32, a.L - q0);
    q.load(make_buf(qp, static_cast<uint32_t>(((rows - 1) * a.q_st + D) * ES)),
           static_cast<uint32_t>(min(i, rows - 1) * a.q_st) * ES, h);
  }
  if (w < ntiles) k.load(tile_buf(kp, a.k_st, w), koff, h);

  const float mul = a.ssmax[head] * a.log_n[b * a.ln_sb + int64_t(min(my_q, a.L - 1)) * a.ln_st];
  const float c_qk = mul * a.scale * kLog2e, c_b = mul * kLog2e;  // logits in log2 units
  const float al = a.alpha[head], be = a.beta[head], mu = a.mu[head];

  extern __shared__ __attribute__((aligned(16))) float smem[];
  float *win = smem + 64 * w;                 // [NW][64]: the bias of distance base + j
  float *sml = smem + 64 * NW;                // [NW][2][32] max and sum of each wave
  float *tile = sml + 64 * NW;                // [NW][16][64] one output tile of each wave
  const float *winr = win + 4 * h - i + 31;   // + key offset inside the tile

  float m = -INFINITY, l = 0.f;
  f32x16 o[VD];
#pragma unroll
  for (int t = 0; t < VD; ++t) o[t] = f32x16{};

  for (int t = w; t < ntiles; t += NW) {
    const int n0 = 32 * t;
    Piece<T, VD> v[16];
    const buf_t vb = tile_buf(vp, a.v_st, t);
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r].load(vb, voff + static_cast<uint32_t>(8 * (r >> 2) + (r & 3)) * vrow);
    win[lane] = ggd_bias(static_cast<float>(n0 - a.q_start - q0 - 31 + lane), al, be, mu, a.eps);
    __builtin_amdgcn_sched_barrier(0);
    f32x16 sc[NS];
    score<D>(k, q, sc);
    float bias[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bias[r] = winr[8 * (r >> 2) + (r & 3)];
    __builtin_amdgcn_sched_barrier(0);
    k.load(tile_buf(kp, a.k_st, t + NW), koff, h);  // (past the last tile: an empty buffer, zeros)
    __builtin_amdgcn_sched_barrier(0);
    const bool masked = n0 + 31 > a.q_start + q0 || n0 + 32 > kv_end;  // the diagonal and the last tiles
    auto keep = [&](int r) {
      const int key = n0 + 8 * (r >> 2) + 4 * h + (r & 3);
      return key <= q_abs && key < kv_end;
    };
    // a logit plus `off`: the fp32 form adds the large terms first, so with off = -max they cancel
    // before the small result is rounded
    auto logit = [&](int r, float off) {
      float x = ES == 4 ? fmaf(c_b, bias[r], off) : c_b * bias[r];
#pragma unroll
      for (int n = 0; n < NS; ++n) x = fmaf(sc[n][r], c_qk, x);
      return ES == 4 ? x : x + off;
    };
    float mx = -INFINITY, s[16];
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, keep(r) ? logit(r, 0.f) : -INFINITY);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, logit(r, 0.f));
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    if (__ballot(m_new > m)) {
      const float resc = m == -INFINITY ? 0.f : fast_exp2(m - m_use);
      l *= resc;
#pragma unroll
      for (int t2 = 0; t2 < VD; ++t2)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t2][r] *= resc;
      m = m_new;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = logit(r, -m_use);
    if (masked) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = keep(r) ? s[r] : -INFINITY;
    }
    float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r]);
      ps[r & 3] += s[r];
    }
    l += (ps[0] + ps[1]) + (ps[2] + ps[3]);
    if constexpr (ES == 4) {  // four fresh chains per tile, as for the scores
#pragma unroll
      for (int t2 = 0; t2 < VD; ++t2) {
        f32x16 c[4] = {};
#pragma unroll
        for (int r = 0; r < 16; ++r) c[r >> 2] = mfma32_f32(v[r].get(t2), s[r], c[r >> 2]);
        o[t2] += (c[0] + c[1]) + (c[2] + c[3]);
      }
    } else {  // (16-bit results: one ulp of theirs covers a chain's rounding)
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int t2 = 0; t2 < VD; ++t2) o[t2] = mfma32_f32(v[r].get(t2), s[r], o[t2]);
    }
  }

  // the waves' partials: l over the two lane halves, then every wave scaled to the common max
  l += __shfl_xor(l, 32, 64);
  if (h == 0) {
    sml[64 * w + i] = m;
    sml[64 * w + 32 + i] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int x = 0; x < NW; ++x) M = fmaxf(M, sml[64 * x + i]);
  const float f = m == -INFINITY ? 0.f : fast_exp2(m - M);
  // threads tid, tid + 64 NW, ... of an output tile: register r = e / 64 of lane e % 64
  constexpr int kE = 16 / NW;
  float sum[kE][VD];
#pragma unroll
  for (int t = 0; t < VD; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) tile[(16 * w + r) * 64 + lane] = o[t][r] * f;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kE; ++e) {
      float x[NW];
#pragma unroll
      for (int y = 0; y < NW; ++y) x[y] = tile[(16 * y + w + NW * e) * 64 + lane];
#pragma unroll
      for (int n = NW / 2; n > 0; n /= 2)
#pragma unroll
        for (int y = 0; y < n; ++y) x[y] += x[y + n];
      sum[e][t] = x[0];
    }
    __syncthreads();
  }
  if (my_q >= a.L) return;
  float Ls = 0.f;
#pragma unroll
  for (int x = 0; x < NW; ++x) {
    const float mx = sml[64 * x + i];
    if (mx != -INFINITY) Ls = fmaf(sml[64 * x + 32 + i], fast_exp2(mx - M), Ls);
  }
  T *op = static_cast<T *>(a.out) + b * a.o_sb + head * a.o_sh + int64_t(my_q) * a.o_st;
#pragma unroll
  for (int e = 0; e < kE; ++e) {
    const int row = acc_row32(w + NW * e, h);
    if (D < 32 && row >= D) continue;
#pragma unroll
    for (int t = 0; t < VD; ++t) st(op + VD * row + t, sum[e][t] / fmaxf(Ls, 1e-20f));
  }
  if (a.lse && w == 0 && h == 0) a.lse[(static_cast<size_t>(b) * a.H + head) * a.L + my_q] = M + fast_log2(Ls);
}

template <typename T, int D, int NW>
int launch_wide(const ChordArgs &a, hipStream_t s) {
  constexpr int smem = (2 * 64 * NW + NW * 16 * 64) * static_cast<int>(sizeof(float));
  const dim3 grid(a.H, (a.L + 31) / 32, a.B), block(64 * NW);
  chord_wide_kernel<T, D, NW><<<grid, block, smem, s>>>(a);
  return check_launch("chord_wide_kernel");
}

template <typename T>
int launch_wide_t(const ChordArgs &a, int D, hipStream_t s) {
  switch (D) {
    case 16: return launch_wide<T, 16, 8>(a, s);
    case 32: return launch_wide<T, 32, 8>(a, s);
    case 64: return launch_wide<T, 64, 8>(a, s);
    // (fp32 rows of 128 features leave no registers for a second wave per SIMD)
    default: return launch_wide<T, 128, sizeof(T) == 4 ? 4 : 8>(a, s);
  }
}

}  // namespace

// 32-bit byte offsets inside a 32-row tile, and grid dimensions within the launch limits.
bool chord_wide_serves(const ChordArgs &a) {
  const int64_t st = std::max({a.q_st, a.k_st, a.v_st}), lo = std::min({a.q_st, a.k_st, a.v_st});
  return a.log_n && lo >= 0 && st < (int64_t(1) << 24) && a.B <= 65535 && (a.L + 31) / 32 <= 65535 &&
         int64_t(a.q_start) + a.L < (int64_t(1) << 30);
}

int launch_chord_wide(const ChordArgs &a, int dtype, int D, hipStream_t s) {
  if (dtype == MOTIF_BF16) return launch_wide_t<bf16_t>(a, D, s);
  if (dtype == MOTIF_F16) return launch_wide_t<f16_t>(a, D, s);
  return launch_wide_t<float>(a, D, s);
}

}  // namespace motif
