// GatedDeltaNet chunk backward (gfx950): the whole backward of the chunked rule from the caller's
// own tensors (fp32 or bf16; unit feature strides, rows of q, k, v and dout apart and on
// four-element boundaries, row strides below 2^23; any batch and head strides on such boundaries)
// to their gradients, fp32 inside, in three launches:
//   gdn_bwd_operators   one workgroup per (chunk, batch * head): T = (I - A)^{-1} and the two scans'
//                       per-chunk operators
//                         A_n = e^{gamma_C} I - M1 K',  H_n = M1 V',  G_n = Q'^T dO,
//                       M1 = K~^T T, M2 = Attn T, Q' = Q e^gamma - M2 K', K' = beta e^gamma K,
//                       V' = beta V (the forward's operators, gdn_f32.hip; O = O' + Q' S, so the
//                       output's gradient enters the state's as Q'^T dO);
//   both scans          S <- A_n S + H_n forward and gS <- A_n^T gS + G_n in reverse, side by side
//                       (gdn_bwd.hip), recording P_n over H_n and dS_n over G_n;
//   gdn_bwd_grads       one workgroup per (chunk, batch * head): every gradient.  With
//                         Y = V' - K' P,  X = T Y,  Z = Attn^T dO + K~ dS,  B = T^T Z
//                       the inverse's own gradient needs no product with T: d/dA = B X^T
//                       (T^T (Z Y^T) T^T), d/dK' = -B P^T, d/dV' = B.
// Reference: motif/ops/gated_deltanet.py:180-260, :727-765 and the autograd of :830-855.
//
// The form this replaced converted and re-chunked every input to fp32 in separate passes (17
// launches, 110 us at H = 12, T = 4096, dv = 128), wrote T, W, U and dX per chunk (96 KB) for the
// last kernel to read, ran its 24 64 x 64 x 64 products per chunk on one wave per SIMD (121 + 177
// us), each operand read right before its use.  Here eight waves share a chunk (two per SIMD),
// products are read a block ahead (gdn_tiles.h) and the last kernel needs only T, P and dS.
// H = 12, T = 4096, dv = 128, bf16: operators 71 us, scans 44 us, gradients 143 us; forward and
// backward through the op 509 -> 298 us.  Code a workgroup runs once is kept small (range-checked
// loads and stores instead of per-row selects, row vectors read four at a time): with a select per
// element the last kernel's 93 KB of code outran the 64 KB instruction cache, 206 us.
// Bound: the phases' chains.  The 8.5 + 22 such products per chunk keep the matrix pipe busy 31% (operators)
// and 41% (gradients) of the time; with one workgroup per CU (120-155 KB of LDS) nothing else runs
// while its waves wait at a barrier or for a phase's LDS round trips.
#include <algorithm>
#include <type_traits>

#include "gdn_internal.h"
#include "gdn_tiles.h"

namespace motif {

namespace {

constexpr int kC = 64, kDK = 64, kLD = 65, kThreads = 512;
constexpr int kPlane = kC * kLD;
constexpr int kMaxGrid = 65535;  // second and third grid dimensions

struct View {  // [B, H, L, (features)] tensor
  const void *p;
  int64_t sb, sh, st;
};

struct BwdArgs {
  View q, k, v, beta, g, dout;
  View dq, dk, dv, dbeta, dg;  // (written)
  float *T, *A, *P, *dS;       // [BH * N][64][64], [..][dk][dk], [..][dk][dv] (H_n, then P_n), [..][dk][dv] (G_n, then dS_n)
  int H, L, N;
  int b0;                      // first batch row of the launch
};

template <typename T>
__device__ __forceinline__ const T *at(const View &v, int b, int h, int64_t t) {
  return static_cast<const T *>(v.p) + b * v.sb + h * v.sh + t * v.st;
}

// gates of the chunk for lane = row: (gamma, beta), zero gates past len
template <typename T>
__device__ __forceinline__ void chunk_gates(const BwdArgs &a, int b, int hd, int t0, int len, float &gam, float &beta) {
  const int lane = threadIdx.x & 63, row = t0 + min(lane, len - 1);
  const float gv = ld(at<T>(a.g, b, hd, row)), bv = ld(at<T>(a.beta, b, hd, row));
  float s = lane < len ? gv : 0.f;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float y = __shfl_up(s, off, 64);
    if (lane >= off) s += y;
  }
  gam = s;
  beta = lane < len ? bv : 0.f;
}

// Lane pointers of a 32 x 32 x k product's operands inside a plane of row stride LDP: element
// (first + l % 32, k + l / 32) of the rows, or of the columns, k two apart per step.
template <int LDP>
__device__ __forceinline__ const float *by_row(const float *plane, int first, int k0 = 0) {
  const int lane = threadIdx.x & 63;
  return plane + (first + (lane & 31)) * LDP + k0 + (lane >> 5);
}
template <int LDP>
__device__ __forceinline__ const float *by_col(const float *plane, int first, int k0 = 0) {
  const int lane = threadIdx.x & 63;
  return plane + (k0 + (lane >> 5)) * LDP + first + (lane & 31);
}

template <int DV>
struct OpLds {
  static constexpr int LV = DV + 1;
  static constexpr int k = 0, q = k + kPlane, v = q + kPlane, d = v + kC * LV, n = d + kC * LV, t = n + kPlane, at = t + kPlane;
  static constexpr int gam = at + kPlane, eg = gam + kC, kd = eg + kC, be = kd + kC, xs = be + kC;
  static constexpr int floats = xs + 32 * 33;
};

template <typename T, int DV>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) gdn_bwd_operators(BwdArgs a) {
  using LD = OpLds<DV>;
  constexpr int LV = LD::LV;
  extern __shared__ float sm[];
  float *sK = sm + LD::k, *sQ = sm + LD::q, *sV = sm + LD::v, *sDo = sm + LD::d, *sN = sm + LD::n, *sT = sm + LD::t,
        *sAt = sm + LD::at;
  float *sGam = sm + LD::gam, *sE = sm + LD::eg, *sKd = sm + LD::kd, *sB = sm + LD::be, *xs = sm + LD::xs;
  const int n = blockIdx.x, hd = blockIdx.y, b = a.b0 + blockIdx.z, t0 = n * kC, len = min(kC, a.L - t0);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, h = lane >> 5;
  const size_t cell = (static_cast<size_t>(b) * a.H + hd) * a.N + n;
  {
    BufRows<T, kDK, kThreads> rk, rq;
    BufRows<T, DV, kThreads> rv, rd;
    rk.fetch(at<T>(a.k, b, hd, t0), a.k.st, len);
    rq.fetch(at<T>(a.q, b, hd, t0), a.q.st, len);
    rv.fetch(at<T>(a.v, b, hd, t0), a.v.st, len);
    rd.fetch(at<T>(a.dout, b, hd, t0), a.dout.st, len);
    float gam, beta;
    chunk_gates<T>(a, b, hd, t0, len, gam, beta);
    if (w == 0) {
      sGam[lane] = gam;
      sE[lane] = exp_fast(gam);
      sKd[lane] = exp_fast(__shfl(gam, 63, 64) - gam);
      sB[lane] = beta;
    }
    rk.put(sK, kLD);
    rq.put(sQ, kLD);
    rv.put(sV, LV);
    rd.put(sDo, LV);
  }
  __syncthreads();
  // A = -strict(beta K K^T * D) (waves 0-2) and Attn = (Q K^T) * D (waves 4-6): lower 32 x 32 tiles
  if ((w & 3) < 3) {
    const int r0 = (w & 3) ? 32 : 0, c0 = (w & 3) == 2 ? 32 : 0;
    const bool attn = w >= 4;
    const float *pa = by_row<kLD>(attn ? sQ : sK, r0), *pb = by_row<kLD>(sK, c0);
    f32x16 c[2] = {};
    mm_pipe<kDK / 4, 2>(c, [&](int p, int s, float &x, float &y) {
      x = pa[p * (kDK / 2) + 2 * s];
      y = pb[p * (kDK / 2) + 2 * s];
    });
    const int C = c0 + i;
    const float gc = sGam[C];
    float gr[16], x[16];
    acc_rows(gr, sGam, r0);
    acc_rows(x, sB, r0);
    float *dst = (attn ? sAt : sN) + r0 * kLD + C;
    const int lim = C - r0 + (attn ? 0 : 1);  // first kept row of the tile
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float d = (attn ? 1.f : -x[r]) * (c[0][r] + c[1][r]) * exp_fast(gr[r] - gc);
      dst[acc_row32(r, h) * kLD] = acc_row32(r, h) >= lim ? d : 0.f;
    }
  }
  invert_unit_lower64<kLD>(sN, sT, xs);

  // M1 = K~^T T (waves 0-3, over the dead A) and M2 = Attn T (waves 4-6, over Attn once it is read);
  // T goes out (its upper right tile, never read, as it is).  T vanishes above its diagonal: column
  // tile 1 starts at k = 32, Attn's rows 0-31 end there.
  f32x16 m[2] = {};
  const int mt = w < 4 ? w : w - 4;
  const int mr = w < 4 ? 32 * (mt >> 1) : (mt ? 32 : 0), mc = w < 4 ? 32 * (mt & 1) : (mt == 2 ? 32 : 0);
  if (w < 4) {
    const float *pa = by_col<kLD>(sK, mr, mc), *pb = by_col<kLD>(sT, mc, mc), *pd = sKd + mc + h;
    auto op = [&](int k, float &x, float &y) { x = pa[k * kLD] * pd[k]; y = pb[k * kLD]; };
    if (mc) mm_pipe<8, 2>(m, [&](int p, int s, float &x, float &y) { op(16 * p + 2 * s, x, y); });
    else mm_pipe<16, 2>(m, [&](int p, int s, float &x, float &y) { op(32 * p + 2 * s, x, y); });
#pragma unroll
    for (int r = 0; r < 16; ++r) sN[(mr + acc_row32(r, h)) * kLD + mc + i] = m[0][r] + m[1][r];
  } else if (w < 7) {
    const float *pa = by_row<kLD>(sAt, mr, mc), *pb = by_col<kLD>(sT, mc, mc);
    auto op = [&](int k, float &x, float &y) { x = pa[k]; y = pb[k * kLD]; };
    if (mr && !mc) mm_pipe<16, 2>(m, [&](int p, int s, float &x, float &y) { op(32 * p + 2 * s, x, y); });
    else mm_pipe<8, 2>(m, [&](int p, int s, float &x, float &y) { op(16 * p + 2 * s, x, y); });
  }
  for (int e = tid; e < kC * kC / 4; e += kThreads) {
    const int r = e >> 4, c = 4 * (e & 15);
    *reinterpret_cast<f32x4 *>(a.T + cell * kC * kC + 4 * e) =
        f32x4{sT[r * kLD + c], sT[r * kLD + c + 1], sT[r * kLD + c + 2], sT[r * kLD + c + 3]};
  }
  __syncthreads();
  if (w >= 4 && w < 7) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sAt[(mr + acc_row32(r, h)) * kLD + mc + i] = m[0][r] + m[1][r];
  }
  for (int e = tid; e < kC * kDK; e += kThreads) sK[(e >> 6) * kLD + (e & 63)] *= sB[e >> 6] * sE[e >> 6];  // K'
  for (int e = tid; e < kC * DV; e += kThreads) sV[e / DV * LV + e % DV] *= sB[e / DV];                      // V'
  __syncthreads();

  // M1 [K' | V'] (A_n, H_n): waves 0 .. NT - 1, a row tile and two column tiles each; M2 K' (Q',
  // over the Q rows): the next two waves
  constexpr int NT = 2 + DV / 32;  // top waves: 2 row tiles x (64 + DV) / 64 column pairs
  if (w < NT + 2) {
    const bool top = w < NT;
    const int r0 = 32 * (top ? w & 1 : w - NT), cp = top ? w >> 1 : 0;  // column pair
    const float *pa = by_row<kLD>(top ? sN : sAt, r0);
    const float *pb = cp == 0 ? by_col<kLD>(sK, 0) : by_col<LV>(sV, 64 * (cp - 1));
    f32x16 c[4] = {};
    auto run = [&](auto ldc, auto kc) {
      constexpr int LB = decltype(ldc)::value, K = decltype(kc)::value;
      mm_pipe<K / 4, 4>(c, [&](int p, int s, float &x, float &y) {
        const int k = (p & 1) * (K / 2) + 2 * s;
        x = pa[k];
        y = pb[k * LB + 32 * (p >> 1)];
      });
    };
    if (!top && r0 == 0) run(std::integral_constant<int, kLD>(), std::integral_constant<int, 32>());  // (M2's rows 0-31)
    else if (cp == 0) run(std::integral_constant<int, kLD>(), std::integral_constant<int, 64>());
    else run(std::integral_constant<int, LV>(), std::integral_constant<int, 64>());
    const float ec = sE[kC - 1];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int R = r0 + acc_row32(r, h), col = 32 * ct + i;
        const float x = c[2 * ct][r] + c[2 * ct + 1][r];
        if (!top) sQ[R * kLD + col] = sQ[R * kLD + col] * sE[R] - x;
        else if (cp == 0) a.A[(cell * kDK + R) * kDK + col] = (R == col ? ec : 0.f) - x;
        else a.P[(cell * kDK + R) * DV + 64 * (cp - 1) + col] = x;
      }
  }
  __syncthreads();
  // G = Q'^T dO: a 32 x 32 tile per wave
  if (w < DV / 16) {
    const int r0 = 32 * (w & 1), c0 = 32 * (w >> 1);
    const float *pa = by_col<kLD>(sQ, r0), *pb = by_col<LV>(sDo, c0);
    f32x16 c[2] = {};
    mm_pipe<kC / 4, 2>(c, [&](int p, int s, float &x, float &y) {
      const int k = p * (kC / 2) + 2 * s;
      x = pa[k * kLD];
      y = pb[k * LV];
    });
#pragma unroll
    for (int r = 0; r < 16; ++r) a.dS[(cell * kDK + r0 + acc_row32(r, h)) * DV + c0 + i] = c[0][r] + c[1][r];
  }
}

// Sums of 16 per-lane values over the 32 lanes of each half: the returned value is the total of
// index 8 b4 + 4 b3 + 2 b2 + b1 (b = bits of lane % 32), the same in lanes that differ in bit 0.
__device__ __forceinline__ float half_sums(const float *v) {
  float x[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = v[r];
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int n = 8, off = 16; n > 0; n /= 2, off /= 2) {
    const bool hi = lane & off;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const float give = hi ? x[r] : x[r + n], keep = hi ? x[r + n] : x[r];
      x[r] = keep + __shfl_xor(give, off, 64);
    }
  }
  return x[0] + __shfl_xor(x[0], 1, 64);
}

struct GradLds {
  static constexpr int k = 0, t = kPlane, at = 2 * kPlane, b0 = 3 * kPlane, b1 = 4 * kPlane, b2 = 5 * kPlane,
                       b3 = 6 * kPlane, b4 = 7 * kPlane, gam = 8 * kPlane, eg = gam + kC, dec = eg + kC, be = dec + kC;
  static constexpr int row_g = be + kC, row_b = row_g + 4 * kC, col = row_b + 4 * kC, red = col + 4 * kC, floats = red + 8;
};

template <typename T, int DV>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) gdn_bwd_grads(BwdArgs a) {
  using LD = GradLds;
  extern __shared__ float sm[];
  float *sK = sm + LD::k, *sT = sm + LD::t, *sAt = sm + LD::at, *b0 = sm + LD::b0, *b1 = sm + LD::b1, *b2 = sm + LD::b2,
        *b3 = sm + LD::b3, *b4 = sm + LD::b4;
  float *sGam = sm + LD::gam, *sE = sm + LD::eg, *sDec = sm + LD::dec, *sB = sm + LD::be;
  const int n = blockIdx.x, hd = blockIdx.y, b = a.b0 + blockIdx.z, t0 = n * kC, len = min(kC, a.L - t0);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, h = lane >> 5;
  // each wave owns the 32 x 32 tile (r0, c0) of every 64 x 64 result of its group (waves 0-3, 4-7)
  const int tr = (w >> 1) & 1, tc = w & 1, r0 = 32 * tr, c0 = 32 * tc;
  const bool low = tr >= tc;  // the tile reaches below the diagonal
  const int own = (r0 + 4 * h) * kLD + c0 + i;  // this lane's elements: register r is el(r)
  auto el = [&](int r) { return own + (8 * (r >> 2) + (r & 3)) * kLD; };
  auto row = [&](int r) { return r0 + acc_row32(r, h); };
  // this lane's tile elements into an output's chunk columns col0 + c0 + i, rows past len dropped by
  // the buffer's range check
  auto put_out = [&](const View &v, int col0, const f32x16 &x) {
    const uint32_t sb = static_cast<uint32_t>(v.st * sizeof(T));
    const buf_t buf = make_buf(at<T>(v, b, hd, t0) + col0, (len - 1) * sb + 64 * sizeof(T));
    const uint32_t off = static_cast<uint32_t>(r0 + 4 * h) * sb + (c0 + i) * sizeof(T);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t o = off + static_cast<uint32_t>(8 * (r >> 2) + (r & 3)) * sb;
      if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[r]), buf, o, 0, 0);
      else __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(x[r]), buf, o, 0, 0);
    }
  };
  const size_t cell = (static_cast<size_t>(b) * a.H + hd) * a.N + n;

  // the value columns 64 j .. of b0 = dO, b1 = P, b2 = dS, b3 = v (all loads in flight together)
  auto stage_half = [&](int j) {
    BufRows<T, 64, kThreads> rd, rv;
    BufRows<float, 64, kThreads> rp, rs;
    rd.fetch(at<T>(a.dout, b, hd, t0) + 64 * j, a.dout.st, len);
    rv.fetch(at<T>(a.v, b, hd, t0) + 64 * j, a.v.st, len);
    rp.fetch(a.P + cell * kDK * DV + 64 * j, DV, 64);
    rs.fetch(a.dS + cell * kDK * DV + 64 * j, DV, 64);
    rd.put(b0, kLD);
    rp.put(b1, kLD);
    rs.put(b2, kLD);
    rv.put(b3, kLD);
  };
  {
    BufRows<T, kDK, kThreads> rk, rq;
    BufRows<float, kC, kThreads> rt;
    rk.fetch(at<T>(a.k, b, hd, t0), a.k.st, len);
    rq.fetch(at<T>(a.q, b, hd, t0), a.q.st, len);
    rt.fetch(a.T + cell * kC * kC, kC, 64);
    float gam, beta;
    chunk_gates<T>(a, b, hd, t0, len, gam, beta);
    if (w == 0) {
      sGam[lane] = gam;
      sE[lane] = exp_fast(gam);
      sDec[lane] = exp_fast(__shfl(gam, 63, 64) - gam);
      sB[lane] = beta;
    }
    rk.put(sK, kLD);
    rq.put(b4, kLD);
    rt.put(sT, kLD);
    stage_half(0);
  }
  __syncthreads();

  // The two groups of waves run the same barriers in code of their own (each with its own registers).
  // Group 0: Attn = (Q K^T) * D; Y; B and dv; T1 = dO X^T, T2 = dO P^T, T3 = X dS^T; dq and a part of dk.
  // Group 1: A (in T3); Z; X; T1 = B X^T, T2 = B P^T; the rest of dk.
  float *sRowG = sm + LD::row_g, *sRowB = sm + LD::row_b, *sCol = sm + LD::col, *sRed = sm + LD::red;
  auto decay = [&](float (&D)[16]) {  // D of the tile's elements, zero above the diagonal
    acc_rows(D, sGam, r0);
    const float gc = sGam[c0 + i];
#pragma unroll
    for (int r = 0; r < 16; ++r) D[r] = row(r) >= c0 + i ? exp_fast(D[r] - gc) : 0.f;
  };
  auto group = [&](auto g0c) {
    constexpr bool g0 = decltype(g0c)::value;
    f32x16 T1 = {}, T2 = {}, T3 = {};
    float rowB[16], rowG[16], bsum = 0.f;
    {
      f32x16 c[1] = {};
      if (low) {
        const float *pa = by_row<kLD>(g0 ? b4 : sK, r0), *pb = by_row<kLD>(sK, c0);
        mm_loop<kDK / 2, 1>(c, [&](int, int s, float &x, float &y) { x = pa[2 * s]; y = pb[2 * s]; });
      }
      float D[16], be[16];
      decay(D);
      if constexpr (!g0) acc_rows(be, sB, r0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        rowB[r] = 0.f;
        if constexpr (g0) sAt[el(r)] = c[0][r] * D[r];
        else T3[r] = row(r) > c0 + i ? -be[r] * c[0][r] * D[r] : 0.f;
      }
    }
    __syncthreads();

#pragma unroll 1
    for (int j = 0; j < DV / 64; ++j) {
      float vv[16];
      if constexpr (g0) {  // Y = beta (v - e^gamma K P) over v
        f32x16 c[2] = {};
        const float *pa = by_row<kLD>(sK, r0), *pb = by_col<kLD>(b1, c0);
        mm_loop<kDK / 4, 2>(c, [&](int p, int s, float &x, float &y) {
          x = pa[32 * p + 2 * s];
          y = pb[(32 * p + 2 * s) * kLD];
        });
        float be[16], eg[16];
        acc_rows(be, sB, r0);
        acc_rows(eg, sE, r0);
#pragma unroll
        for (int r = 0; r < 16; ++r) vv[r] = b3[el(r)];
#pragma unroll
        for (int r = 0; r < 16; ++r) b3[el(r)] = be[r] * (vv[r] - eg[r] * (c[0][r] + c[1][r]));
      } else {  // Z = Attn^T dO + e^{gamma_C - gamma} (K dS) over b4 (Attn^T: rows 32.. start at k = 32)
        f32x16 kd[1] = {}, x1[1] = {};
        const float *pa = by_row<kLD>(sK, r0), *pb = by_col<kLD>(b2, c0);
        mm_loop<kDK / 2, 1>(kd, [&](int, int s, float &x, float &y) { x = pa[2 * s]; y = pb[2 * s * kLD]; });
        const float *qa = by_col<kLD>(sAt, r0, r0), *qb = by_col<kLD>(b0, c0, r0);
        auto op = [&](int, int s, float &x, float &y) { x = qa[2 * s * kLD]; y = qb[2 * s * kLD]; };
        if (tr) mm_loop<16, 1>(x1, op);
        else mm_loop<32, 1>(x1, op);
        float dec[16];
        acc_rows(dec, sDec, r0);
#pragma unroll
        for (int r = 0; r < 16; ++r) b4[el(r)] = fmaf(kd[0][r], dec[r], x1[0][r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) bsum = fmaf(b2[el(r)], b1[el(r)], bsum);
      }
      __syncthreads();
      f32x16 c[1] = {};
      if constexpr (g0) {  // B = T^T Z
        const float *pa = by_col<kLD>(sT, r0, r0), *pb = by_col<kLD>(b4, c0, r0);
        auto op = [&](int, int s, float &x, float &y) { x = pa[2 * s * kLD]; y = pb[2 * s * kLD]; };
        if (tr) mm_loop<16, 1>(c, op);
        else mm_loop<32, 1>(c, op);
      } else {  // X = T Y
        const float *pa = by_row<kLD>(sT, r0), *pb = by_col<kLD>(b3, c0);
        auto op = [&](int, int s, float &x, float &y) { x = pa[2 * s]; y = pb[2 * s * kLD]; };
        if (tr) mm_loop<32, 1>(c, op);
        else mm_loop<16, 1>(c, op);
      }
      __syncthreads();  // Z and Y are read: B and X over them
#pragma unroll
      for (int r = 0; r < 16; ++r) (g0 ? b4 : b3)[el(r)] = c[0][r];
      if constexpr (g0) {
        float be[16];
        acc_rows(be, sB, r0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          rowB[r] = fmaf(c[0][r], vv[r], rowB[r]);
          c[0][r] *= be[r];
        }
        put_out(a.dv, 64 * j, c[0]);
      }
      __syncthreads();
      const float *pa = by_row<kLD>(g0 ? b0 : b4, r0), *px = by_row<kLD>(b3, c0), *pp = by_row<kLD>(b1, c0);
      if (low) {
        f32x16 x[2] = {T1, T2};
        mm_loop<32, 2>(x, [&](int p, int s, float &u, float &v) { u = pa[2 * s]; v = (p ? pp : px)[2 * s]; });
        T1 = x[0];
        T2 = x[1];
      } else {
        f32x16 x[1] = {T2};
        mm_loop<32, 1>(x, [&](int, int s, float &u, float &v) { u = pa[2 * s]; v = pp[2 * s]; });
        T2 = x[0];
      }
      if constexpr (g0) {
        const float *qa = by_row<kLD>(b3, r0), *qb = by_row<kLD>(b2, c0);
        f32x16 x[1] = {T3};
        mm_loop<32, 1>(x, [&](int, int s, float &u, float &v) { u = qa[2 * s]; v = qb[2 * s]; });
        T3 = x[0];
      }
      __syncthreads();
      if (j + 1 < DV / 64) {
        stage_half(j + 1);
        __syncthreads();
      }
    }

    // b0 = q, b1 = dAttn = (dO X^T) * D, b2 = -d(K K^T) / beta = -strict(B X^T) * D.  The row and
    // column sums of (d/dD) * D, dAttn * Attn and dA * A, are d gamma's.
    {
      BufRows<T, kDK, kThreads> rq;
      rq.fetch(at<T>(a.q, b, hd, t0), a.q.st, len);
      rq.put(b0, kLD);
    }
    float D[16];
    decay(D);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float x = T1[r] * D[r];
      if constexpr (g0) {
        rowG[r] = low ? T1[r] * sAt[el(r)] : 0.f;
        b1[el(r)] = x;
      } else {
        const bool in = row(r) > c0 + i;
        rowG[r] = in ? T1[r] * T3[r] : 0.f;
        b2[el(r)] = in ? -x : 0.f;
      }
    }
    float colG = 0.f;  // (pairwise)
    {
      float x[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = rowG[2 * r] + rowG[2 * r + 1];
      colG = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    }
    __syncthreads();
    f32x16 dkp[1] = {};
    if constexpr (g0) {  // dq = (dO P^T) e^gamma + dAttn k;  of dk: dAttn^T q + (X dS^T) e^{gamma_C - gamma}
      f32x16 dq[1] = {};
      const float *pa = by_row<kLD>(b1, r0), *pb = by_col<kLD>(sK, c0);
      auto op = [&](int, int s, float &x, float &y) { x = pa[2 * s]; y = pb[2 * s * kLD]; };
      if (tr) mm_loop<32, 1>(dq, op);
      else mm_loop<16, 1>(dq, op);
      const float *qa = by_col<kLD>(b1, r0, r0), *qb = by_col<kLD>(b0, c0, r0);
      auto op2 = [&](int, int s, float &x, float &y) { x = qa[2 * s * kLD]; y = qb[2 * s * kLD]; };
      if (tr) mm_loop<16, 1>(dkp, op2);
      else mm_loop<32, 1>(dkp, op2);
      float eg[16], dec[16];
      acc_rows(eg, sE, r0);
      acc_rows(dec, sDec, r0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float qe = T2[r] * eg[r];
        dq[0][r] += qe;
        const float t = T3[r] * dec[r], kd = t * sK[el(r)];
        rowG[r] += fmaf(qe, b0[el(r)], -kd);
        bsum += kd;
        b3[el(r)] = dkp[0][r] + t;
      }
      put_out(a.dq, 0, dq[0]);
      __syncthreads();
    } else {  // dkb = d(beta k): -(B P^T) e^gamma + dG k;  of dk: dG^T (beta k) + beta dkb
      f32x16 gk[1] = {};
      const float *pa = by_row<kLD>(b2, r0), *pb = by_col<kLD>(sK, c0);
      auto op = [&](int, int s, float &x, float &y) { x = pa[2 * s]; y = pb[2 * s * kLD]; };
      if (tr) mm_loop<32, 1>(gk, op);
      else mm_loop<16, 1>(gk, op);
      const float *qa = by_col<kLD>(b2, r0, r0), *qb = by_col<kLD>(sK, c0, r0), *qs = sB + r0 + h;
      auto op2 = [&](int, int s, float &x, float &y) { x = qa[2 * s * kLD] * qs[2 * s]; y = qb[2 * s * kLD]; };
      if (tr) mm_loop<16, 1>(dkp, op2);
      else mm_loop<32, 1>(dkp, op2);
      float eg[16], be[16];
      acc_rows(eg, sE, r0);
      acc_rows(be, sB, r0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float kv = sK[el(r)], z = -T2[r] * eg[r], dkb = z + gk[0][r];
        rowG[r] = fmaf(z * be[r], kv, rowG[r]);
        rowB[r] = dkb * kv;
        dkp[0][r] = fmaf(dkb, be[r], dkp[0][r]);
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 16; ++r) dkp[0][r] += b3[el(r)];
      put_out(a.dk, 0, dkp[0]);
    }

    // row sums over the tile's 32 columns, column sums over its 32 rows, block sums; wave 0 adds the
    // slots of (group, column tile) / (group, row tile)
    const float sg = half_sums(rowG), sb = half_sums(rowB);
    const int ri = (lane >> 1) & 15;  // half_sums' index of this lane
    constexpr int gi = g0 ? 0 : 2;
    if (!(lane & 1)) {
      sRowG[(gi + tc) * kC + r0 + acc_row32(ri, h)] = sg;
      sRowB[(gi + tc) * kC + r0 + acc_row32(ri, h)] = sb;
    }
    colG += __shfl_xor(colG, 32, 64);
    if (h == 0) sCol[(gi + tr) * kC + c0 + i] = colG;
    bsum = wave_sum(bsum);
    if (lane == 0) sRed[w] = bsum;
  };
  if (w < 4) group(std::true_type());
  else group(std::false_type());
  __syncthreads();
  if (w == 0) {
    // (the row and column sums cancel in the cumulative sum: 64 bits for these few terms)
    double dgam = 0.0;
    float db = 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      dgam += double(sRowG[x * kC + lane]) - double(sCol[x * kC + lane]);
      db += sRowB[x * kC + lane];
    }
    if (lane == kC - 1)
      dgam += (sRed[0] + sRed[1] + sRed[2] + sRed[3]) + sE[kC - 1] * (sRed[4] + sRed[5] + sRed[6] + sRed[7]);
    double s = dgam;  // dg: the reverse cumulative sum of d gamma (gamma = cumsum g)
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double y = __shfl_down(s, off, 64);
      if (lane + off < 64) s += y;
    }
    if (lane < len) {
      st(const_cast<T *>(at<T>(a.dg, b, hd, t0 + lane)), static_cast<float>(s));
      st(const_cast<T *>(at<T>(a.dbeta, b, hd, t0 + lane)), db);
    }
  }
}

template <typename K>
int set_smem(K kern, size_t smem, const char *what) {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(smem));
  return e == hipSuccess ? MOTIF_OK : set_error(MOTIF_ERR_HIP, std::string(what) + " smem: " + hipGetErrorString(e));
}

// workspace: T, A, H_n / P_n, G_n / dS_n per cell, then the forward scan's final state (not used)
size_t ws_floats(int64_t BH, int N, int dv) {
  const size_t cells = static_cast<size_t>(BH) * N;
  return cells * (kC * kC + kDK * kDK + 2 * kDK * size_t(dv)) + static_cast<size_t>(BH) * kDK * dv;
}

template <typename T, int DV>
int launch_bwd(BwdArgs a, int B, const float *S0, const float *dS_final, float *dS0, float *s_scratch, hipStream_t s) {
  const dim3 block(kThreads);
  // (a launch takes 65535 batch rows)
  auto grid = [&] { return dim3(a.N, a.H, std::min(B - a.b0, kMaxGrid)); };
  constexpr size_t smem1 = OpLds<DV>::floats * 4, smem2 = GradLds::floats * 4;
  if (int rc = set_smem(gdn_bwd_operators<T, DV>, smem1, "gdn_bwd_operators")) return rc;
  for (a.b0 = 0; a.b0 < B; a.b0 += kMaxGrid) {
    gdn_bwd_operators<T, DV><<<grid(), block, smem1, s>>>(a);
    if (int rc = check_launch("gdn_bwd_operators")) return rc;
  }
  if (int rc = motif_gdn_opscan_pair_f32(a.A, a.P, S0, a.P, s_scratch, a.dS, dS_final, a.dS, dS0, B * a.H, a.N, kDK, DV, s))
    return rc;
  if (int rc = set_smem(gdn_bwd_grads<T, DV>, smem2, "gdn_bwd_grads")) return rc;
  for (a.b0 = 0; a.b0 < B; a.b0 += kMaxGrid) {
    gdn_bwd_grads<T, DV><<<grid(), block, smem2, s>>>(a);
    if (int rc = check_launch("gdn_bwd_grads")) return rc;
  }
  return MOTIF_OK;
}

}  // namespace

}  // namespace motif

extern "C" size_t motif_gdn_chunk_bwd_workspace_bytes(int B, int H, int L, int dk, int dv) {
  using namespace motif;
  if (B <= 0 || H <= 0 || L <= 0 || dk != kDK || (dv != 64 && dv != 128)) return 0;
  return ws_floats(int64_t(B) * H, (L + kC - 1) / kC, dv) * sizeof(float);
}

extern "C" int motif_gdn_chunk_bwd(
    const void *q, int64_t q_sb, int64_t q_sh, int64_t q_st, const void *k, int64_t k_sb, int64_t k_sh, int64_t k_st,
    const void *v, int64_t v_sb, int64_t v_sh, int64_t v_st, const void *beta, int64_t b_sb, int64_t b_sh, int64_t b_st,
    const void *g, int64_t g_sb, int64_t g_sh, int64_t g_st, const void *dout, int64_t o_sb, int64_t o_sh, int64_t o_st,
    const float *state_in, const float *dstate_out,
    void *dq, int64_t dq_sb, int64_t dq_sh, int64_t dq_st, void *dk_, int64_t dk_sb, int64_t dk_sh, int64_t dk_st,
    void *dv_, int64_t dv_sb, int64_t dv_sh, int64_t dv_st, void *dbeta, int64_t db_sb, int64_t db_sh, int64_t db_st,
    void *dg, int64_t dg_sb, int64_t dg_sh, int64_t dg_st, float *dstate_in,
    int B, int H, int L, int dk, int dv, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
  using namespace motif;
  if (B < 0 || H < 0 || L < 0 || dk <= 0 || dv <= 0) return set_error(MOTIF_ERR_INVALID, "gdn_chunk_bwd: bad sizes");
  if (dk != kDK || (dv != 64 && dv != 128))
    return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: needs dk == 64 and dv in {64, 128}");
  if (dtype != MOTIF_F32 && dtype != MOTIF_BF16) return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: unsupported dtype");
  if (B == 0 || H == 0) return MOTIF_OK;
  if (L == 0) {  // (no step to go through: the state's gradient is the final state's)
    if (!dstate_in) return set_error(MOTIF_ERR_INVALID, "gdn_chunk_bwd: NULL pointer");
    return motif_gdn_opscan_f32(nullptr, nullptr, dstate_out, nullptr, dstate_in, B * H, 0, dk, dv, 1, 0, stream);
  }
  if (!q || !k || !v || !beta || !g || !dout || !dq || !dk_ || !dv_ || !dbeta || !dg || !dstate_in)
    return set_error(MOTIF_ERR_INVALID, "gdn_chunk_bwd: NULL pointer");
  const int N = (L + kC - 1) / kC;
  if (H > kMaxGrid || int64_t(B) * H * N >= (int64_t(1) << 31))
    return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: too many chunks");
  const size_t need = motif_gdn_chunk_bwd_workspace_bytes(B, H, L, dk, dv);
  if (!workspace || workspace_bytes < need)
    return set_error(MOTIF_ERR_INVALID, "gdn_chunk_bwd: workspace too small (need " + std::to_string(need) + " bytes)");
  if (reinterpret_cast<uintptr_t>(workspace) & 15)
    return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: the workspace needs 16-byte alignment");
  // four-element row loads, 32-bit offsets inside a chunk
  const uintptr_t p = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                      reinterpret_cast<uintptr_t>(dout);
  const int64_t st = q_sb | q_sh | q_st | k_sb | k_sh | k_st | v_sb | v_sh | v_st | o_sb | o_sh | o_st;
  if ((st & 3) || (p & (dtype == MOTIF_F32 ? 15 : 7)))
    return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: q, k, v and dout rows need four-element alignment");
  for (int64_t x : {q_st, k_st, dq_st, dk_st})
    if (x < dk || x >= kTileMaxStride) return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: row stride out of range");
  for (int64_t x : {v_st, o_st, dv_st})
    if (x < dv || x >= kTileMaxStride) return set_error(MOTIF_ERR_UNSUPPORTED, "gdn_chunk_bwd: row stride out of range");
  const size_t cells = static_cast<size_t>(B) * H * N;
  float *T = static_cast<float *>(workspace), *A = T + cells * kC * kC, *P = A + cells * kDK * kDK, *dS = P + cells * kDK * dv;
  const BwdArgs a{{q, q_sb, q_sh, q_st}, {k, k_sb, k_sh, k_st}, {v, v_sb, v_sh, v_st}, {beta, b_sb, b_sh, b_st},
                  {g, g_sb, g_sh, g_st}, {dout, o_sb, o_sh, o_st}, {dq, dq_sb, dq_sh, dq_st}, {dk_, dk_sb, dk_sh, dk_st},
                  {dv_, dv_sb, dv_sh, dv_st}, {dbeta, db_sb, db_sh, db_st}, {dg, dg_sb, dg_sh, dg_st},
                  T, A, P, dS, H, L, N};
  float *scratch = dS + cells * kDK * dv;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MOTIF_F32)
    return dv == 64 ? launch_bwd<float, 64>(a, B, state_in, dstate_out, dstate_in, scratch, s)
                    : launch_bwd<float, 128>(a, B, state_in, dstate_out, dstate_in, scratch, s);
  return dv == 64 ? launch_bwd<bf16_t, 64>(a, B, state_in, dstate_out, dstate_in, scratch, s)
                  : launch_bwd<bf16_t, 128>(a, B, state_in, dstate_out, dstate_in, scratch, s);
}
