// GDN chunked prefill for fp32 inputs on the fp32 matrix instructions (gfx950), chunk 64.
//
// The same three-kernel form as the bf16 path (gdn_chunk.hip), every operand, product and
// sum in fp32 (v_mfma_f32_32x32x2_f32 / 16x16x4_f32: an fp32 multiply and add per term):
//   gdn_f32_prep  one workgroup per (chunk, head): T = (I - A)^{-1},
//                 A = -strict(beta K K^T * D), then with M1 = K~^T T, M2 = Attn T
//                 (K~ = K e^{gamma_C - gamma}, Attn = (Q K^T) * D) and the scaled rows
//                 K' = beta e^gamma K, V' = beta V
//                   A_n = e^{gamma_C} I - M1 K',  H_n = M1 V',
//                   Q'  = Q e^gamma - M2 K',      O'  = M2 V';
//   the operator scan of gdn_bwd.hip  S_{n+1} = A_n S_n + H_n, recording every S_n;
//   gdn_f32_out   O_n = O' + Q' S_n for all chunks in parallel.
// The form this replaced (row-by-row substitution of [W | U] and a scan holding three
// products per chunk, on the vector unit) put every chunk's products into the serial chain:
// 17 us a chunk.  Here only one dk x dk x dv product per chunk is serial.  Measured (prep +
// scan + output): 30 us at B = 1, H = 4, T = 256, dk = dv = 64 (19.4 + 5.2 + 5.7; was 110), 138 us
// at H = 12, T = 4096, dv = 128 (77 + 41 + 20; was 1220).  The prep is bound by its MFMA chains (32
// terms each) and the LDS round trips between its phases (one workgroup per CU; the matrix pipe is
// busy 27% of the time), the scan by the chain.  Its error against 64 bits is the smaller one too
// (4.0e-7 against 4.5e-7 relative at T = 256).
#include <algorithm>
#include <type_traits>

#include "gdn_internal.h"
#include "gdn_tiles.h"

namespace motif {

namespace {

constexpr int kC = 64;         // chunk length
constexpr int kLT = 65;        // LDS row stride of a 64-column matrix (floats)
constexpr int kThreads = 512;  // prep: 8 waves, two per SIMD, so one's operand reads hide under the other's MFMAs

// Workspace: per (head, chunk) cell, fp32 and row-major, one array per operand.
struct F32Ws {
  float *A, *Hn, *Qp;  // [cells][dk][dk], [cells][dk][dv] (the scan puts S_n in H_n's place), [cells][64][dk]
  static size_t cell_floats(int dk, int dv) { return size_t(dk) * dk + size_t(dk) * dv + size_t(kC) * dk; }
  F32Ws(float *ws, size_t cells, int dk, int dv) : A(ws), Hn(A + cells * dk * dk), Qp(Hn + cells * dk * dv) {}
};

template <int DK, int DV>
struct F32Lds {
  static constexpr int LK = DK + 1, LV = DV + 1;
  static constexpr int k = 0, q = k + kC * LK, v = q + kC * LK, n = v + kC * LV, t = n + kC * kLT, at = t + kC * kLT;
  static constexpr int gam = at + kC * kLT, eg = gam + kC, kd = eg + kC, be = kd + kC, xs = be + kC;
  static constexpr int floats = xs + 32 * 33;
};

// sum over k in [0, K) of fa(k) fb(k) for a 32x32 tile, fa / fb the lane's row and column
// (offset by the lane half): the two halves of the range in two independent chains, which
// halves both the chain and the rounding a chain of 64 sums collects.
template <int K, typename FA, typename FB>
__device__ __forceinline__ f32x16 dot2(FA fa, FB fb) {
  f32x16 c[2] = {};
  mm_pipe<K / 4, 2>(c, [&](int p, int s, float &a, float &b) {
    const int k = p * (K / 2) + 2 * s;
    a = fa(k);
    b = fb(k);
  });
  return c[0] + c[1];
}

template <int DK, int DV>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) gdn_f32_prep(GdnArgs a, ChunkArgs ca, F32Ws ws, int vec) {
  using LD = F32Lds<DK, DV>;
  constexpr int LK = LD::LK, LV = LD::LV;
  extern __shared__ float sm[];
  float *sK = sm + LD::k, *sQ = sm + LD::q, *sV = sm + LD::v, *sN = sm + LD::n, *sT = sm + LD::t, *sAt = sm + LD::at;
  float *sGam = sm + LD::gam, *sE = sm + LD::eg, *sKd = sm + LD::kd, *sB = sm + LD::be, *xs = sm + LD::xs;

  const int chunk = blockIdx.x, hd = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 31, h = lane >> 5;
  const ChunkInfo ci = resolve_chunk(chunk, kC, a.L, ca);
  const float *kb = static_cast<const float *>(a.k) + ci.batch * a.k_sb + hd * a.k_sh + int64_t(ci.t0) * a.k_st;
  const float *qb = static_cast<const float *>(a.q) + ci.batch * a.q_sb + hd * a.q_sh + int64_t(ci.t0) * a.q_st;
  const float *vb = static_cast<const float *>(a.v) + ci.batch * a.v_sb + hd * a.v_sh + int64_t(ci.t0) * a.v_st;
  {
    // gates: every wave computes the prefix sum (lane = chunk row), wave 0 stores it
    const int64_t row = min(lane, ci.len - 1);
    const float gr = static_cast<const float *>(a.g)[ci.batch * a.g_sb + hd * a.g_sh + (ci.t0 + row) * a.g_st];
    const float br = static_cast<const float *>(a.beta)[ci.batch * a.b_sb + hd * a.b_sh + (ci.t0 + row) * a.b_st];
    TileRows<float, DK, kThreads> rk, rq;
    TileRows<float, DV, kThreads> rv;
    if (vec) {
      rk.fetch(kb, a.k_st, ci.len, DK);
      rq.fetch(qb, a.q_st, ci.len, DK);
      rv.fetch(vb, a.v_st, ci.len, a.dv);
    } else {
      rk.template fetch<false>(kb, a.k_st, ci.len, DK);
      rq.template fetch<false>(qb, a.q_st, ci.len, DK);
      rv.template fetch<false>(vb, a.v_st, ci.len, a.dv);
    }
    float s = lane < ci.len ? gr : 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float y = __shfl_up(s, off, 64);
      if (lane >= off) s += y;
    }
    const float be = lane < ci.len ? br : 0.f;
    if (w == 0) {
      sGam[lane] = s;
      sE[lane] = exp_f(s);
      sKd[lane] = exp_f(__shfl(s, 63, 64) - s);
      sB[lane] = be;
    }
    rk.put(sK, LK, ci.len, DK);
    rq.put(sQ, LK, ci.len, DK);
    __syncthreads();
    rv.put(sV, LV, ci.len, a.dv, [&](int r) { return sB[r]; });  // V' = beta V
  }

  // N = -strict(beta K K^T * D) (waves 0-2) and Attn = (Q K^T) * D (waves 4-6), the lower
  // 32 x 32 tiles (0, 0), (1, 0), (1, 1); the upper right tiles are never read
  if ((w & 3) < 3) {
    const int r0 = (w & 3) ? 32 : 0, c0 = (w & 3) == 2 ? 32 : 0;
    const bool attn = w >= 4;
    const float *sL = attn ? sQ : sK;
    const float *la = sL + (r0 + i) * LK + h, *lb = sK + (c0 + i) * LK + h;
    const f32x16 acc = dot2<DK>([&](int k) { return la[k]; }, [&](int k) { return lb[k]; });
    const int C = c0 + i;
    const float gc = sGam[C];
    float gr[16], x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) gr[r] = sGam[r0 + acc_row32(r, h)];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = attn ? 1.f : -sB[r0 + acc_row32(r, h)];
    float *dst = (attn ? sAt : sN) + r0 * kLT + C;
    const int lim = C - r0 - (attn ? 0 : -1);  // first kept row of the tile
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float d = x[r] * acc[r] * exp_f(gr[r] - gc);
      dst[acc_row32(r, h) * kLT] = acc_row32(r, h) >= lim ? d : 0.f;
    }
  }
  invert_unit_lower64<kLT>(sN, sT, xs);

  // M1 = K~^T T over the dead N, M2 = Attn T (kept in registers until Attn is dead): 32 x 32
  // tiles, T's zero blocks skipped (column tile 1 starts at k = 32; Attn's rows 0-31 end there)
  constexpr int RT1 = DK / 32;
  f32x16 m2;
  int mr = 0, mc = 0;
  const bool has1 = w < 2 * RT1, has2 = w >= 2 * RT1 && w < 2 * RT1 + 3;
  if (has1) {
    mr = 32 * (w >> 1), mc = 32 * (w & 1);
    const float *la = sK + (mc + h) * LK + mr + i, *lb = sT + (mc + h) * kLT + mc + i, *ld = sKd + mc + h;
    auto fa = [&](int k) { return la[k * LK] * ld[k]; };
    auto fb = [&](int k) { return lb[k * kLT]; };
    m2 = mc ? dot2<32>(fa, fb) : dot2<kC>(fa, fb);
#pragma unroll
    for (int r = 0; r < 16; ++r) sN[(mr + acc_row32(r, h)) * kLT + mc + i] = m2[r];
  } else if (has2) {
    const int t = w - 2 * RT1;
    mr = t ? 32 : 0, mc = t == 2 ? 32 : 0;
    const float *la = sAt + (mr + i) * kLT + mc + h, *lb = sT + (mc + h) * kLT + mc + i;
    auto fa = [&](int k) { return la[k]; };
    auto fb = [&](int k) { return lb[k * kLT]; };
    m2 = mr && !mc ? dot2<kC>(fa, fb) : dot2<32>(fa, fb);
  }
  __syncthreads();
  if (has2) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sAt[(mr + acc_row32(r, h)) * kLT + mc + i] = m2[r];
  }
  for (int e = tid; e < kC * DK; e += kThreads) {  // K' = beta e^gamma K
    const int r = e / DK;
    sK[r * LK + e % DK] *= sB[r] * sE[r];
  }
  __syncthreads();

  // [M1; M2] [K' | V']: wave w takes row tile w % RT and its share of the column tiles, all in
  // one k loop (the row operand is read once for them)
  constexpr int RT = RT1 + 2, CT = (DK + DV) / 32, NG = 8 / RT, NCT = (CT + NG - 1) / NG;
  if (w >= RT * NG) return;
  const int rt = w % RT, ct0 = (w / RT) * NCT;
  const bool top = rt < RT1;
  const int row0 = 32 * (top ? rt : rt - RT1);
  const float *mrow = (top ? sN : sAt) + (row0 + i) * kLT;
  const float *colp[NCT];
  int cst[NCT];
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int ct = min(ct0 + c, CT - 1);
    colp[c] = 32 * ct < DK ? sK + 32 * ct + i : sV + 32 * ct - DK + i;
    cst[c] = 32 * ct < DK ? LK : LV;
  }
  f32x16 acc[NCT];
  auto products = [&](auto kc) {
    constexpr int K = decltype(kc)::value;
    f32x16 x[2 * NCT] = {};  // the two halves of the k sum
    mm_pipe<K / 4, 2 * NCT>(x, [&](int p, int s, float &av, float &bv) {
      const int k = (p & 1) * (K / 2) + 2 * s + h;
      av = mrow[k];
      bv = colp[p >> 1][k * cst[p >> 1]];
    });
#pragma unroll
    for (int c = 0; c < NCT; ++c) acc[c] = x[2 * c] + x[2 * c + 1];
  };
  if (top || row0) products(std::integral_constant<int, kC>());
  else products(std::integral_constant<int, 32>());  // M2's rows 0-31 vanish past column 31
  const size_t cell = static_cast<size_t>(hd) * ca.total_chunks + chunk;
  const float ec = sE[kC - 1];
  float *ob = static_cast<float *>(a.o) + ci.batch * a.o_sb + hd * a.o_sh + int64_t(ci.t0) * a.o_st;
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int ct = ct0 + c, col = 32 * ct + i;
    if (ct >= CT) break;
    if (col < DK) {  // (wave-uniform: whole tiles)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int R = row0 + acc_row32(r, h);
        if (top) ws.A[(cell * DK + R) * DK + col] = (R == col ? ec : 0.f) - acc[c][r];
        else ws.Qp[(cell * kC + R) * DK + col] = sQ[R * LK + col] * sE[R] - acc[c][r];
      }
    } else if (col - DK < a.dv) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int R = row0 + acc_row32(r, h);
        if (top) ws.Hn[(cell * DK + R) * a.dv + col - DK] = acc[c][r];
        else if (R < ci.len) ob[int64_t(R) * a.o_st + col - DK] = acc[c][r];  // O' waits in the output
      }
    }
  }
}

// O_n += Q' S_n: a wave per 32 x 32 tile of the chunk's output (rows 32 (w % 2), columns
// 32 (w / 2)), operands straight from global memory in 4-k groups: lane l holds row (or
// column) l % 32 at k = 8 j + 4 (l / 32) + 0..3.  HBM bound (O' and S_n read, O written).
template <int DK>
__global__ void __launch_bounds__(512) gdn_f32_out(GdnArgs a, ChunkArgs ca, F32Ws ws) {
  const int chunk = blockIdx.x, hd = blockIdx.y;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 31, h = lane >> 5, r0 = 32 * (w & 1), c0 = 32 * (w >> 1);
  const ChunkInfo ci = resolve_chunk(chunk, kC, a.L, ca);
  if (c0 >= a.dv || r0 >= ci.len) return;
  const size_t cell = static_cast<size_t>(hd) * ca.total_chunks + chunk;
  const float *qp = ws.Qp + (cell * kC + r0 + i) * DK + 4 * h;
  const float *sn = ws.Hn + (cell * DK + 4 * h) * a.dv + c0 + i;
  float *ob = static_cast<float *>(a.o) + ci.batch * a.o_sb + hd * a.o_sh + int64_t(ci.t0) * a.o_st + c0 + i;
  f32x4 q[DK / 8];
  float s[DK / 2];
#pragma unroll
  for (int j = 0; j < DK / 8; ++j) q[j] = *reinterpret_cast<const f32x4 *>(qp + 8 * j);
#pragma unroll
  for (int j = 0; j < DK / 8; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t) s[4 * j + t] = sn[static_cast<size_t>(8 * j + t) * a.dv];
  float op[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) op[r] = ob[int64_t(min(r0 + acc_row32(r, h), ci.len - 1)) * a.o_st];
  f32x16 acc = {}, acc1 = {};
#pragma unroll
  for (int j = 0; j < DK / 16; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc = mfma32_f32(q[j][t], s[4 * j + t], acc);
      acc1 = mfma32_f32(q[j + DK / 16][t], s[4 * (j + DK / 16) + t], acc1);
    }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int R = r0 + acc_row32(r, h);
    if (R < ci.len) ob[int64_t(R) * a.o_st] = op[r] + (acc[r] + acc1[r]);
  }
}

template <int DK, int DV>
int launch_f32_prep(const GdnArgs &a, const ChunkArgs &ca, const F32Ws &ws, int vec, hipStream_t s) {
  constexpr int smem = F32Lds<DK, DV>::floats * 4;
  auto kern = gdn_f32_prep<DK, DV>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e != hipSuccess) return set_error(MOTIF_ERR_HIP, std::string("gdn_f32_prep smem: ") + hipGetErrorString(e));
  kern<<<dim3(ca.total_chunks, a.H), dim3(kThreads), smem, s>>>(a, ca, ws, vec);
  return check_launch("gdn_f32_prep");
}

}  // namespace

// The MFMA form takes chunk 64, dk 32 / 64 and whole 32-column tiles of dv up to 128; the
// vector kernels of gdn.hip keep the other shapes.
bool chunk_f32_supported(int dk, int dv, int chunk) {
  return chunk == kC && (dk == 32 || dk == 64) && dv % 32 == 0 && dv > 0 && dv <= 128;
}
bool chunk_f32_eligible(const GdnArgs &a, int chunk, const void *workspace) {
  const int64_t lo = std::min({a.q_st, a.k_st, a.v_st}), hi = std::max({a.q_st, a.k_st, a.v_st});
  return chunk_f32_supported(a.dk, a.dv, chunk) && lo >= 0 && hi < kTileMaxStride &&
         (reinterpret_cast<uintptr_t>(workspace) & 15) == 0;
}

size_t chunk_f32_workspace_bytes(int H, int dk, int dv, int total_chunks) {
  return F32Ws::cell_floats(dk, dv) * sizeof(float) * static_cast<size_t>(H) * total_chunks;
}

int launch_chunk_f32(const GdnArgs &a, const ChunkArgs &ca, void *workspace, hipStream_t s) {
  const F32Ws ws(static_cast<float *>(workspace), static_cast<size_t>(a.H) * ca.total_chunks, a.dk, a.dv);
  // 16-byte row loads where every row starts on a 16-byte boundary
  const int64_t st = a.q_sb | a.q_sh | a.q_st | a.k_sb | a.k_sh | a.k_st | a.v_sb | a.v_sh | a.v_st;
  const uintptr_t p = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) | reinterpret_cast<uintptr_t>(a.v);
  const int vec = (st & 3) == 0 && (p & 15) == 0;
  int rc;
  if (a.dk == 64) rc = a.dv <= 64 ? launch_f32_prep<64, 64>(a, ca, ws, vec, s) : launch_f32_prep<64, 128>(a, ca, ws, vec, s);
  else rc = a.dv <= 64 ? launch_f32_prep<32, 64>(a, ca, ws, vec, s) : launch_f32_prep<32, 128>(a, ca, ws, vec, s);
  if (rc) return rc;
  if ((rc = launch_opscan_cells(ws.A, ws.Hn, a.s_in, a.s_out, a.H, ca, a.dk, a.dv, s))) return rc;
  const dim3 grid(ca.total_chunks, a.H), block(4 * a.dv);  // a wave per 32 x 32 tile
  if (a.dk == 64) gdn_f32_out<64><<<grid, block, 0, s>>>(a, ca, ws);
  else gdn_f32_out<32><<<grid, block, 0, s>>>(a, ca, ws);
  return check_launch("gdn_f32_out");
}

}  // namespace motif
