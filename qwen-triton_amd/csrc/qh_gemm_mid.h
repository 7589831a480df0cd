// MFMA GEMM for outputs of at most one small or medium tile per CU, and fp32 products.
//
// C[M,N] = A(M,K) B(N,K)^T (+ bias), each operand k-contiguous ("N") or k-outer ("T"): the products
// of prompts, small training batches and weight gradients of a few hundred to a few thousand tokens,
// whose outputs are too small for 256x256 tiles, and every product of 128 rows or fewer that the
// decode kernels do not take.
//
// What bounds it: a CU takes in 64 bytes of operands per clock from L2 and multiplies 4096 bf16 flop
// per clock, so a BM x BN tile needs (BM + BN) / 32 clocks of loads and BM BN / 2048 of MFMA per k:
// below 128 x 128 the loads are longer, and one workgroup on its own also waits for its barriers.
//  * The tile is the smallest of 32x64 .. 256x128 whose count is at most 256, one workgroup per CU
//    (the rule is in mid_pick, qh_gemm_mid.hip): more, smaller tiles load more bytes for the same
//    output, fewer leave CUs idle.
//  * WK groups of WM x WN wavefronts split the tile's k-tiles between them, each with its own ring of
//    NS LDS stages filled by direct-to-LDS loads NS - 1 k-tiles ahead. A round's loads are thus in
//    flight for WK k-tiles at once and a group's LDS reads overlap another's MFMAs, without which a
//    64x64 tile took 0.44 us per k-tile of 64 and now takes 0.27. The groups' sums are added through
//    LDS in a fixed order.
//  * 16-bit rows leave through LDS as 16-byte stores.
// fp32 operands go through the same kernel: a 16-byte chunk is then 4 k's and a fragment pair four
// v_mfma_f32_32x32x2_f32 (fp32 products and sums, 256 flop per clock and CU, twice the unpacked
// vector ALU's rate), which bounds them.
//
// Measured, us per launch replayed from a graph over distinct buffers, with the 128x128-tile kernel
// (fp32: vector ALU kernel) that took these products before: bf16 517x1024x1024 18.4 -> 7.4,
// 517x3072x1024 18.8 -> 9.8, 2000x1024x3072 38.9 -> 22.1; input gradient 517x2048x1024 28.8 -> 9.7;
// weight gradient 1024x3072 of 2000 rows 74.3 -> 22.5, of 200 rows 15.1 -> 8.2; fp32 384x1024x3072
// 439 -> 36, 384x3072x1024 193 -> 33, its weight gradient 79 -> 29 (83 of 157 TFLOP/s).
#pragma once

#include "qh_lds_limit.h"
#include "qh_tile_layout.h"

namespace {

// Products that share A in one launch. MID_GROUP: tile column tn belongs to the last product i with
// tile0[i] <= tn. MID_GATED: B[0] and B[1] (gate and up, equal N, a multiple of 64) alternate in blocks
// of 32 weight rows, so a wavefront's two column blocks are the same columns of both and its lanes
// write C[0] = silu(gate) * up, each product rounded first.
enum { MID_ONE, MID_GROUP, MID_GATED };
constexpr int kMidProducts = 3;
template <typename T>
struct MidGroup {
  const T* B[kMidProducts];
  int64_t ldb[kMidProducts];
  T* C[kMidProducts];
  int64_t ldc[kMidProducts];
  const T* bias[kMidProducts];
  int N[kMidProducts], tile0[kMidProducts];
};

template <typename T, typename OT, int BM, int BN, int WM, int WN, int WK, int NS, bool AT, bool BT, int MODE = MID_ONE>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_mid_kernel(const T* __restrict__ A, int64_t lda,
                                                                     const T* __restrict__ B, int64_t ldb,
                                                                     OT* __restrict__ C, int64_t ldc,
                                                                     const T* __restrict__ bias, int M, int N, int K,
                                                                     int tiles_m, int tiles_n, MidGroup<T> grp) {
  static_assert(MODE == MID_ONE || (!AT && !BT && std::is_same<T, OT>::value), "grouped products: forward layout");
  static_assert(MODE != MID_GATED || (BN == 128 && WN == 2), "gated tiles: a wavefront holds one block of each");
  constexpr int NW = WM * WN, BK = 128 / (int)sizeof(T), KS = 4;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
  using TA = OpTile<T, BM, BK, AT, NW>;
  using TB = OpTile<T, BN, BK, BT, NW>;
  constexpr int STAGE = TA::ELEMS + TB::ELEMS;
  constexpr int NPT = TA::PW + TB::PW;  // DMA instructions per wave and k-tile
  static_assert((NS - 1) * NPT <= 63 && NS <= 4, "vmcnt");
  extern __shared__ __attribute__((aligned(1024))) unsigned char qh_mid_smem[];

  int tm, tn;
  tile_order(tiles_m, tiles_n, tm, tn);
  if constexpr (MODE == MID_GROUP) {
    const int i = (tn >= grp.tile0[1]) + (tn >= grp.tile0[2]);
    B = grp.B[i], ldb = grp.ldb[i], C = grp.C[i], ldc = grp.ldc[i], bias = grp.bias[i], N = grp.N[i];
    tn -= grp.tile0[i];
  }
  constexpr int OBN = MODE == MID_GATED ? BN / 2 : BN;  // output columns of a tile
  const int m0 = tm * BM, n0 = tn * OBN;
  const int vm = M - m0, vn = MODE == MID_GATED ? BN : N - n0;
  const int lane = threadIdx.x & 63;
  const int wg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ks = wg / NW, wid = wg % NW;  // k slice, wavefront in it
  const int wm = wid / WN, wn = wid % WN;
  T* smem = reinterpret_cast<T*>(qh_mid_smem) + ks * (NS * STAGE);  // the slice's stages
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t voa = TA::voff(lda, wid), vob = TB::voff(ldb, wid);
  auto a_at = [&](int i, int k) { return AT ? A + (int64_t)k * lda + (m0 + i) : A + (int64_t)(m0 + i) * lda + k; };
  auto b_at = [&](int i, int k) {
    if constexpr (MODE == MID_GATED)
      return ((i >> 5) & 1 ? grp.B[1] : B) + (int64_t)(n0 + ((i >> 6) << 5) + (i & 31)) * ldb + k;
    return BT ? B + (int64_t)k * ldb + (n0 + i) : B + (int64_t)(n0 + i) * ldb + k;
  };
  // slice ks takes k-tiles ks, ks + WK, ...: its t-th is k-tile ks + WK t
  auto issue = [&](int t) {
    const int k0 = (ks + WK * t) * BK;
    const uint32_t base = lds0 + (uint32_t)((t % NS) * STAGE * (int)sizeof(T));
    TA::issue(base, a_at, k0, vm, K - k0, voa, wid);
    TB::issue(base + (uint32_t)(TA::ELEMS * sizeof(T)), b_at, k0, vn, K - k0, vob, wid);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = zero16();

  const int nkt = (K + BK - 1) / BK;
  const int nr = (nkt + WK - 1) / WK;        // rounds of the workgroup
  const int nk = (nkt - ks + WK - 1) / WK;   // k-tiles of this slice: nr or nr - 1
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nk) issue(t);
  for (int t = 0; t < nr; ++t) {
    // k-tiles issued after t: min(NS - 2, nk - 1 - t)
    const int after = nk - 1 - t;
    if (NS > 3 && after >= 2) __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * NPT));
    else if (NS > 2 && after >= 1) __builtin_amdgcn_s_waitcnt(waitcnt_vm(NPT));
    else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __syncthreads();  // round t's k-tiles are in LDS for every wave, and every wave has read round t - 1's
    T* S = smem + (t % NS) * STAGE;
    if (K - WK * t * BK < WK * BK) {  // (uniform) the round with the last k-tile: K may end inside one
      const int vk = K - (ks + WK * t) * BK;
      if (vk > 0 && vk < BK) {
        TA::zero_k_tail(S, vk, threadIdx.x % (64 * NW));
        TB::zero_k_tail(S + TA::ELEMS, vk, threadIdx.x % (64 * NW));
      }
      __syncthreads();
      if (vk <= 0) break;  // no k-tile for this slice in the last round
    }
    if (t + NS - 1 < nk) issue(t + NS - 1);  // into the stage of round t - 1
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      V8<T> af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = TA::frag(S, wm * WTM + 32 * i, kk);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = TB::frag(S + TA::ELEMS, wn * WTN + 32 * j, kk);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MfmaOf<T>::mma(af[i], bf[j], acc[i][j]);
    }
  }

  if constexpr (WK > 1) {
    // the slices' sums, added in slice order by slice 0
    constexpr int WAVE = TM * TN * 16 * 64;
    float* R = reinterpret_cast<float*>(qh_mid_smem);
    static_assert((WK - 1) * NW * WAVE * 4 <= WK * NS * STAGE * (int)sizeof(T), "partial sums");
    __syncthreads();  // every wave is done with the operand stages
    if (ks > 0) {
      float* P = R + ((ks - 1) * NW + wid) * WAVE + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) P[((i * TN + j) * 16 + e) * 64] = acc[i][j][e];
    }
    __syncthreads();
    if (ks == 0)
#pragma unroll
    for (int s = 0; s < WK - 1; ++s) {
      const float* P = R + (s * NW + wid) * WAVE + lane;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] += P[((i * TN + j) * 16 + e) * 64];
    }
  }

  if constexpr (sizeof(OT) == 2) {
    // 16-byte row stores through LDS (rows of BN + 8 elements keep the staging writes of rows r and
    // r + 4 in different banks)
    if ((N & 7) == 0 && (ldc & 7) == 0 && ((uintptr_t)C & 15) == 0) {
      constexpr int LD = OBN + 8;
      static_assert(BM * LD * (int)sizeof(OT) <= WK * NS * STAGE * (int)sizeof(T), "staged tile");
      OT* E = reinterpret_cast<OT*>(qh_mid_smem);
      __syncthreads();  // every wave is done with the operand stages and the partial sums
      if (MODE == MID_GATED && ks == 0) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float gt = to_f32((T)acc[i][0][4 * g + r]), up = to_f32((T)acc[i][TN - 1][4 * g + r]);
              E[(wm * WTM + 32 * i + 4 * (lane >> 5) + 8 * g + r) * LD + 32 * wn + (lane & 31)] =
                  from_f32<OT>(gt * sigmoidf_(gt) * up);
            }
      } else if (ks == 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int cl = wn * WTN + 32 * j + (lane & 31);
          const float bv = bias && n0 + cl < N ? to_f32(bias[n0 + cl]) : 0.f;
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                E[(wm * WTM + 32 * i + 4 * (lane >> 5) + 8 * g + r) * LD + cl] =
                    from_f32<OT>(acc[i][j][4 * g + r] + bv);
        }
      }
      __syncthreads();
      constexpr int CPR = OBN / 8, NTH = 64 * NW * WK, NV = (BM * CPR + NTH - 1) / NTH;
      Vec16<OT> v[NV];
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int idx = threadIdx.x + NTH * u;
        if (BM * CPR % NTH == 0 || idx < BM * CPR) v[u] = ld16(E + (idx / CPR) * LD + 8 * (idx % CPR));
      }
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int idx = threadIdx.x + NTH * u;
        const int r = idx / CPR, c = 8 * (idx % CPR);
        if (r < vm && r < BM && (MODE == MID_GATED || c < vn)) st16(C + (int64_t)(m0 + r) * ldc + n0 + c, v[u]);
      }
      return;
    }
  }
  if (MODE == MID_GATED || ks > 0) return;  // (gated products always have 16-byte rows)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + wn * WTN + 32 * j + (lane & 31);
    if (col >= N) continue;
    const float bv = bias ? to_f32(bias[col]) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r0 = m0 + wm * WTM + 32 * i + 4 * (lane >> 5);
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (r0 + 8 * g + r < M) C[(int64_t)(r0 + 8 * g + r) * ldc + col] = from_f32<OT>(acc[i][j][4 * g + r] + bv);
    }
  }
}

template <typename T, typename OT, int BM, int BN, int WM, int WN, int WK, int NS, bool AT, bool BT>
int mid_run(const T* A, int64_t lda, const T* B, int64_t ldb, OT* C, int64_t ldc, const T* bias, int M, int N, int K,
            hipStream_t st) {
  constexpr int lds = WK * NS * (BM + BN) * 128;
  static_assert(lds <= 160 * 1024, "LDS");
  auto* kern = gemm_mid_kernel<T, OT, BM, BN, WM, WN, WK, NS, AT, BT>;
  static qh::LdsLimit limit;
  if (const int rc = limit.raise(reinterpret_cast<const void*>(kern), lds, "qh_gemm")) return rc;
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  kern<<<(unsigned)(tm * tn), 64 * WM * WN * WK, lds, st>>>(A, lda, B, ldb, C, ldc, bias, M, N, K, tm, tn, MidGroup<T>{});
  return QH_OK;
}

template <typename T, int BM, int BN, int WK, int NS, int MODE>
int mid_group_run(const T* A, int64_t lda, const MidGroup<T>& grp, int M, int K, int tiles_n, hipStream_t st) {
  constexpr int lds = WK * NS * (BM + BN) * 128;
  auto* kern = gemm_mid_kernel<T, T, BM, BN, 2, 2, WK, NS, false, false, MODE>;
  static qh::LdsLimit limit;
  if (const int rc = limit.raise(reinterpret_cast<const void*>(kern), lds, "qh_gemm_group")) return rc;
  const int tm = (M + BM - 1) / BM;
  kern<<<(unsigned)(tm * tiles_n), 64 * 4 * WK, lds, st>>>(A, lda, grp.B[0], grp.ldb[0], grp.C[0], grp.ldc[0], nullptr,
                                                           M, grp.N[0], K, tm, tiles_n, grp);
  return QH_OK;
}

template <typename T, typename OT, int BM, int BN, int WM, int WN, int WK, int NS>
int mid_layout(int ta, int tb, const T* A, int64_t lda, const T* B, int64_t ldb, OT* C, int64_t ldc, const T* bias,
               int M, int N, int K, hipStream_t st) {
#define QH_MID_GO(AT, BT) mid_run<T, OT, BM, BN, WM, WN, WK, NS, AT, BT>(A, lda, B, ldb, C, ldc, bias, M, N, K, st)
  if (!ta && !tb) return QH_MID_GO(false, false);
  if (!ta && tb) return QH_MID_GO(false, true);
  if (ta && tb) return QH_MID_GO(true, true);
  return QH_MID_GO(true, false);
#undef QH_MID_GO
}

}  // namespace
