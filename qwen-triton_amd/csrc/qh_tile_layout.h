// LDS layouts of the 16-bit GEMM operand tiles, shared by the large-tile and the small-tile kernels:
// direct-to-LDS loads of a tile by NW wavefronts, and the MFMA fragment reads. The layouts and why
// they are free of bank conflicts are described at the top of qh_gemm_tile.hip.
#pragma once

#include "qh_lds.h"
#include "qh_mfma.h"

namespace {

// One lane's 16-byte MFMA operand fragment, and the product of a fragment pair: for fp32 the four
// k's of a lane's chunk go through four 32x32x2 products (k 8 g + i and 8 g + 4 + i in product i).
struct MfmaF32 {
  typedef f32x4 v8;
  static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
};
template <typename T>
using MfmaOf = typename std::conditional<std::is_same<T, float>::value, MfmaF32, Mfma<T>>::type;
template <typename T>
using V8 = typename MfmaOf<T>::v8;

// ---------------------------------------------------------------------------
// LDS tile layouts (BK = k extent of one tile: 32 or 64)
// ---------------------------------------------------------------------------
// "N" tile: ROWS x BK elements. W = 256 / (2 BK) rows share one 256-byte bank
// window, so chunk c of row r is stored at c ^ ((r / W) mod CPR): the 16 rows
// of a 16-lane fragment read then cover every bank exactly once.
template <typename T, int ROWS, int BK, int NW>
struct NTile {
  static constexpr int E = 16 / sizeof(T);  // elements per 16-byte chunk
  static constexpr int ELEMS = ROWS * BK;
  static constexpr int CPR = BK / E;       // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;     // rows per 1 KiB DMA instruction
  static constexpr int W = 16 / CPR;       // rows per 256-byte bank window
  static constexpr int PW = ROWS / RPI / NW;  // DMA instructions per wave
  static_assert(PW >= 1 && (ROWS / RPI) % NW == 0, "tile height");
  static_assert(tile_reach_ok(RPI - 1, kTileMaxLd, sizeof(T)), "lane offset");
  static constexpr int64_t kMaxLdSplit = kTileMaxLdSplit;

  static __device__ __forceinline__ int sw(int r) { return (r / W) & (CPR - 1); }
  // Rows of instruction n are RPI n + lane / CPR with n = wid + NW i; RPI / W
  // is 4 and NW is even, so sw(row) is fixed per lane across instructions.
  static __device__ __forceinline__ uint32_t voff(int64_t ld, int wid) {
    const int lane = threadIdx.x & 63;
    const int rin = lane / CPR, c = (lane % CPR) ^ sw(RPI * wid + rin);
    return (uint32_t)(((int64_t)rin * ld + E * c) * (int64_t)sizeof(T));
  }
  // at(i, k): address of element (tile row i, k). Rows RPI n .. RPI n + RPI-1
  // must share one stride ld. vrows: valid rows; vk: valid k from k0.
  template <class AT>
  static __device__ __forceinline__ void issue(uint32_t lds, const AT& at, int k0, int vrows, int vk, uint32_t vo,
                                               int wid) {
    if (vrows >= ROWS && vk >= BK) {
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        lds_dma16_s(vo, at(RPI * n, k0), lds + (uint32_t)n * 1024u);
      }
    } else {
      // (the empty asm keeps the lane's clamped addresses inside this rarely taken
      // branch: hoisted out of the k-loop they stay live in registers through it)
      int lane = threadIdx.x & 63;
      asm volatile("" : "+v"(lane));
      const int rin = lane / CPR;
      int kc = E * ((lane % CPR) ^ sw(RPI * wid + rin));
      if (kc > vk - E) kc = vk - E;  // vk is a positive multiple of E
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        int r = RPI * n + rin;
        if (r > vrows - 1) r = vrows - 1;
        lds_dma16(at(r, k0 + kc), lds + (uint32_t)n * 1024u);
      }
    }
  }
  // Split roles: wave wid also issues the instructions of wave wid + NW/2, whose
  // rows lie NW/2 RPI rows further on at the same swizzle, so they take the same
  // scalar row address with the lane offset vo2 = vo + shift(ld) (at() linear in the
  // row with stride ld).
  static __device__ __forceinline__ uint32_t shift(int64_t ld) {
    static_assert(tile_reach_ok(RPI - 1 + (NW / 2) * RPI, kMaxLdSplit, sizeof(T)), "lane offset");
    return (uint32_t)((int64_t)(NW / 2) * RPI * ld * (int64_t)sizeof(T));
  }
  template <class AT>
  static __device__ __forceinline__ void issue2(uint32_t lds, const AT& at, int k0, int vrows, int vk, uint32_t vo,
                                                uint32_t vo2, int wid) {
    if (vrows >= ROWS && vk >= BK) {
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        const T* base = at(RPI * n, k0);
        lds_dma16_s(vo, base, lds + (uint32_t)n * 1024u);
        lds_dma16_s(vo2, base, lds + (uint32_t)(n + NW / 2) * 1024u);
      }
    } else {
      issue(lds, at, k0, vrows, vk, vo, wid);
      issue(lds, at, k0, vrows, vk, vo2, wid + NW / 2);
    }
  }
  // Row of the tile that this lane loads in DMA instruction i (its row pointer
  // is fixed for the whole tile when rows are gathered).
  static __device__ __forceinline__ int lane_row(int wid, int i) {
    return RPI * (wid + NW * i) + (int)(threadIdx.x & 63) / CPR;
  }
  // Rows reached through per-lane row pointers (gathered operands): rowp[i] is
  // the lane's row lane_row(wid, i), already clamped to a valid row.
  static __device__ __forceinline__ void issue_rows(uint32_t lds, const T* const (&rowp)[PW], int k0, int vk, int wid) {
    const int lane = threadIdx.x & 63;
    int kc = E * ((lane % CPR) ^ sw(RPI * wid + lane / CPR));
    if (kc > vk - E) kc = vk - E;  // vk is a positive multiple of E
#pragma unroll
    for (int i = 0; i < PW; ++i) lds_dma16(rowp[i] + k0 + kc, lds + (uint32_t)(wid + NW * i) * 1024u);
  }
  // Zero the k chunks at or past vk (all rows); tid: the thread among the tile's 64 NW.
  static __device__ __forceinline__ void zero_k_tail(T* S, int vk, int tid) {
    for (int idx = tid; idx < ROWS * CPR; idx += 64 * NW) {
      const int r = idx / CPR, c = idx % CPR;
      if (E * c >= vk) *reinterpret_cast<uint4*>(S + r * BK + E * (c ^ sw(r))) = make_uint4(0, 0, 0, 0);
    }
  }
  // Fragment of rows r0 .. r0+31 at step kk (the k's of two chunks, one per 32-lane half).
  static __device__ __forceinline__ V8<T> frag(const T* S, int r0, int kk) {
    const int lane = threadIdx.x & 63;
    const int row = r0 + (lane & 31);
    const int ch = (2 * kk + (lane >> 5)) ^ sw(row);
    return *reinterpret_cast<const V8<T>*>(S + row * BK + ch * E);
  }
};

// "T" tile: BK k-rows x COLS elements.
template <typename T, int COLS, int BK, int NW>
struct TTile {
  static_assert(sizeof(T) == 2, "16-bit operands");
  static constexpr int ELEMS = BK * COLS;
  static constexpr int CPR = COLS / 8;   // 16-byte chunks per k-row
  static constexpr int RPI = 64 / CPR;   // k-rows per 1 KiB instruction (64 lanes x 16 bytes)
  static constexpr int NI = BK / RPI;
  static constexpr int PW = NI / NW;
  static constexpr int64_t kMaxLdSplit = kTileMaxLd;
  static_assert(CPR >= 4 && CPR <= 64 && PW >= 1 && NI % NW == 0 && NW * RPI % 4 == 0, "tile width");
  static_assert(tile_reach_ok(RPI - 1, kTileMaxLd, sizeof(T)), "lane offset");
  // A fragment read touches 64 bytes of four k-rows. A k-row of 32 columns is a quarter of a
  // 256-byte bank window, so the four fill it; one of 64 columns is half, so rows kr and kr + 2
  // share banks; a wider one fills it, so all four do.
  static __device__ __forceinline__ int sw(int kr) {
    return CPR == 4 ? 0 : CPR == 8 ? 4 * ((kr >> 1) & 1) : 4 * (kr & 3);
  }

  // k-row of this lane in instruction n is n*RPI + lane/CPR; n = wid + NW i
  // and NW*RPI is a multiple of 4, so (k-row & 3) is fixed per lane and so
  // is its swizzled chunk.
  static __device__ __forceinline__ uint32_t voff(int64_t ld, int wid) {
    const int lane = threadIdx.x & 63;
    const int kin = lane / CPR, slot = lane % CPR;
    const int c = slot ^ sw(wid * RPI + kin);
    return (uint32_t)(((int64_t)kin * ld + 8 * c) * (int64_t)sizeof(T));
  }
  // at(i, k): address of element (tile column i, k). k-rows RPI n .. RPI n +
  // RPI-1 must share one stride ld. vcols: valid columns; vk: valid k-rows.
  template <class AT>
  static __device__ __forceinline__ void issue(uint32_t lds, const AT& at, int k0, int vcols, int vk, uint32_t vo,
                                               int wid) {
    if (vcols >= COLS && vk >= BK) {
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        lds_dma16_s(vo, at(0, k0 + n * RPI), lds + (uint32_t)n * 1024u);
      }
    } else {
      int lane = threadIdx.x & 63;
      asm volatile("" : "+v"(lane));  // (as in NTile::issue)
      const int kin = lane / CPR, slot = lane % CPR;
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        int kr = n * RPI + kin;
        int col = 8 * (slot ^ sw(kr));
        if (col > vcols - 8) col = vcols - 8;  // vcols is a positive multiple of 8
        if (kr > vk - 1) kr = vk - 1;
        lds_dma16(at(col, k0 + kr), lds + (uint32_t)n * 1024u);
      }
    }
  }
  // Split roles (as NTile::issue2): the instructions of wave wid + NW/2 read the
  // k-rows NW/2 RPI further on at the same swizzle.
  static __device__ __forceinline__ uint32_t shift(int64_t ld) {
    static_assert(tile_reach_ok(RPI - 1 + (NW / 2) * RPI, kMaxLdSplit, sizeof(T)), "lane offset");
    return (uint32_t)((int64_t)(NW / 2) * RPI * ld * (int64_t)sizeof(T));
  }
  template <class AT>
  static __device__ __forceinline__ void issue2(uint32_t lds, const AT& at, int k0, int vcols, int vk, uint32_t vo,
                                                uint32_t vo2, int wid) {
    if (vcols >= COLS && vk >= BK) {
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int n = wid + NW * i;
        const T* base = at(0, k0 + n * RPI);
        lds_dma16_s(vo, base, lds + (uint32_t)n * 1024u);
        lds_dma16_s(vo2, base, lds + (uint32_t)(n + NW / 2) * 1024u);
      }
    } else {
      issue(lds, at, k0, vcols, vk, vo, wid);
      issue(lds, at, k0, vcols, vk, vo2, wid + NW / 2);
    }
  }
  static __device__ __forceinline__ void zero_k_tail(T* S, int vk, int tid) {
    for (int idx = tid; idx < BK * CPR; idx += 64 * NW) {
      const int kr = idx / CPR;
      if (kr >= vk) *reinterpret_cast<uint4*>(S + idx * 8) = make_uint4(0, 0, 0, 0);
    }
  }
  // Fragment of rows (tile columns) r0 .. r0+31 at k16 step kk.
  static __device__ __forceinline__ V8<T> frag(const T* S, int r0, int kk) {
    const int lane = threadIdx.x & 63;
    const int grp = lane >> 4, j = lane & 15;
    const int m = r0 + 16 * (grp & 1) + 4 * (j & 3);
    const int kr0 = 16 * kk + 8 * (grp >> 1) + (j >> 2);
    const int kr1 = kr0 + 4;
    const T* s0 = S + kr0 * COLS + 8 * ((m >> 3) ^ sw(kr0)) + (m & 7);
    const T* s1 = S + kr1 * COLS + 8 * ((m >> 3) ^ sw(kr1)) + (m & 7);
    const qh_v4i16 w0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) qh_v4i16*)(s0));
    const qh_v4i16 w1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) qh_v4i16*)(s1));
    const qh_v8i16 w = __builtin_shufflevector(w0, w1, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(V8<T>, w);
  }
};

// "T" tile of fp32: BK k-rows x COLS elements. A lane's four k's 8 g + 4 (lane / 32) + i are four
// 4-byte reads; the 32-lane halves read k-rows 4 apart, which must lie in different halves of the
// 256-byte bank window: for rows of 64 or 128 columns chunk c of k-row kr is stored at
// c ^ 8((kr >> 2) & 1); for rows of 32 columns (half a window) the k-rows of a group of 8 are
// stored in the order 0 4 1 5 2 6 3 7, so rows 4 apart are neighbours.
template <int COLS, int BK, int NW>
struct TTileF32 {
  static constexpr int ELEMS = BK * COLS;
  static constexpr int CPR = COLS / 4;
  static constexpr int RPI = 64 / CPR;  // k-rows per 1 KiB instruction
  static constexpr int NI = BK / RPI;
  static constexpr int PW = NI / NW;
  static_assert((CPR == 8 || CPR == 16 || CPR == 32) && PW >= 1 && NI % NW == 0, "tile width");
  static __device__ __forceinline__ int sw(int kr) { return CPR == 8 ? 0 : 8 * ((kr >> 2) & 1); }
  // k-row stored at line `line` of the tile (an involution is not needed: pos() is its inverse)
  static __device__ __forceinline__ int krow(int line) {
    return CPR == 8 ? (line & ~7) + 4 * (line & 1) + ((line >> 1) & 3) : line;
  }
  static __device__ __forceinline__ int pos(int kr) {
    return CPR == 8 ? (kr & ~7) + 2 * (kr & 3) + ((kr >> 2) & 1) : kr;
  }
  // (the swizzle of a line depends on the instruction, so the loads take per-lane addresses)
  static __device__ __forceinline__ uint32_t voff(int64_t, int) { return 0; }
  template <class AT>
  static __device__ __forceinline__ void issue(uint32_t lds, const AT& at, int k0, int vcols, int vk, uint32_t,
                                               int wid) {
    const int lane = threadIdx.x & 63;
    const int lin = lane / CPR, slot = lane % CPR;
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int n = wid + NW * i;
      int kr = krow(n * RPI + lin);
      int col = 4 * (slot ^ sw(kr));
      if (col > vcols - 4) col = vcols - 4;  // vcols is a positive multiple of 4
      if (kr > vk - 1) kr = vk - 1;
      lds_dma16(at(col, k0 + kr), lds + (uint32_t)n * 1024u);
    }
  }
  static __device__ __forceinline__ void zero_k_tail(float* S, int vk, int tid) {
    for (int idx = tid; idx < BK * CPR; idx += 64 * NW)
      if (krow(idx / CPR) >= vk) *reinterpret_cast<uint4*>(S + idx * 4) = make_uint4(0, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 frag(const float* S, int r0, int g) {
    const int lane = threadIdx.x & 63;
    const int col = r0 + (lane & 31);
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kr = 8 * g + 4 * (lane >> 5) + i;
      v[i] = S[pos(kr) * COLS + 4 * ((col >> 2) ^ sw(kr)) + (col & 3)];
    }
    return v;
  }
};

template <typename T, int ROWS, int BK, int NW>
struct TTileOf {
  typedef TTile<T, ROWS, BK, NW> type;
};
template <int ROWS, int BK, int NW>
struct TTileOf<float, ROWS, BK, NW> {
  typedef TTileF32<ROWS, BK, NW> type;
};

template <typename T, int ROWS, int BK, bool TR, int NW>
using OpTile = typename std::conditional<TR, typename TTileOf<T, ROWS, BK, NW>::type, NTile<T, ROWS, BK, NW>>::type;

}  // namespace
