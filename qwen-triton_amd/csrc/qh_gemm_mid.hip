// Tile choice and dispatch of the small- and medium-output GEMM (kernel and measurements:
// qh_gemm_mid.h); bf16 products. The other types are in qh_gemm_mid_f16.hip.
#include "qh_gemm_mid_run.h"

int qh_gemm_splitk_count(int64_t M, int64_t N, int64_t K);
int qh_gemm_mid_f16(int v, int ta, int tb, int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb,
                    void* C, int64_t ldc, const void* bias, int out_dtype, hipStream_t st);

// Variant for an M x N output of 16-bit operands, -1 when the 256x256-tile kernel takes it. One
// workgroup per CU: the first tile of the list with at most 256 tiles. Each was the fastest of 16
// tile and wave shapes where the rule takes it (M = 136 .. 4000, N = 1024 .. 6144, K = 1024 .. 6144,
// all layouts); e.g. 2000x1024x1024: 64x128 10.0 us, 64x64 13.7, 128x128 13.2; 4000x1024x3072:
// 128x128 33.2, 64x128 42.2, 256x128 49.1, split-K over 256x256 50.5; 2800x3072x1024: 256x256 29.7,
// 128x128 37.4. Wide outputs of few rows (the LM head of a decode batch) stream their weights over
// several rounds of tiles, where one group of waves and a deeper ring read fastest: 64 x 151936 x 1024
// 65.7 us against 69.7 before, 128 rows 83 against 87.
static int mid_pick(int64_t M, int64_t N) {
  auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (tiles(32, 64) <= 256) return MID_32x64;
  if (tiles(64, 64) <= 256) return MID_64x64;
  if (tiles(64, 128) <= 256) return MID_64x128;
  if (tiles(128, 128) <= 256) return MID_128x128;
  if (tiles(256, 128) <= 256) return MID_256x128;
  if (M >= 256 && N >= 256) return -1;
  return M <= 64 ? MID_STREAM_64x128 : MID_STREAM_128x128;
}

// 16-bit operands, 16-byte aligned along their contiguous dimension. QH_GEMM_MID_NONE: not taken.
int qh_gemm_mid_dispatch(int ta, int tb, int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb,
                         void* C, int64_t ldc, const void* bias, int dtype, int out_dtype, hipStream_t st) {
  const int v = mid_pick(M, N);
  if (v < 0) return QH_GEMM_MID_NONE;
  if (dtype == QH_F16) return qh_gemm_mid_f16(v, ta, tb, M, N, K, A, lda, B, ldb, C, ldc, bias, out_dtype, st);
  return mid_out<bf16_t>(v, ta, tb, M, N, K, A, lda, B, ldb, C, ldc, bias, out_dtype, st);
}

// Several products of 128 to about 1000 rows that share A (q/k/v; gate/up with SiLU-mul), one launch.
// All of the tiles it uses, and those the products take on their own where it is taken, split k over
// two wave groups in the same way, so each output has the bits of the separate products: a product
// that would go to a tile with another split, or whose K would be split over workgroups, keeps its own
// launch. 0: not taken, else the tile.
static int group_pick(int64_t M, int64_t K, int count, const int64_t* N, bool gated) {
  if (M <= 128 || count < 2 || count > kMidProducts) return 0;
  int64_t t64 = 0, t64128 = 0, t128 = 0;
  for (int i = 0; i < count; ++i) {
    if (N[i] <= 0 || N[i] >= (1ll << 31)) return 0;
    const int v = mid_pick(M, N[i]);
    if (v != MID_64x64 && v != MID_64x128 && v != MID_128x128) return 0;
    if (qh_gemm_splitk_count(M, N[i], K) > 1) return 0;
    t64 += ((M + 63) / 64) * ((N[i] + 63) / 64);
    t64128 += ((M + 63) / 64) * ((N[i] + 127) / 128);
    t128 += ((M + 127) / 128) * ((N[i] + 127) / 128);
  }
  if (gated && (count != 2 || N[0] != N[1] || N[0] % 64 != 0)) return 0;
  if (!gated && t64 <= 256) return MID_64x64;
  if (t64128 <= 256) return MID_64x128;
  return t128 <= 256 ? MID_128x128 : 0;
}

extern "C" int64_t qh_gemm_group_ok(int64_t M, int64_t K, int count, const int64_t* N, int gated) {
  return group_pick(M, K, count, N, gated != 0) > 0;
}

template <typename T>
static int group_typed(int v, const T* A, int64_t lda, const void* const* B, const int64_t* ldb, const int64_t* N,
                       void* const* C, const int64_t* ldc, const void* const* bias, int count, bool gated, int M,
                       int K, hipStream_t st) {
  MidGroup<T> g = {};
  const int bn = v == MID_64x64 ? 64 : 128;
  int tiles = 0;
  for (int i = 0; i < kMidProducts; ++i) {
    g.tile0[i] = i < count ? tiles : (1 << 30);
    if (i >= count) continue;
    g.B[i] = (const T*)B[i];
    g.ldb[i] = ldb[i];
    g.C[i] = (T*)C[i];
    g.ldc[i] = ldc[i];
    g.bias[i] = bias ? (const T*)bias[i] : nullptr;
    g.N[i] = (int)N[i];
    tiles += (int)((N[i] + bn - 1) / bn);
  }
  if (gated) {
    const int tn = (int)(N[0] / 64);
    return v == MID_64x128 ? mid_group_run<T, 64, 128, 2, 3, MID_GATED>(A, lda, g, M, K, tn, st)
                           : mid_group_run<T, 128, 128, 2, 2, MID_GATED>(A, lda, g, M, K, tn, st);
  }
  if (v == MID_64x64) return mid_group_run<T, 64, 64, 2, 4, MID_GROUP>(A, lda, g, M, K, tiles, st);
  if (v == MID_64x128) return mid_group_run<T, 64, 128, 2, 3, MID_GROUP>(A, lda, g, M, K, tiles, st);
  return mid_group_run<T, 128, 128, 2, 2, MID_GROUP>(A, lda, g, M, K, tiles, st);
}

extern "C" int qh_gemm_group(int64_t M, int64_t K, const void* A, int64_t lda, int count, const void* const* B,
                             const int64_t* ldb, const int64_t* N, void* const* C, const int64_t* ldc,
                             const void* const* bias, int gated, int dtype, void* stream) {
  QH_CHECK_ARG(K > 0 && K < (1ll << 31) && M < (1ll << 31), "qh_gemm_group: bad shape");
  const int v = group_pick(M, K, count, N, gated != 0);
  QH_CHECK_ARG(v > 0, "qh_gemm_group: shape not served (see qh_gemm_group_ok)");
  QH_CHECK_ARG(dtype == QH_BF16 || dtype == QH_F16, "qh_gemm_group: bf16/f16 only");
  QH_CHECK_ARG(aligned16(A) && lda % 8 == 0 && lda >= K && K % 8 == 0,
               "qh_gemm_group: A must be 16-byte aligned with K, lda multiples of 8");
  QH_CHECK_ARG(lda < kTileMaxLd, "qh_gemm_group: rows of A 2^27 or more elements apart");
  QH_CHECK_ARG(!gated || ldb[0] == ldb[1], "qh_gemm_group: gated products need one weight stride");
  for (int i = 0; i < count; ++i) {
    QH_CHECK_ARG(aligned16(B[i]) && ldb[i] % 8 == 0 && ldb[i] >= K, "qh_gemm_group: product %d: bad B", i);
    QH_CHECK_ARG(ldb[i] < kTileMaxLd, "qh_gemm_group: product %d: rows of B 2^27 or more elements apart", i);
    QH_CHECK_ARG((gated && i == 1) || (C[i] != nullptr && ldc[i] >= N[i]), "qh_gemm_group: product %d: bad C", i);
    QH_CHECK_ARG(!gated || bias == nullptr || bias[i] == nullptr, "qh_gemm_group: gated products take no bias");
  }
  QH_CHECK_ARG(!gated || (ldc[0] % 8 == 0 && aligned16(C[0])), "qh_gemm_group: gated output rows must be 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const int rc = dtype == QH_BF16 ? group_typed<bf16_t>(v, (const bf16_t*)A, lda, B, ldb, N, C, ldc, bias, count,
                                                        gated != 0, (int)M, (int)K, st)
                                  : group_typed<f16_t>(v, (const f16_t*)A, lda, B, ldb, N, C, ldc, bias, count,
                                                       gated != 0, (int)M, (int)K, st);
  if (rc) return rc;
  QH_CHECK_LAUNCH("qh_gemm_group");
  return QH_OK;
}
