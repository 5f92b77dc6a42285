// Launches of the 16-bit matrix-core GEMM (gemm16.hpp) for nvf_matmul on activations
// and weights of one 16-bit type.

#include <mutex>

#include "gemm16.hpp"

namespace nvf {

template <typename T, typename TO, int BM, int BN, int WM, int WN, int KG, int NS, int OCC>
int launch_tile16(const void* x, const void* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  constexpr int BK = 64;
  constexpr int kLds = KG * NS * (BM + BN) * BK * 2;
  auto kern = gemm16_kernel<T, TO, BM, BN, WM, WN, KG, BK, NS, OCC>;
  static std::once_flag attr_once;
  std::call_once(attr_once, [&] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  });
  const int tiles_n = (int)((n + BN - 1) / BN);
  const int vec_out = aligned16(out) && n % (16 / (int64_t)sizeof(TO)) == 0;
  const dim3 grid((unsigned)(((m + BM - 1) / BM) * tiles_n));
  kern<<<grid, WM * WN * KG * 64, kLds, st>>>(static_cast<const T*>(x), static_cast<const T*>(w),
                                              static_cast<TO*>(out), m, n, k, tiles_n, vec_out);
  return launch_status("dense_gemm (16-bit)");
}

// The tile: the one whose estimated time for a 64-deep K step of the whole output is
// least, from the tiles per CU r = tiles / 256.  Up to one per CU a step takes `alone`
// (the latency of its load, wait and barrier); beyond, tiles whose LDS lets two share a
// CU add `busy` for each further tile per CU, and the others run in whole rounds of
// `busy`.  Measured in us per step at bf16 (launch time / K steps), on:
//   256 x 256      alone 1.60 (300 x 24576 x 4096)   round 1.74 (4096 x 24576 x 4096: 669 us on that box)
//   128 x 128      0.64 (1021 x 3584 x 18944)        + 0.60 (1021 x 37888 x 3584: 345 us)
//   the same, 2 K groups   0.55 (1021 x 3584 x 18944: 163 us against 190)
//   64 x 128       0.41 (200 x 3584 x 18944)         + 0.35 (4096 x 24576 x 4096: 1080 us)
//   64 x 64        0.29 (200 x 3584 x 18944)         + 0.234 (1021 x 37888 x 3584: 485 us)
//   the same, 2 K groups   0.21 (200 x 3584 x 18944: 62 us against 82)
//   64 x 32, 4 K groups    0.14 (64 x 3584 x 3584: 10.6 us)  round 0.145
//   32 x 32, 4 K groups    0.105 (24 x 3584 x 18944: 30.5 us; 24 x 4608 x 3584: 8.3 us)  round 0.16
// Each is the fastest on some sizes: 1021 x 37888 x 3584 288 us at 256 x 256, 345 at 128 x 128; 300 x
// 24576 x 4096 79 us at 64 x 128, 94 to 102 at the others; 24 x 151936 x 4096 215 us at 64 x
// 128, 222 at 32 x 32; 200 x 4608 x 3584 21 us at 64 x 64, 26 at 64 x 128, 38 at 128 x 128.
// Up to 32 rows the weights' stream is what counts, and the 32-row tiles keep more of
// it in flight (weights not in the cache, m = 8): 3584 x 18944 38.6 us at 32 x 32
// against 48.7 at 64 x 32; 37888 x 3584 49.5 us at 32 x 64 (2 K groups, 2 stages: three
// workgroups per CU) against 53.7 at 32 x 32 and 58.2 at 64 x 128.  The widest outputs
// (LM heads) have tiles enough for the choice above.
// (A short K leaves the 32 x 32 tiles' fixed costs bare once a CU runs two of them: 9728 x
// 896 8.2 us against 6.0.)
int gemm16_tile(int64_t m, int64_t n, int64_t k) {
  if (m <= 32 && n < 65536) return n <= 8192 || (n <= 24576 && k >= 2048) ? 7 : 8;
  constexpr struct {
    int bm, bn;
    bool rounds;
    double alone, busy;
  } kTile[8] = {{256, 256, true, 1.60, 1.74}, {128, 128, false, 0.64, 0.60}, {128, 128, true, 0.55, 0.55},
                {64, 128, false, 0.41, 0.35}, {64, 64, false, 0.29, 0.234},  {64, 64, true, 0.21, 0.21},
                {64, 32, true, 0.14, 0.145},  {32, 32, true, 0.105, 0.16}};
  int best = 0;
  double best_t = 0.0;
  for (int i = 0; i < 8; ++i) {
    const int64_t tiles = ((m + kTile[i].bm - 1) / kTile[i].bm) * ((n + kTile[i].bn - 1) / kTile[i].bn);
    if (i > 0 && tiles > INT32_MAX) continue;
    const double r = (double)tiles / 256.0;
    const double t = r <= 1.0          ? kTile[i].alone
                     : kTile[i].rounds ? (double)((tiles + 255) / 256) * kTile[i].busy
                                       : kTile[i].alone + (r - 1.0) * kTile[i].busy;
    if (i == 0 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

template <typename T, typename TO>
int launch_gemm16(const void* x, const void* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  switch (gemm16_tile(m, n, k)) {
    case 0:
      return launch_tile16<T, TO, 256, 256, 2, 4, 1, 2, 2>(x, w, out, m, n, k, st);
    case 1:
      return launch_tile16<T, TO, 128, 128, 2, 2, 1, 2, 2>(x, w, out, m, n, k, st);
    case 2:
      return launch_tile16<T, TO, 128, 128, 2, 2, 2, 2, 2>(x, w, out, m, n, k, st);
    case 3:
      return launch_tile16<T, TO, 64, 128, 2, 2, 1, 3, 2>(x, w, out, m, n, k, st);
    case 4:
      return launch_tile16<T, TO, 64, 64, 2, 2, 1, 4, 2>(x, w, out, m, n, k, st);
    case 5:
      return launch_tile16<T, TO, 64, 64, 2, 2, 2, 4, 2>(x, w, out, m, n, k, st);
    case 6:
      return launch_tile16<T, TO, 64, 32, 2, 1, 4, 3, 2>(x, w, out, m, n, k, st);
    case 8:
      return launch_tile16<T, TO, 32, 64, 1, 2, 2, 2, 3>(x, w, out, m, n, k, st);
    default:
      return launch_tile16<T, TO, 32, 32, 1, 1, 4, 3, 1>(x, w, out, m, n, k, st);
  }
}

int gemm16(const void* x, const void* w, bool bf16, void* out, int out_dtype, int64_t m, int64_t n, int64_t k,
           hipStream_t st) {
  int rc = NVF_OK;
  if (bf16)
    NVF_DISPATCH_DTYPE(out_dtype, TO, rc = (launch_gemm16<__bf16, TO>(x, w, out, m, n, k, st)));
  else
    NVF_DISPATCH_DTYPE(out_dtype, TO, rc = (launch_gemm16<_Float16, TO>(x, w, out, m, n, k, st)));
  return rc;
}

}  // namespace nvf
