// GEMM on K-quant weights (Q4_K, Q5_K, Q6_K) with 16-bit activations on the 16-bit
// matrix cores: out[m][n] = x[m][k] . W[n][k]^T, k a multiple of 256 (whole superblocks
// per weight row), m > 16.
//
// A weight of a superblock is d sc_j q - dmin m_j with 6-bit whole sc_j, m_j of its sub-block and
// a whole q.  With the sub-block's centre c_j (kq_centre: the quant nearest to where the weight
// is 0) it is d sc_j (q - c_j) + r_j, r_j = d sc_j c_j - dmin m_j in fp32; Q6_K is d sc_j (q - 32),
// sc_j signed 8-bit.  The integer P = sc_j (q - c_j) has at most 11 significant bits (Q6_K 13), so
// it is one fp16 value exactly, or the exact sum of two 16-bit values.  Per superblock the matrix
// cores sum
//   B = sum_k x_k P_k                (exact products, fp32 sums)
//   R = sum_j r_j (sum_{k in j} x_k) (the sub-block sums of x and the r_j as three bf16 pieces
//                                    each, the six products down to 2^-24 of the largest)
// and the accumulator takes R, and d B by one fused multiply-add per output and 256 K, where a
// scale per sub-block would cost one per 32 K and decoding each weight to fp32
// leaves only the fp32 matrix cores, 16 times slower.  P and r_j are at most twice and once
// their weight, so the result is within three times the bound of fp32 sums of x w.
//
// 1021 x 37888 x 3584, fp16 x, Q4_K: the fp32 matrix-core tile kernel takes 2487 us (111
// TFLOP/s), this one 407 (681; 399 with c_j = 0, whose two parts can cancel: then the error is
// bounded by sums of |x| (d sc q + dmin m) alone; 421 with the centres found behind the products).
// Activations reach LDS by DMA; a weight stage is loaded to registers two stages ahead,
// decoded once per workgroup and stored to LDS as 16-bit operands.
//
// Infinities and NaN: x and P are multiplied apart from the weight's scale and offset, so a
// non-finite activation or superblock scale (or an activation beyond 1e35) can give NaN
// where the plain product has an infinity or a number.  Any of them leaves the output
// non-finite, and such outputs are made again from the decoded weights on the fp32 matrix
// cores, by the waves that hold them (1021 x 4096 x 3584, every activation NaN: 13.8 ms one
// output after the other, 520 us so, 315 on the fp32 tile kernel).

#include <array>
#include <mutex>
#include <type_traits>

#include "gemm16.hpp"
#include "gemm_tile.hpp"

namespace nvf {

constexpr int kKqBN = 128, kKqBK = 64;

// One stage of one thread: NB bytes of quants of column c, part p of its 64 K values.  Head is
// what a superblock's four stages share, loaded once for them: read again in every
// stage, the compiler merges it with the older copy and waits for the newest load.  run() gives (8 integers q as
// bytes, chunk, scale index).
template <int KIND, int LAYOUT, int NB>
struct KqRaw;

template <int LAYOUT, int NB>
struct KqRaw<NVF_Q4_K, LAYOUT, NB> {
  static constexpr int kBlock = 144;
  struct Head {
    u32x4 w;
    __device__ __forceinline__ void load(const uint8_t* blk, int) { w = ld16(blk); }
  } hd;
  uint32_t q[NB / 4];
  __device__ __forceinline__ void load(const uint8_t* blk, int quarter, int part) {
    const uint8_t* p = blk + 16 + 32 * quarter + NB * part;
    if constexpr (NB == 16) {
      const u32x4 v = ld16(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = v[i];
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      q[0] = v.x;
      q[1] = v.y;
    }
  }
  // run r (8 values) of this thread: its bytes, its chunk of the stage, its sub-block
  static constexpr int kRuns = NB / 4;
  __device__ __forceinline__ void run(int r, int quarter, int part, uint32_t* b, int& chunk, int& j) const {
    const int u = r >> 1, nib = r & 1, byte8 = part * (NB / 8) + u;  // the 8-byte group and the nibble
    b[0] = (q[2 * u] >> (4 * nib)) & 0x0f0f0f0fu;
    b[1] = (q[2 * u + 1] >> (4 * nib)) & 0x0f0f0f0fu;
    if constexpr (LAYOUT == NVF_QK_LAYOUT_GGML) {  // element 64 p + 32 nib + k
      chunk = 4 * nib + byte8;
      j = 2 * quarter + nib;
    } else {  // element 32 j + 16 nib + k is byte 16 j + k
      chunk = 4 * (byte8 >> 1) + 2 * nib + (byte8 & 1);
      j = 2 * quarter + (byte8 >> 1);
    }
  }
  __device__ __forceinline__ void scale_min(int j, uint32_t& sc, uint32_t& mn) const {
    q4k_sm(hd.w[1], hd.w[2], hd.w[3], j, sc, mn);
  }
  __device__ __forceinline__ float d() const { return half_bits_to_f32(hd.w[0] & 0xffffu); }
  __device__ __forceinline__ float dmin() const { return half_bits_to_f32(hd.w[0] >> 16); }
};

template <int LAYOUT, int NB>
struct KqRaw<NVF_Q5_K, LAYOUT, NB> {
  static constexpr int kBlock = 176;
  struct Head {
    u32x4 w;
    uint32_t h[NB / 4];
    __device__ __forceinline__ void load(const uint8_t* blk, int part) {
      w = ld16(blk);
      const uint8_t* p = blk + 16 + NB * part;
      if constexpr (NB == 16) {
        const u32x4 g = ld16(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = g[i];
      } else {
        const uint2 g = *reinterpret_cast<const uint2*>(p);
        h[0] = g.x;
        h[1] = g.y;
      }
    }
  } hd;
  uint32_t q[NB / 4];
  __device__ __forceinline__ void load(const uint8_t* blk, int quarter, int part) {
    const uint8_t* p = blk + 48 + 32 * quarter + NB * part;
    if constexpr (NB == 16) {
      const u32x4 v = ld16(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = v[i];
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      q[0] = v.x;
      q[1] = v.y;
    }
  }
  static constexpr int kRuns = NB / 4;
  __device__ __forceinline__ void run(int r, int quarter, int part, uint32_t* b, int& chunk, int& j) const {
    const int u = r >> 1, nib = r & 1;
    chunk = 4 * nib + part * (NB / 8) + u;
    j = 2 * quarter + nib;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      b[i] = ((q[2 * u + i] >> (4 * nib)) & 0x0f0f0f0fu) | (((hd.h[2 * u + i] >> j) & 0x01010101u) << 4);
  }
  __device__ __forceinline__ void scale_min(int j, uint32_t& sc, uint32_t& mn) const {
    q4k_sm(hd.w[1], hd.w[2], hd.w[3], j, sc, mn);
  }
  __device__ __forceinline__ float d() const { return half_bits_to_f32(hd.w[0] & 0xffffu); }
  __device__ __forceinline__ float dmin() const { return half_bits_to_f32(hd.w[0] >> 16); }
};

template <int NB>
__device__ __forceinline__ void kq_load_a2(const uint8_t* p, uint32_t* out) {  // NB bytes at a 2-byte aligned address
#pragma unroll
  for (int i = 0; i < NB / 8; ++i) load_a2<8>(p + 8 * i, out + 2 * i);
}

template <int LAYOUT, int NB>
struct KqRaw<NVF_Q6_K, LAYOUT, NB> {  // element 128 h + 32 s + l: ql[64 h + 32 (s & 1) + l] nibble s / 2, qh[32 h + l]
  static constexpr int kBlock = 210;
  struct Head {  // its header bytes differ between the stages
    __device__ __forceinline__ void load(const uint8_t*, int) {}
  } hd;
  uint32_t q[2][NB / 4], h[NB / 4];
  uint32_t sc[2];  // the int8 scales of slots s = 2 (quarter & 1), + 1 at this thread's l
  uint32_t dbits;
  __device__ __forceinline__ void load(const uint8_t* blk, int quarter, int part) {
    const int half = quarter >> 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      kq_load_a2<NB>(blk + 64 * half + 32 * s + NB * part, q[s]);
      sc[s] = blk[192 + 8 * half + 2 * (2 * (quarter & 1) + s) + (NB * part >= 16 ? 1 : 0)];
    }
    kq_load_a2<NB>(blk + 128 + 32 * half + NB * part, h);
    dbits = *reinterpret_cast<const uint16_t*>(blk + 208);
  }
  static constexpr int kRuns = NB / 4;
  __device__ __forceinline__ void run(int r, int quarter, int part, uint32_t* b, int& chunk, int& j) const {
    const int u = r >> 1, s = r & 1, nib = quarter & 1, slot = 2 * nib + s;
    chunk = 4 * s + part * (NB / 8) + u;
    j = s;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      b[i] = ((q[s][2 * u + i] >> (4 * nib)) & 0x0f0f0f0fu) | (((h[2 * u + i] >> (2 * slot)) & 0x03030303u) << 4);
  }
  __device__ __forceinline__ void scale_min(int j, uint32_t& s, uint32_t& mn) const {
    s = sc[j];
    mn = 0;
  }
  __device__ __forceinline__ float d() const { return half_bits_to_f32(dbits); }
  __device__ __forceinline__ float dmin() const { return 0.0f; }
};

// 16-bit operand planes of 8 integers P = sc (q - q0) (Q6_K: sc (q - 32), sc signed), the q as
// bytes and q0 the sub-block's centre: the planes sum to P exactly.
template <typename T, int KIND>
struct KqPlanes {
  static constexpr int value = __is_same(T, _Float16) && KIND != NVF_Q6_K ? 1 : 2;
};
// 1 / the planes' unit.
template <typename T, int KIND>
constexpr float kKqUnit = __is_same(T, _Float16) && KIND != NVF_Q6_K ? 0x1p14f : 1.0f;
template <int KIND>
__device__ __forceinline__ void kq_planes(const uint32_t* b, uint32_t sc, uint32_t q0, u32x4* p, _Float16) {
  // Q4_K, Q5_K: a byte under a zero one is the subnormal q 2^-24, and one exact multiply-add
  // makes it sc (q - q0) 2^-14.  Q6_K: bytes under 0x64 are the fp16 values 1024 + q.
  const uint32_t top = KIND == NVF_Q6_K ? 0x64646464u : 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = b[i >> 1];
    const f16x2 t = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(top, w, (i & 1) ? 0x07030602u : 0x05010400u));
    if constexpr (KIND == NVF_Q6_K) {
      const int s = (int8_t)sc, lo = s & 15, hi = s - lo;  // s = hi + lo, hi a multiple of 16
      const f16x2 q = t - f16x2{(_Float16)1056.0f, (_Float16)1056.0f};
      const f16x2 l2 = {(_Float16)(float)lo, (_Float16)(float)lo}, h2 = {(_Float16)(float)hi, (_Float16)(float)hi};
      p[0][i] = __builtin_bit_cast(uint32_t, q * h2);
      p[1][i] = __builtin_bit_cast(uint32_t, q * l2);
    } else {
      const _Float16 s = (_Float16)(1024.0f * (float)sc), c = (_Float16)(-0x1p-14f * (float)sc * (float)q0);
      const f16x2 s2 = {s, s}, c2 = {c, c};
      p[0][i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(t, s2, c2));
    }
  }
}
template <int KIND>
__device__ __forceinline__ void kq_planes(const uint32_t* b, uint32_t sc, uint32_t q0, u32x4* p, __bf16) {
  const float s = KIND == NVF_Q6_K ? (float)(int8_t)sc : (float)sc, c = s * (KIND == NVF_Q6_K ? -32.0f : -(float)q0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t hi[2], lo[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float v = fmaf((float)byte_of(b[i >> 1], 2 * (i & 1) + e), s, c);  // a whole number below 2^13
      hi[e] = __builtin_bit_cast(uint32_t, v) & 0xffff0000u;
      lo[e] = __builtin_bit_cast(uint32_t, v - __builtin_bit_cast(float, hi[e]));  // at most 8 bits: exact in bf16
    }
    p[0][i] = (hi[0] >> 16) | hi[1];
    p[1][i] = (lo[0] >> 16) | (lo[1] & 0xffff0000u);
  }
}

// The weights one by one (8 at a time).
template <int KIND, int LAYOUT>
struct KqPlain : Q4K<8, LAYOUT> {};
template <int LAYOUT>
struct KqPlain<NVF_Q5_K, LAYOUT> : Q5K<8> {};
template <int LAYOUT>
struct KqPlain<NVF_Q6_K, LAYOUT> : Q6K<8> {};

// Sum of 8 16-bit values, added to s in order.
__device__ __forceinline__ float kq_sum8(u32x4 v, float s, _Float16) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = v[i];
    const f16x2 h = __builtin_bit_cast(f16x2, w);
    s += (float)h[0];
    s += (float)h[1];
  }
  return s;
}
__device__ __forceinline__ float kq_sum8(u32x4 v, float s, __bf16) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s += __builtin_bit_cast(float, v[i] << 16);
    s += __builtin_bit_cast(float, v[i] & 0xffff0000u);
  }
  return s;
}

template <typename T, int KIND, int BM, int WM, int WN>
struct KqLds {  // byte offsets; two stage buffers, two tables of x's sums (superblock parity)
  static constexpr int kPlanes = KqPlanes<T, KIND>::value;
  static constexpr int kX = BM * kKqBK * 2, kW = kKqBN * kKqBK * 2;
  static constexpr int kStage = kX + kPlanes * kW;
  static constexpr bool kMin = KIND != NVF_Q6_K;
  static constexpr int kXs = kMin ? BM * 48 : 0;     // x sub-block sums: [piece][row][8 j] bf16
  static constexpr int kR = kMin ? kKqBN * 48 : 0;   // r_j: [piece][column][8 j] bf16
  static constexpr int kD = kKqBN * 4;               // d
  static constexpr int kXsAt = 2 * kStage, kRAt = kXsAt + 2 * kXs, kDAt = kRAt + kR;
  static constexpr int kBytes = kDAt + (kMin ? kD : 2 * kD);
};

template <typename T, int KIND, int LAYOUT, typename TO, int BM, int WM, int WN>
__global__ __launch_bounds__(WM* WN * 64) __attribute__((amdgpu_waves_per_eu(2))) void kq_gemm_kernel(
    const T* __restrict__ x, const uint8_t* __restrict__ wq, TO* __restrict__ out, int64_t m, int64_t n, int64_t k,
    int tiles_n, int vec_out) {
  using L = KqLds<T, KIND, BM, WM, WN>;
  constexpr int kThreads = WM * WN * 64, kWaves = WM * WN;
  constexpr int TM = BM / WM / 32, TN = kKqBN / WN / 32;
  constexpr int kRowB = kKqBK * 2;
  constexpr int kDma = BM * kRowB / 1024 / kWaves;  // 1 KB transfers (8 activation rows) per wave and stage
  constexpr int kTpc = kThreads / kKqBN, kNb = 32 / kTpc;  // threads per column, quant bytes per thread
  static_assert(kDma >= 1 && (kNb == 8 || kNb == 16), "staging");
  using Raw = KqRaw<KIND, LAYOUT, kNb>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  int tm, tn;
  g16_tile<8>(tiles_n, tm, tn);
  const int64_t row0 = (int64_t)tm * BM, col0 = (int64_t)tn * kKqBN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int nsb = (int)(k >> 8), nst = 4 * nsb;

  // activations: rows past m fall outside the resource and read zero
  const int64_t a_rows = m - row0 < BM ? m - row0 : BM;
  const __amdgpu_buffer_rsrc_t ra = g16_rsrc(x + row0 * k, a_rows * k * 2);
  uint32_t off[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = (wave * kDma + i) * 8 + (lane >> 3);
    off[i] = (uint32_t)(r * k * 2) + (uint32_t)(((lane & 7) ^ g16_key<64>(r)) * 16);
  }
  auto issue = [&](int st, int buf) {  // a stage past the end reads the last one again (never used)
    const uint32_t kb = (uint32_t)(st < nst ? st : nst - 1) * kRowB;
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      g16_dma(ra, lds + buf * L::kStage + (wave * kDma + i) * 1024, off[i], kb);
  };

  // weights: this thread's column (one past n repeats the last: its outputs are not stored)
  const int wc = tid / kTpc, part = tid % kTpc;
  const int64_t wcol = col0 + wc < n ? col0 + wc : n - 1;
  const uint8_t* wrow = wq + wcol * nsb * Raw::kBlock;
  const int wkey = g16_key<64>(wc);
  Raw raw[2];
  auto load = [&](Raw& r, int st) {
    const int s = st < nst ? st : nst - 1;
    r.load(wrow + (int64_t)(s >> 2) * Raw::kBlock, s & 3, part);
  };
  typename Raw::Head head, next;  // of the stage that is decoded, and of the superblock after it
  uint32_t cen[2] = {};           // its centres c_j, one per byte
  uint32_t rem[4 / kTpc][3] = {};  // the r_j that this thread finds, in pairs: three pieces
  // the column's threads find 8 / kTpc centres each and hand them round (quad_perm)
  auto centres = [&](const Raw& r) {
    if constexpr (L::kMin) {
      constexpr int kOwn = 8 / kTpc;
      uint32_t sc[2], mn[2];
      q4k_tables(r.hd.w, sc, mn);
      const int sh = kTpc == 2 ? 0 : 16 * (part & 1);
      const bool low = part < kTpc / 2;  // this thread's are among c_0 .. c_3
      const uint32_t sw = (low ? sc[0] : sc[1]) >> sh, mw = (low ? mn[0] : mn[1]) >> sh;
      const float d = r.d(), dmin = r.dmin();
      uint32_t own = 0, pc[kOwn][3];
#pragma unroll
      for (int i = 0; i < kOwn; ++i) {
        const float p = d * (float)byte_of(sw, i), o = dmin * (float)byte_of(mw, i);
        const float c = kq_centre(p, o, KIND == NVF_Q4_K ? 15.0f : 31.0f);
        own |= (uint32_t)c << (8 * i);
        bf16_pieces(fmaf(p, c, -o), pc[i]);
      }
#pragma unroll
      for (int i = 0; i < kOwn / 2; ++i)
#pragma unroll
        for (int q = 0; q < 3; ++q) rem[i][q] = pc[2 * i][q] | pc[2 * i + 1][q] << 16;
      auto swap = [](uint32_t v, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false);
      };
      uint32_t other;
      if constexpr (kTpc == 2) {
        other = swap(own, std::integral_constant<int, 0xb1>{});
      } else {
        own <<= sh;
        own |= swap(own, std::integral_constant<int, 0xb1>{});
        other = swap(own, std::integral_constant<int, 0x4e>{});
      }
      cen[0] = low ? own : other;
      cen[1] = low ? other : own;
    }
  };
  auto store_w = [&](const Raw& r, int st, int quarter, int buf) {
    uint8_t* base = lds + buf * L::kStage + L::kX + wc * kRowB;
#pragma unroll
    for (int u = 0; u < Raw::kRuns; ++u) {
      uint32_t b[2], sc, mn;
      int chunk, j;
      r.run(u, quarter, part, b, chunk, j);
      r.scale_min(j, sc, mn);
      u32x4 p[2];
      kq_planes<KIND>(b, sc, byte_of(cen[j >> 2], j & 3), p, T{});
#pragma unroll
      for (int i = 0; i < L::kPlanes; ++i) st16(base + i * L::kW + ((chunk ^ wkey) << 4), p[i]);
    }
    // the superblock's d and r_j: after quarter 0, in which the last superblock's are still read
    if (quarter == 2) {
      if constexpr (L::kMin) {
#pragma unroll
        for (int i = 0; i < 4 / kTpc; ++i)
#pragma unroll
          for (int q = 0; q < 3; ++q)
            *reinterpret_cast<uint32_t*>(lds + L::kRAt + q * (kKqBN * 16) + wc * 16 + (part * (4 / kTpc) + i) * 4) =
                rem[i][q];
      }
      if (L::kMin && part == 0) *reinterpret_cast<float*>(lds + L::kDAt + wc * 4) = r.d() * kKqUnit<T, KIND>;
    }
    if (!L::kMin && quarter == 0 && part == 0)
      *reinterpret_cast<float*>(lds + L::kDAt + ((st >> 2) & 1) * (kKqBN * 4) + wc * 4) = r.d();
  };

  // sub-block sums of the stage's activations, as three bf16 pieces
  auto sums = [&](int st, int buf) {
    if constexpr (!L::kMin) return;
    const int quarter = st & 3, par = (st >> 2) & 1;
    for (int t = tid; t < 2 * BM; t += kThreads) {
      const int r = t & (BM - 1), s = t / BM, key = g16_key<64>(r);
      const uint8_t* p = lds + buf * L::kStage + r * kRowB;
      float v = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c) v = kq_sum8(ld16(p + (((4 * s + c) ^ key) << 4)), v, T{});
      uint32_t pc[3];
      bf16_pieces(v, pc);
      uint16_t* d = reinterpret_cast<uint16_t*>(lds + L::kXsAt + par * L::kXs) + r * 8 + 2 * quarter + s;
#pragma unroll
      for (int q = 0; q < 3; ++q) d[q * BM * 8] = (uint16_t)pc[q];
    }
  };

  f32x16 acc[TM][TN], blk[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) acc[a][b] = f32x16{};
  const int half = lane >> 5, lr = lane & 31;
  const int ar = wm * TM * 32 + lr, br = wn * TN * 32 + lr;
  const int a0 = ar * kRowB + ((half ^ g16_key<64>(ar)) << 4);
  const int b0 = L::kX + br * kRowB + ((half ^ g16_key<64>(br)) << 4);

  auto apply = [&](int sb) {  // acc += R + d B (the next superblock's first products start from 0)
    const int par = sb & 1;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      const float d = *reinterpret_cast<const float*>(lds + L::kDAt + (L::kMin ? 0 : par * L::kD) + (br + 32 * b) * 4);
      u32x4 r0 = {}, r1 = {}, r02 = {};
      if constexpr (L::kMin) {  // k slots 0-7 (half 0) and 8-15 (half 1) of an MFMA
        const uint8_t* rt = lds + L::kRAt + (br + 32 * b) * 16;
        r0 = ld16(rt);
        r1 = ld16(rt + kKqBN * 16);
        r02 = ld16(rt + half * (2 * kKqBN * 16));
      }
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        if constexpr (L::kMin) {
          const uint8_t* xs = lds + L::kXsAt + par * L::kXs + (ar + 32 * a) * 16;
          const u32x4 x01 = ld16(xs + half * (BM * 16)), x20 = ld16(xs + (1 - half) * (2 * BM * 16));
          acc[a][b] = mfma16(x20, r02, acc[a][b], __bf16{});
          acc[a][b] = mfma16(x01, r1, acc[a][b], __bf16{});
          acc[a][b] = mfma16(x01, r0, acc[a][b], __bf16{});
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[a][b][j] = fmaf(d, blk[a][b][j], acc[a][b][j]);
      }
    }
  };

  issue(0, 0);
  load(raw[0], 0);
  load(raw[1], 1);
  head.load(wrow, part);
  next = raw[0].hd = head;
  centres(raw[0]);
  store_w(raw[0], 0, 0, 0);
#pragma unroll 1
  for (int sb = 0; sb < nsb; ++sb) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int st = 4 * sb + q;
      wait_vm<0>();                        // this stage's transfers (and the next stage's weights)
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this stage's weights are written, the last one's reads done
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (q == 0 && sb > 0) apply(sb - 1);
      issue(st + 1, (q + 1) & 1);
      load(raw[q & 1], st + 2);
      if (q == 2) next.load(wrow + (int64_t)(sb + 1 < nsb ? sb + 1 : sb) * Raw::kBlock, part);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products, not after
      if (q == 3) head = next;
      raw[(q + 1) & 1].hd = head;
      if (q == 3) centres(raw[(q + 1) & 1]);
      const uint8_t* s = lds + (q & 1) * L::kStage;
#pragma unroll
      for (int kk = 0; kk < kKqBK / 16; ++kk) {
        u32x4 xa[TM];
#pragma unroll
        for (int a = 0; a < TM; ++a) xa[a] = ld16(s + (a0 ^ (kk << 5)) + a * 32 * kRowB);
#pragma unroll
        for (int p = L::kPlanes - 1; p >= 0; --p) {
          u32x4 wb[TN];
#pragma unroll
          for (int b = 0; b < TN; ++b) wb[b] = ld16(s + p * L::kW + (b0 ^ (kk << 5)) + b * 32 * kRowB);
#pragma unroll
          for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b)
              blk[a][b] = mfma16(xa[a], wb[b], q == 0 && kk == 0 && p == L::kPlanes - 1 ? f32x16{} : blk[a][b], T{});
        }
      }
      sums(st, q & 1);
      store_w(raw[(q + 1) & 1], st + 1, (q + 1) & 3, (q + 1) & 1);
    }
  }
  wait_vm<0>();
  __syncthreads();
  apply(nsb - 1);
  __syncthreads();

  // D layout: lane l, value j -> x row 8 (j / 4) + 4 (l / 32) + j % 4, output column l % 32.  Each
  // wave passes 32 output rows at a time through its own LDS.
  constexpr int kCols = TN * 32, kPitch = kCols * (int)sizeof(TO) + 16;
  static_assert(kWaves * 32 * kPitch <= 2 * L::kStage, "epilogue LDS");
  uint8_t* mine = lds + wave * (32 * kPitch);
  constexpr int kVec = 16 / (int)sizeof(TO), kVpr = kCols / kVec;
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int j = 0; j < 16; ++j)
        *reinterpret_cast<TO*>(mine + (8 * (j >> 2) + 4 * half + (j & 3)) * kPitch + (32 * b + lr) * (int)sizeof(TO)) =
            from_f32<TO>(acc[a][b][j]);
    __builtin_amdgcn_wave_barrier();
    const int64_t r0 = row0 + wm * TM * 32 + 32 * a, c0 = col0 + wn * kCols;
#pragma unroll
    for (int u0 = 0; u0 < 32 * kVpr; u0 += 64) {
      const int u = u0 + lane, r = u / kVpr, c = (u % kVpr) * kVec;
      const u32x4 v = ld16(mine + r * kPitch + c * (int)sizeof(TO));
      if (r0 + r < m) {
        TO* p = out + (r0 + r) * n + c0 + c;
        if (vec_out && c0 + c + kVec <= n) {
          st16(p, v);
        } else {
          const auto e = __builtin_bit_cast(std::array<TO, kVec>, v);
#pragma unroll
          for (int i = 0; i < kVec; ++i)
            if (c0 + c + i < n) p[i] = e[i];
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }

  // outputs that came out infinite or NaN, again on the fp32 matrix cores: the 32 x 32 results that hold one
  uint64_t bad = 0;
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (!__builtin_isfinite(acc[a][b][j])) bad |= 1ull << ((a * TN + b) * 16 + j);
  static_assert(TM * TN * 16 <= 64, "one bit per accumulator");
  if (!__any(bad != 0)) return;
  wait_vm<0>();  // the stores above come first
#pragma unroll 1
  for (int t = 0; t < TM * TN; ++t) {
    const int64_t r0 = row0 + wm * TM * 32 + 32 * (t / TN), c = col0 + wn * kCols + 32 * (t % TN) + lr;
    uint32_t mine = c < n ? (uint32_t)(bad >> (16 * t)) & 0xffffu : 0u;
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (r0 + 8 * (j >> 2) + 4 * half + (j & 3) >= m) mine &= ~(1u << j);
    if (!__any(mine != 0)) continue;
    const Table<8, T> xs{x};
    const KqPlain<KIND, LAYOUT> ws{wq};
    const int64_t x0 = (r0 + lr < m ? r0 + lr : m - 1) * k + 8 * half, w0 = (c < n ? c : n - 1) * k + 8 * half;
    f32x16 v = f32x16{};
#pragma unroll 1
    for (int64_t e = 0; e < k; e += 32) {  // the loads of two steps go out together
      typename Table<8, T>::Raw xr[2];
      typename KqPlain<KIND, LAYOUT>::Raw wr[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        xr[u] = xs.load(x0 + e + 16 * u);
        wr[u] = ws.load(w0 + e + 16 * u);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float xv[8], wv[8];
        xs.decode(xr[u], xv);
        ws.decode(wr[u], wv);
#pragma unroll
        for (int i = 0; i < 8; ++i) v = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i], wv[i], v, 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (mine >> j & 1) out[(r0 + 8 * (j >> 2) + 4 * half + (j & 3)) * n + c] = from_f32<TO>(v[j]);
  }
}

template <typename T, int KIND, int LAYOUT, typename TO, int BM, int WM, int WN>
int launch_kq_tile(const void* x, const uint8_t* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  constexpr int kLds = KqLds<T, KIND, BM, WM, WN>::kBytes;
  static_assert(kLds <= 160 * 1024, "LDS");
  auto kern = kq_gemm_kernel<T, KIND, LAYOUT, TO, BM, WM, WN>;
  static std::once_flag attr_once;
  std::call_once(attr_once, [&] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  });
  const int tiles_n = (int)((n + kKqBN - 1) / kKqBN);
  const int vec_out = aligned16(out) && n % (16 / (int64_t)sizeof(TO)) == 0;
  kern<<<dim3((unsigned)(((m + BM - 1) / BM) * tiles_n)), WM * WN * 64, kLds, st>>>(
      static_cast<const T*>(x), w, static_cast<TO*>(out), m, n, k, tiles_n, vec_out);
  return launch_status("dense_gemm (K-quant)");
}

// The tile: the one whose estimated time per superblock of the whole output is least, from the
// tiles that the fullest of the 256 CUs gets (c).  One takes `alone`; where the LDS lets several
// share a CU each further one adds `busy`, else c of them take `busy` each.  us per superblock
// (launch time at k = 3584 over 14; 32-, 64-, 128-, 256-row tiles):
//                      alone                     busy                        from
//   fp16 Q4_K, Q5_K    2.75 3.25 3.86 5.00       1.3  2.0  3.86 5.35         16 to 4096 x 3584, 4608, 37888 x 3584
//   bf16 Q4_K, Q5_K    4.25 5.00 6.25 7.80       4.1  5.0  6.25 8.00         32 to 2048 x 4608, 37888 x 3584
//   Q6_K               4.70 5.40 7.00 6.85       3.55 6.2  7.50 7.20         as the first, and 3584 x 18944
// (Q6_K is never best at 128 rows: not built.)
// So 128 rows on 4608 columns take 39 us at 32 rows per tile against 46 to 70 at the others, 1021 rows
// there 77 at 256 against 102 to 110, 64 x 37888 62 at 64 rows; Q6_K, 1021 x 4608, 107 at 256
// against 210 to 261.  At each of these sizes the choice is the best tile or within 3% of it.
template <typename T, int KIND>
int kq_tile(int64_t m, int64_t n) {
  constexpr int kCls = KIND == NVF_Q6_K ? 2 : __is_same(T, _Float16) ? 0 : 1;
  constexpr double kAlone[3][4] = {{2.75, 3.25, 3.86, 5.0}, {4.25, 5.0, 6.25, 7.8}, {4.7, 5.4, 7.0, 6.85}};
  constexpr double kBusy[3][4] = {{1.3, 2.0, 3.86, 5.35}, {4.1, 5.0, 6.25, 8.0}, {3.55, 6.2, 7.5, 7.2}};
  int best = 3;
  double best_t = 0.0;
  for (int i = 3; i >= 0; --i) {
    const int64_t bm = 32ll << i, tiles = ((m + bm - 1) / bm) * ((n + kKqBN - 1) / kKqBN);
    if ((i < 3 && tiles > INT32_MAX) || (i == 2 && KIND == NVF_Q6_K)) continue;
    const double c = (double)((tiles + 255) / 256);
    const bool share = i == 0 || (i == 1 && kCls == 0);
    const double t = c == 1.0 ? kAlone[kCls][i] : share ? kAlone[kCls][i] + (c - 1.0) * kBusy[kCls][i] : c * kBusy[kCls][i];
    if (i == 3 || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

template <typename T, int KIND, int LAYOUT, typename TO>
int launch_kq(const void* x, const uint8_t* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  switch (kq_tile<T, KIND>(m, n)) {
    case 3:
      return launch_kq_tile<T, KIND, LAYOUT, TO, 256, 4, 2>(x, w, out, m, n, k, st);
    case 2:
      return launch_kq_tile<T, KIND, LAYOUT, TO, KIND == NVF_Q6_K ? 256 : 128, KIND == NVF_Q6_K ? 4 : 2, 2>(x, w, out, m,
                                                                                                          n, k, st);
    case 1:
      return launch_kq_tile<T, KIND, LAYOUT, TO, 64, 2, 2>(x, w, out, m, n, k, st);
    default:
      return launch_kq_tile<T, KIND, LAYOUT, TO, 32, 1, 4>(x, w, out, m, n, k, st);
  }
}

template <typename T, typename TO>
int dispatch_kq(const void* x, const uint8_t* w, int kind, int layout, void* out, int64_t m, int64_t n, int64_t k,
                hipStream_t st) {
  switch (kind) {
    case NVF_W_Q4_K:
      if (layout == NVF_QK_LAYOUT_HIP_LEGACY)
        return launch_kq<T, NVF_Q4_K, NVF_QK_LAYOUT_HIP_LEGACY, TO>(x, w, out, m, n, k, st);
      return launch_kq<T, NVF_Q4_K, NVF_QK_LAYOUT_GGML, TO>(x, w, out, m, n, k, st);
    case NVF_W_Q5_K:
      return launch_kq<T, NVF_Q5_K, NVF_QK_LAYOUT_GGML, TO>(x, w, out, m, n, k, st);
    default:
      return launch_kq<T, NVF_Q6_K, NVF_QK_LAYOUT_GGML, TO>(x, w, out, m, n, k, st);
  }
}

int kq_gemm(const void* x, bool bf16, const void* w, int kind, int layout, void* out, int out_dtype, int64_t m,
            int64_t n, int64_t k, hipStream_t st) {
  int rc = NVF_OK;
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  if (bf16)
    NVF_DISPATCH_DTYPE(out_dtype, TO, rc = (dispatch_kq<__bf16, TO>(x, wb, kind, layout, out, m, n, k, st)));
  else
    NVF_DISPATCH_DTYPE(out_dtype, TO, rc = (dispatch_kq<_Float16, TO>(x, wb, kind, layout, out, m, n, k, st)));
  return rc;
}

}  // namespace nvf
