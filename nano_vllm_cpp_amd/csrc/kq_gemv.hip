// Decode product on Q4_K and Q5_K weights: out[m][n] = x[m][k] . W[n][k]^T,
// m <= 16, k a multiple of 256, on the 16-bit matrix cores.
//
// Bound by the weights' stream from HBM as long as decoding them costs about 2 VALU
// instructions per weight; decoding each to fp32 and multiplying on the VALU takes 5.2 at one
// row, and the fp32 matrix cores are slower still.  Here c_j is a sub-block's centre
// (kq_centre) and r_j = d sc_j c_j - dmin m_j its remainder, as in kq_gemm.hip.  fp16 x: a weight's
// quant is masked out as a subnormal and one packed multiply-add makes it the exact operand
// sc_j (q - c_j) 2^-14, so v_mfma_f32_16x16x32 sums whole superblocks for 16 rows and 16 columns,
// and d takes one fused multiply-add per four rows and 4096 weights.  bf16 x (and fp32 x as
// three exact bf16 pieces): the operand is q - c_j, and sc_j takes one multiply-add per four rows
// and 512 weights.  The r_j times the sub-blocks' sums of x are 8 multiply-adds per superblock up to
// 4 rows, else two MFMAs (both as three bf16 pieces).  The result is within three times the bound of fp32 sums of x w.
//
// A wave owns 16 columns: lane l holds column l % 16 and, of every sub-block, the values
// 8 (l / 16) .. + 7.  Read straight from memory in that layout a superblock takes 5 loads that
// each touch 16 cache lines, and the L1's line rate bounds the kernel (1 x 151936 x 4096 Q4_K
// 119 us); so the weights go HBM -> LDS by DMA, whole runs of each column at a time, into
// a ring of kKvStages superblocks that is the wave's own.  WC waves of a
// workgroup on other columns share the staged x; KG groups of them split K for
// narrow outputs.
//
// fp16 x, Q4_K: 1 x 151936 x 4096 (350 MB) 136 us on decoded weights -> 80 (4.4 TB/s); 1 x
// 37888 x 3584 26.4 -> 22.5 us, 8 x 37888 x 3584 56 -> 29.3.  146 VALU instructions per
// superblock of a wave's 16 columns (2.3 per weight); with the remainders by MFMAs at one row too
// 160 and 22.8 us; with a subtraction of c_j and a multiply-add per sub-block 174 and 23.6; with
// c_j = 0 (no centres: the bound then lies over the two parts, however they cancel) the three
// take 73, 21.0 and 26.5 us.  bf16 x, 2 x 37888 x 3584: 29.3 us, 34.6 with the subtraction in
// fp32 after the conversion.
//
// Infinities and NaN: sums that come out non-finite are made again from the decoded weights,
// as in kq_gemm.hip (8 x 37888 x 3584, every activation NaN: 1040 us one
// output after the other, 127 so).

#include <mutex>
#include <type_traits>

#include "gemm16.hpp"
#include "gemm_tile.hpp"

namespace nvf {

__device__ __forceinline__ f32x4 mfma16x16(const u32x4 a, const u32x4 b, const f32x4 c, __bf16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}
__device__ __forceinline__ f32x4 mfma16x16(const u32x4 a, const u32x4 b, const f32x4 c, _Float16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

constexpr int kKvStages = 4;  // weight stages (superblocks) of a wave's ring

// (An ext_vector type: HIP's own uint2 carries alias information that makes the compiler drain
// every LDS DMA transfer in flight before a read of it.)
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// One superblock of a lane's column, as read from LDS: bytes(s) gives the quants 8 g .. 8 g + 7 of
// sub-block s (32 values).
template <int KIND, int LAYOUT>
struct KvRaw;

template <int LAYOUT>
struct KvRaw<NVF_Q4_K, LAYOUT> {
  static constexpr int kBlock = 144;
  static constexpr int kLoads = LAYOUT == NVF_QK_LAYOUT_GGML ? 4 : 8;
  u32x4 hdr;
  u32x2 q[kLoads];
  __device__ __forceinline__ void load(const uint8_t* blk, int g) {
    hdr = ld16(blk);
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      q[i] = *reinterpret_cast<const u32x2*>(blk + 16 + (LAYOUT == NVF_QK_LAYOUT_GGML ? 32 * i + 8 * g
                                                                                     : 16 * i + 8 * (g & 1)));
  }
  __device__ __forceinline__ void bytes(int s, int g, uint32_t* b) const {
    if constexpr (LAYOUT == NVF_QK_LAYOUT_GGML) {
      b[0] = (q[s >> 1].x >> (4 * (s & 1))) & 0x0f0f0f0fu;
      b[1] = (q[s >> 1].y >> (4 * (s & 1))) & 0x0f0f0f0fu;
    } else {
      const int sh = 4 * (g >> 1);
      b[0] = (q[s].x >> sh) & 0x0f0f0f0fu;
      b[1] = (q[s].y >> sh) & 0x0f0f0f0fu;
    }
  }
  // The same as fp16 operands, without a conversion: a quant under a zero exponent is the
  // subnormal q 2^-24 (q 2^-20 where the nibble stays in its upper place: odd sub-blocks),
  // exact, and the matrix cores take subnormals as they are.  The halves of a dword hold
  // bytes two apart, so the values come in the order 0 2 1 3 4 6 5 7, as x is staged.
  __device__ __forceinline__ u32x4 halves(int s, int g) const {
    if constexpr (LAYOUT == NVF_QK_LAYOUT_GGML) {
      const uint32_t mask = (s & 1) ? 0x00f000f0u : 0x000f000fu;
      const u32x2 w = q[s >> 1];
      return {w.x & mask, (w.x >> 8) & mask, w.y & mask, (w.y >> 8) & mask};
    } else {
      const uint32_t a = q[s].x >> (4 * (g >> 1)), b = q[s].y >> (4 * (g >> 1));
      return {a & 0x000f000fu, (a >> 8) & 0x000f000fu, b & 0x000f000fu, (b >> 8) & 0x000f000fu};
    }
  }
  static constexpr float kOdd = LAYOUT == NVF_QK_LAYOUT_GGML ? 0x1p20f : 0x1p24f;  // odd sub-blocks' 1 / unit
  static constexpr float kTop = 15.0f;                                             // the largest quant
  __device__ __forceinline__ float d() const { return half_bits_to_f32(hdr[0] & 0xffffu); }
  __device__ __forceinline__ float dmin() const { return half_bits_to_f32(hdr[0] >> 16); }
};

template <int LAYOUT>
struct KvRaw<NVF_Q5_K, LAYOUT> : KvRaw<NVF_Q4_K, NVF_QK_LAYOUT_GGML> {
  using Base = KvRaw<NVF_Q4_K, NVF_QK_LAYOUT_GGML>;
  static constexpr int kBlock = 176;
  static constexpr float kTop = 31.0f;
  u32x2 h;
  __device__ __forceinline__ void load(const uint8_t* blk, int g) {
    hdr = ld16(blk);
    h = *reinterpret_cast<const u32x2*>(blk + 16 + 8 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const u32x2*>(blk + 48 + 32 * i + 8 * g);
  }
  __device__ __forceinline__ void bytes(int s, int g, uint32_t* b) const {
    Base::bytes(s, g, b);
    b[0] |= ((h.x >> s) & 0x01010101u) << 4;
    b[1] |= ((h.y >> s) & 0x01010101u) << 4;
  }
  // the fifth bit joins the nibble where it is: bit 4, or 8 for odd sub-blocks
  __device__ __forceinline__ u32x4 halves(int s, int g) const {
    u32x4 v = Base::halves(s, g);
    const int to = (s & 1) ? 8 : 4;
    const uint32_t bit = (s & 1) ? 0x01000100u : 0x00100010u;
    const uint32_t hw[2] = {h.x, h.y};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int from = s + 8 * (i & 1);  // bit s of bytes 0 and 2, then of bytes 1 and 3
      v[i] |= (from >= to ? hw[i >> 1] >> (from - to) : hw[i >> 1] << (to - from)) & bit;
    }
    return v;
  }
};

// Sub-block s's quants 8 g .. + 7 as 16-bit operands.  sub is what kv_sub made of the sub-block.
// fp16: sc (q - c) 2^-14 by one exact multiply-add of the subnormal q (at most 11 bits).
template <typename Raw>
__device__ __forceinline__ u32x4 kv_operand(const Raw& r, int s, int g, uint32_t sub, _Float16) {
  const f16x2 m = __builtin_bit_cast(f16x2, sub);
  u32x4 p = r.halves(s, g);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = p[i];
    p[i] = __builtin_bit_cast(
        uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, w), f16x2{m[0], m[0]}, f16x2{m[1], m[1]}));
  }
  return p;
}
// The multiplier and the addend (exact in fp16); q's unit is 1 / kOdd in odd sub-blocks.
template <typename Raw>
__device__ __forceinline__ uint32_t kv_sub(float sc, float c, bool odd, _Float16) {
  const float mul = odd ? 0x1p-14f * Raw::kOdd : 1024.0f;
  const f16x2 m = {(_Float16)(mul * sc), (_Float16)(-0x1p-14f * sc * c)};
  return __builtin_bit_cast(uint32_t, m);
}
// bf16: q - c (the scale would take a second operand)
template <typename Raw>
__device__ __forceinline__ u32x4 kv_operand(const Raw& r, int s, int g, uint32_t sub, __bf16) {
  uint32_t b[2];
  r.bytes(s, g, b);
  // four weights at a time as signed bytes: 128 + q - c leaves no borrow, then the top bit flips
#pragma unroll
  for (int i = 0; i < 2; ++i) b[i] = (b[i] + sub) ^ 0x80808080u;
  u32x4 p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // at most 5 significant bits: the upper halves of the fp32 values
    const float v0 = sbyte(b[i >> 1], 2 * (i & 1)), v1 = sbyte(b[i >> 1], 2 * (i & 1) + 1);
    p[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, v1), __builtin_bit_cast(uint32_t, v0), 0x07060302u);
  }
  return p;
}
template <typename Raw>
__device__ __forceinline__ uint32_t kv_sub(float, float c, bool, __bf16) {
  const uint32_t b = (uint32_t)c;
  return 0x80808080u - b * 0x01010101u;
}

// v of the 16-lane group i in o[i], in every group.
__device__ __forceinline__ void kv_gather(uint32_t v, uint32_t* o) {
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);              // groups 0 0 2 2, 1 1 3 3
  const auto a = __builtin_amdgcn_permlane32_swap(r[0], r[0], false, false);        // 0 0 0 0, 2 2 2 2
  const auto b = __builtin_amdgcn_permlane32_swap(r[1], r[1], false, false);        // 1 1 1 1, 3 3 3 3
  o[0] = a[0];
  o[1] = b[0];
  o[2] = a[1];
  o[3] = b[1];
}

// x as staged: XP planes of 16-bit values (fp32: three exact bf16 pieces), rows of a
// superblock 528 bytes apart (the 16 rows of a read phase on distinct banks), then the
// sub-blocks' sums: as bf16 pieces, [row][8 j][x0 x0 x0 x1 x1 x2 0 0], rows 144 bytes apart, or
// up to 4 rows as they are, [8 j][4 rows].
template <typename TX>
struct KvX {
  using T = TX;
  static constexpr int kPlanes = 1;
};
template <>
struct KvX<float> {
  using T = __bf16;
  static constexpr int kPlanes = 3;
};
constexpr int kKvRow = 528, kKvSums = 144;
template <typename TX>
constexpr int kv_sb_bytes(int m) {
  return m * KvX<TX>::kPlanes * kKvRow + (m <= 4 ? 128 : m * kKvSums);
}

// A weight stage in LDS: one superblock of 16 columns, column after column.  A column is 9 or
// 11 units of 16 bytes, an odd number, so the 16 columns' reads of one unit fall in distinct
// bank groups.
template <int BLOCK>
struct KvStage {
  static constexpr int kUnits = BLOCK / 16, kAll = 16 * kUnits;
  static constexpr int kDma = (kAll + 63) / 64;  // transfers; the last one of fewer lanes
  static constexpr int kBytes = kAll * 16;
  static_assert(kUnits % 2 == 1, "bank groups");
};

template <typename TX, int KIND, int LAYOUT, typename TO, int WC, int KG, int NE>
__global__ __launch_bounds__(WC* KG * 64) __attribute__((amdgpu_waves_per_eu(2, 4))) void kq_gemv_kernel(
    const TX* __restrict__ x, const uint8_t* __restrict__ wq, TO* __restrict__ out, int m, int64_t n, int64_t k,
    int chunk) {
  using T = typename KvX<TX>::T;
  using Raw = KvRaw<KIND, LAYOUT>;
  using Stage = KvStage<Raw::kBlock>;
  constexpr int XP = KvX<TX>::kPlanes;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kg = wave / WC, wc = wave % WC;
  const int gt = threadIdx.x - kg * WC * 64;  // thread of the K group
  const int64_t col0 = ((int64_t)blockIdx.x * WC + wc) * 16;
  const int nsb = (int)(k >> 8);
  const int per = (nsb + KG - 1) / KG;  // superblocks per K group
  const int sb0 = kg * per, cnt = nsb - sb0 < per ? nsb - sb0 : per;    // (cnt may be <= 0)
  const int sbb = kv_sb_bytes<TX>(m);
  uint8_t* const ring = lds + wave * (kKvStages * Stage::kBytes);
  uint8_t* const xl = lds + WC * KG * (kKvStages * Stage::kBytes) + kg * chunk * sbb;

  // this lane's units of a stage; a column past n falls outside the resource and reads zero
  const int64_t row_bytes = (int64_t)nsb * Raw::kBlock;
  const int64_t cols = col0 >= n ? 0 : n - col0 < 16 ? n - col0 : 16;
  const __amdgpu_buffer_rsrc_t rw = g16_rsrc(wq + (cols > 0 ? col0 : 0) * row_bytes, cols * row_bytes);
  uint32_t off[Stage::kDma];
#pragma unroll
  for (int i = 0; i < Stage::kDma; ++i) {
    const int p = i * 64 + lane;
    off[i] = (uint32_t)((p / Stage::kUnits) * row_bytes + (int64_t)sb0 * Raw::kBlock + (p % Stage::kUnits) * 16);
  }
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int i = 0; i < Stage::kDma; ++i) {
      const uint32_t o = st < cnt ? off[i] : 0x80000000u;  // a superblock past the group's: zeros
      if (i * 64 + lane < Stage::kAll)
        g16_dma(rw, ring + slot * Stage::kBytes + i * 1024, o, (uint32_t)(st * Raw::kBlock));
    }
  };
#pragma unroll
  for (int st = 0; st < kKvStages - 1; ++st) issue(st, st);

  // stages x of superblocks [i, i + chunk) of this group
  auto stage = [&](int i) {
    const int have = cnt - i < chunk ? cnt - i : chunk;
    for (int t = gt; t < have * m * 32; t += WC * 64) {
      const int ch = t & 31, rs = t >> 5, r = rs % m, s = rs / m;
      const TX* p = x + (int64_t)r * k + (int64_t)(sb0 + i + s) * 256 + 8 * ch;
      uint8_t* d = xl + s * sbb + r * kKvRow + 16 * ch;
      float v[8], sum = 0.0f;
      if constexpr (sizeof(TX) == 2) {
        const u32x4 w = ld16(p);
        // fp16: in the order of the fp16 operands
        if constexpr (__is_same(TX, _Float16))
          st16(d, u32x4{__builtin_amdgcn_perm(w[1], w[0], 0x05040100u), __builtin_amdgcn_perm(w[1], w[0], 0x07060302u),
                        __builtin_amdgcn_perm(w[3], w[2], 0x05040100u), __builtin_amdgcn_perm(w[3], w[2], 0x07060302u)});
        else
          st16(d, w);
        Pack<TX>::unpack(w, v);
      } else {
        const Table<8, float> xs{x};
        xs.decode(xs.load(p - x), v);
        bf16x8 pc[3];
        split3(v, pc);
#pragma unroll
        for (int q = 0; q < 3; ++q) st16(d + q * m * kKvRow, __builtin_bit_cast(u32x4, pc[q]));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += v[e];
      sum = group_sum<4>(sum);
      if ((ch & 3) == 0) {
        uint8_t* ds = xl + s * sbb + XP * m * kKvRow;
        if constexpr (NE == 1) {
          reinterpret_cast<float*>(ds)[ch + r] = sum;
        } else {
          uint32_t pc[3];
          bf16_pieces(sum, pc);
          st16(ds + r * kKvSums + 4 * ch,
               u32x4{pc[0] | pc[0] << 16, pc[0] | pc[1] << 16, pc[1] | pc[2] << 16, 0u});
        }
      }
    }
  };

  // Row r of x is operand row 4 (r % 4) + r / 4, so that lane group g's results e < NE are
  // rows g + 4 e: up to 4 NE rows cost NE multiply-adds per sub-block.  Operand rows of no
  // row of x repeat row 0; their results are not stored.
  f32x4 tot = {};
  const int xr = (c >> 2) + 4 * (c & 3), xrow = xr < m ? xr : 0;
  const uint8_t* const xa = xl + xrow * kKvRow + 16 * g;
  const uint8_t* const xs = xl + XP * m * kKvRow + (NE == 1 ? 0 : xrow * kKvSums) + 32 * g;
  float rt[4] = {};  // NE = 1: the remainders' part of rows 0 .. 3, of this lane group's sub-blocks
  auto compute = [&](const Raw& r, int s) {  // superblock s of the staged chunk
    const uint8_t* xb = xa + s * sbb;
    const float d = r.d();
    uint32_t sc[2], mn[2];
    q4k_tables(r.hdr, sc, mn);
    // lane group g finds the centres of sub-blocks 2 g and 2 g + 1 and takes their remainders: up to
    // 4 rows times the sums of x as they are (8 multiply-adds), else by an MFMA over the pieces
    // [r0 r1 r2 r0 r1 r0 0 0]
    const uint32_t sg = (g < 2 ? sc[0] : sc[1]) >> (16 * (g & 1)), mg = (g < 2 ? mn[0] : mn[1]) >> (16 * (g & 1));
    uint32_t sub[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float sf = (float)byte_of(sg, i), p = d * sf, o = r.dmin() * (float)byte_of(mg, i);
      const float q0 = kq_centre(p, o, Raw::kTop);
      kv_gather(kv_sub<Raw>(sf, q0, i == 1, T{}), sub[i]);
      const float rem = fmaf(p, q0, -o);
      if constexpr (NE == 1) {
        float xj[4];
        Pack<float>::unpack(ld16(xs + s * sbb + 16 * i), xj);
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) rt[r4] = fmaf(rem, xj[r4], rt[r4]);
      } else {
        uint32_t pc[3];
        bf16_pieces(rem, pc);
        const u32x4 rb = {pc[0] | pc[1] << 16, pc[2] | pc[0] << 16, pc[1] | pc[0] << 16, 0u};
        tot = mfma16x16(ld16(xs + s * sbb + 16 * i), rb, tot, __bf16{});
      }
    }
    if constexpr (__is_same(T, _Float16)) {  // the operands hold the scales
      f32x4 a[2] = {};
#pragma unroll
      for (int j = 0; j < 8; ++j)
        a[j & 1] = mfma16x16(ld16(xb + 64 * j), kv_operand(r, j, g, sub[j & 1][j >> 1], T{}), a[j & 1], T{});
#pragma unroll
      for (int e = 0; e < NE; ++e) tot[e] = fmaf(d * 0x1p14f, a[0][e] + a[1][e], tot[e]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const u32x4 w = kv_operand(r, j, g, sub[j & 1][j >> 1], T{});
        f32x4 a = {};
#pragma unroll
        for (int p = XP - 1; p >= 0; --p) a = mfma16x16(ld16(xb + p * m * kKvRow + 64 * j), w, a, T{});
        const float sj = d * (float)byte_of(sc[j >> 2], j & 3);
#pragma unroll
        for (int e = 0; e < NE; ++e) tot[e] = fmaf(sj, a[e], tot[e]);
      }
    }
  };

  // a barrier that leaves the weights' transfers in flight (a workgroup fence would drain them)
  auto barrier = [] {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  int c0 = 0, slot = 0;  // the staged chunk's first superblock
  const uint8_t* const wl = ring + c * Raw::kBlock;
#pragma unroll 1
  for (int i = 0; i < per; ++i) {
    if (i == 0 || i - c0 == chunk) {
      if (i > 0) barrier();  // everyone is done with the previous chunk
      c0 = i;
      if (i < cnt) stage(i);
      barrier();
    }
    const int prev = slot == 0 ? kKvStages - 1 : slot - 1;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the previous stage's reads are done
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    issue(i + kKvStages - 1, prev);
    wait_vm<(kKvStages - 1) * Stage::kDma>();  // this stage's transfers have landed
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (i < cnt) {  // uniform
      Raw raw;
      raw.load(wl + slot * Stage::kBytes, g);
      compute(raw, i - c0);
    }
    slot = slot == kKvStages - 1 ? 0 : slot + 1;
  }
  wait_vm<0>();
  if constexpr (NE == 1) {  // row g: its remainders' part from all lane groups
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      float v = rt[r4] + __shfl_xor(rt[r4], 16);
      v += __shfl_xor(v, 32);
      if (g == r4) tot[0] += v;
    }
  }

  // lane l, value e: row l / 16 + 4 e, column l % 16.  Sums that came out infinite or NaN, again
  // on the fp32 matrix cores (v_mfma_f32_16x16x4: value i of the four lane groups at a time).
  const int64_t col = col0 + c;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < NE; ++e) bad = bad || (g + 4 * e < m && col < n && !__builtin_isfinite(tot[e]));
  if (__any(bad)) {
    const Table<8, TX> xt{x};
    using Plain = std::conditional_t<KIND == NVF_Q4_K, Q4K<8, LAYOUT>, Q5K<8>>;
    const Plain wt{wq};
    const int64_t x0 = (int64_t)xrow * k + 8 * g, w0 = (col < n ? col : n - 1) * k + 8 * g;
    f32x4 v = {};
#pragma unroll 1
    for (int64_t i = (int64_t)sb0 * 256; i < (int64_t)(sb0 + cnt) * 256; i += 128) {
      typename Table<8, TX>::Raw xr4[4];
      typename Plain::Raw wr4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // the loads of four steps go out together
        xr4[u] = xt.load(x0 + i + 32 * u);
        wr4[u] = wt.load(w0 + i + 32 * u);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float xv[8], wv[8];
        xt.decode(xr4[u], xv);
        wt.decode(wr4[u], wv);
#pragma unroll
        for (int q = 0; q < 8; ++q) v = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[q], wv[q], v, 0, 0, 0);
      }
    }
#pragma unroll
    for (int e = 0; e < NE; ++e)
      if (!__builtin_isfinite(tot[e])) tot[e] = v[e];
  }
  if constexpr (KG > 1) {  // the K groups' sums, in group order
    __syncthreads();
    float* part = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int e = 0; e < NE; ++e)
      if (kg > 0) part[(((kg - 1) * WC + wc) * NE + e) * 64 + lane] = tot[e];
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int q = 1; q < KG; ++q)
#pragma unroll
      for (int e = 0; e < NE; ++e) tot[e] += part[(((q - 1) * WC + wc) * NE + e) * 64 + lane];
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int r = g + 4 * e;
    if (r < m && col < n) out[(int64_t)r * n + col] = from_f32<TO>(tot[e]);
  }
}

constexpr int kKvLds = 160 * 1024;
template <typename TX, int BLOCK>
int kv_lds(int m, int waves, int kg, int chunk) {  // the rings and x; the groups' partial sums reuse the rings
  static_assert(KvStage<BLOCK>::kBytes * kKvStages >= 64 * 16, "partial sums");
  return waves * kKvStages * KvStage<BLOCK>::kBytes + kg * chunk * kv_sb_bytes<TX>(m);
}

// (A function per kernel, so that each has a flag of its own: the kernels are of one type.)
template <typename TX, int KIND, int LAYOUT, typename TO, int WC, int KG, int NE>
int launch_kv_kernel(const TX* x, const uint8_t* w, TO* out, int m, int64_t n, int64_t k, int chunk, int lds,
                     hipStream_t st) {
  auto kern = kq_gemv_kernel<TX, KIND, LAYOUT, TO, WC, KG, NE>;
  static std::once_flag attr_once;
  static hipError_t attr = hipSuccess;
  std::call_once(attr_once, [&] {
    attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kKvLds);
  });
  if (attr != hipSuccess)
    return fail(NVF_ERR_LAUNCH, "dense_gemv (K-quant): %d bytes of LDS: %s", kKvLds, hipGetErrorString(attr));
  kern<<<dim3((unsigned)((n + 16 * WC - 1) / (16 * WC))), WC * KG * 64, lds, st>>>(x, w, out, m, n, k, chunk);
  return launch_status("dense_gemv (K-quant)");
}

// Narrow outputs split K over the workgroup's 8 waves, where kq_gemv_wins sends up to 8 rows (fp32 x:
// 4) here; x then fits the LDS (145 KB at most, 4 rows of fp32 x on Q5_K).
template <typename TX>
constexpr int kKvSplitRows = sizeof(TX) == 4 ? 4 : 8;

template <typename TX, int KIND, int LAYOUT, typename TO, int WC, int KG>
int launch_kv(const TX* x, const uint8_t* w, TO* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  constexpr int kBlock = KvRaw<KIND, LAYOUT>::kBlock;
  // x: the group's whole K where it is small, else chunks of about 16 KB per workgroup (three
  // workgroups of four waves per CU)
  const int per = ((int)(k >> 8) + KG - 1) / KG;
  const int room = kKvLds - WC * KG * kKvStages * KvStage<kBlock>::kBytes;
  const int most = ((room < 16 * 1024 ? room : 16 * 1024) / KG) / kv_sb_bytes<TX>((int)m);
  const int chunk = most < 1 ? 1 : most < per ? most : per;
  const int lds = kv_lds<TX, kBlock>((int)m, WC * KG, KG, chunk);
  constexpr int kMost = KG == 1 ? 16 : kKvSplitRows<TX>;
  if constexpr (kMost > 8)
    if (m > 8) return launch_kv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 4>(x, w, out, (int)m, n, k, chunk, lds, st);
  if constexpr (kMost > 4)
    if (m > 4) return launch_kv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 2>(x, w, out, (int)m, n, k, chunk, lds, st);
  return launch_kv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 1>(x, w, out, (int)m, n, k, chunk, lds, st);
}

template <typename TX, int KIND, int LAYOUT, typename TO>
int launch_kv_split(const void* x, const uint8_t* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  const TX* xp = static_cast<const TX*>(x);
  TO* op = static_cast<TO*>(out);
  if (n < 16384 && m <= kKvSplitRows<TX>) return launch_kv<TX, KIND, LAYOUT, TO, 1, 8>(xp, w, op, m, n, k, st);
  return launch_kv<TX, KIND, LAYOUT, TO, 4, 1>(xp, w, op, m, n, k, st);
}

template <typename TX, typename TO>
int dispatch_kv(const void* x, const uint8_t* w, int kind, int layout, void* out, int64_t m, int64_t n, int64_t k,
                hipStream_t st) {
  switch (kind) {
    case NVF_W_Q4_K:
      if (layout == NVF_QK_LAYOUT_HIP_LEGACY)
        return launch_kv_split<TX, NVF_Q4_K, NVF_QK_LAYOUT_HIP_LEGACY, TO>(x, w, out, m, n, k, st);
      return launch_kv_split<TX, NVF_Q4_K, NVF_QK_LAYOUT_GGML, TO>(x, w, out, m, n, k, st);
    default:
      return launch_kv_split<TX, NVF_Q5_K, NVF_QK_LAYOUT_GGML, TO>(x, w, out, m, n, k, st);
  }
}

int kq_gemv(const void* x, int x_dtype, const void* w, int kind, int layout, void* out, int out_dtype, int64_t m,
            int64_t n, int64_t k, hipStream_t st) {
  int rc = NVF_OK;
  const uint8_t* wb = static_cast<const uint8_t*>(w);
  NVF_DISPATCH_DTYPE(x_dtype, TX,
                     NVF_DISPATCH_DTYPE(out_dtype, TO, rc = (dispatch_kv<TX, TO>(x, wb, kind, layout, out, m, n, k,
                                                                                 st))));
  return rc;
}

}  // namespace nvf
