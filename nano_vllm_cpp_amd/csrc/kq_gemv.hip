// Decode product on Q4_K and Q5_K weights: out[m][n] = x[m][k] . W[n][k]^T,
// m <= 16, k a multiple of 256, on the 16-bit matrix cores.
//
// Bound by the weights' stream from HBM as long as decoding them costs about 2 VALU
// instructions per weight; decoding each to fp32 and multiplying on the VALU takes 5.2 at one
// row, and the fp32 matrix cores are slower still.  Here only the whole quant q becomes a
// 16-bit operand (for fp16 a mask: a subnormal; for bf16 a conversion), one
// v_mfma_f32_16x16x32 sums a sub-block's 32 exact products x q for 16 rows and 16 columns, and
// the sub-block's scale takes one fused multiply-add per four rows and 512 weights.  The
// minimum's part is one MFMA per superblock, over the sub-blocks' sums of x (three exact bf16
// pieces) and the m_j.  fp16 x takes fp16 operands; bf16 x bf16; fp32 x three exact
// bf16 pieces.
//
// A wave owns 16 columns: lane l holds column l % 16 and, of every sub-block, the values
// 8 (l / 16) .. + 7.  Read straight from memory in that layout a superblock takes 5 loads that
// each touch 16 cache lines, and the L1's line rate bounds the kernel (1 x 151936 x 4096 Q4_K
// 119 us); so the weights go HBM -> LDS by DMA, whole runs of each column at a time, into
// a ring of kKvStages superblocks that is the wave's own.  WC waves of a
// workgroup on other columns share the staged x; KG groups of them split K for
// narrow outputs.
//
// fp16 x, Q4_K: 1 x 151936 x 4096 (350 MB) 136 us on decoded weights -> 67 (5.2 TB/s); 1 x
// 37888 x 3584 29.5 -> 22.5 us, 8 x 37888 x 3584 59 -> 27.  With the quants read in that
// layout straight from memory the first took 119 us, with fp16 conversions instead of
// subnormals 74, and with every LDS read draining the transfers (see u32x2) 96.
//
// Infinities and NaN: outputs that come out non-finite are recomputed weight by weight, as
// in kq_gemm.hip.

#include <mutex>

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
  __device__ __forceinline__ float d() const { return half_bits_to_f32(hdr[0] & 0xffffu); }
  __device__ __forceinline__ float dmin() const { return half_bits_to_f32(hdr[0] >> 16); }
  // the eight 6-bit scales and minima, one per byte
  __device__ __forceinline__ void tables(uint32_t* sc, uint32_t* mn) const {
    sc[0] = hdr[1] & 0x3f3f3f3fu;
    mn[0] = hdr[2] & 0x3f3f3f3fu;
    sc[1] = (hdr[3] & 0x0f0f0f0fu) | ((hdr[1] >> 2) & 0x30303030u);
    mn[1] = ((hdr[3] >> 4) & 0x0f0f0f0fu) | ((hdr[2] >> 2) & 0x30303030u);
  }
};

template <int LAYOUT>
struct KvRaw<NVF_Q5_K, LAYOUT> : KvRaw<NVF_Q4_K, NVF_QK_LAYOUT_GGML> {
  using Base = KvRaw<NVF_Q4_K, NVF_QK_LAYOUT_GGML>;
  static constexpr int kBlock = 176;
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

// The quants 8 g .. + 7 of sub-block s as 16-bit operands, and 1 / their unit.
template <typename Raw>
__device__ __forceinline__ u32x4 kv_operand(const Raw& r, int s, int g, float& unit, _Float16) {
  unit = (s & 1) ? Raw::kOdd : 0x1p24f;
  return r.halves(s, g);
}
template <typename Raw>
__device__ __forceinline__ u32x4 kv_operand(const Raw& r, int s, int g, float& unit, __bf16) {
  unit = 1.0f;
  uint32_t b[2];
  r.bytes(s, g, b);
  u32x4 p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // at most 5 significant bits: the upper halves of the fp32 values
    const float v0 = (float)byte_of(b[i >> 1], 2 * (i & 1)), v1 = (float)byte_of(b[i >> 1], 2 * (i & 1) + 1);
    p[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, v1), __builtin_bit_cast(uint32_t, v0), 0x07060302u);
  }
  return p;
}

// x as staged: XP planes of 16-bit values (fp32: three exact bf16 pieces), rows of a
// superblock 528 bytes apart (the 16 rows of a read phase on distinct banks), then the
// sub-blocks' sums as three bf16 pieces, [row][piece][8].
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
constexpr int kKvRow = 528, kKvZero = 16;  // kKvZero bytes of zeros lead the LDS
template <typename TX>
constexpr int kv_sb_bytes(int m) {
  return m * (KvX<TX>::kPlanes * kKvRow + 48);
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
  uint8_t* const ring = lds + kKvZero + wave * (kKvStages * Stage::kBytes);
  uint8_t* const xl = lds + kKvZero + WC * KG * (kKvStages * Stage::kBytes) + kg * chunk * sbb;

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
  if (threadIdx.x < kKvZero / 4) reinterpret_cast<uint32_t*>(lds)[threadIdx.x] = 0;

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
        const uint32_t h = __builtin_bit_cast(uint32_t, sum) & 0xffff0000u;
        const float r1 = sum - __builtin_bit_cast(float, h);
        const __bf16 b1 = (__bf16)r1, b2 = (__bf16)(r1 - (float)b1);
        uint16_t* xs = reinterpret_cast<uint16_t*>(xl + s * sbb + XP * m * kKvRow + r * 48) + (ch >> 2);
        xs[0] = (uint16_t)(h >> 16);
        xs[8] = __builtin_bit_cast(uint16_t, b1);
        xs[16] = __builtin_bit_cast(uint16_t, b2);
      }
    }
  };

  // Row r of x is operand row 4 (r % 4) + r / 4, so that lane group g's results e < NE are
  // rows g + 4 e: up to 4 NE rows cost NE multiply-adds per sub-block.  Operand rows of no
  // row of x repeat row 0; their results are not stored.
  float tot[NE] = {};
  const int xr = (c >> 2) + 4 * (c & 3), xrow = xr < m ? xr : 0;
  const uint8_t* const xa = xl + xrow * kKvRow + 16 * g;
  const uint8_t* const xs = xl + XP * m * kKvRow + xrow * 48 + 16 * g;
  auto compute = [&](const Raw& r, int s) {  // superblock s of the staged chunk
    const uint8_t* xb = xa + s * sbb;
    const float d = r.d();
    uint32_t sc[2], mn[2];
    r.tables(sc, mn);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float unit;
      const u32x4 w = kv_operand(r, j, g, unit, T{});
      f32x4 a = {};
#pragma unroll
      for (int p = XP - 1; p >= 0; --p) a = mfma16x16(ld16(xb + p * m * kKvRow + 64 * j), w, a, T{});
      const float sj = (d * unit) * (float)byte_of(sc[j >> 2], j & 3);
#pragma unroll
      for (int e = 0; e < NE; ++e) tot[e] = fmaf(sj, a[e], tot[e]);
    }
    u32x4 mb;  // m_j in bf16 (6 bits)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float m0 = (float)byte_of(mn[i >> 1], 2 * (i & 1)), m1 = (float)byte_of(mn[i >> 1], 2 * (i & 1) + 1);
      mb[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, m1), __builtin_bit_cast(uint32_t, m0), 0x07060302u);
    }
    const f32x4 mm = mfma16x16(ld16(g < 3 ? xs + s * sbb : lds), mb, f32x4{}, __bf16{});
    const float dm = -r.dmin();
#pragma unroll
    for (int e = 0; e < NE; ++e) tot[e] = fmaf(dm, mm[e], tot[e]);
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

  // lane l, value e: row l / 16 + 4 e, column l % 16
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
  const int64_t col = col0 + c;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int r = g + 4 * e;
    if (r >= m || col >= n) continue;
    float v = tot[e];
    if (!__builtin_isfinite(v)) {
      v = 0.0f;
#pragma unroll 1
      for (int64_t i = 0; i < k; i += 4) {
        float wv[4];
        if constexpr (KIND == NVF_Q4_K) {
          const Q4K<4, LAYOUT> w{wq};
          w.decode(w.load(col * k + i), wv);
        } else {
          const Q5K<4> w{wq};
          w.decode(w.load(col * k + i), wv);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) v = fmaf(to_f32(x[(int64_t)r * k + i + q]), wv[q], v);
      }
    }
    out[(int64_t)r * n + col] = from_f32<TO>(v);
  }
}

constexpr int kKvLds = 160 * 1024;
template <typename TX, int BLOCK>
int kv_lds(int m, int waves, int kg, int chunk) {
  const int part = (waves - waves / kg) * 64 * 16;
  const int bytes = kKvZero + waves * kKvStages * KvStage<BLOCK>::kBytes + kg * chunk * kv_sb_bytes<TX>(m);
  return bytes > part ? bytes : part;
}

template <typename TX, int KIND, int LAYOUT, typename TO, int WC, int KG>
int launch_kv(const TX* x, const uint8_t* w, TO* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  constexpr int kBlock = KvRaw<KIND, LAYOUT>::kBlock;
  // x: the group's whole K where it is small, else chunks of about 16 KB per workgroup (three
  // workgroups of four waves per CU)
  const int per = ((int)(k >> 8) + KG - 1) / KG;
  const int room = kKvLds - kKvZero - WC * KG * kKvStages * KvStage<kBlock>::kBytes;
  const int most = ((room < 16 * 1024 ? room : 16 * 1024) / KG) / kv_sb_bytes<TX>((int)m);
  const int chunk = most < 1 ? 1 : most < per ? most : per;
  const int lds = kv_lds<TX, kBlock>((int)m, WC * KG, KG, chunk);
  const dim3 grid((unsigned)((n + 16 * WC - 1) / (16 * WC)));
  auto launch = [&](auto kern) {
    static std::once_flag attr_once;
    std::call_once(attr_once, [&] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kKvLds);
    });
    kern<<<grid, WC * KG * 64, lds, st>>>(x, w, out, (int)m, n, k, chunk);
  };
  if (m <= 4)
    launch(kq_gemv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 1>);
  else if (m <= 8)
    launch(kq_gemv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 2>);
  else
    launch(kq_gemv_kernel<TX, KIND, LAYOUT, TO, WC, KG, 4>);
  return launch_status("dense_gemv (K-quant)");
}

template <typename TX, int KIND, int LAYOUT, typename TO>
int launch_kv_split(const void* x, const uint8_t* w, void* out, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  constexpr int kBlock = KvRaw<KIND, LAYOUT>::kBlock;
  const TX* xp = static_cast<const TX*>(x);
  TO* op = static_cast<TO*>(out);
  if (n < 16384) {
    if (kv_lds<TX, kBlock>((int)m, 8, 8, 1) <= kKvLds)
      return launch_kv<TX, KIND, LAYOUT, TO, 1, 8>(xp, w, op, m, n, k, st);
    if (kv_lds<TX, kBlock>((int)m, 4, 4, 1) <= kKvLds)
      return launch_kv<TX, KIND, LAYOUT, TO, 1, 4>(xp, w, op, m, n, k, st);
  }
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
