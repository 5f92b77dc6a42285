// The 16-bit matrix-core GEMM: out[m][n] = x[m][k] . W[n][k]^T with x and W both
// fp16 or both bf16, products exact in fp32, fp32 sums (v_mfma_f32_32x32x16).
//
// Bound by the matrix cores and the LDS reads that feed them; small m by the weights'
// stream.  Both operands go HBM -> LDS by DMA (no VALU and no registers in between: a
// 16-bit operand needs no conversion), K in 64-value stages in a ring of NS, one barrier
// per stage.  A wave of the 256 x 256 tile owns 128 x 64 outputs: 6 KB of LDS reads per 8
// MFMAs, three quarters of the LDS rate that a 64 x 64 wave would need.  4096 x 24576 x
// 4096 bf16: 2298 us on the three-piece split tile kernel (which takes any activation
// type) -> 690 us, 1195 TFLOP/s (670 to 725 over boxes); other shapes of the tile and of the
// stages, where this one took 669: 4 stages of 32 K-values 697 us, 4 waves of 128 x 128 755, 256 x 128 760.
// 24 x 151936 x 4096 (LM head): 447 -> 215 us, 5.8 TB/s of weights.
#pragma once

#include "nvf_device.hpp"
#include "nvf_host.hpp"

#include <array>

namespace nvf {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16 mfma16(const u32x4 a, const u32x4 b, const f32x16 c, __bf16) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}
__device__ __forceinline__ f32x16 mfma16(const u32x4 a, const u32x4 b, const f32x16 c, _Float16) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t g16_rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// One 1 KB transfer HBM -> LDS: lane l's 16 bytes at r[off + soff] go to dst + 16 l.  (A
// function of its own: kernels that call the builtin from a template can lose their
// launch stubs in the host pass.)
__device__ __forceinline__ void g16_dma(__amdgpu_buffer_rsrc_t r, uint8_t* dst, uint32_t off, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, off, soff, 0, 0);
}

// Waits until at most N of this wave's vector-memory operations are outstanding
// (lgkmcnt and expcnt untouched).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

constexpr int kG16Xcds = 8;

// Workgroup -> output tile, XCD-aware (as dg_tile): each XCD takes a contiguous
// range of an order that walks GM tile rows at a time column by column.
template <int GM>
__device__ __forceinline__ void g16_tile(int tiles_n, int& tm, int& tn) {
  const int tiles = (int)gridDim.x;
  const int tiles_m = tiles / tiles_n;
  const int xcd = (int)blockIdx.x % kG16Xcds, local = (int)blockIdx.x / kG16Xcds;
  const int per = tiles / kG16Xcds, extra = tiles % kG16Xcds;
  const int id = xcd * per + (xcd < extra ? xcd : extra) + local;
  const int gsz = GM * tiles_n;
  const int first = (id / gsz) * GM;
  const int rows_g = tiles_m - first < GM ? tiles_m - first : GM;
  const int in_g = id % gsz;
  tm = first + in_g % rows_g;
  tn = in_g / rows_g;
}

// Rows of a stage: BK 16-bit values in 16-byte chunks, chunk c of row r at position
// c ^ g16_key(r): the 16 consecutive rows of a ds_read_b128 phase then cover all 64
// banks (BK = 64: two rows per 256 bytes, BK = 32: four).
template <int BK>
__device__ __forceinline__ int g16_key(int row) {
  return BK == 64 ? (row >> 1) & 7 : (row >> 2) & 3;
}

// BM x BN outputs per workgroup, WM x WN waves in each of KG groups that split K (each
// with its own ring; for outputs with too few tiles to fill the GPU), NS stages of BK
// K-values per ring, OCC waves per SIMD asked of the compiler.  vec_out: rows of out are
// 16-byte aligned.  Needs k % 8 == 0, 16-byte aligned x and w, BM k and BN k < 2^30.
template <typename T, typename TO, int BM, int BN, int WM, int WN, int KG, int BK, int NS, int OCC>
__global__ __launch_bounds__(WM* WN* KG * 64) __attribute__((amdgpu_waves_per_eu(OCC))) void gemm16_kernel(
    const T* __restrict__ x, const T* __restrict__ w, TO* __restrict__ out, int64_t m, int64_t n, int64_t k,
    int tiles_n, int vec_out) {
  constexpr int kWaves = WM * WN;                      // of one K group
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // 32 x 32 MFMA tiles of a wave
  constexpr int kRowB = BK * 2, kCpr = kRowB / 16;     // bytes and chunks of a staged row
  constexpr int kRpi = 1024 / kRowB;                   // rows one 1 KB transfer moves
  constexpr int kStage = (BM + BN) * kRowB;
  constexpr int kDma = kStage / 1024 / kWaves;  // transfers per wave and stage
  static_assert(kStage % (1024 * kWaves) == 0 && BM % kRpi == 0, "stage transfers");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  int tm, tn;
  g16_tile<8>(tiles_n, tm, tn);
  const int64_t row0 = (int64_t)tm * BM, col0 = (int64_t)tn * BN;
  const int lane = threadIdx.x & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int group = KG == 1 ? 0 : wave_id / kWaves, wave = KG == 1 ? wave_id : wave_id % kWaves;
  const int wm = wave / WN, wn = wave % WN;
  uint8_t* const ring = lds + group * (NS * kStage);  // this K group's stages

  // tile-local buffer resources: rows past m / n fall outside and read zero
  const int64_t a_rows = m - row0 < BM ? m - row0 : BM;
  const int64_t b_rows = n - col0 < BN ? n - col0 : BN;
  const __amdgpu_buffer_rsrc_t ra = g16_rsrc(x + row0 * k, a_rows * k * 2);
  const __amdgpu_buffer_rsrc_t rb = g16_rsrc(w + col0 * k, b_rows * k * 2);

  // transfer t = wave * kDma + i of a stage: staged rows [t kRpi, +kRpi), activation rows first
  uint32_t off[kDma];
  int kchunk[kDma];  // element offset of this lane's chunk inside the stage
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = (wave * kDma + i) * kRpi + lane / kCpr;
    const int c = (lane % kCpr) ^ g16_key<BK>(r);
    kchunk[i] = c * 8;
    off[i] = (uint32_t)((r < BM ? r : r - BM) * k * 2) + (uint32_t)(c * 16);
  }
  // group g takes stages g, g + KG, ...; all make the same number of steps, the last
  // ones past the end and all zeros where KG does not divide the stages
  const int nst = (int)((k + BK - 1) / BK), steps = (nst + KG - 1) / KG;
  auto issue = [&](int step, int buf) {
    const int st = step * KG + group;
    const uint32_t kb = (uint32_t)st * kRowB;
    const bool tail = (int64_t)(st + 1) * BK > k;  // a partial stage, or one past the end: zeros
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const int t = wave * kDma + i;  // uniform
      uint32_t o = off[i];
      if (tail) o = (int64_t)st * BK + kchunk[i] < k ? o : 0x80000000u;
      g16_dma(t * kRpi < BM ? ra : rb, ring + buf * kStage + t * 1024, o, kb);
    }
  };

  f32x16 acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = f32x16{};

  // fragment addresses: lane l reads chunk 2 kk + l / 32 of row l % 32
  const int half = lane >> 5, lr = lane & 31;
  const int ar = wm * TM * 32 + lr, br = BM + wn * TN * 32 + lr;
  const int a0 = ar * kRowB + ((half ^ g16_key<BK>(ar)) << 4);
  const int b0 = br * kRowB + ((half ^ g16_key<BK>(br)) << 4);

#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, s);
  int buf = 0;
#pragma unroll 1
  for (int st = 0; st < steps; ++st) {
    wait_vm<(NS - 2) * kDma>();  // this wave's transfers of stage st have landed
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_barrier();  // everyone's have, and everyone is done with stage st - 1
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int nb = buf == 0 ? NS - 1 : buf - 1;  // the slot of stage st - 1
    issue(st + NS - 1, nb);
    const uint8_t* s = ring + buf * kStage;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      u32x4 xa[TM], wb[TN];
#pragma unroll
      for (int b = 0; b < TM; ++b) xa[b] = ld16(s + (a0 ^ (kk << 5)) + b * 32 * kRowB);
#pragma unroll
      for (int a = 0; a < TN; ++a) wb[a] = ld16(s + (b0 ^ (kk << 5)) + a * 32 * kRowB);
#pragma unroll
      for (int b = 0; b < TM; ++b)
#pragma unroll
        for (int a = 0; a < TN; ++a) acc[a][b] = mfma16(wb[a], xa[b], acc[a][b], T{});
    }
    buf = buf == NS - 1 ? 0 : buf + 1;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this stage's reads are done before the barrier
  }
  wait_vm<0>();
  __syncthreads();
  if constexpr (KG > 1) {  // the groups' partial sums meet in group order
    float* part = reinterpret_cast<float*>(lds);
    static_assert((KG - 1) * kWaves * TM * TN * 4096 <= KG * NS * kStage, "partial sums in LDS");
    if (group > 0) {
      u32x4* d = reinterpret_cast<u32x4*>(part) + ((group - 1) * kWaves + wave) * (TM * TN * 256) + lane;
#pragma unroll
      for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float v[4] = {acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
            d[((a * TM + b) * 4 + q) * 64] = Pack<float>::pack(v);
          }
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int g = 1; g < KG; ++g) {
        const u32x4* d = reinterpret_cast<const u32x4*>(part) + ((g - 1) * kWaves + wave) * (TM * TN * 256) + lane;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
          for (int b = 0; b < TM; ++b)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float v[4];
              Pack<float>::unpack(d[((a * TM + b) * 4 + q) * 64], v);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[a][b][4 * q + e] += v[e];
            }
      }
    }
    __syncthreads();
    if (group > 0) return;
  }

  // D layout: lane l, value j -> W row (output column) 8 (j / 4) + 4 (l / 32) + j % 4, x row
  // l % 32.  Each wave passes 32 output rows at a time through its own LDS so that a
  // store instruction writes whole 128-byte runs.
  constexpr int kCols = TN * 32, kPitch = kCols * (int)sizeof(TO) + 16;
  static_assert(kWaves * 32 * kPitch <= KG * NS * kStage, "epilogue LDS");
  uint8_t* mine = lds + wave * (32 * kPitch);
  constexpr int kVec = 16 / (int)sizeof(TO), kVpr = kCols / kVec;  // elements per vector, vectors per row
#pragma unroll
  for (int b = 0; b < TM; ++b) {
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[a][b][4 * jq + e];
        uint8_t* d = mine + lr * kPitch + (32 * a + 8 * jq + 4 * half) * (int)sizeof(TO);
        if constexpr (sizeof(TO) == 4) {
          st16(d, Pack<float>::pack(v));
        } else {
          TO t[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] = from_f32<TO>(v[e]);
          *reinterpret_cast<uint2*>(d) = __builtin_bit_cast(uint2, t);
        }
      }
    __builtin_amdgcn_wave_barrier();
    const int64_t r0 = row0 + wm * TM * 32 + 32 * b, c0 = col0 + wn * kCols;
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
}

}  // namespace nvf
