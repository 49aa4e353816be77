// Projections of a longer prompt over f16 weights, y[t][n] = x[t] . W[n], where
// the output is too small for the library's tiles to fill the GPU: 512 tokens
// of a 2560 x 9728 matrix are 80 tiles of 128 x 128 for 256 CUs, and the
// library's kernel runs at 500 TFLOP/s there.  K is split over the grid as well.
//
// Split: 32 TB tokens x 128 weight rows x a range of K per workgroup of 4 waves
// (16 TB x 64 each), `splits` ranges; the ranges' fp32 sums are added by the
// projection's consumer as tok_gemm.hip's are.  Weight rows are the MFMA's A
// operand (v_mfma_f32_16x16x32_f16), tokens its B operand: a lane ends with 4
// consecutive outputs of one token.
//
// What bounds it: a step of 64 k needs 32 KB from L2 and 64 KB out of LDS per
// 512 MFMA cycles of a SIMD, so the load path and LDS run as long as the matrix
// cores.  Two workgroups per CU with two steps of LDS each hide each other's
// barrier (512 x 2560 x 9728: 39.4 us; one workgroup with three or four steps 40.0;
// 256 weight rows per workgroup, a third less LDS traffic per MFMA, 40.1).
// Against the library, us: Qwen3-4B down 512 tokens 50.9 -> 39.4, o_proj 21.5
// -> 19.3, 131 tokens 28.6 -> 22.6, qkv 19.1 -> 13.0; Qwen3-32B down 200 tokens
// 255 -> 85, 512 tokens 270 -> 171.
// Prefill of 4 layers, us: Qwen3-4B 131 tokens 642 -> 581, 200 748 -> 614, 512
// 931 -> 870; Qwen3-32B 200 tokens 2272 -> 1487, 512 3048 -> 2595; Qwen3-0.6B
// 200 tokens 486 -> 348.
#include "common.hpp"
#include "kernels.hpp"

namespace grout {

namespace {

typedef __attribute__((address_space(3))) void lds_void;

constexpr int kStep = 64;  // k per step: 128-byte LDS rows
constexpr int kRowBytes = 2 * kStep;
constexpr int kTileN = 128;               // weight rows per workgroup
constexpr int kBufferWord3 = 0x00020000;  // raw 32-bit buffer access
constexpr unsigned kOob = 0x80000000u;    // past every buffer: loads return zero
constexpr int kMaxBuffer = 0x7ffffff0;
constexpr int kSlots = 2;       // steps of LDS: one is read while the next one's loads are in flight
constexpr int kVmcnt0 = 0x0F70;  // s_waitcnt immediate: vmcnt(0) alone

struct TileArgs {
  const half_t* W;  // [N][K]
  const half_t* x;  // [M][K]
  half_t* y;        // one range of K: f16 rows ldy apart
  float* part;      // more: [range][M][ldy] fp32
  int M, N, K;
  long ldy;
  int steps;    // steps per range of K
  int tiles_m;  // token tiles
  int units;    // weight tiles times ranges
  int tiles_n;
  DivBy div_m, div_n;
};

}  // namespace

// TB: 16-token blocks per wave (32 TB tokens per workgroup).
template <int TB>
__global__ __launch_bounds__(256, 2) void tile_gemm_kernel(TileArgs A) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = 32 * TB;
  constexpr int kW = BM * kRowBytes;  // weights follow the tokens in a slot
  constexpr int kSlot = kW + kTileN * kRowBytes;
  // one LDS object per slot: a read of one does not wait for loads into another
  __shared__ __attribute__((aligned(1024))) unsigned char s_a[kSlot];
  __shared__ __attribute__((aligned(1024))) unsigned char s_b[kSlot];
  const int id = (int)blockIdx.x;
  // XCD id % 8 takes every eighth (weight tile, range), all its token tiles in
  // turn: the weights of a tile are read into one L2 only
  const int local = id >> 3;
  const int lu = (int)div_by((uint32_t)local, A.div_m);
  const int tm = local - lu * A.tiles_m;
  const int unit = 8 * lu + (id & 7);
  if (unit >= A.units) return;
  const int range = (int)div_by((uint32_t)unit, A.div_n);
  const int tn = unit - range * A.tiles_n;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  const int wm = w & 1, wn = w >> 1;
  const int t0 = tm * BM, n0 = tn * kTileN;
  const int K = A.K;
  const int s0 = range * A.steps, s1 = min(s0 + A.steps, K / kStep);

  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<half_t*>(A.x) + (size_t)t0 * K, (short)0,
      (int)min((long)(A.M - t0) * K * 2, (long)kMaxBuffer), kBufferWord3);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<half_t*>(A.W) + (size_t)n0 * K, (short)0,
      (int)min((long)(A.N - n0) * K * 2, (long)kMaxBuffer), kBufferWord3);
  // A load instruction fills 8 rows: lane l row l / 8, stored chunk l % 8 =
  // logical chunk (l % 8) ^ (row % 8).  Rows past the end arrive as zeros.
  const unsigned lo = (unsigned)(lane >> 3) * (unsigned)K * 2u +
                      16u * (unsigned)((lane & 7) ^ (lane >> 3));
  const unsigned row8 = 16u * (unsigned)K;  // bytes of 8 rows
  auto issue = [&](int s, unsigned char* slot) __attribute__((always_inline)) {
    const unsigned o = s < s1 ? lo + (unsigned)s * kRowBytes : kOob;
#pragma unroll
    for (int i = 0; i < TB; ++i) {
      const unsigned j = (unsigned)(w * TB + i);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(slot + j * 1024), 16, o + j * row8,
                                               0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned j = (unsigned)(w * 4 + i);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(slot + kW + j * 1024), 16,
                                               o + j * row8, 0, 0, 0);
    }
  };

  floatx4 acc[4][TB];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int c0 = (kb ^ (col & 7)) << 4, c1 = c0 ^ 64;  // chunks kb and 4 + kb
  const int xo = (wm * 16 * TB + col) * kRowBytes, wo = kW + (wn * 64 + col) * kRowBytes;

  auto compute = [&](const unsigned char* slot) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = kk ? c1 : c0;
      half8 f[4], g[TB];
#pragma unroll
      for (int a = 0; a < 4; ++a)
        f[a] = as_half8(*reinterpret_cast<const u32x4*>(slot + wo + c + a * 16 * kRowBytes));
#pragma unroll
      for (int b = 0; b < TB; ++b)
        g[b] = as_half8(*reinterpret_cast<const u32x4*>(slot + xo + c + b * 16 * kRowBytes));
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a) acc[a][b] = mfma16x16x32(f[a], g[b], acc[a][b]);
    }
  };
  auto slot_at = [&](int u) __attribute__((always_inline)) -> unsigned char* {
    return u == 0 ? s_a : s_b;
  };
  issue(s0, s_a);
  for (int i = s0; i < s1; i += kSlots) {
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const int s = i + u;
      if (s >= s1) break;  // uniform over the workgroup
      __builtin_amdgcn_s_waitcnt(kVmcnt0);  // this step's loads
      // every wave's share has landed, and the other slot's reads are done
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      issue(s + 1, slot_at(u ^ 1));
      __builtin_amdgcn_sched_barrier(0);
      compute(slot_at(u));
    }
  }
  __builtin_amdgcn_s_waitcnt(kVmcnt0);  // no load into LDS outlives the workgroup

#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int t = t0 + (wm * TB + b) * 16 + col;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int n = n0 + wn * 64 + 16 * a + 4 * kb;  // N % 4 == 0: four outputs or none
      if (t >= A.M || n >= A.N) continue;
      if (A.part != nullptr) {
        *reinterpret_cast<floatx4*>(A.part + ((size_t)range * A.M + t) * A.ldy + n) = acc[a][b];
      } else {
        half4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (half_t)acc[a][b][e];
        *reinterpret_cast<u32x2*>(A.y + (size_t)t * A.ldy + n) = __builtin_bit_cast(u32x2, o);
      }
    }
  }
#endif
}

constexpr int kTileMaxSplits = 12;

// 16-token blocks per wave: the fewest that cover M in tiles of at most 128
// tokens.
static int tile_tb(int M) {
  const int tiles = (M + 127) / 128;
  return (M + 32 * tiles - 1) / (32 * tiles);
}

// Shapes this kernel takes.
bool tile_gemm_ok(int M, int N, int K) {
  return M >= 1 && N >= 4 && N % 4 == 0 && K >= 128 && K % kStep == 0 && K <= 32768;
}

static long tile_workgroups(int M, int N) {
  const int bm = 32 * tile_tb(M);
  return (long)((M + bm - 1) / bm) * ((N + kTileN - 1) / kTileN);
}

// Where this kernel is the faster route for a projection of N rows in all: at
// least three ranges of K at two workgroups per CU.  us, library / here: 4B
// o_proj 800 tokens (140 tiles) 30.5 / 26.6, 1024 (160) 30.9 / 29.8; 32B qkv
// 200 (160) 50.3 / 39.6; with more tiles 4B qkv 512 (192) 25.4 / 26.2, 1024
// (384) 34.7 / 43.3, 4B gate_up 512 (608) 57 / 88.
bool tile_gemm_pays(int M, int N) {
  return M > 64 && M <= kTileMax && tile_workgroups(M, N) * 3 <= 512;
}

// Ranges of K.  Estimated time in units of 0.1 us: a step takes 0.8 us with a CU
// to itself and 1.2 where two workgroups share it, and every range's sums are
// written and read again at ~5 TB/s.
int tile_gemm_splits(int M, int N, int K) {
  const long wgs = tile_workgroups(M, N);
  const int steps = K / kStep;
  long best = 0;
  int pick = 1;
  for (int s = 1; s <= kTileMaxSplits && s * 4 <= steps; ++s) {
    const int per = (steps + s - 1) / s;
    if ((long)per * (s - 1) >= steps) continue;  // an empty range
    const long n = wgs * s, rounds = (n + 511) / 512;
    const long t = per * (n <= 256 ? 8 : 12 * rounds) +
                   (s > 1 ? (long)s * M * N / 62500 : 0);
    if (s == 1 || t < best) {
      best = t;
      pick = s;
    }
  }
  return pick;
}

hipError_t launch_tile_gemm(const void* W, const void* x, void* y, float* part, long ldy, int M,
                            int N, int K, int splits, hipStream_t stream) {
  if (!tile_gemm_ok(M, N, K) || splits < 1 || (splits > 1 && part == nullptr) || ldy % 4)
    return hipErrorInvalidValue;
  const int tb = tile_tb(M);
  TileArgs a{};
  a.W = (const half_t*)W;
  a.x = (const half_t*)x;
  a.y = (half_t*)y;
  a.part = splits > 1 ? part : nullptr;
  a.M = M;
  a.N = N;
  a.K = K;
  a.ldy = ldy;
  a.steps = (K / kStep + splits - 1) / splits;
  if ((long)a.steps * (splits - 1) >= K / kStep) return hipErrorInvalidValue;  // an empty range
  a.tiles_m = (M + 32 * tb - 1) / (32 * tb);
  a.tiles_n = (N + kTileN - 1) / kTileN;
  const long units = (long)a.tiles_n * splits;
  const long grid = (units + 7) / 8 * 8 * a.tiles_m;
  if (grid > 0x3fffffff) return hipErrorInvalidValue;
  a.units = (int)units;
  a.div_m = make_div(a.tiles_m);
  a.div_n = make_div(a.tiles_n);
  switch (tb) {
    case 1: tile_gemm_kernel<1><<<(unsigned)grid, 256, 0, stream>>>(a); break;
    case 2: tile_gemm_kernel<2><<<(unsigned)grid, 256, 0, stream>>>(a); break;
    case 3: tile_gemm_kernel<3><<<(unsigned)grid, 256, 0, stream>>>(a); break;
    default: tile_gemm_kernel<4><<<(unsigned)grid, 256, 0, stream>>>(a); break;
  }
  return hipGetLastError();
}

}  // namespace grout
