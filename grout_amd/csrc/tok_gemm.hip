// Projections of a few tokens (a short prompt, the next turn of a chat) over
// f16 or low-bit weights: y[t][n] = x[t] . W[n] for 2 .. a few hundred tokens.
//
// What bounds it: up to ~64 tokens the weight bytes, as in a decode step (the
// library's GEMMs stream them at 1.9-4.1 TB/s for 18 tokens); a low-bit matrix
// is read in its own format and dequantized in registers, where the library
// needs a dequantized f16 copy written and read back first (7x the bytes of
// Q4_K).  Above that the x fragments that every wave reads from LDS.
//
// Split: a workgroup of 4 waves takes 64 weight rows (16 per wave) and a range
// of K; the grid covers the rows times `splits` ranges of K (about two
// workgroups per CU, so one computes while the other's loads are in flight)
// times blocks of 16 MT tokens.  Weight rows are the MFMA's A operand, tokens
// its B operand (v_mfma_f32_16x16x32_f16), so each lane ends with 4
// consecutive outputs of one token.  x is staged once per workgroup into
// LDS (direct-to-LDS, 16-byte chunks XOR-swizzled by the row, as the prefill
// attention's K tiles) and shared by the four waves: reading it per wave from
// L2 cost more than the weights themselves (18 tokens, 2560 x 9728: 18-19 us
// against 11.3).  f16 weights go the same way, 4 rows x 256 B per load
// instruction (16 rows x 64 B, which is the A operand's own order, streamed at
// 3.0 TB/s against 5.0 for 19456 x 2560); low-bit weights are loaded in the
// operand's order, 64 B of a row per instruction, and dequantized in
// registers.  Steps of SUB x 128 k are double-buffered.
//
// With more than one range of K the workgroups write fp32 partial sums that
// the projection's consumer (the norm, the norm/RoPE/KV write, SiLU * up) adds
// in range order and rounds to f16 once, so no launch is spent on the sum and
// the result does not depend on scheduling.
//
// Numerics: fp32 accumulation; a low-bit weight is the f16 rounding of the
// decode layout's fp32 value d*sc*q (- dmin*m), as the dequantized copy holds.
#include "common.hpp"
#include "kernels.hpp"
#include "quant_layout.hpp"

#include <type_traits>

namespace grout {

namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kF16 = 0;
constexpr int kWaves = 4;
constexpr int kRowsPerWg = 16 * kWaves;
constexpr int kSub = 128;           // k per sub-step: one 256-byte LDS row
constexpr int kSubBytes = 2 * kSub;
constexpr int kBufferWord3 = 0x00020000;  // raw 32-bit buffer access
constexpr unsigned kOob = 0x80000000u;    // past every buffer: loads return zero
constexpr int kMaxBuffer = 0x7ffffff0;
constexpr int kVmcnt0 = 0x0F70;  // s_waitcnt immediate: vmcnt(0) alone

struct TokArgs {
  const uint8_t* W;
  const half_t* x;  // [M][K]
  half_t* y;        // one range: f16 rows ldy apart
  float* part;      // more: [range][M][ldy] fp32
  int M, N, K;
  long ldy;
  int subs;  // sub-steps per range of K
  QLayout L;
};

// One row's raw bytes of a sub-step in one lane (32 weights).
template <int FMT>
struct Raw {};
template <>
struct Raw<8> {
  u32x4 a, b;  // q[16 kb ..], q[64 + 16 kb ..]
  u32x2 d;     // the sub-step's four block scales
};
template <>
struct Raw<12> {
  u32x4 a, h;  // qs[16 kb ..], header
};
template <>
struct Raw<13> {
  u32x4 a, b, h;  // qs, qh[16 (kb & 1) ..], header
};
template <>
struct Raw<14> {
  u32x4 a, b;   // ql[16 kb ..], qh[16 (kb & 1) ..]
  u32x2 sc;     // the sub-step's eight scales
  uint32_t d;
};

__device__ __forceinline__ float h2f_bits(uint32_t b) {
  return (float)__builtin_bit_cast(half_t, (uint16_t)b);
}

// Bytes 0, 1 (or 2, 3) of v as an f16 pair of denormals, byte * 2^-24.
__device__ __forceinline__ half2v dpair(uint32_t v, uint32_t sel) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(v, v, sel));
}

// Eight bytes q -> f16(q * s + c) in byte order; s carries the 2^24.
__device__ __forceinline__ half8 deq8(uint32_t w0, uint32_t w1, float s, float c) {
  half8 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2v p = dpair(i < 2 ? w0 : w1, (i & 1) ? 0x0C030C02u : 0x0C010C00u);
    o[2 * i] = (half_t)__builtin_fmaf((float)p[0], s, c);
    o[2 * i + 1] = (half_t)__builtin_fmaf((float)p[1], s, c);
  }
  return o;
}

// The four A fragments of sub-step s (of K) from a lane's raw bytes; fragment
// j holds the weights whose x chunk frag_chunk<FMT>(j, kb) names.
template <int FMT>
__device__ __forceinline__ void dequant_frags(int s, int kb, const Raw<FMT>& r, half8 (&f)[4]) {
  if constexpr (FMT == 8) {
    // blocks kb / 2 and 2 + kb / 2; bytes held as q + 128
    const float d0 = h2f_bits((kb >> 1) ? r.d[0] >> 16 : r.d[0] & 0xffffu);
    const float d1 = h2f_bits((kb >> 1) ? r.d[1] >> 16 : r.d[1] & 0xffffu);
    constexpr uint32_t flip = 0x80808080u;
    f[0] = deq8(r.a[0] ^ flip, r.a[1] ^ flip, d0 * 0x1p24f, -128.f * d0);
    f[1] = deq8(r.a[2] ^ flip, r.a[3] ^ flip, d0 * 0x1p24f, -128.f * d0);
    f[2] = deq8(r.b[0] ^ flip, r.b[1] ^ flip, d1 * 0x1p24f, -128.f * d1);
    f[3] = deq8(r.b[2] ^ flip, r.b[3] ^ flip, d1 * 0x1p24f, -128.f * d1);
  } else if constexpr (FMT == 12 || FMT == 13) {
    // 64-weight group g = 2 (s & 1) + kb / 2 of the superblock: sub-blocks 2g
    // (low nibbles) and 2g + 1 (high)
    const float d = h2f_bits(r.h[0] & 0xffffu), dmin = h2f_bits(r.h[0] >> 16);
    const int sh = 16 * (kb >> 1);
    uint32_t sc, mn;  // two 6-bit values, in bytes 0 and 1
    if (s & 1) {
      const uint32_t q8 = r.h[3] >> sh;
      sc = (q8 & 0x0f0fu) | (((r.h[1] >> sh) & 0xc0c0u) >> 2);
      mn = ((q8 >> 4) & 0x0f0fu) | (((r.h[2] >> sh) & 0xc0c0u) >> 2);
    } else {
      sc = (r.h[1] >> sh) & 0x3f3fu;
      mn = (r.h[2] >> sh) & 0x3f3fu;
    }
    float slo = d * (float)(sc & 0xff), mlo = dmin * (float)(mn & 0xff);
    float shi = d * (float)(sc >> 8), mhi = dmin * (float)(mn >> 8);
    uint32_t lo[4], hi[4];
    if constexpr (FMT == 12) {  // the decode layout's effective scales
      slo = (float)(half_t)slo;
      mlo = (float)(half_t)mlo;
      shi = (float)(half_t)shi * 0x1p-4f;  // hi bytes hold 16 q
      mhi = (float)(half_t)mhi;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = r.a[i] & 0x0F0F0F0Fu;
        hi[i] = r.a[i] & 0xF0F0F0F0u;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t t = r.b[i] >> (4 * (s & 1) + 2 * (kb >> 1));
        lo[i] = (r.a[i] & 0x0F0F0F0Fu) | ((t << 4) & 0x10101010u);
        hi[i] = ((r.a[i] >> 4) & 0x0F0F0F0Fu) | ((t << 3) & 0x10101010u);
      }
    }
    f[0] = deq8(lo[0], lo[1], slo * 0x1p24f, -mlo);
    f[1] = deq8(lo[2], lo[3], slo * 0x1p24f, -mlo);
    f[2] = deq8(hi[0], hi[1], shi * 0x1p24f, -mhi);
    f[3] = deq8(hi[2], hi[3], shi * 0x1p24f, -mhi);
  } else if constexpr (FMT == 14) {
    // half s & 1 of the superblock: 16-runs 2 ilo + (kb & 1) and 4 further
    const int ilo = kb >> 1, sb = 8 * (2 * ilo + (kb & 1));
    const float d = h2f_bits(r.d);
    const float slo = d * (float)(int8_t)((r.sc[0] >> sb) & 0xff);
    const float shi = d * (float)(int8_t)((r.sc[1] >> sb) & 0xff);
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t t = r.b[i] >> (2 * ilo);
      lo[i] = (r.a[i] & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u);
      hi[i] = ((r.a[i] >> 4) & 0x0F0F0F0Fu) | (t & 0x30303030u);
    }
    f[0] = deq8(lo[0], lo[1], slo * 0x1p24f, -32.f * slo);
    f[1] = deq8(lo[2], lo[3], slo * 0x1p24f, -32.f * slo);
    f[2] = deq8(hi[0], hi[1], shi * 0x1p24f, -32.f * shi);
    f[3] = deq8(hi[2], hi[3], shi * 0x1p24f, -32.f * shi);
  }
}

// 16-byte x chunk (8 k) of a sub-step that lane group kb multiplies with its
// fragment j.
template <int FMT>
__device__ __forceinline__ int frag_chunk(int j, int kb) {
  const int h = j & 1, hi = j >> 1;
  return FMT == kF16 ? 4 * j + kb
         : FMT == 8  ? 8 * hi + 2 * kb + h
         : FMT == 14 ? 8 * hi + 4 * (kb >> 1) + 2 * (kb & 1) + h
                     : 8 * (kb >> 1) + 4 * hi + 2 * (kb & 1) + h;
}

// LDS-only workgroup barrier (the loads of the next step stay in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

#ifdef __HIP_DEVICE_COMPILE__
// LDS of a workgroup: two slots of x, and of f16 weights.
constexpr int x_slot(int mt, int sub) { return sub * mt * 16 * kSubBytes; }
constexpr int w_slot(int fmt, int sub) { return fmt == kF16 ? kWaves * sub * 4096 : 16; }

template <int FMT, int MT, int SUB>
__device__ __forceinline__ void tok_gemm_rows(const TokArgs& A, int row_group,
                                              unsigned char (&s_x)[2][x_slot(MT, SUB)],
                                              unsigned char (&s_w)[2][w_slot(FMT, SUB)]) {
  constexpr bool WL = FMT == kF16;  // weights through LDS
  constexpr int XI = SUB * MT;      // x staging: 1 KiB instructions per wave and step
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, kb = lane >> 4;
  const int row0 = (row_group * kWaves + w) * 16;
  const int t0 = (int)blockIdx.z * MT * 16;
  const int K = A.K, N = A.N;
  const int s0 = (int)blockIdx.y * A.subs, s1 = min(s0 + A.subs, K / kSub);

  // Wave instruction i stages rows 4j .. 4j+3 (j = XI w + i counted over the
  // step's sub-steps), lane l row 4j + l/16, stored chunk l%16 = logical chunk
  // (l%16) ^ (row%16).  Rows past M lie past the buffer and arrive as zeros.
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<half_t*>(A.x) + (size_t)t0 * K, (short)0,
      (int)min((long)(A.M - t0) * K * 2, (long)kMaxBuffer), kBufferWord3);
  auto stage_x = [&](int s, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int j = w * XI + i;
      const int sub = j / (4 * MT), r = 4 * (j % (4 * MT)) + kb;
      unsigned o = (unsigned)r * (unsigned)K * 2u + 16u * (unsigned)(col ^ (r & 15)) +
                   (unsigned)(s + sub) * kSubBytes;
      o = s + sub < s1 ? o : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(s_x[slot] + j * 1024), 16, o, 0, 0,
                                               0);
    }
  };

  // Row strides (bytes) of the matrix's arrays; each array's buffer starts at
  // this wave's first row and ends with the matrix (rows past N read zeros).
  constexpr int NA = FMT == kF16 ? 1 : FMT == 8 || FMT == 12 ? 2 : FMT == 13 ? 3 : 4;
  unsigned rs[4] = {};
  if constexpr (FMT == kF16) {
    rs[0] = 2 * K;
  } else if constexpr (FMT == 8) {
    rs[0] = K;
    rs[1] = K / 16;
  } else {
    rs[0] = K / 2;
    rs[1] = FMT == 14 ? K / 4 : K / 16;
    rs[2] = FMT == 14 ? K / 16 : K / 8;
    rs[3] = K / 128;
  }
  __amdgpu_buffer_rsrc_t wr[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const long left = row0 < N ? (long)(N - row0) * (long)rs[i] : 0;
    wr[i] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(A.W) + A.L.off[i] + (size_t)row0 * rs[i], (short)0,
        (int)min(left, (long)kMaxBuffer), kBufferWord3);
  }
  auto stage_w = [&](int s, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int r = 4 * c + kb;
        unsigned o = (unsigned)r * rs[0] + 16u * (unsigned)(col ^ r) +
                     (unsigned)(s + sub) * kSubBytes;
        o = s + sub < s1 ? o : kOob;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            wr[0], (lds_void*)(s_w[slot] + (w * SUB + sub) * 4096 + c * 1024), 16, o, 0, 0, 2);
      }
  };
  auto load16b = [&](const __amdgpu_buffer_rsrc_t& r, unsigned o) __attribute__((always_inline)) {
    return (u32x4)__builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0);
  };
  auto load_raw = [&](int s, Raw<FMT>& r) __attribute__((always_inline)) {
    const bool live = s < s1;
    const unsigned us = (unsigned)s, kq = 16u * (unsigned)kb, kh = 16u * (unsigned)(kb & 1);
    if constexpr (FMT == 8) {
      const unsigned o = live ? (unsigned)col * rs[0] + kq + us * 128u : kOob;
      r.a = load16b(wr[0], o);
      r.b = load16b(wr[0], o + 64u);
      r.d = __builtin_amdgcn_raw_buffer_load_b64(
          wr[1], live ? (unsigned)col * rs[1] + us * 8u : kOob, 0, 0);
    } else if constexpr (FMT == 12 || FMT == 13) {
      r.a = load16b(wr[0], live ? (unsigned)col * rs[0] + kq + us * 64u : kOob);
      r.h = load16b(wr[1], live ? (unsigned)col * rs[1] + (us >> 1) * 16u : kOob);
      if constexpr (FMT == 13)
        r.b = load16b(wr[2], live ? (unsigned)col * rs[2] + kh + (us >> 1) * 32u : kOob);
    } else if constexpr (FMT == 14) {
      r.a = load16b(wr[0], live ? (unsigned)col * rs[0] + kq + us * 64u : kOob);
      r.b = load16b(wr[1], live ? (unsigned)col * rs[1] + kh + us * 32u : kOob);
      r.sc = __builtin_amdgcn_raw_buffer_load_b64(
          wr[2], live ? (unsigned)col * rs[2] + us * 8u : kOob, 0, 0);
      r.d = __builtin_amdgcn_raw_buffer_load_b16(
          wr[3], live ? (unsigned)col * rs[3] + (us >> 1) * 2u : kOob, 0, 0);
    }
  };

  int xf[4];  // LDS offset of fragment j's chunk in a 16-row tile
#pragma unroll
  for (int j = 0; j < 4; ++j) xf[j] = col * kSubBytes + ((frag_chunk<FMT>(j, kb) ^ col) << 4);

  floatx4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};

  Raw<FMT> raw[2][SUB];
  auto issue = [&](int s, int slot) __attribute__((always_inline)) {
    stage_x(s, slot);
    if constexpr (WL) {
      stage_w(s, slot);
    } else {
#pragma unroll
      for (int sub = 0; sub < SUB; ++sub) load_raw(s + sub, raw[slot][sub]);
    }
  };
  issue(s0, 0);
  for (int i = s0; i < s1; i += 2 * SUB) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int s = i + u * SUB;
      // Everything in flight is this step's.  The builtin, not inline asm: the
      // compiler then knows that the raw registers have landed and puts no
      // wait for the next step's loads in front of their use.
      __builtin_amdgcn_s_waitcnt(kVmcnt0);
      lds_barrier();  // every wave's share landed; the other slot is free
      if (s >= s1) break;  // uniform over the workgroup
      if (s + SUB < s1) issue(s + SUB, u ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int sub = 0; sub < SUB; ++sub) {
        half8 f[4];
        if constexpr (WL) {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            f[c] = as_half8(*reinterpret_cast<const u32x4*>(s_w[u] + (w * SUB + sub) * 4096 + xf[c]));
        } else {
          dequant_frags<FMT>(s + sub, kb, raw[u][sub], f);
        }
        const unsigned char* xs = s_x[u] + sub * MT * 16 * kSubBytes;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt] = mfma16x16x32(
                f[j], as_half8(*reinterpret_cast<const u32x4*>(xs + xf[j] + mt * 16 * kSubBytes)),
                acc[mt]);
      }
    }
  }

#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int t = t0 + 16 * mt + col, n = row0 + 4 * kb;  // N % 4 == 0: four outputs or none
    if (t >= A.M || n >= N) continue;
    if (A.part != nullptr) {
      *reinterpret_cast<floatx4*>(A.part + ((size_t)blockIdx.y * A.M + t) * A.ldy + n) = acc[mt];
    } else {
      half4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (half_t)acc[mt][e];
      *reinterpret_cast<u32x2*>(A.y + (size_t)t * A.ldy + n) = __builtin_bit_cast(u32x2, o);
    }
  }
}
#endif

template <int FMT, int MT, int SUB>
__global__ __launch_bounds__(kWaves * 64, 2) void tok_gemm_kernel(TokArgs A) {
#ifdef __HIP_DEVICE_COMPILE__
  __shared__ __attribute__((aligned(1024))) unsigned char s_x[2][x_slot(MT, SUB)];
  __shared__ __attribute__((aligned(1024))) unsigned char s_w[2][w_slot(FMT, SUB)];
  tok_gemm_rows<FMT, MT, SUB>(A, (int)blockIdx.x, s_x, s_w);
#endif
}

// Two matrices over the same x in one grid, low-bit formats: row groups
// [0, groups_a) of the first, the rest of the second.  The Q6_K V rows of a
// Q4_K_M layer are 16 row groups: a launch of their own left most CUs idle
// (Qwen3-4B, 131 tokens 9.2 us after the 16.3 us of Q and K).
template <int FA, int FB, int MT, int SUB>
__global__ __launch_bounds__(kWaves * 64, 2) void tok_gemm_pair_kernel(TokArgs A, TokArgs B,
                                                                      int groups_a) {
#ifdef __HIP_DEVICE_COMPILE__
  __shared__ __attribute__((aligned(1024))) unsigned char s_x[2][x_slot(MT, SUB)];
  __shared__ __attribute__((aligned(1024))) unsigned char s_w[2][w_slot(FA, SUB)];
  const int g = (int)blockIdx.x;
  if (g < groups_a)
    tok_gemm_rows<FA, MT, SUB>(A, g, s_x, s_w);
  else
    tok_gemm_rows<FB, MT, SUB>(B, g - groups_a, s_x, s_w);
#endif
}

// Token tiles of 16 per workgroup: the fewest that cover M in blocks of at
// most kMaxTiles.
constexpr int kMaxTiles = 10;
int tiles_for(int M) {
  const int all = (M + 15) / 16, blocks = (all + kMaxTiles - 1) / kMaxTiles;
  const int mt = (all + blocks - 1) / blocks;
  return mt;
}

}  // namespace

// Most tokens for which this kernel is the faster route.  Prefill of 4 layers
// (us) against the library's GEMMs over f16 or freshly dequantized weights:
// f16 4B 64 tokens 430 / 530, 96 496 / 553, 112 605 / 591; 32B 96 1176 / 1620;
// Q8_0 8B 300 1027 / 1260, 350 1346 / 1307; Q4_K_M 4B 480 856 / 1120; Q5_K_M
// 32B 480 3034 / 4242.
static int tok_max(int fmt) { return fmt == 0 ? 96 : fmt == 8 ? 320 : kTokMax; }

// Token counts and shapes this kernel takes.
bool tok_gemm_ok(int fmt, int M, int N, int K) {
  if (fmt != 0 && fmt != 8 && fmt != 12 && fmt != 13 && fmt != 14) return false;
  return M >= 2 && M <= tok_max(fmt) && N >= 4 && N % 4 == 0 && K >= kSub && K % (fmt == 0 || fmt == 8 ? kSub : 256) == 0 && K <= 32768;
}

// Ranges of K for a projection of N rows in all.
int tok_gemm_splits(int M, int N, int K) {
  const int mt = tiles_for(M);
  const long wgs = (long)((N + kRowsPerWg - 1) / kRowsPerWg) * ((M + 16 * mt - 1) / (16 * mt));
  const int units = (K / kSub + 1) / 2;  // pairs of sub-steps
  long s = (512 + wgs / 2) / wgs;
  s = s < 1 ? 1 : s > units ? units : s;
  const int per = (int)((units + s - 1) / s);
  return (units + per - 1) / per;
}

static unsigned row_groups(int N) { return (unsigned)((N + kRowsPerWg - 1) / kRowsPerWg); }

// SUB for MT token tiles: two sub-steps per barrier while x stays small
// (low-bit only: with f16 weights in LDS as well, one workgroup per CU would
// be left).
template <int FMT, int MT>
constexpr int sub_steps() { return FMT != kF16 && MT <= 2 ? 2 : 1; }

// Calls f(integral_constant<MT>) for the tile count of M tokens.
template <class F>
static hipError_t for_tiles(int M, F f) {
  switch (tiles_for(M)) {
#define GROUT_TILES(mt) case mt: f(std::integral_constant<int, mt>{}); break;
    GROUT_TILES(1) GROUT_TILES(2) GROUT_TILES(3) GROUT_TILES(4) GROUT_TILES(5)
    GROUT_TILES(6) GROUT_TILES(7) GROUT_TILES(8) GROUT_TILES(9) GROUT_TILES(10)
#undef GROUT_TILES
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int FMT>
static hipError_t tok_launch(const TokArgs& a, int splits, hipStream_t stream) {
  return for_tiles(a.M, [&](auto t) {
    constexpr int MT = decltype(t)::value;
    if constexpr (FMT != kF16 || MT <= 6) {  // f16: at most 96 tokens
      const dim3 grid(row_groups(a.N), (unsigned)splits, (unsigned)((a.M + 16 * MT - 1) / (16 * MT)));
      tok_gemm_kernel<FMT, MT, sub_steps<FMT, MT>()><<<grid, kWaves * 64, 0, stream>>>(a);
    }
  });
}

template <int FA, int FB>
static hipError_t tok_launch_pair(const TokArgs& a, const TokArgs& b, int splits,
                                  hipStream_t stream) {
  return for_tiles(a.M, [&](auto t) {
    constexpr int MT = decltype(t)::value;
    const unsigned ga = row_groups(a.N);
    const dim3 grid(ga + row_groups(b.N), (unsigned)splits,
                    (unsigned)((a.M + 16 * MT - 1) / (16 * MT)));
    tok_gemm_pair_kernel<FA, FB, MT, sub_steps<FA, MT>()>
        <<<grid, kWaves * 64, 0, stream>>>(a, b, (int)ga);
  });
}

static bool tok_args(TokArgs& a, int fmt, const void* W, const void* x, void* y, float* part,
                     long ldy, int M, int N, int K, int splits) {
  if (!tok_gemm_ok(fmt, M, N, K) || splits < 1 || (splits > 1 && part == nullptr) || ldy % 4)
    return false;
  a = TokArgs{};
  a.W = (const uint8_t*)W;
  a.x = (const half_t*)x;
  a.y = (half_t*)y;
  a.part = splits > 1 ? part : nullptr;
  a.M = M;
  a.N = N;
  a.K = K;
  a.ldy = ldy;
  const int units = (K / kSub + 1) / 2;
  a.subs = 2 * ((units + splits - 1) / splits);
  if (fmt != 0) a.L = qlayout(fmt, (size_t)N, (size_t)K);
  return (long)a.subs * (splits - 1) < K / kSub;  // no empty range
}

hipError_t launch_tok_gemm(int fmt, const void* W, const void* x, void* y, float* part, long ldy,
                           int M, int N, int K, int splits, hipStream_t stream) {
  TokArgs a;
  if (!tok_args(a, fmt, W, x, y, part, ldy, M, N, K, splits)) return hipErrorInvalidValue;
  switch (fmt) {
    case 0: return tok_launch<0>(a, splits, stream);
    case 8: return tok_launch<8>(a, splits, stream);
    case 12: return tok_launch<12>(a, splits, stream);
    case 13: return tok_launch<13>(a, splits, stream);
    default: return tok_launch<14>(a, splits, stream);
  }
}

bool tok_gemm_pair_ok(int fmt_a, int fmt_b) { return (fmt_a == 12 || fmt_a == 13) && fmt_b == 14; }

hipError_t launch_tok_gemm_pair(int fmt_a, const void* Wa, int Na, int fmt_b, const void* Wb,
                                int Nb, const void* x, void* y, float* part, long ldy, int M,
                                int K, int splits, hipStream_t stream) {
  TokArgs a, b;
  if (!tok_gemm_pair_ok(fmt_a, fmt_b) || Na % 4 ||
      !tok_args(a, fmt_a, Wa, x, y, part, ldy, M, Na, K, splits) ||
      !tok_args(b, fmt_b, Wb, x, y ? (half_t*)y + Na : nullptr, part ? part + Na : nullptr, ldy, M,
                Nb, K, splits))
    return hipErrorInvalidValue;
  return fmt_a == 12 ? tok_launch_pair<12, 14>(a, b, splits, stream)
                     : tok_launch_pair<13, 14>(a, b, splits, stream);
}

}  // namespace grout
