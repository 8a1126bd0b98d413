// dm_gguf_mm.hip -- GGUF MoE layers for many tokens per call on the matrix
// cores, without giving up 32-bit precision.
//
// A GGUF weight is a small integer times a scale of its block: Q3_K
// d (s - 32) (q - 4), Q4_K d s q - dmin m, Q8_0 d q.  The integers
// (s - 32)(q - 4) (at most 892 in magnitude), s q (at most 945) and q (8
// bits) are exact in f16, so they enter v_mfma_f32_16x16x32_f16 as they are,
// and the block scale d multiplies the fp32 partial sum of its columns.  An
// fp32 activation enters whole, as three f16 parts (two hold 23 of its 24
// bits): with s such that the row's largest value lies in [2^14, 2^15),
// hi = f16(x 2^s), mid = f16(2^12 (x 2^s - hi)) and lo = 2^12 (x 2^s - hi) -
// mid.  mid and lo meet the integers times 2^-12, exact in f16 too, so all
// products go into one fp32 accumulator, and a value far below its row's
// largest keeps its bits: hi + 2^-12 (mid + lo) is x 2^s exactly down to 2^-27
// of the largest value, and within 2^-51 of that value below.  (hi and a lo
// part unscaled lose bits from 2^-16 on, which counts where the weight at the
// largest value is zero: relative errors of 3e-4 to 2e-3 in a block's outputs
// against 2e-7 to 1e-6, and of the whole result where the leading bits of two
// activations cancel.)  Against 64 bits the block's outputs are as far off as
// those of the fp32 lane sums of dm_gguf.hip, or closer
// (tests/test_gpu_gguf_mm.py).
//
//   k_gguf_tile   (at upload) expert payloads -> records of 16 rows x 64
//                 columns in the order the matrix cores read them
//   k_gguf_split  fp32 rows -> f16 parts, the three of 64 columns side by
//                 side, and the row's exponent; Q4_K: the sums of 32 columns
//   k_gguf_mm     gate/up (h = SiLU(g) u) and down products over the units of
//                 launch_group_build
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dm_device.h"
#include "dm_gguf.h"
#include "dm_grouped.h"
#include "dm_layout.h"

namespace dm {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kMmCols = 64;                   // columns of a record and of a stage
constexpr int kMmThreads = 512;               // 8 waves
constexpr int kMmRowBytes = kMmCols * 2 * 2;  // a token row's hi and mid parts of a stage
constexpr int kMmRow3 = kMmCols * 3;          // elements of a token row and stage, all parts
constexpr float kMmMid = 4096.0f;             // scale of mid and lo

// Bytes of a record: the codes (lane l of a wave: row l & 15, columns
// 8 (l >> 4) .. + 7 of each 32), then the scales.
//   Q3_K  512 codes (4 bits) | f16 s - 32 [16 rows][2 halves of 32][2] | fp32 d [16]
//   Q4_K  512 codes | f16 s [16][2], padded to 8 bytes a row | even records:
//         f16 m [16][4] of the 128 columns from here; odd: fp32 d [16], dmin [16]
//   Q8_0  1024 codes (8 bits, + 128) | fp32 d [2][16]
template <int TY>
struct Rec {
  static constexpr int kCodes = TY == kGgmlQ8_0 ? 1024 : 512;
  static constexpr int kRest = TY == kGgmlQ3_K ? 192 : TY == kGgmlQ4_K ? 256 : 128;
  static constexpr int kBytes = kCodes + kRest;
  static constexpr bool kSums = TY == kGgmlQ4_K;  // column sums in a stage
  // direct-to-LDS loads of a wave and stage besides those of the token rows
  static constexpr int kDma = kCodes / 512 + 1 + (kSums ? 1 : 0);
};
// Tokens per unit: 64, where two workgroups' stages fit a CU (160 KB); the
// codes of Q8_0 leave room for 48.
constexpr int mm_tok(int type) { return type == kGgmlQ8_0 ? 48 : 64; }
// Stages of NCT column tiles: token rows (hi and mid, then lo), the 16 tiles'
// codes, their scales, the column sums.
template <int TY, int NCT>
struct MmBuf {
  // stages in flight
  static constexpr int kAhead = NCT > 2 || (NCT == 2 && TY == kGgmlQ8_0) ? 1 : 2;
  static constexpr int kBufs = kAhead + 1;
  static constexpr int kLoAt = 16 * NCT * kMmRowBytes;
  static constexpr int kB = kLoAt + kLoAt / 2;
  static constexpr int kSumsAt = kB + 16 * Rec<TY>::kBytes;
  static constexpr int kBytes = kSumsAt + (Rec<TY>::kSums ? 16 * NCT * 32 : 0);
  static constexpr int kRowLoads = NCT > 2 ? 2 : 1;  // of 32 rows over the 8 waves
  // The lo parts lie two rows to a line of 256 bytes.  Four column tiles: line r
  // holds rows r and r + 32, segment c of row r + 32 m at (8 m + c) ^ (r & 15), so
  // that the addresses are those of the hi and mid parts; else line l holds rows
  // 2 l + m, segment c at 8 m + (c ^ (l & 7)).
  static constexpr bool kLoFar = NCT == 4;
};
int rec_bytes(int type) {
  switch (type) {
    case kGgmlQ3_K: return Rec<kGgmlQ3_K>::kBytes;
    case kGgmlQ4_K: return Rec<kGgmlQ4_K>::kBytes;
    case kGgmlQ8_0: return Rec<kGgmlQ8_0>::kBytes;
    default: return 0;
  }
}

__device__ __forceinline__ float h2f_bits(uint32_t h) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
__device__ __forceinline__ uint32_t f16_bits(float v) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}

// Byte offset of matrix k (gate, up, down) of expert e (E: shared).
__host__ __device__ __forceinline__ size_t tile_offset(int E, int H, int I, int Ish, int rec,
                                                       int e, int k) {
  const size_t routed = (size_t)(I / 16) * (H / kMmCols) * rec;
  const size_t shared = (size_t)(Ish / 16) * (H / kMmCols) * rec;
  return e < E ? ((size_t)e * 3 + k) * routed : (size_t)E * 3 * routed + (size_t)k * shared;
}

// ---- upload ------------------------------------------------------------------
// Wave per record; grid.y = 3 e + k.
template <int TY>
__global__ __launch_bounds__(256) void k_gguf_tile(GgufMoeDev L, uint8_t* __restrict__ out) {
  const int m = blockIdx.y, e = m / 3, k = m % 3;
  const int n = e < L.E ? L.I : L.Ish;
  const int C = k < 2 ? L.H : n, R = k < 2 ? n : L.H;
  const int nS = C / kMmCols, i = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= (R / 16) * nS) return;
  const int s = i % nS, lane = threadIdx.x & 63, row = lane & 15, q = lane >> 4;
  const uint8_t* raw = L.raw + L.off[m];
  uint8_t* rec = out + tile_offset(L.E, L.H, L.I, L.Ish, Rec<TY>::kBytes, e, k) +
                 (size_t)i * Rec<TY>::kBytes;
  uint8_t* rest = rec + Rec<TY>::kCodes;
  const int64_t e0 = (int64_t)(16 * (i / nS) + row) * C + (int64_t)kMmCols * s;
  if constexpr (TY == kGgmlQ8_0) {
    uint8_t c[16];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const uint8_t* blk = raw + ((e0 >> 5) + kk) * 34;
#pragma unroll
      for (int b = 0; b < 8; ++b) c[8 * kk + b] = blk[2 + 8 * q + b] ^ 0x80;
      if (q == 0)
        reinterpret_cast<float*>(rest)[16 * kk + row] =
            h2f_bits(blk[0] | (uint32_t)blk[1] << 8);
    }
    uint32_t w[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      w[b] = c[4 * b] | (uint32_t)c[4 * b + 1] << 8 | (uint32_t)c[4 * b + 2] << 16 |
             (uint32_t)c[4 * b + 3] << 24;
    reinterpret_cast<uint4*>(rec)[lane] = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    constexpr int kBlk = TY == kGgmlQ3_K ? 114 : 144;
    const uint8_t* blk = raw + (e0 >> 8) * kBlk;
    // Q4_K: scale and min of sub-block j of the block (the packings of values4)
    auto q4_sm = [&](int j, int& sc, int& mn) {
      const uint8_t* p = blk + 4;
      if (j < 4) {
        sc = p[j] & 63;
        mn = p[j + 4] & 63;
      } else {
        const int lo = L.layout ? p[j + 4] : p[j];
        sc = (lo & 15) | ((p[j - 4] >> 6) << 4);
        mn = (lo >> 4) | ((p[j] >> 6) << 4);
      }
    };
    uint32_t w[2], sc2 = 0;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int el = (int)(e0 & 255) + 32 * kk + 8 * q;  // in the block (64 | e0)
      w[kk] = 0;
      int sc;
      if constexpr (TY == kGgmlQ3_K) {
        const uint32_t hm = blk[el >> 3];
        const uint32_t qs = blk[32 + (el >> 2)] | (uint32_t)blk[33 + (el >> 2)] << 8;
#pragma unroll
        for (int b = 0; b < 8; ++b)
          w[kk] |= ((((hm >> b) & 1) << 2) | ((qs >> (2 * b)) & 3)) << (4 * (b >> 1) + 16 * (b & 1));
        sc = (int)blk[96 + (el >> 4)] - 32;
      } else {
        const int j = el >> 5, r = el & 31;
#pragma unroll
        for (int b = 0; b < 8; ++b)
          w[kk] |= (uint32_t)((blk[16 + 16 * j + (r & 15) + b] >> (r < 16 ? 0 : 4)) & 15)
                   << (4 * (b >> 1) + 16 * (b & 1));
        int mn;
        q4_sm(j, sc, mn);
      }
      sc2 |= f16_bits((float)sc) << (16 * kk);
    }
    reinterpret_cast<uint2*>(rec)[lane] = make_uint2(w[0], w[1]);
    if constexpr (TY == kGgmlQ3_K) {
      if ((q & 1) == 0) reinterpret_cast<uint32_t*>(rest)[2 * row + (q >> 1)] = sc2;
      if (q == 0)
        reinterpret_cast<float*>(rest + 128)[row] = h2f_bits(blk[112] | (uint32_t)blk[113] << 8);
    } else if (q == 0) {
      reinterpret_cast<uint2*>(rest)[row] = make_uint2(sc2, 0);
      if ((s & 1) == 0) {
        uint32_t mm[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          int sc, mn;
          q4_sm((int)((e0 & 255) >> 5) + jj, sc, mn);
          mm[jj] = f16_bits((float)mn);
        }
        reinterpret_cast<uint2*>(rest + 128)[row] = make_uint2(mm[0] | mm[1] << 16, mm[2] | mm[3] << 16);
      } else {
        reinterpret_cast<float*>(rest + 128)[row] = h2f_bits(blk[0] | (uint32_t)blk[1] << 8);
        reinterpret_cast<float*>(rest + 192)[row] = h2f_bits(blk[2] | (uint32_t)blk[3] << 8);
      }
    }
  }
}

// ---- activations ---------------------------------------------------------------
struct F16Parts {
  _Float16 hi, mid, lo;
};
__device__ __forceinline__ F16Parts split3(float x) {
  F16Parts p;
  p.hi = (_Float16)x;
  const float r = (x - (float)p.hi) * kMmMid;  // exact
  p.mid = (_Float16)r;
  p.lo = (_Float16)(r - (float)p.mid);
  return p;
}

// Wave per row: rows [0, na) of a (width wa), then rows of b (width wb), the
// parts one after the other in out, exponents in ex.  Row layout: per 64
// columns 64 hi, 64 mid, 64 lo parts.  sums (Q4_K): per 128 columns the f16
// parts [4 hi][4 mid][4 lo][4 zeros] of the sums of 32 columns.
template <bool SUMS>
__global__ __launch_bounds__(256) void k_gguf_split(const float* __restrict__ a, int64_t na, int wa,
                                                    const float* __restrict__ b, int64_t nb, int wb,
                                                    uint16_t* __restrict__ out,
                                                    int32_t* __restrict__ ex,
                                                    uint16_t* __restrict__ sums) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= na + nb) return;
  const int lane = threadIdx.x & 63;
  const bool first = row < na;
  const int n = first ? wa : wb;
  const float* src = first ? a + row * wa : b + (row - na) * wb;
  const int64_t o = first ? row * wa : na * wa + (row - na) * wb;  // elements before the row
  float mx = 0.0f;
  for (int c = lane * 8; c < n; c += 512) {
    const f32x4 u = *reinterpret_cast<const f32x4*>(src + c);
    const f32x4 v = *reinterpret_cast<const f32x4*>(src + c + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      mx = __builtin_fmaxf(mx, __builtin_fmaxf(__builtin_fabsf(u[i]), __builtin_fabsf(v[i])));
  }
  mx = __ockl_wfred_max_f32(mx);
  // 2^s takes the largest value to [2^14, 2^15); 0 for a row of zeros or one
  // that holds an infinity (its parts are then not finite either)
  const int s = mx > 0.0f && finite_f(mx) ? 15 - __builtin_amdgcn_frexp_expf(mx) : 0;
  if (lane == 0) ex[row] = s;
  for (int c0 = 0; c0 < n; c0 += 512) {
    const int c = c0 + lane * 8;
    const bool in = c < n;
    f16x8 hi, mid, lo;
    float sum = 0.0f;
    const f32x4 u = *reinterpret_cast<const f32x4*>(src + (in ? c : 0));
    const f32x4 v = *reinterpret_cast<const f32x4*>(src + (in ? c + 4 : 4));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = __builtin_amdgcn_ldexpf(i < 4 ? u[i & 3] : v[i & 3], s);
      const F16Parts p = split3(x);
      hi[i] = p.hi;
      mid[i] = p.mid;
      lo[i] = p.lo;
      sum = sum + x;
    }
    if (in) {
      uint16_t* dst = out + 3 * (o + (c & ~63)) + (c & 63);
      *reinterpret_cast<f16x8*>(dst) = hi;
      *reinterpret_cast<f16x8*>(dst + 64) = mid;
      *reinterpret_cast<f16x8*>(dst + 128) = lo;
    }
    if constexpr (SUMS) {
      // sums of 32 columns: four lanes; sixteen lanes hold the four of 128.
      // Scaled by 2^-5, within f16's range.
      sum = sum + __shfl_xor(sum, 1, 64);
      sum = sum + __shfl_xor(sum, 2, 64);
      const float q = sum * 0.03125f;
      f16x8 p, p2{};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const F16Parts t = split3(__shfl(q, (lane & 48) + 4 * j, 64));
        p[j] = t.hi;
        p[4 + j] = t.mid;
        p2[j] = t.lo;
      }
      if (in && (lane & 15) == 0) {
        f16x8* dst = reinterpret_cast<f16x8*>(sums + (o + c) / 128 * 16);
        dst[0] = p;
        dst[1] = p2;
      }
    }
  }
}

// ---- the products ----------------------------------------------------------------
struct MmArgs {
  GgufMoeDev L;
  const uint8_t* tiles;
  const int32_t* off;
  const int32_t* perm;
  const int2* units;
  const int32_t* meta;
  int T;
  const uint16_t* b;     // token rows in f16 parts: x by token, or h by position (shared rows last)
  const uint16_t* sums;  // their column sums (Q4_K)
  const int32_t* ex;     // their exponents
  float* out;            // gate/up: h [T K][I] by position; down: r [T K][H] by assignment
  float* outs;           // shared expert: h [T][Ish]; [T][H]
  unsigned long long* status;
};

struct MmUnit {
  bool shared;
  int e, p0, n;  // expert, first position (shared: first token), tokens
  int rows, fb;  // I or Ish, block of rows
};

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
// N B fragments of a staged k-group at byte AT from a as LDS reads in flight
// together, PITCH bytes apart; not valid before lds_wait.
template <int AT, int PITCH, int N>
__device__ __forceinline__ void lds_read_b(uint32_t a, f16x8 (&b)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(b[i]) : "v"(a), "n"(AT + i * PITCH));
}
// until at most M LDS operations are in flight; b's registers tied
template <int N, int M>
__device__ __forceinline__ void lds_wait_b(f16x8 (&b)[N]) {
  if constexpr (N == 3)
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]) : "n"(M));
  else if constexpr (N == 2)
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(b[0]), "+v"(b[1]) : "n"(M));
  else
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(b[0]) : "n"(M));
}

__device__ __forceinline__ f32x4 mfma_f16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Eight 4-bit codes times their scale as exact f16 integers: a code at
// mantissa bits 6 .. 9 under the exponent of 16 is 16 + code, and
// s (16 + code) - s (16 + bias) is one fused operation with an exact result.
__device__ __forceinline__ f16x8 codes4(uint32_t w, f16x2 s, f16x2 ns) {
  constexpr uint32_t kM = 0x03C003C0u, kB = 0x4C004C00u;
  const uint32_t v[4] = {((w << 6) & kM) | kB, ((w << 2) & kM) | kB, ((w >> 2) & kM) | kB,
                         ((w >> 6) & kM) | kB};
  f16x8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f16x2 p = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, v[i]), s, ns);
    r[2 * i] = p.x;
    r[2 * i + 1] = p.y;
  }
  return r;
}
// eight 8-bit codes (+ 128) as exact f16 integers: 1024 + byte - 1152
__device__ __forceinline__ f16x8 codes8(uint32_t w0, uint32_t w1) {
  f16x8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i < 2 ? w0 : w1;
    const uint32_t v = __builtin_amdgcn_perm(0x64646464u, w, i & 1 ? 0x04030402u : 0x04010400u);
    const f16x2 p = __builtin_bit_cast(f16x2, v) + f16x2{(_Float16)-1152.0f, (_Float16)-1152.0f};
    r[2 * i] = p.x;
    r[2 * i + 1] = p.y;
  }
  return r;
}
__device__ __forceinline__ f16x2 splat_lo(uint32_t w) {
  const f16x2 v = __builtin_bit_cast(f16x2, w);
  return f16x2{v.x, v.x};
}
__device__ __forceinline__ f16x2 splat_hi(uint32_t w) {
  const f16x2 v = __builtin_bit_cast(f16x2, w);
  return f16x2{v.y, v.y};
}

template <int NCT>
struct MmAcc {
  f32x4 m[2][NCT];  // sums in units of the activations' scale
  f32x4 c[2][NCT];  // K-quants: the integer products of the columns that share a d
};

// One stage: 2 tiles x NCT column tiles x 64 columns x (hi, mid, lo).  ODD: the
// second stage of 128 columns, which ends the K-quants' partial sums.
//
// Its steps Z: column group kg of 32, part (hi, mid, lo), group of up to three
// column tiles, running fastest; the B fragments of step Z + 1 are read
// while step Z multiplies.
template <int TY, int NCT, bool ODD>
struct MmStage {
  using R = Rec<TY>;
  using S = MmBuf<TY, NCT>;
  static constexpr int kG = NCT < 4 ? NCT : 2, kNG = NCT / kG, kSteps = 6 * kNG;
  static constexpr int kg(int z) { return z / (3 * kNG); }
  static constexpr int part(int z) { return z / kNG % 3; }
  static constexpr int ct0(int z) { return z % kNG * kG; }

  const unsigned char* st;
  const unsigned char* rs;
  uint32_t bp, bl;  // row j's hi and mid parts, its line of lo parts
  int q, j;
  uint4 cw[2];
  uint32_t sc[2];
  f16x8 a[2];
  f16x8 b[2][kG];

  template <int Z>
  __device__ __forceinline__ void read() {
    constexpr int ct = ct0(Z), k = 4 * kg(Z);
    if constexpr (part(Z) < 2)
      lds_read_b<ct * 16 * kMmRowBytes, 16 * kMmRowBytes>(
          bp + (uint32_t)(((8 * part(Z) + k + q) ^ j) * 16), b[Z & 1]);
    else if constexpr (S::kLoFar)
      lds_read_b<S::kLoAt, 16 * kMmRowBytes>(bp + (uint32_t)(((4 * ct + k + q) ^ j) * 16), b[Z & 1]);
    else
      lds_read_b<S::kLoAt + ct * 8 * kMmRowBytes, 8 * kMmRowBytes>(
          bl + (uint32_t)((8 * (j & 1) + ((k + q) ^ (j >> 1))) * 16), b[Z & 1]);
  }

  template <int Z>
  __device__ __forceinline__ void steps(MmAcc<NCT>& A) {
    if constexpr (Z < kSteps) {
      if constexpr (Z % (3 * kNG) == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if constexpr (TY == kGgmlQ8_0) {
            a[t] = kg(Z) ? codes8(cw[t].z, cw[t].w) : codes8(cw[t].x, cw[t].y);
          } else {
            const f16x2 s = kg(Z) ? splat_hi(sc[t]) : splat_lo(sc[t]);
            constexpr float kBias = TY == kGgmlQ3_K ? -20.0f : -16.0f;
            a[t] = codes4(kg(Z) ? cw[t].y : cw[t].x, s, s * f16x2{(_Float16)kBias, (_Float16)kBias});
          }
        }
      }
      if constexpr (part(Z) == 1 && ct0(Z) == 0) {  // for mid and lo
#pragma unroll
        for (int t = 0; t < 2; ++t) a[t] = a[t] * (_Float16)(1.0f / kMmMid);
      }
      if constexpr (Z + 1 < kSteps) {
        read<Z + 1>();
        lds_wait_b<kG, kG>(b[Z & 1]);
      } else {
        lds_wait_b<kG, 0>(b[Z & 1]);
      }
      // the columns' partial sums start at zero
      constexpr bool kStart = part(Z) == 0 && (TY == kGgmlQ8_0 || (!ODD && kg(Z) == 0));
#pragma unroll
      for (int i = 0; i < kG; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          f32x4& c = A.c[t][ct0(Z) + i];
          c = mfma_f16(a[t], b[Z & 1][i], kStart ? f32x4{0, 0, 0, 0} : c);
        }
      if constexpr (TY == kGgmlQ8_0 && part(Z) == 2) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 d = *reinterpret_cast<const f32x4*>(rs + t * R::kRest + kg(Z) * 64 + 16 * q);
#pragma unroll
          for (int i = 0; i < kG; ++i) {
            f32x4& m = A.m[t][ct0(Z) + i];
            fma4(m, d, A.c[t][ct0(Z) + i]);
            // (left alone, the additions sink to the stage's end, every step's
            // products kept: 169 registers instead of 120)
            asm volatile("" : "+v"(m));
          }
        }
      }
      steps<Z + 1>(A);
    }
  }
  static __device__ __forceinline__ uint32_t mul_mid(uint32_t w) {
    constexpr _Float16 k = (_Float16)(1.0f / kMmMid);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, w) * f16x2{k, k});
  }
  static __device__ __forceinline__ void fma4(f32x4& m, const f32x4& d, const f32x4& c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = __builtin_fmaf(d[i], c[i], m[i]);
  }

  __device__ __forceinline__ void run(const unsigned char* lds, int off, int w, int lane,
                                      MmAcc<NCT>& A, uint2 (&mn)[2]) {
    q = lane >> 4;
    j = lane & 15;
    st = lds + off;
    rs = st + S::kB + 16 * R::kCodes + w * 2 * R::kRest;
    bp = lds_u32(lds) + (uint32_t)(off + j * kMmRowBytes);
    bl = lds_u32(lds) + (uint32_t)(off + (j >> 1) * kMmRowBytes);
    const unsigned char* cd = st + S::kB + w * 2 * R::kCodes;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (TY == kGgmlQ8_0) {
        cw[t] = *reinterpret_cast<const uint4*>(cd + t * R::kCodes + lane * 16);
      } else {
        const uint2 c2 = *reinterpret_cast<const uint2*>(cd + t * R::kCodes + lane * 8);
        cw[t] = make_uint4(c2.x, c2.y, 0, 0);
        sc[t] = *reinterpret_cast<const uint32_t*>(rs + t * R::kRest + j * 8 +
                                                   (TY == kGgmlQ3_K ? (q >> 1) * 4 : 0));
        if (TY == kGgmlQ4_K && !ODD)
          mn[t] = *reinterpret_cast<const uint2*>(rs + t * R::kRest + 128 + j * 8);
      }
    }
    read<0>();
    steps<0>(A);
    if constexpr (TY != kGgmlQ8_0 && ODD) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(rs + t * R::kRest + 128 + 16 * q);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) fma4(A.m[t][ct], d, A.c[t][ct]);
        if constexpr (TY == kGgmlQ4_K) {
          // - dmin sum_j m_j (sum of sub-block j's activations): the mins of
          // the four sub-blocks against the parts of 2^-5 the sums (lanes 0 .. 15
          // hi and mid, 16 .. 31 lo)
          const f32x4 dm = *reinterpret_cast<const f32x4*>(rs + t * R::kRest + 192 + 16 * q);
          const f32x4 dn = dm * -32.0f;
          const uint2 z = q < 2 ? mn[t] : make_uint2(0, 0);
          const uint2 y = make_uint2(mul_mid(z.x), mul_mid(z.y));
          const f16x8 am = __builtin_bit_cast(
              f16x8, q == 0 ? make_uint4(z.x, z.y, y.x, y.y) : make_uint4(y.x, y.y, 0, 0));
#pragma unroll
          for (int ct = 0; ct < NCT; ++ct) {
            const f16x8 bs = *reinterpret_cast<const f16x8*>(st + S::kSumsAt +
                                                             (16 * ct + j) * 32 + (q & 1) * 16);
            fma4(A.m[t][ct], dn, mfma_f16(am, bs, f32x4{0, 0, 0, 0}));
          }
        }
      }
    }
  }
};

constexpr int kMmInfo = 64 * (int)sizeof(int2);
template <int TY>
constexpr int mm_lds() {
  constexpr int kMax = mm_tok(TY) / 16;
  constexpr int a = MmBuf<TY, kMax>::kBufs * MmBuf<TY, kMax>::kBytes;
  constexpr int b = MmBuf<TY, 2>::kBufs * MmBuf<TY, 2>::kBytes;
  constexpr int c = MmBuf<TY, 1>::kBufs * MmBuf<TY, 1>::kBytes;
  constexpr int n = (a > b ? a > c ? a : c : b > c ? b : c) + kMmInfo;
  static_assert(2 * n <= 160 * 1024, "two workgroups per CU");
  return n;
}
// A unit's block of rows with NCT column tiles, kAhead stages in flight.
template <int TY, bool GU, int NCT>
struct MmRun {
  using R = Rec<TY>;
  using S = MmBuf<TY, NCT>;
  const uint8_t* t0;  // this wave's two tiles
  const uint8_t* t1;
  const uint16_t* b[S::kRowLoads];  // this lane's segment of its token rows: hi or mid
  const uint16_t* bl;               // lo (unless kLoFar)
  const uint16_t* sums;             // and (Q4_K) half a row of column sums
  uint32_t l0;
  int w, lane, nst, nload;          // stages; loads of this wave and stage

  // row of token rows of position r (0 .. n - 1) of a unit
  static __device__ __forceinline__ int row_of(const MmArgs& g, const MmUnit& u, int r) {
    const int p = u.p0 + min(r, u.n - 1);
    return GU && !u.shared ? g.perm[p] / g.L.K : p;
  }

  // This wave's loads of stage s.
  __device__ __forceinline__ void issue(int s) {
    const uint32_t st = l0 + (uint32_t)(s % S::kBufs * S::kBytes);
#pragma unroll
    for (int m = 0; m < S::kRowLoads; ++m)
      if (w + 8 * m < 4 * NCT)  // uniform
        dma16_lds(b[m] + s * kMmRow3, st + (uint32_t)((w + 8 * m) * 1024));
    if (w < 2 * NCT) {
      const uint16_t* src = bl;
      if constexpr (S::kLoFar)  // segment c of row 4 w + q + 32 m, where 8 m + c is b's segment
        src = ((lane ^ (4 * w + (lane >> 4))) & 8) ? b[S::kRowLoads - 1] + kMmCols : b[0] + 2 * kMmCols;
      dma16_lds(src + s * kMmRow3, st + (uint32_t)(S::kLoAt + w * 1024));
    }
    const uint8_t* r0 = t0 + (size_t)s * R::kBytes;
    const uint8_t* r1 = t1 + (size_t)s * R::kBytes;
    const uint32_t ca = st + S::kB + (uint32_t)(w * 2 * R::kCodes);
    if (R::kCodes == 512) {
      dma16_lds((lane < 32 ? r0 : r1) + (lane & 31) * 16, ca);
    } else {
      dma16_lds(r0 + lane * 16, ca);
      dma16_lds(r1 + lane * 16, ca + 1024);
    }
    constexpr int kl = R::kRest / 16;  // lanes per tile
    if (lane < 2 * kl)
      dma16_lds((lane < kl ? r0 : r1) + R::kCodes + (lane < kl ? lane : lane - kl) * 16,
                st + S::kB + 16 * R::kCodes + (uint32_t)(w * 2 * R::kRest));
    if (R::kSums && w < NCT && lane < 32)  // (w uniform)
      dma16_lds(sums + (s >> 1) * 16, st + S::kSumsAt + (uint32_t)(w * 512));
  }

  // Stage s is complete everywhere, and nobody reads stage s - 1 any more,
  // whose buffer stage s + kAhead takes; the stage's byte offset.
  __device__ __forceinline__ int turn(int s) {
    // this wave's loads of stage s have landed (those of the next stage may
    // be in flight where two are ahead) ...
    constexpr int kA = R::kDma - (R::kSums ? 1 : 0);
    if (S::kAhead == 1 || s + 1 >= nst) {
      vm_wait<0>();
    } else {
      if (nload == kA + 3) vm_wait<kA + 3>();  // uniform
      else if (nload == kA + 2) vm_wait<kA + 2>();
      else if (nload == kA + 1) vm_wait<kA + 1>();
      else vm_wait<kA>();
    }
    __builtin_amdgcn_s_barrier();  // ... and every wave's
    if (s + S::kAhead < nst) issue(s + S::kAhead);
    return s % S::kBufs * S::kBytes;
  }

  __device__ __forceinline__ void run(const MmArgs& g, const MmUnit& cur,
                                      const unsigned char* lds) {
    const GgufMoeDev& L = g.L;
    const int K = L.K, H = L.H;
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    l0 = lds_u32(lds);
    const int q = lane >> 4, j = lane & 15;
    const int KD = GU ? H : cur.rows;
    nst = KD / kMmCols;
    const uint8_t* m0 = g.tiles + tile_offset(L.E, H, L.I, L.Ish, R::kBytes, cur.e, GU ? 0 : 2);
    const size_t rb = (size_t)nst * R::kBytes;  // bytes of 16 rows
    if (GU) {
      t0 = m0 + (size_t)(cur.fb * 8 + w) * rb;
      t1 = t0 + (size_t)(cur.rows / 16) * rb;
    } else {
      // H is a multiple of 128: waves past it (in the last block) load rows
      // 0 .. 31 and store nothing
      t0 = m0 + (size_t)(cur.fb * 256 + 32 * w < H ? cur.fb * 16 + 2 * w : 0) * rb;
      t1 = t0 + rb;
    }
    const size_t before = !GU && cur.shared ? (size_t)g.T * K * L.I : 0;
    // load m carries rows 4 (w + 8m) .. + 3, stored segment lane & 15 of row r
    // being its segment (lane & 15) ^ (r & 15) of hi and mid; the load of the lo
    // parts lines 4 w .. + 3
    nload = (w < 4 * NCT ? 1 : 0) + (w < 2 * NCT ? 1 : 0) + (R::kSums && w < NCT ? 1 : 0) +
            R::kDma - (R::kSums ? 1 : 0);  // (kAhead 2: one row load)
    const int sg = j ^ ((4 * w + q) & 15);
#pragma unroll
    for (int m = 0; m < S::kRowLoads; ++m)
      b[m] = g.b + 3 * before + (size_t)row_of(g, cur, 4 * (w + 8 * m) + q) * (3 * KD) + sg * 8;
    if (!S::kLoFar)
      bl = g.b + 3 * before + (size_t)row_of(g, cur, 8 * w + 2 * q + (j >> 3)) * (3 * KD) +
           2 * kMmCols + ((j & 7) ^ ((4 * w + q) & 7)) * 8;
    if (R::kSums)
      sums = g.sums + before / 8 + (size_t)row_of(g, cur, 16 * w + (lane >> 1)) * (KD / 8) +
             (lane & 1) * 8;
    issue(0);
    if (S::kAhead > 1) issue(1);  // (128 columns: nst is even)
    // the epilogue's words of a position: assignment, exponent (written before
    // the first barrier)
    int2* info = reinterpret_cast<int2*>(const_cast<unsigned char*>(lds) + mm_lds<TY>() - kMmInfo);
    if (threadIdx.x < mm_tok(TY)) {
      const int p = cur.p0 + min((int)threadIdx.x, cur.n - 1);
      const int a = cur.shared ? p : g.perm[p];
      info[threadIdx.x] =
          make_int2(a, g.ex[GU ? (cur.shared ? p : a / K) : (cur.shared ? g.T * K + p : p)]);
    }
    MmAcc<NCT> A;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) A.m[t][ct] = A.c[t][ct] = f32x4{0, 0, 0, 0};
    uint2 mn[2] = {make_uint2(0, 0), make_uint2(0, 0)};
    for (int s = 0; s < nst; s += 2) {
      int o = turn(s);
      MmStage<TY, NCT, false>().run(lds, o, w, lane, A, mn);
      o = turn(s + 1);
      MmStage<TY, NCT, true>().run(lds, o, w, lane, A, mn);
    }
    // rows fr .. fr + 3 of the lane in its column of each column tile
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      const int c = 16 * ct + j;
      if (c < cur.n) {
        const int2 in = info[c];
        const int p = cur.p0 + c, a = in.x, x = in.y;
        const uint32_t ph = cur.shared ? kPhShared : kPhExpert;
        if (GU) {
          const int fr = cur.fb * 128 + 16 * w + 4 * q;
          f32x4 gv, uv, hv;
          bool bad = false;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gv[i] = __builtin_amdgcn_ldexpf(A.m[0][ct][i], -x);
            uv[i] = __builtin_amdgcn_ldexpf(A.m[1][ct][i], -x);
            hv[i] = dm_silu(gv[i]) * uv[i];
            bad |= !finite_f(gv[i]) || !finite_f(uv[i]) || !finite_f(hv[i]);
          }
          *reinterpret_cast<f32x4*>((cur.shared ? g.outs : g.out) + (size_t)p * cur.rows + fr) = hv;
          if (bad) {
            const int t = cur.shared ? p : a / K, k = cur.shared ? 0 : a % K;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (!finite_f(gv[i]) || !finite_f(uv[i]) || !finite_f(hv[i]))
                record_err(g.status, err_key(ph, t, k, fr + i, !finite_f(gv[i])   ? kEkGate
                                                               : !finite_f(uv[i]) ? kEkUp
                                                                                  : kEkH));
          }
        } else if (cur.fb * 256 + 32 * w < H) {
          float* dst = cur.shared ? g.outs + (size_t)p * H : g.out + (size_t)a * H;
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int d0 = cur.fb * 256 + 32 * w + 16 * t + 4 * q;
            f32x4 v;
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              v[i] = __builtin_amdgcn_ldexpf(A.m[t][ct][i], -x);
              bad |= !finite_f(v[i]);
            }
            *reinterpret_cast<f32x4*>(dst + d0) = v;
            if (bad) {
              const int tk = cur.shared ? p : a / K, k = cur.shared ? 0 : a % K;
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (!finite_f(v[i])) record_err(g.status, err_key(ph, tk, k, cur.rows + d0 + i, kEkDown));
            }
          }
        }
      }
    }
  }
};

// Workgroup b: unit and block of rows in 8 classes (b % 8 is the XCD the
// dispatcher places it on: a unit's row blocks share that XCD's L2 for its
// token rows, as in k_experts).  A unit of n tokens runs with the column tiles
// it needs; at most 128 registers and 80 KB of LDS, so that two workgroups
// share a CU (see k_experts; one persistent workgroup on 128-token units took 1.2
// times as long).  At hidden 2048, inter 512, 256 experts, top 8, per call of 256 /
// 2048 tokens: Q3_K 229 / 588 us, Q4_K 247 / 682, Q8_0 259 / 642 (with two parts of
// 23 bits 197 / 515, 218 / 568, 245 / 549).  Bound by the matrix units' three
// passes and, between them, the codes' conversion and the fp32 scaling of the
// partial sums.
template <int TY, bool GU>
__global__ __launch_bounds__(kMmThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_gguf_mm(const int32_t* meta, const int2* units, const int32_t* off, const int32_t* perm,
               int nblk, MmArgs gk) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ldsm[];
  MmArgs g = gk;
  g.perm = perm;
  const int nall = meta[0], span = (nall + 7) >> 3, idx = (int)blockIdx.x >> 3;
  const int ul = idx / nblk, u = ((int)blockIdx.x & 7) * span + ul;
  MmUnit it;
  it.fb = idx - ul * nblk;
  if (ul >= span || u >= nall) return;
  const int2 v = units[u];
  it.shared = v.x >= g.L.E;
  it.e = it.shared ? g.L.E : v.x;
  it.p0 = it.shared ? v.y : off[v.x] + v.y;
  it.n = min(mm_tok(TY), (it.shared ? g.T : off[v.x + 1]) - it.p0);
  it.rows = it.shared ? g.L.Ish : g.L.I;
  if (GU && it.fb * 128 >= it.rows) return;  // uniform per workgroup
  if (it.n <= 16) MmRun<TY, GU, 1>().run(g, it, ldsm);
  else if (it.n <= 32) MmRun<TY, GU, 2>().run(g, it, ldsm);
  else MmRun<TY, GU, mm_tok(TY) / 16>().run(g, it, ldsm);
}

template <int TY>
hipError_t mm_attrs() {
  const int lds = mm_lds<TY>();
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_gguf_mm<TY, true>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_gguf_mm<TY, false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  return e;
}

template <int TY>
hipError_t run_mm(const GgufMoeDev& L, const uint8_t* tiles, const float* x, int T, const int32_t* off,
                  const int32_t* perm, const int2* units, const int32_t* meta, int nunits,
                  const GgufMmScratch& s, float* r, float* rs, unsigned long long* status,
                  hipStream_t st) {
  constexpr bool kSums = Rec<TY>::kSums > 0;
  const int64_t TK = (int64_t)T * L.K;
  const size_t lds = mm_lds<TY>();
  float* hs = s.h + TK * L.I;
  const int imax = L.I > L.Ish ? L.I : L.Ish, classes = 8 * ((nunits + 7) / 8);
  const int gb = (imax + 127) / 128, db = (L.H + 255) / 256;
  hipLaunchKernelGGL(k_gguf_split<kSums>, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, st, x,
                     (int64_t)T, L.H, nullptr, (int64_t)0, L.H, s.xs, s.ex, s.xsum);
  MmArgs g{L, tiles, off, perm, units, meta, T, s.xs, s.xsum, s.ex, s.h, hs, status};
  hipLaunchKernelGGL((k_gguf_mm<TY, true>), dim3(classes * gb), dim3(kMmThreads), lds, st, meta,
                     units, off, perm, gb, g);
  hipLaunchKernelGGL(k_gguf_split<kSums>, dim3((unsigned)((TK + T + 3) / 4)), dim3(256), 0, st,
                     s.h, TK, L.I, hs, (int64_t)T, L.Ish, s.hs, s.ex + T, s.hsum);
  g.b = s.hs;
  g.sums = s.hsum;
  g.ex = s.ex + T;
  g.out = r;
  g.outs = rs;
  hipLaunchKernelGGL((k_gguf_mm<TY, false>), dim3(classes * db), dim3(kMmThreads), lds, st, meta,
                     units, off, perm, db, g);
  return hipGetLastError();
}

}  // namespace

size_t gguf_tiles_bytes(const GgufMoeDev& L) {
  const int rec = rec_bytes(L.type);
  if (!rec || L.H % 128 || L.I % 128 || L.Ish % 128) return 0;
  return tile_offset(L.E, L.H, L.I, L.Ish, rec, L.E, 3);
}

hipError_t launch_gguf_tiles(const GgufMoeDev& L, uint8_t* out, hipStream_t st) {
  if (!gguf_tiles_bytes(L)) return hipErrorInvalidValue;
  const int imax = L.I > L.Ish ? L.I : L.Ish;
  const dim3 grid((unsigned)(((imax / 16) * (L.H / kMmCols) + 3) / 4), (unsigned)(3 * (L.E + 1)));
  hipError_t e;
  switch (L.type) {
    case kGgmlQ3_K:
      if ((e = mm_attrs<kGgmlQ3_K>()) != hipSuccess) return e;
      k_gguf_tile<kGgmlQ3_K><<<grid, 256, 0, st>>>(L, out);
      break;
    case kGgmlQ4_K:
      if ((e = mm_attrs<kGgmlQ4_K>()) != hipSuccess) return e;
      k_gguf_tile<kGgmlQ4_K><<<grid, 256, 0, st>>>(L, out);
      break;
    default:
      if ((e = mm_attrs<kGgmlQ8_0>()) != hipSuccess) return e;
      k_gguf_tile<kGgmlQ8_0><<<grid, 256, 0, st>>>(L, out);
      break;
  }
  return hipGetLastError();
}

int gguf_mm_tok(const GgufMoeDev& L) { return mm_tok(L.type); }

bool gguf_mm_ok(const GgufMoeDev& L, int T) {
  // (calls of 2^31 activations and more: not measured, the grouped form)
  const uint64_t n = L.I > L.Ish ? L.I : L.Ish;
  return gguf_tiles_bytes(L) && T >= kGgufMmMinT && 2ull * T * L.H < (1ull << 32) &&
         2ull * T * L.K * n < (1ull << 32);
}

size_t gguf_mm_sums(const GgufMoeDev& L, int64_t elements) {
  return L.type == kGgmlQ4_K ? (size_t)elements / 8 : 0;
}

hipError_t launch_gguf_mm(const GgufMoeDev& L, const uint8_t* tiles, const float* x, int T, const int32_t* off,
                          const int32_t* perm, const int2* units, const int32_t* meta, int nunits,
                          const GgufMmScratch& s, float* r, float* rs, unsigned long long* status,
                          hipStream_t st) {
  if (!tiles || !gguf_mm_ok(L, T) || nunits <= 0) return hipErrorInvalidValue;
  switch (L.type) {
    case kGgmlQ3_K:
      return run_mm<kGgmlQ3_K>(L, tiles, x, T, off, perm, units, meta, nunits, s, r, rs, status, st);
    case kGgmlQ4_K:
      return run_mm<kGgmlQ4_K>(L, tiles, x, T, off, perm, units, meta, nunits, s, r, rs, status, st);
    default:
      return run_mm<kGgmlQ8_0>(L, tiles, x, T, off, perm, units, meta, nunits, s, r, rs, status, st);
  }
}

}  // namespace dm
