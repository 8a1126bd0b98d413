// dm_grouped.hip -- the MoE block for several tokens at once (small batches
// and prefill): tokens are grouped by expert on the GPU and every expert runs
// as a grouped GEMM on MFMA.
//
// Reference composition (src/layers/moe_block.mojo:20-138): router for all
// tokens, then the routed experts per (token, k) with
// src/layers/swiglu.mojo:52-230, then the shared expert for all tokens, then
// the combine of src/layers/moe.mojo:105-177.  Here:
//
//   k_router_mfma / k_router_dec, k_router_select (dm_kernels.hip)  logits
//                   (matrix cores for bf16 activations), softmax, top-k
//   k_group_build   one workgroup: count assignments per expert, scan,
//                   scatter them into expert order, emit the work units
//                   (expert, up to 64 or 16 of its tokens); the shared expert is
//                   expert E over all tokens
//   k_split_rows    activations -> bf16 hi / lo rows
//   k_experts<true>  h = SiLU(W_g x) * (W_u x): token rows, 4-bit weights and
//                   scales all staged in LDS by direct-to-LDS loads, weights
//                   dequantised from LDS (16 features x 32 k per MFMA)
//   k_experts<false> r = W_d h, B = h as bf16 hi + lo parts
//   k_gu_small, k_down_small  the same for calls of a few tokens: operands
//                   straight from memory, no LDS and no barriers
//   k_combine       y = sum_k p_k r_k + g r_sh (+ residual), reference order
//
// Each token's outputs depend only on its own column of the MFMA tiles, so
// the placement of tokens inside an expert's tiles (atomic scatter) does not
// change any result bit.
#include <hip/hip_runtime.h>

#include <atomic>

#include "dm_device.h"
#include "dm_grouped.h"

namespace dm {

constexpr int kGThreads = 256;

// ---------------------------------------------------------------------------
// One workgroup of 1024 threads.  ids [T*K] in the reference order (slot k of
// token t at t*K + k).  Outputs: off [E+1] expert offsets into perm, perm
// [T*K] assignment indices grouped by expert, units = (expert, first position
// within the expert) of up to tok positions each, meta[0] = number of units:
// the shared expert's first (they are full), then the routed ones in expert
// order.
// The grouping on one workgroup of 1024 threads, lds: (2 E + 32) ints.
// COH: ids are read with agent-scope loads (written in the same launch).
template <bool COH>
__device__ __forceinline__ void group_build_wg(const int32_t* __restrict__ ids, int T, int K, int E,
                                               int tok, int32_t* __restrict__ off,
                                               int32_t* __restrict__ perm,
                                               int2* __restrict__ units,
                                               int32_t* __restrict__ meta, int* lds) {
  // cnt[E] | cur[E] | wave totals of the 2 scans (counts, units), 16 waves each
  int* cnt = lds;
  int* cur = lds + E;
  int* sc = lds + 2 * E;
  const int tid = threadIdx.x, TK = T * K;
  for (int e = tid; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  // the first kCache expert ids of this thread stay in registers for the
  // scatter below (a load issued after the stores of the units would wait
  // for them)
  constexpr int kCache = 16;
  int ec[kCache];
#pragma unroll
  for (int i = 0; i < kCache; ++i) {
    const int a = tid + 1024 * i;
    ec[i] = a < TK ? min(max((int)(COH ? ld_coh_i32(ids + a) : ids[a]), 0), E - 1) : 0;
  }
#pragma unroll
  for (int i = 0; i < kCache; ++i)
    if (tid + 1024 * i < TK) atomicAdd(&cnt[ec[i]], 1);
  for (int a = tid + 1024 * kCache; a < TK; a += 1024) {
    const int e = min(max((int)(COH ? ld_coh_i32(ids + a) : ids[a]), 0), E - 1);
    atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  // thread tid owns experts [e0, e1)
  const int per = (E + 1023) / 1024, e0 = min(tid * per, E), e1 = min(e0 + per, E);
  int v[2] = {0, 0};
  for (int e = e0; e < e1; ++e) {
    v[0] += cnt[e];
    v[1] += (cnt[e] + tok - 1) / tok;
  }
  // exclusive prefix sums of the two counts over the threads: inclusive
  // scans inside each wave (shuffles), then the 16 wave totals from LDS
  const int lane = tid & 63, wv = tid >> 6;
  int incl[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int a = v[i];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(a, d, 64);
      a += lane >= d ? o : 0;
    }
    incl[i] = a;
    if (lane == 63) sc[i * 16 + wv] = a;
  }
  __syncthreads();
  int pre[2], tot[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int p = 0, t = 0;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int wt = sc[i * 16 + u];
      p += u < wv ? wt : 0;
      t += wt;
    }
    pre[i] = p + incl[i] - v[i];
    tot[i] = t;
  }
  const int nsh = (T + tok - 1) / tok;
  int base = pre[0], un = nsh + pre[1];
  for (int e = e0; e < e1; ++e) {
    off[e] = base;
    cur[e] = base;
    for (int i = 0; i < cnt[e]; i += tok) units[un++] = make_int2(e, i);
    base += cnt[e];
  }
  if (tid == 0) off[E] = TK;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kCache; ++i) {
    const int a = tid + 1024 * i;
    if (a < TK) perm[atomicAdd(&cur[ec[i]], 1)] = a;
  }
  for (int a = tid + 1024 * kCache; a < TK; a += 1024) {
    const int e = min(max((int)(COH ? ld_coh_i32(ids + a) : ids[a]), 0), E - 1);
    perm[atomicAdd(&cur[e], 1)] = a;
  }
  for (int i = tid; i < nsh; i += 1024) units[i] = make_int2(E, tok * i);
  if (tid == 0) meta[0] = nsh + tot[1];
}

__global__ __launch_bounds__(1024) void k_group_build(const int32_t* __restrict__ ids, int T, int K,
                                                      int E, int tok, int32_t* __restrict__ off,
                                                      int32_t* __restrict__ perm,
                                                      int2* __restrict__ units,
                                                      int32_t* __restrict__ meta) {
  extern __shared__ int lds[];
  group_build_wg<false>(ids, T, K, E, tok, off, perm, units, meta, lds);
}

hipError_t launch_group_build(const int32_t* ids, int T, int K, int E, int tok, int32_t* off,
                              int32_t* perm, int2* units, int32_t* meta, hipStream_t st) {
  const size_t lds = (size_t)(2 * E + 32) * sizeof(int);
  hipLaunchKernelGGL(k_group_build, dim3(1), dim3(1024), lds, st, ids, T, K, E, tok, off,
                     perm, units, meta);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The front end of a small batch in one launch (T tokens, 2 <= T < 64):
// workgroup (b, t) stages token t's x in LDS, computes router rows
// 64 b .. 64 b + 63 (16 lanes each, the chains of router_chain and the
// halving tree of k_router_dec: the same logits bit for bit), and workgroup
// (0, t) also writes t's bf16 hi / lo rows and the need-lo flag.  Each
// workgroup then counts itself in token t's counter flags[2 + t]; the last
// of them (the logits are written and read at the device-coherent level, so
// that those of workgroups on other XCDs are visible) runs t's softmax /
// top-k on one wave (route_select_token) and counts the token in flags[1];
// the last token's workgroup groups the assignments (group_build_wg).  Each
// counter is reset by the workgroup that saw it complete.  No workgroup
// waits for another.
template <int NE>
__global__ __launch_bounds__(1024) void k_front(const float* __restrict__ x,
                                                const uint16_t* __restrict__ router_, int H_,
                                                int E_, LayerDev Lk, int T,
                                                float* __restrict__ z, uint4* __restrict__ xhi,
                                                uint4* __restrict__ xlo, int* flags,
                                                int32_t* __restrict__ ids,
                                                float* __restrict__ probs,
                                                float* __restrict__ shg, int32_t* __restrict__ off,
                                                int32_t* __restrict__ perm,
                                                int2* __restrict__ units,
                                                int32_t* __restrict__ meta,
                                                unsigned long long* status) {
  extern __shared__ __attribute__((aligned(16))) float fl[];
  __shared__ int last, last_tok;
  LayerDev L = Lk;  // the entry fields from the preloaded leading arguments
  L.H = H_;
  L.E = E_;
  L.router = router_;
  const int tid = threadIdx.x, H = L.H, E = L.E, t = blockIdx.y;
  const float* xr = x + (size_t)t * H;
  bool bad = false;
  for (int i = tid; i < H; i += 1024) {
    const float v = xr[i];
    bad |= !finite_f(v);
    fl[i] = v;
  }
  if (bad && blockIdx.x == 0) record_err(status, err_key(kPhX, 0, 0, 0, 0));
  if (blockIdx.x == 0) {
    bool nz = false;
    for (int i = tid; i < H / 8; i += 1024) {
      uint4 h, l;
      split8(xr + 8 * i, h, l);
      xhi[(size_t)t * (H / 8) + i] = h;
      xlo[(size_t)t * (H / 8) + i] = l;
      nz |= (l.x | l.y | l.z | l.w) != 0u;
    }
    if (__builtin_amdgcn_ballot_w64(nz) != 0 && (tid & 63) == 0) atomicOr(&flags[0], 1);
  }
  __syncthreads();
  const int l = tid & 15, e = blockIdx.x * 64 + (tid >> 4);
  float acc = e <= E ? router_chain(L.router, H, e, l, fl) : 0.0f;
#pragma unroll
  for (int wdt = 8; wdt >= 1; wdt >>= 1) acc = acc + __shfl_down(acc, wdt, 16);
  // logits to the device-coherent level (agent-scope stores, complete before
  // the count), read back by the last workgroup with agent-scope loads: no
  // write-back or invalidation of the whole L2
  if (l == 0 && e <= E) st_coh(z + (size_t)t * (E + 1) + e, acc);
  wait_stores();
  __syncthreads();
  // the last of token t's workgroups selects its experts (wave 0) ...
  if (tid == 0) last = atomicAdd(&flags[2 + t], 1) == (int)gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  const int lane = tid & 63, w = tid >> 6, K = L.K;
  auto wsync = [] {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  // Two waves at once: wave 0 picks the top K on the logits (topk_on_logits:
  // the same set as the reference's rounds on the probabilities whenever its
  // margin check passes), wave 1 forms the softmax terms (max, the
  // exponentials, their sum in expert order) and the shared gate, as
  // router_softmax does (src/layers/router.mojo:140-183).  Then wave 0
  // forms the K probabilities e_k * (1/S) and orders them (p desc, id asc),
  // as select_topk (src/layers/topk.mojo:79-128).  On a near tie at the
  // boundary wave 0 runs the exact rounds (route_select_token) instead.
  constexpr int R = NE <= 4 ? 1 : 2;
  __shared__ float sm_terms[2];  // max, 1/S
  __shared__ int sm_unsafe;
  float* sev = fl;               // [E] exponentials (the staged x is no longer read)
  const float* zr = z + (size_t)t * (E + 1);
  int myid = 0;
  float zk = 0.0f;
  if (w == 0) {
    if (tid == 0) atomicExch(&flags[2 + t], 0);
    float zv[4 * R];
#pragma unroll
    for (int i = 0; i < 4 * R; ++i) {
      const int e = lane + 64 * i;
      zv[i] = e < E ? ld_coh(zr + e) : -__builtin_inff();
    }
    uint32_t fk[4 * R];
    const bool unsafe = topk_on_logits<R>(zv, E, K, lane, fk, myid);
    myid = min(max(myid, 0), E - 1);
    // the logit of expert myid sits in lane myid & 63, entry myid >> 6
#pragma unroll
    for (int i = 0; i < 4 * R; ++i) {
      const float zo = u2f((uint32_t)__builtin_amdgcn_ds_bpermute(4 * (myid & 63), (int)f2u(zv[i])));
      zk = (myid >> 6) == i ? zo : zk;
    }
    if (lane == 0) sm_unsafe = unsafe || K > 8 ? 1 : 0;  // (the ranks below take K <= 8)
  } else if (w == 1) {
    const float lg = lane == 0 ? ld_coh(zr + E) : 0.0f;
    float zv[NE];
    float m = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = lane + 64 * i;
      zv[i] = e < E ? ld_coh(zr + e) : -__builtin_inff();
      if (e < E && !finite_f(zv[i])) record_err(status, err_key(kPhLogit, t, 0, e, 0));
      m = zv[i] > m ? zv[i] : m;
    }
    m = __ockl_wfred_max_f32(m);
    if (lane == 0 && !finite_f(m)) record_err(status, err_key(kPhSoftmax, t, 0, 0, 0));
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = lane + 64 * i;
      if (e < E) {
        const float ev = dm_expf(zv[i] - m);
        if (!finite_f(ev)) record_err(status, err_key(kPhSoftmax, t, 0, 1 + e, 0));
        sev[e] = ev;
      }
    }
    wsync();
    if (lane == 0) {
      const float sum = seq_sum(sev, E);
      if (!(sum > 0.0f) || !finite_f(sum)) record_err(status, err_key(kPhSoftmax, t, 0, 1 + E, 0));
      sm_terms[0] = m;
      sm_terms[1] = 1.0f / sum;
      if (!finite_f(lg)) record_err(status, err_key(kPhGate, t, 0, 0, kGkLogit));
      const float g = dm_sigmoid(lg);
      if (!finite_f(g) || g < 0.0f || g > 1.0f) record_err(status, err_key(kPhGate, t, 0, 0, kGkRange));
      shg[t] = g;
    }
  }
  __syncthreads();
  if (w == 0) {
    if (sm_unsafe) {
      route_select_token<NE, true>(z, E + 1, E, K, 1, t, lane, fl, ids, probs, shg, status, wsync);
    } else {
      const float m = sm_terms[0], inv = sm_terms[1];
      const float pk = lane < K ? dm_expf(zk - m) * inv : 0.0f;
      // rank of slot k: (p desc, id asc); the ids are distinct
      const uint32_t kk = f2key(pk);
      int rank = 0;
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        const uint32_t kj = (uint32_t)__builtin_amdgcn_readlane((int)kk, jj);
        const int ij = __builtin_amdgcn_readlane(myid, jj);
        if (jj < K && lane < K) rank += (kj > kk || (kj == kk && ij < myid)) ? 1 : 0;
      }
      if (lane < K) {
        st_coh_i32(ids + (size_t)t * K + rank, myid);
        probs[(size_t)t * K + rank] = pk;
      }
      // the checks of select_topk in rank order
      float* sp = sev + ((E + 3) & ~3);  // [8] probabilities by rank
      if (lane < K) sp[rank] = pk;
      wsync();
      if (lane == 0) {
        float sum_topk = 0.0f;
        for (int r = 0; r < K; ++r) sum_topk = sum_topk + sp[r];
        if (sum_topk > 1.00001f) record_err(status, err_key(kPhTopk, t, 0, 0, kTkSum));
        if (K < E && __builtin_fabsf(sum_topk - 1.0f) < 1e-6f) {
          float sum_all = 0.0f;
          for (int e = 0; e < E; ++e) sum_all = sum_all + sev[e] * inv;
          if (sum_all - sum_topk > 1e-5f) record_err(status, err_key(kPhTopk, t, 0, 0, kTkLeak));
        }
      }
    }
    wait_stores();
    // ... and the last token to be selected groups the assignments
    if (tid == 0) last_tok = atomicAdd(&flags[1], 1) == T - 1;
  }
  __syncthreads();
  if (!last_tok) return;
  if (tid == 0) atomicExch(&flags[1], 0);
  group_build_wg<true>(ids, T, L.K, E, unit_tok(T), off, perm, units, meta, reinterpret_cast<int*>(fl));
}

bool front_supported(const LayerDev& L, int T) {
  return T >= 2 && T <= kFrontMaxT && L.E <= kFrontMaxE && L.H % 128 == 0;
}

hipError_t launch_front(const LayerDev& L, const float* x, int T, float* z, uint16_t* xhi,
                        uint16_t* xlo, int* flags, int32_t* ids, float* probs, float* shg,
                        int32_t* off, int32_t* perm, int2* units, int32_t* meta,
                        unsigned long long* status, hipStream_t st) {
  if (!front_supported(L, T)) return hipErrorInvalidValue;
  const size_t sel = (size_t)(((L.E + 3) & ~3) + 8) * sizeof(float);
  const size_t bld = (size_t)(2 * L.E + 32) * sizeof(int);
  const size_t xs = (size_t)L.H * sizeof(float);
  const size_t lds = sel > bld ? (sel > xs ? sel : xs) : (bld > xs ? bld : xs);
  const dim3 grid((L.E + 1 + 63) / 64, T);
  uint4* hi = reinterpret_cast<uint4*>(xhi);
  uint4* lo = reinterpret_cast<uint4*>(xlo);
  const int ne = (L.E + 63) / 64;
#define DM_FRONT(N)                                                                             \
  hipLaunchKernelGGL(k_front<N>, grid, dim3(1024), lds, st, x, L.router, L.H, L.E, L, T, z, hi, \
                     lo, flags, ids, probs, shg, off, perm, units, meta, status)
  if (ne <= 1) DM_FRONT(1);
  else if (ne <= 2) DM_FRONT(2);
  else if (ne <= 4) DM_FRONT(4);
  else DM_FRONT(8);
#undef DM_FRONT
  return hipGetLastError();
}

int group_units_max(int T, int K, int E, int tok) {
  // an expert of c tokens has ceil(c / tok): at most c, and at most c / tok + 1
  const long tk = (long)T * K, n = tk / tok + (tk < E ? tk : E);
  return (int)(tk < n ? tk : n) + (T + tok - 1) / tok;
}

// ---------------------------------------------------------------------------
// rows [T][n] fp32 -> bf16 hi / lo; *need_lo |= 1 when some lo part is nonzero.
__global__ __launch_bounds__(256) void k_split_rows(const float* __restrict__ x, int64_t count8,
                                                    uint4* __restrict__ hi, uint4* __restrict__ lo,
                                                    int* __restrict__ need_lo) {
  bool nz = false;
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < count8; i += (int64_t)gridDim.x * 256) {
    const float4 a = reinterpret_cast<const float4*>(x)[2 * i];
    const float4 b = reinterpret_cast<const float4*>(x)[2 * i + 1];
    const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint4 h, l;
    split8(f, h, l);
    hi[i] = h;
    lo[i] = l;
    nz |= (l.x | l.y | l.z | l.w) != 0u;
  }
  // a plain store of 1, not an atomic: thousands of waves may set the flag,
  // and same-address atomics would be serialised one after another
  if (__builtin_amdgcn_ballot_w64(nz) != 0 && (threadIdx.x & 63) == 0) *need_lo = 1;
}

hipError_t launch_split_rows(const float* x, int64_t n, uint16_t* hi, uint16_t* lo, int* need_lo,
                             hipStream_t st) {
  const int64_t c8 = n / 8;
  const int blocks = (int)((c8 + 255) / 256 < 2048 ? (c8 + 255) / 256 : 2048);
  hipLaunchKernelGGL(k_split_rows, dim3(blocks > 0 ? blocks : 1), dim3(256), 0, st, x, c8,
                     reinterpret_cast<uint4*>(hi), reinterpret_cast<uint4*>(lo), need_lo);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Token rows of a unit (e, start): row r is position p = off[e] + start + r
// of the expert order, i.e. assignment a = perm[p] of token a / K; for the
// shared expert (e == E) row r is token start + r itself.
struct UnitTokens {
  int e, p0, n;   // expert, first position, tokens in this unit
  bool shared;
};
__device__ __forceinline__ UnitTokens unit_tokens(int2 u, const int32_t* off, int E, int T,
                                                  int size) {
  UnitTokens r;
  r.e = u.x;
  r.shared = u.x >= E;
  if (r.shared) {
    r.p0 = u.y;
    r.n = min(size, T - r.p0);
  } else {
    r.p0 = off[u.x] + u.y;
    r.n = min(size, off[u.x + 1] - r.p0);
  }
  return r;
}

struct GroupArgs {
  LayerDev L;
  const uint16_t* xhi;   // [T][H] bf16 parts of the activations
  const uint16_t* xlo;
  const int* need_lo;    // nonzero: some activation is not a bf16 value
  const int32_t* off;
  const int32_t* perm;
  const int2* units;
  const int32_t* meta;
  int T;
  uint16_t* hrh;         // h of routed positions [T*K][I], bf16 hi / lo
  uint16_t* hrl;
  uint16_t* hsh;         // h of the shared expert [T][Ish]
  uint16_t* hsl;
  float* r;              // routed down outputs [T*K][H] by assignment
  float* rs;             // shared down outputs [T][H]
  unsigned long long* status;
};

__device__ __forceinline__ int gwave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// The A chunks (16 rows x 128 columns, 4-bit + scales) of NT tiles for one
// k-step.  Gate/up (GU): tiles 0..NT/2-1 are gate tiles rb0 + t, tiles
// NT/2.. the up tiles at the same rows; down: tiles rb0 + t of one matrix.
template <int NT>
struct AChunks {
  uint4 w[NT];
  uint2 s[NT];
};

template <int NT, bool GU>
__device__ __forceinline__ void load_a(const ExpertView& v0, const ExpertView& v1, int rb0, int s,
                                       int lane, AChunks<NT>& a) {
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (GU)
      load_chunk_nt(t < NT / 2 ? v0 : v1, rb0 + (t % (NT / 2)), s, lane, a.w[t], a.s[t]);
    else
      load_chunk_nt(v0, rb0 + t, s, lane, a.w[t], a.s[t]);
  }
}

template <int NT>
__device__ __forceinline__ void dequant_a(const AChunks<NT>& a, int kk, bf16x8 (&av)[NT]) {
#pragma unroll
  for (int tl = 0; tl < NT; ++tl) av[tl] = dequant8(word_of(a.w[tl], kk), scale_of(a.s[tl], kk));
}

__device__ __forceinline__ void split4(const float* v, uint2& hi, uint2& lo) {
  float h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t hb = pack_bf16x2(v[i], 0.0f) & 0xFFFFu;
    h[i] = u2f(hb << 16);
    l[i] = v[i] - h[i];
  }
  hi = make_uint2(pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3]));
  lo = make_uint2(pack_bf16x2(l[0], l[1]), pack_bf16x2(l[2], l[3]));
}

// ---- epilogues -------------------------------------------------------------
// Gate/up: tile t < NT/2 holds gate features f0 + 16 t + 4q + i, tile
// NT/2 + t the same up features; h = SiLU(g) * u with the reference's checks
// (src/layers/swiglu.mojo:191-201), stored as bf16 hi / lo.
// The assignment (token * K + slot; the token for the shared expert) of
// column j of each of the unit's NC column tiles, all requested before the
// first store: a load issued after stores waits for them to complete (one
// counter covers both), which would serialise the epilogue on store latency.
template <int NC>
__device__ __forceinline__ void unit_assignments(const GroupArgs& g, const UnitTokens& ut, int j,
                                                 int (&aa)[NC]) {
// (The load is unconditional — perm has T * K >= T entries — so that no
// path joins with loads of unknown count in flight.)
#pragma unroll
  for (int ct = 0; ct < NC; ++ct) {
    const int p = ut.p0 + min(16 * ct + j, ut.n - 1);
    const int a = g.perm[p];
    aa[ct] = ut.shared ? p : a;
  }
}

// (aa: the unit's assignments of column j, unit_assignments)
template <int NT, int NC>
__device__ __forceinline__ void gu_epilogue(const GroupArgs& g, const UnitTokens& ut, int I,
                                            int f0, int q, int j, const f32x4 (&acc)[NT][NC],
                                            const int (&aa)[NC]) {
  const int K = g.L.K;
#pragma unroll
  for (int ct = 0; ct < NC; ++ct) {
    const int c = 16 * ct + j;
    if (c < ut.n) {
      const int p = ut.p0 + c;
#pragma unroll
      for (int half = 0; half < NT / 2; ++half) {
        const int fr = f0 + 16 * half + 4 * q;
        float hv[4];
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gg = acc[half][ct][i], u = acc[NT / 2 + half][ct][i];
          hv[i] = dm_silu(gg) * u;
          bad |= !finite_f(gg) || !finite_f(u) || !finite_f(hv[i]);
        }
        uint2 h2, l2;
        split4(hv, h2, l2);
        const size_t o = (size_t)p * I + fr;
        *reinterpret_cast<uint2*>((ut.shared ? g.hsh : g.hrh) + o) = h2;
        *reinterpret_cast<uint2*>((ut.shared ? g.hsl : g.hrl) + o) = l2;
        if (bad) {  // the error key needs token and slot (a division by K): only here
          const int a = aa[ct];
          const int t = ut.shared ? p : a / K, k = ut.shared ? 0 : a % K;
          const uint32_t ph = ut.shared ? kPhShared : kPhExpert;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float gg = acc[half][ct][i], u = acc[NT / 2 + half][ct][i];
            if (!finite_f(gg) || !finite_f(u) || !finite_f(hv[i])) {
              const uint32_t kind = !finite_f(gg) ? kEkGate : !finite_f(u) ? kEkUp : kEkH;
              record_err(g.status, err_key(ph, t, k, fr + i, kind));
            }
          }
        }
      }
    }
  }
}

// Down: tile tl holds output rows row0 + 16 tl + 4q + i of column j.
template <int NT, int NC>
__device__ __forceinline__ void down_epilogue(const GroupArgs& g, const UnitTokens& ut, int I,
                                              int row0, int q, int j, const f32x4 (&acc)[NT][NC],
                                              const int (&aa)[NC]) {
  const int H = g.L.H, K = g.L.K;
#pragma unroll
  for (int ct = 0; ct < NC; ++ct) {
    const int c = 16 * ct + j;
    if (c < ut.n) {
      const int p = ut.p0 + c;
      const int a = aa[ct];
      float* dst = ut.shared ? g.rs + (size_t)p * H : g.r + (size_t)a * H;
#pragma unroll
      for (int tl = 0; tl < NT; ++tl) {
        const int d0 = row0 + 16 * tl + 4 * q;
        const float* v = reinterpret_cast<const float*>(&acc[tl][ct]);
        *reinterpret_cast<float4*>(dst + d0) = make_float4(v[0], v[1], v[2], v[3]);
        if (!finite_f(v[0]) || !finite_f(v[1]) || !finite_f(v[2]) || !finite_f(v[3])) {
          // the error key needs token and slot (a division by K): only here
          const int t = ut.shared ? p : a / K, k = ut.shared ? 0 : a % K;
          const uint32_t ph = ut.shared ? kPhShared : kPhExpert;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!finite_f(v[i])) record_err(g.status, err_key(ph, t, k, I + d0 + i, kEkDown));
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k_experts<GU>: a workgroup of 8 waves takes one unit (up to 64 tokens) and
// 128 features (gate/up: gate and up tile 8 f + w of wave w, so that h =
// SiLU(g) * u is formed in its registers) or 256 output rows (down: tiles
// 16 f + 2w, 16 f + 2w + 1 of wave w).  A unit of n tokens runs with the
// column tiles it needs (NCT: 1, 2 or 4 of 16 tokens).  Every operand is
// staged in LDS by direct-to-LDS loads (global_load_lds_dwordx4: 16 bytes per
// lane land in LDS without passing through registers), D stages ahead:
//   - B rows: 256 bytes per token and stage, segment sigma of row r stored at
//     position sigma ^ (r & 15) of its row, so that the 16 rows of one MFMA B
//     operand read distinct LDS banks;
//   - A: a k-step's 16 A16 chunks (16 rows x 128 columns, 2 per wave) as they
//     lie in memory, and their scales.
// A stage is 128 columns of the bf16 hi parts, or, when the activations are
// not all bf16 values (LO: h always; x when the need-lo flag is set), 64
// columns of the hi and of the lo parts: then a chunk serves two stages, its
// weights dequantised once for both parts.  One barrier per stage: after it,
// stage s is complete everywhere and the buffer of stage s - 1 is free.
//
// At most 128 registers and 78 KB of LDS, so that two workgroups share a CU:
// one's matrix instructions run while the other waits for its stage or its
// first loads (one workgroup per CU on 128-token units waited for a third of
// its time and lost a quarter of the launch to the last round of items).
// Workgroups are dispatched as others end; they come in classes b % 8, which
// the dispatcher places on one XCD each (it hands a launch's workgroups to the
// XCDs in rotation).  The units are cut into 8 contiguous ranges (the units of
// an expert are adjacent) and range c runs in class c with each unit's blocks
// next to each other: they share that XCD's L2 for the unit's token rows, and
// the units of an expert for its weights.
//
// Bound by the matrix and vector units together from some 32 tokens a unit
// (every weight is rounded to bf16 on the way, 1.75 operations), below by the
// weights' bytes.  Against that former kernel, at hidden 2048, inter 512, 256
// experts: 1533 fp32 tokens, gate/up 291 -> 168 us and down 166 + 13 -> 95; 2048
// bf16 tokens (Zipf) 152 -> 134 and 125 + 24 -> 108; 131 tokens 91 -> 70 and 23 + 47
// -> 45 (290 MB of weights in the 70: 4.1 TB/s; a copy reaches 5.1).
constexpr int kExThreads = 512;
constexpr int kExRowBytes = 256;                        // a token row of a stage
constexpr int kExChunks = 16 * 1024;                    // 16 A16 chunks
constexpr int kExABytes = kExChunks + 16 * 128;         // and their scales
constexpr int kExADma = 3;                              // loads of a chunk pair per wave
template <int NCT>
struct ExStages {
  static constexpr int kAhead = NCT == 4 ? 1 : 2;       // stages in flight
  static constexpr int kBufs = kAhead + 1;
  static constexpr int kB = 16 * NCT * kExRowBytes;
  static constexpr int kBuf = kB + kExABytes;
  static constexpr int kRowLoads = NCT == 4 ? 2 : 1;    // of 32 rows over the 8 waves
};
constexpr int cmax(int a, int b) { return a > b ? a : b; }
constexpr int kExLds = cmax(ExStages<4>::kBufs * ExStages<4>::kBuf,
                            cmax(ExStages<2>::kBufs * ExStages<2>::kBuf,
                                 ExStages<1>::kBufs * ExStages<1>::kBuf));
static_assert(2 * kExLds <= 160 * 1024, "two workgroups per CU");

// The B fragments of N column tiles (rows 16 ct + j of a stage, 16 * 256 bytes
// apart) as N LDS reads in flight together.  Inline assembly: the compiler
// would otherwise sink each read next to its first use.  Their registers are
// not valid before lds_wait.
template <int N>
__device__ __forceinline__ void lds_read(uint32_t a, bf16x8 (&b)[N]) {
#pragma unroll
  for (int ct = 0; ct < N; ++ct)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(b[ct]) : "v"(a), "n"(ct * 16 * kExRowBytes));
}
// Wait until at most M LDS operations are in flight (LDS operations complete
// in order, so every read issued before the last M has landed); b's
// registers are tied to the wait, so no use of them moves above it.
template <int M, int N>
__device__ __forceinline__ void lds_wait(bf16x8 (&b)[N]) {
  if constexpr (N == 4)
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]) : "n"(M));
  else if constexpr (N == 2)
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(b[0]), "+v"(b[1]) : "n"(M));
  else
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(b[0]) : "n"(M));
}
// Until at most n of this wave's memory operations are in flight (uniform).
__device__ __forceinline__ void vm_wait(int n) {
  static_assert(kExADma == 3, "0, a stage's row load, a chunk pair, or both");
  if (n == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  else if (n == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
  else if (n == 1) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One unit's block on NCT column tiles.
template <bool GU, bool LO, int NCT>
struct ExRun {
  using S = ExStages<NCT>;
  const uint8_t* a0;  // this wave's two tiles
  const uint8_t* a1;
  const uint8_t* sc;  // this lane's 16 bytes of their scales (lanes 0 .. 15)
  const uint16_t* b[S::kRowLoads];  // this lane's 8 columns of its token rows
  uint32_t l0;
  int w, lane, nst, nrow;           // stages; row loads of this wave and stage
  uint4 c0, c1;
  uint2 s0, s1;
  f32x4 acc[2][NCT];

  __device__ __forceinline__ void issue_b(int s) {
    const uint32_t st = l0 + (uint32_t)(s % S::kBufs * S::kBuf);
    if (NCT > 1 || nrow) {  // uniform
#pragma unroll
      for (int m = 0; m < S::kRowLoads; ++m)
        dma16_lds(b[m] + s * (LO ? 64 : 128), st + (uint32_t)((w + 8 * m) * 1024));
    }
  }
  __device__ __forceinline__ void issue_a(int c) {
    const uint32_t st = l0 + (uint32_t)(c % S::kBufs * S::kBuf + S::kB);
    dma16_lds(a0 + (c * 64 + lane) * 16, st + (uint32_t)(2 * w * 1024));
    dma16_lds(a1 + (c * 64 + lane) * 16, st + (uint32_t)((2 * w + 1) * 1024));
    // scales of the two chunks: 128 bytes each, lanes 0..7 and 8..15
    if (lane < 16) dma16_lds(sc + c * 128, st + (uint32_t)(kExChunks + w * 256));
  }

  // Stage s (LO: ODD: the second one of its chunk).  The B fragments of step
  // z + 1 (a group of 32 columns; LO: of its hi, then its lo part) are read
  // while step z multiplies.
  template <bool ODD>
  __device__ __forceinline__ void stage(int s, const unsigned char* lds) {
    // this wave's loads of stage s have landed; in flight may be those of
    // stage s + 1 (where two are ahead) and, at the odd stage of a chunk, the
    // next chunk's
    const bool more = s + 1 < nst;
    int n = S::kAhead > 1 && more ? nrow : 0;
    if (LO ? ODD && more : S::kAhead > 1 && more) n += kExADma;
    vm_wait(n);
    // ... and after the barrier every wave's, and nobody reads stage s - 1
    __builtin_amdgcn_s_barrier();
    if (s + S::kAhead < nst) {
      issue_b(s + S::kAhead);
      if (!LO) issue_a(s + S::kAhead);
    }
    const int c = LO ? s >> 1 : s;
    if (LO && !ODD && s + 2 < nst) issue_a(c + 1);
    const int q = lane >> 4, j = lane & 15;
    if (!LO || !ODD) {
      const unsigned char* a = lds + c % S::kBufs * S::kBuf + S::kB;
      c0 = *reinterpret_cast<const uint4*>(a + 2 * w * 1024 + lane * 16);
      c1 = *reinterpret_cast<const uint4*>(a + (2 * w + 1) * 1024 + lane * 16);
      s0 = *reinterpret_cast<const uint2*>(a + kExChunks + w * 256 + j * 8);
      s1 = *reinterpret_cast<const uint2*>(a + kExChunks + w * 256 + 128 + j * 8);
    }
    const uint32_t bp = l0 + (uint32_t)(s % S::kBufs * S::kBuf + j * kExRowBytes);
    auto seg = [&](int z) { return (uint32_t)(((LO ? 8 * (z & 1) + 4 * (z >> 1) : 4 * z) + q) ^ j) * 16; };
    bf16x8 bb[2][NCT], d0, d1;
    lds_read<NCT>(bp + seg(0), bb[0]);
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      if (z < 3) lds_read<NCT>(bp + seg(z + 1), bb[(z + 1) & 1]);
      if (!LO || !(z & 1)) {
        const int kk = LO ? (ODD ? 2 : 0) + (z >> 1) : z;
        d0 = dequant8(word_of(c0, kk), scale_of(s0, kk));
        d1 = dequant8(word_of(c1, kk), scale_of(s1, kk));
      }
      if (z < 3)
        lds_wait<NCT>(bb[z & 1]);
      else
        lds_wait<0>(bb[z & 1]);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        acc[0][ct] = mfma16(d0, bb[z & 1][ct], acc[0][ct]);
        acc[1][ct] = mfma16(d1, bb[z & 1][ct], acc[1][ct]);
      }
    }
  }

  __device__ __forceinline__ void run(const GroupArgs& g, const UnitTokens& ut, int I, int fb,
                                      const unsigned char* lds) {
    const LayerDev& L = g.L;
    const int H = L.H, K = L.K;
    w = gwave_id();
    lane = threadIdx.x & 63;
    l0 = lds_u32(lds);
    const int q = lane >> 4, j = lane & 15;
    const int KD = GU ? H : I, nGQ = KD / kQuadCols;  // reduction length, chunks
    nst = LO ? 2 * nGQ : nGQ;
    const size_t mat = (size_t)I * H;
    const uint8_t* nib;
    const uint16_t* scl;
    int t0, t1;
    if (GU) {
      nib = ut.shared ? L.sgu_nib : L.gu_nib + (size_t)ut.e * mat;
      scl = ut.shared ? L.sgu_sc : L.gu_sc + (size_t)ut.e * 2 * (mat / kGroup);
      t0 = fb * 8 + w;
      t1 = I / kTileRows + t0;  // the up matrix follows the gate's tiles
    } else {
      nib = ut.shared ? L.sd_nib : L.d_nib + (size_t)ut.e * (mat / 2);
      scl = ut.shared ? L.sd_sc : L.d_sc + (size_t)ut.e * (mat / kGroup);
      // H is a multiple of 128, so the last block may hold 128 rows: waves
      // past H load tiles 0 and 1 (their share of the B rows is still needed)
      // and store nothing
      t0 = fb * 256 + 32 * w < H ? fb * 16 + 2 * w : 0;
      t1 = t0 + 1;
    }
    a0 = nib + a16_nib_offset(nGQ, t0, 0, 0);
    a1 = nib + a16_nib_offset(nGQ, t1, 0, 0);
    sc = reinterpret_cast<const uint8_t*>(scl + a16_sc_offset(nGQ, lane < 8 ? t0 : t1, 0, 0)) +
         (lane & 7) * 16;
    // B rows: load m of wave w carries rows 4 (w + 8m) .. + 3, lane l row
    // 4 (w + 8m) + l / 16, stored segment l % 16 = segment (l % 16) ^ (row & 15)
    // (of 16: 128 hi columns; LO: 64 hi, then 64 lo columns)
    nrow = NCT > 1 || w < 4 ? S::kRowLoads : 0;
    const int sg = (lane & 15) ^ ((4 * w + q) & 15);
    const uint16_t* hi = GU ? g.xhi : (ut.shared ? g.hsh : g.hrh);
    const uint16_t* lo = GU ? g.xlo : (ut.shared ? g.hsl : g.hrl);
    const uint16_t* src = LO ? (sg < 8 ? hi : lo) + (sg & 7) * 8 : hi + sg * 8;
#pragma unroll
    for (int m = 0; m < S::kRowLoads; ++m) {
      const int p = ut.p0 + min(4 * (w + 8 * m) + q, ut.n - 1);
      const int row = !GU || ut.shared ? p : g.perm[p] / K;  // h rows by position, x by token
      b[m] = src + (size_t)row * KD;
    }
    issue_b(0);
    issue_a(0);
    if (S::kAhead > 1 && nst > 1) {
      issue_b(1);
      if (!LO) issue_a(1);
    }
    int aa[NCT];
    unit_assignments<NCT>(g, ut, j, aa);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) acc[t][ct] = f32x4{0, 0, 0, 0};
    if (LO) {
      for (int s = 0; s < nst; s += 2) {
        stage<false>(s, lds);
        stage<true>(s + 1, lds);
      }
    } else {
      for (int s = 0; s < nst; ++s) stage<false>(s, lds);
    }
    if (GU)
      gu_epilogue<2, NCT>(g, ut, I, fb * 128 + 16 * w, q, j, acc, aa);
    else if (fb * 256 + 32 * w < H)
      down_epilogue<2, NCT>(g, ut, I, fb * 256 + 32 * w, q, j, acc, aa);
  }
};

template <bool GU, bool LO>
__device__ __forceinline__ void ex_unit(const GroupArgs& g, const UnitTokens& ut, int I, int fb,
                                        const unsigned char* lds) {
  if (ut.n <= 16) ExRun<GU, LO, 1>().run(g, ut, I, fb, lds);
  else if (ut.n <= 32) ExRun<GU, LO, 2>().run(g, ut, I, fb, lds);
  else ExRun<GU, LO, 4>().run(g, ut, I, fb, lds);
}

// (The grouping's arrays lead the arguments, preloaded at dispatch: they
// start each workgroup's chain of dependent loads.)
template <bool GU>
__global__ __launch_bounds__(kExThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_experts(const int32_t* meta, const int2* units, const int32_t* off, const int32_t* perm,
               const int* need_lo, int nblk, GroupArgs gk) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds2[];
  GroupArgs g = gk;
  g.perm = perm;
  const int nall = meta[0], span = (nall + 7) >> 3, idx = (int)blockIdx.x >> 3;
  const int ul = idx / nblk, fb = idx - ul * nblk, u = ((int)blockIdx.x & 7) * span + ul;
  if (ul >= span || u >= nall) return;
  const UnitTokens ut = unit_tokens(units[u], off, g.L.E, g.T, kUnitTok);
  const int I = ut.shared ? g.L.Ish : g.L.I;
  if (GU && fb * 128 >= I) return;  // uniform per workgroup
  if (!GU || need_lo[0] != 0)
    ex_unit<GU, true>(g, ut, I, fb, lds2);
  else
    ex_unit<GU, false>(g, ut, I, fb, lds2);
}

// k_experts' LDS is above the default limit of a launch: raised once per
// device.
static hipError_t ex_attrs() {
  static std::atomic<uint64_t> done{0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev < 64 ? 1ull << dev : 0;
  if (bit && (done.load() & bit)) return hipSuccess;
  e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_experts<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kExLds);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_experts<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kExLds);
  if (e == hipSuccess) done.fetch_or(bit);
  return e;
}

// ---------------------------------------------------------------------------
// Calls of at most kSmallMaxT tokens: units of up to 16, one column tile.
// Their few workgroups are bound by the latency of their stages, so waves are
// independent (no LDS, no barrier): each wave owns 2 A tiles (gate/up: 16
// features, gate and up tile; down: 32 output rows) and reads its B fragments
// (lane (q, j): token j, columns 8q..8q+7 of each group) straight from memory
// into the same prefetch ring as the A chunks, P k-steps ahead.  At most 168
// registers per lane, so that three waves share a SIMD and their loads
// overlap.  Through k_experts instead, weights from HBM: 2 tokens 46 us per
// call against 37, 12 tokens 68 against 63, 24 tokens 91 against 83 (fp32
// activations 112 against 110), 32 tokens 94 against 90 (115 against 121); at 48
// tokens, where the shared expert fills three units, it is 112 against the 139 of
// one workgroup per CU on 128-token units beside these kernels.
constexpr int kSmallTiles = 2;

template <bool LO>
struct SmallStep {
  AChunks<kSmallTiles> a;
  v4u b[kGroupsPerQuad];
  v4u bl[LO ? kGroupsPerQuad : 1];
};

template <bool LO, bool GU>
__device__ __forceinline__ void small_load(const ExpertView& v0, const ExpertView& v1, int rb0,
                                           int s, int lane, const uint16_t* bh,
                                           const uint16_t* bl, SmallStep<LO>& st) {
  load_a<kSmallTiles, GU>(v0, v1, rb0, s, lane, st.a);
#pragma unroll
  for (int kk = 0; kk < kGroupsPerQuad; ++kk) {
    const int o = s * kQuadCols + kk * kGroup;
    st.b[kk] = *reinterpret_cast<const v4u*>(bh + o);
    if (LO) st.bl[kk] = *reinterpret_cast<const v4u*>(bl + o);
  }
}

template <bool LO>
__device__ __forceinline__ void small_step(const SmallStep<LO>& st,
                                           f32x4 (&acc)[kSmallTiles][1]) {
#pragma unroll
  for (int kk = 0; kk < kGroupsPerQuad; ++kk) {
    bf16x8 av[kSmallTiles];
    dequant_a<kSmallTiles>(st.a, kk, av);
    const bf16x8 b = __builtin_bit_cast(bf16x8, st.b[kk]);
#pragma unroll
    for (int tl = 0; tl < kSmallTiles; ++tl) acc[tl][0] = mfma16(av[tl], b, acc[tl][0]);
    if (LO) {
      const bf16x8 b2 = __builtin_bit_cast(bf16x8, st.bl[kk]);
#pragma unroll
      for (int tl = 0; tl < kSmallTiles; ++tl) acc[tl][0] = mfma16(av[tl], b2, acc[tl][0]);
    }
  }
}

// bh / bl point at this lane's B row (+ 8q) at column 0.  The ring slot of a
// step is a constant of the unrolled body; steps past the last are clamped
// to it (redundant loads only when ns % P != 0).
template <bool LO, bool GU, int P>
__device__ __forceinline__ void small_loop(const ExpertView& v0, const ExpertView& v1, int rb0,
                                           const uint16_t* bh, const uint16_t* bl, int ns,
                                           f32x4 (&acc)[kSmallTiles][1]) {
  const int lane = threadIdx.x & 63;
  SmallStep<LO> ring[P];
#pragma unroll
  for (int u = 0; u < P; ++u) small_load<LO, GU>(v0, v1, rb0, min(u, ns - 1), lane, bh, bl, ring[u]);
#pragma unroll
  for (int tl = 0; tl < kSmallTiles; ++tl) acc[tl][0] = f32x4{0, 0, 0, 0};
  int s0 = 0;
  for (; s0 + P < ns; s0 += P) {
#pragma unroll
    for (int u = 0; u < P; ++u) {
      small_step<LO>(ring[u], acc);
      small_load<LO, GU>(v0, v1, rb0, min(s0 + u + P, ns - 1), lane, bh, bl, ring[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < P; ++u)
    if (s0 + u < ns) small_step<LO>(ring[u], acc);
}

constexpr int kSmallGuCols = 4 * 16;   // features per small gate/up workgroup
constexpr int kSmallDnRows = 4 * 32;   // output rows per small down workgroup

// Gate/up of unit bx, features by * 64 .., on wave w of four.
__device__ __forceinline__ void gu_small_part(const GroupArgs& g, int bx, int by, int w) {
  const int ui = bx;
  if (ui >= g.meta[0]) return;
  const UnitTokens ut = unit_tokens(g.units[ui], g.off, g.L.E, g.T, kUnitSmall);
  const LayerDev& L = g.L;
  const int H = L.H, K = L.K, I = ut.shared ? L.Ish : L.I;
  const int lane = threadIdx.x & 63, q = lane >> 4, j = lane & 15;
  const int f0 = by * kSmallGuCols + 16 * w;
  if (f0 >= I) return;  // uniform per wave
  const size_t mat = (size_t)I * H;
  const ExpertView gv = ut.shared ? ExpertView{L.sgu_nib, L.sgu_sc, I, H}
                                  : ExpertView{L.gu_nib + (size_t)ut.e * mat,
                                               L.gu_sc + (size_t)ut.e * 2 * (mat / kGroup), I, H};
  const ExpertView uv = {gv.nib + mat / 2, gv.sc + mat / kGroup, I, H};
  const int r = min(j, ut.n - 1);
  const int t = ut.shared ? ut.p0 + r : g.perm[ut.p0 + r] / K;
  const size_t o = (size_t)t * H + 8 * q;
  f32x4 acc[kSmallTiles][1];
  const int ns = H / kQuadCols;
  if (g.need_lo[0] != 0)
    small_loop<true, true, 2>(gv, uv, f0 / kTileRows, g.xhi + o, g.xlo + o, ns, acc);
  else
    small_loop<false, true, 4>(gv, uv, f0 / kTileRows, g.xhi + o, g.xlo + o, ns, acc);
  int aa[1];
  unit_assignments<1>(g, ut, j, aa);
  gu_epilogue<kSmallTiles, 1>(g, ut, I, f0, q, j, acc, aa);
}

// Down of unit bx, output rows by * 128 .., on wave w of four.
__device__ __forceinline__ void down_small_part(const GroupArgs& g, int bx, int by, int w) {
  const int ui = bx;
  if (ui >= g.meta[0]) return;
  const UnitTokens ut = unit_tokens(g.units[ui], g.off, g.L.E, g.T, kUnitSmall);
  const LayerDev& L = g.L;
  const int H = L.H, I = ut.shared ? L.Ish : L.I;
  const int lane = threadIdx.x & 63, q = lane >> 4, j = lane & 15;
  const int row0 = by * kSmallDnRows + 32 * w;
  if (row0 >= H) return;
  const size_t mat = (size_t)H * I;
  const ExpertView dv = ut.shared ? ExpertView{L.sd_nib, L.sd_sc, H, I}
                                  : ExpertView{L.d_nib + (size_t)ut.e * (mat / 2),
                                               L.d_sc + (size_t)ut.e * (mat / kGroup), H, I};
  const size_t o = (size_t)(ut.p0 + min(j, ut.n - 1)) * I + 8 * q;
  f32x4 acc[kSmallTiles][1];
  small_loop<true, false, 2>(dv, dv, row0 / kTileRows, (ut.shared ? g.hsh : g.hrh) + o,
                             (ut.shared ? g.hsl : g.hrl) + o, I / kQuadCols, acc);
  int aa[1];
  unit_assignments<1>(g, ut, j, aa);
  down_epilogue<kSmallTiles, 1>(g, ut, I, row0, q, j, acc, aa);
}

// The grouping's arrays come first among the arguments: they start each
// workgroup's chain of dependent loads (meta -> units -> off -> perm) and
// are preloaded into scalar registers at dispatch.
__global__ __launch_bounds__(kGThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_gu_small(
    const int32_t* meta, const int2* units, const int32_t* off, const int32_t* perm,
    GroupArgs gk) {
  GroupArgs g = gk;
  g.meta = meta;
  g.units = units;
  g.off = off;
  g.perm = perm;
  gu_small_part(g, blockIdx.x, blockIdx.y, gwave_id());
}

__global__ __launch_bounds__(kGThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_down_small(
    const int32_t* meta, const int2* units, const int32_t* off, const int32_t* perm,
    GroupArgs gk) {
  GroupArgs g = gk;
  g.meta = meta;
  g.units = units;
  g.off = off;
  g.perm = perm;
  down_small_part(g, blockIdx.x, blockIdx.y, gwave_id());
}

hipError_t launch_experts_grouped(const LayerDev& L, const uint16_t* xhi, const uint16_t* xlo,
                                  const int* need_lo, const int32_t* off, const int32_t* perm,
                                  const int2* units, const int32_t* meta, int T, uint16_t* hrh,
                                  uint16_t* hrl, uint16_t* hsh, uint16_t* hsl, float* r,
                                  float* rs, unsigned long long* status, hipStream_t st) {
  const GroupArgs g = {L, xhi, xlo, need_lo, off, perm, units, meta, T,
                       hrh, hrl, hsh, hsl, r, rs, status};
  if ((size_t)T * L.K * (L.I > L.Ish ? L.I : L.Ish) >= (1ull << 32) ||
      (size_t)T * L.H >= (1ull << 32))
    return hipErrorInvalidValue;
  if (T <= kSmallMaxT) {
    // (workgroups go to the XCDs in rotation: with a multiple of 8 units a row of
    // the grid, all blocks of a unit would run on one XCD; 24 tokens, 32 experts,
    // hidden 4096: 97 -> 93 us per call.  The two more end at once)
    int nu = group_units_max(T, L.K, L.E, kUnitSmall);
    if (nu % 8 == 0) nu += 2;
    const int gy = ((L.I > L.Ish ? L.I : L.Ish) + kSmallGuCols - 1) / kSmallGuCols;
    const int dy = (L.H + kSmallDnRows - 1) / kSmallDnRows;
    hipLaunchKernelGGL(k_gu_small, dim3(nu, gy), dim3(kGThreads), 0, st, meta, units, off, perm, g);
    hipLaunchKernelGGL(k_down_small, dim3(nu, dy), dim3(kGThreads), 0, st, meta, units, off, perm,
                       g);
    return hipGetLastError();
  }
  const hipError_t e = ex_attrs();
  if (e != hipSuccess) return e;
  // a grid for the most units there can be; those past the units end at once
  const int classes = 8 * ((group_units_max(T, L.K, L.E, kUnitTok) + 7) / 8);
  const int gb = ((L.I > L.Ish ? L.I : L.Ish) + 127) / 128, db = (L.H + 255) / 256;
  hipLaunchKernelGGL(k_experts<true>, dim3(classes * gb), dim3(kExThreads), kExLds, st, meta, units,
                     off, perm, need_lo, gb, g);
  hipLaunchKernelGGL(k_experts<false>, dim3(classes * db), dim3(kExThreads), kExLds, st, meta,
                     units, off, perm, need_lo, db, g);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// y[t][d] = (sum_k p[t][k] r[t*K+k][d]) + g[t] rs[t][d] (+ residual[t][d]):
// routed experts in the reference order, then the shared expert, then the
// residual (src/layers/moe.mojo:157-166, src/layers/forward_layer.mojo:226-238).
__global__ __launch_bounds__(256) void k_combine(const float* __restrict__ r,
                                                  const float* __restrict__ rs,
                                                  const float* __restrict__ probs,
                                                  const float* __restrict__ shg,
                                                  const float* __restrict__ residual, int H, int K,
                                                  float* __restrict__ y,
                                                  unsigned long long* status,
                                                  int* __restrict__ clear_flag, int t0) {
  // four consecutive outputs per thread (H % 4 == 0); the slots' rows are
  // requested eight at a time before their products
  const int t = t0 + blockIdx.y, d = (blockIdx.x * 256 + threadIdx.x) * 4;
  // the last kernel of a call clears the call's need-lo flag for the next
  if (clear_flag && t == 0 && d == 0) *clear_flag = 0;
  if (d >= H) return;
  const float* pt = probs + (size_t)t * K;
  float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = 0; k0 < K; k0 += 8) {
    float4 rv[8];
    float pv[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const int k = min(k0 + kk, K - 1);
      rv[kk] = *reinterpret_cast<const float4*>(r + ((size_t)t * K + k) * H + d);
      pv[kk] = pt[k];
    }
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      if (k0 + kk < K) {
        a[0] = a[0] + pv[kk] * rv[kk].x;
        a[1] = a[1] + pv[kk] * rv[kk].y;
        a[2] = a[2] + pv[kk] * rv[kk].z;
        a[3] = a[3] + pv[kk] * rv[kk].w;
      }
    }
  }
  const float g = shg[t];
  const float4 sv = *reinterpret_cast<const float4*>(rs + (size_t)t * H + d);
  float tot[4] = {a[0] + g * sv.x, a[1] + g * sv.y, a[2] + g * sv.z, a[3] + g * sv.w};
  if (residual) {
    const float4 rr = *reinterpret_cast<const float4*>(residual + (size_t)t * H + d);
    tot[0] = tot[0] + rr.x;
    tot[1] = tot[1] + rr.y;
    tot[2] = tot[2] + rr.z;
    tot[3] = tot[3] + rr.w;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (!finite_f(tot[i])) record_err(status, err_key(kPhAgg, t, 0, d + i, 0));
  *reinterpret_cast<float4*>(y + (size_t)t * H + d) = make_float4(tot[0], tot[1], tot[2], tot[3]);
}

hipError_t launch_combine(const float* r, const float* rs, const float* probs, const float* shg,
                          const float* residual, int T, int H, int K, float* y,
                          unsigned long long* status, hipStream_t st, int* clear_flag) {
  if (H % 4) return hipErrorInvalidValue;
  for (int t0 = 0; t0 < T; t0 += 65535) {  // grid.y holds at most 65535 tokens
    const int n = T - t0 < 65535 ? T - t0 : 65535;
    hipLaunchKernelGGL(k_combine, dim3((H / 4 + 255) / 256, n), dim3(256), 0, st, r, rs, probs, shg,
                       residual, H, K, y, status, clear_flag, t0);
  }
  return hipGetLastError();
}

}  // namespace dm
