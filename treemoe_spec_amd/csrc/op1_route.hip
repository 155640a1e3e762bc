// op1 routing on gfx950: router logits + softmax, then op3 budget routing and
// stable (expert, DFS-order) bucketing.
//
// Every floating-point operation here is written out in a fixed order with
// contraction disabled, so that the CPU restatement reproduces the outputs bit
// for bit: expert ids, gate weights, demand and every layout index.
//
// Launch shapes: the router runs one workgroup (8 waves) per token, one wave
// per expert, or from 1024 tokens one wave per token with W_g in LDS.  The
// bucketing runs in one workgroup, from 1024 tokens spread over the chip in two
// or three launches; at one or two tokens it shares the router's launch.
// Otherwise they are separate launches: handing the gates to a last-finishing
// workgroup instead would need a device-scope release fence per workgroup (an
// L2 write-back), which measured slower than the kernel boundary.
#pragma clang fp contract(off)

#include <algorithm>

#include "op1_bucket.h"
#include "tm_common.h"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
// From this many tokens the bucketing is spread over the chip; below, one
// workgroup keeps every per-slot intermediate in LDS.
constexpr int kSpreadMinTokens = 1024;
// Up to this many tokens more than kMaxPaddedRows padded rows are refused: the
// one-workgroup kernel's block table, and above kSpreadMinTokens a limit of the
// entry points that no call with its routing's own max_blocks reaches (2 T rows
// in at most 64 experts).
constexpr int kFewTokens = 4096;
constexpr int kMaxPaddedRows = 16384;
// Tokens from which the row router runs: its per-workgroup W_g copy costs
// ~8 us, so below ~1024 tokens one workgroup per token is faster (T = 512:
// 6.1 against 8.6 us; T = 2048: 14.0 against 9.2 us; T = 4096: 25.4 against
// 13.1 us at H = 4096, E = 8).
constexpr int kRowsMinTokens = 1024;

// The two 16-bit elements of a 32-bit word, widened exactly to fp32 (DT is
// TM_DTYPE_BF16 or TM_DTYPE_F16).
template <int DT>
__device__ __forceinline__ float lo16(uint32_t w) {
  return DT == TM_DTYPE_F16 ? tm_f16_to_f32((uint16_t)(w & 0xffffu)) : __uint_as_float(w << 16);
}
template <int DT>
__device__ __forceinline__ float hi16(uint32_t w) {
  return DT == TM_DTYPE_F16 ? tm_f16_to_f32((uint16_t)(w >> 16))
                            : __uint_as_float(w & 0xffff0000u);
}

template <int DT>
__device__ __forceinline__ float fma8(uint4 xv, uint4 wv, float acc) {
  acc = fmaf(lo16<DT>(xv.x), lo16<DT>(wv.x), acc);
  acc = fmaf(hi16<DT>(xv.x), hi16<DT>(wv.x), acc);
  acc = fmaf(lo16<DT>(xv.y), lo16<DT>(wv.y), acc);
  acc = fmaf(hi16<DT>(xv.y), hi16<DT>(wv.y), acc);
  acc = fmaf(lo16<DT>(xv.z), lo16<DT>(wv.z), acc);
  acc = fmaf(hi16<DT>(xv.z), hi16<DT>(wv.z), acc);
  acc = fmaf(lo16<DT>(xv.w), lo16<DT>(wv.w), acc);
  acc = fmaf(hi16<DT>(xv.w), hi16<DT>(wv.w), acc);
  return acc;
}

// Softmax of one token's E logits (s_logit, bf16-rounded) by one wave: max,
// e^(l - max), a sum in expert order, a correctly rounded division.  Lane e
// returns expert e's gate.
__device__ __forceinline__ float router_softmax(const float* s_logit, float* __restrict__ gates,
                                                int t, int E, int lane) {
  const float my_logit = (lane < E) ? s_logit[lane] : 0.0f;
  float m = (lane < E) ? my_logit : -INFINITY;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  const float ex = (lane < E) ? tm_expf_det(my_logit - m) : 0.0f;
  float s = 0.0f;
  for (int e = 0; e < E; ++e) s = s + __shfl(ex, e);
  const float gate = ex / s;
  if (lane < E) gates[(size_t)t * E + lane] = gate;
  return gate;
}

// One logit by one wave: see router_token.
template <int DT>
__device__ __forceinline__ float router_logit(const uint16_t* __restrict__ x,
                                              const uint16_t* __restrict__ wg, int H, int lane) {
  const int nchunk = H >> 3;
  const uint4* xr = reinterpret_cast<const uint4*>(x);
  const uint4* wr = reinterpret_cast<const uint4*>(wg);
  float acc = 0.0f;
  int c = lane;
  for (; c + 64 * 7 < nchunk; c += 64 * 8) {
    uint4 xv[8], wv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      xv[u] = xr[c + 64 * u];
      wv[u] = wr[c + 64 * u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = fma8<DT>(xv[u], wv[u], acc);
  }
  for (; c < nchunk; c += 64) acc = fma8<DT>(xr[c], wr[c], acc);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) acc = acc + __shfl_xor(acc, off);
  return Half16<DT>::to_f32(Half16<DT>::round(acc));
}

// Router for token t in one workgroup.  Logit (t, e): lane l of the wave that
// owns expert e accumulates the 8-element chunks l, l+64, ... in element order
// (fmaf of exact products of the 16-bit inputs); the 64 lane sums are combined
// by a halving tree (xor butterfly) and rounded to the input type (bf16 or
// fp16), as F.linear on such operands returns (treemoe/kernels/op1_tree_moe.py:676).  Softmax (:677) in fp32: max,
// e^(l - max), a sum in expert order, a correctly rounded division.
template <int DT>
__device__ __forceinline__ void router_token(const uint16_t* __restrict__ x,
                                             const uint16_t* __restrict__ wg,
                                             float* __restrict__ gates, int t, int H, int E,
                                             float* s_logit) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  for (int e = wave; e < E; e += kWaves) {
    const float l = router_logit<DT>(x + (size_t)t * H, wg + (size_t)e * H, H, lane);
    if (lane == 0) s_logit[e] = l;
  }
  __syncthreads();
  if (wave == 0) router_softmax(s_logit, gates, t, E, lane);
}

using tmb::BucketArgs;
constexpr int kMaxBlocks = kMaxPaddedRows / 16;
// gates staged in LDS when T * E fits (64 KB)
using BucketShared = tmb::BucketSharedT<kSpreadMinTokens, 16384, kMaxBlocks>;
using tmb::Top2;
using tmb::wave_exclusive_scan;

template <int DT>
__global__ void __launch_bounds__(kThreads)
tm_router_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg,
                 float* __restrict__ gates, int T, int H, int E) {
  __shared__ float s_logit[TM_MAX_EXPERTS];
  router_token<DT>(x, wg, gates, blockIdx.x, H, E, s_logit);
}

// Router for many tokens: wave w of workgroup b takes token kWaves b + w and
// all E experts.  x stays in registers (XC 16-byte chunks per lane, H = 512
// XC) and W_g in LDS, read once per workgroup instead of once per token.  Lane
// l accumulates its chunks l, l+64, ... of each expert in the order
// router_token uses, then the same xor fold, rounding and softmax, so the
// gates are bit-identical to it.
constexpr int kRowsLdsChunks = 4096;  // W_g staged in LDS: E * H / 8 <= 4096 (64 KB)

template <int DT, int XC>
__global__ void __launch_bounds__(kThreads)
tm_router_rows_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg,
                      float* __restrict__ gates, int T, int H, int E) {
  __shared__ uint4 s_w[kRowsLdsChunks];
  __shared__ float s_logit[kWaves][TM_MAX_EXPERTS];
  const int nchunk = H >> 3;  // = 64 XC
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * kWaves + wave;
  // the token's row is requested before the W_g copy, so the two memory
  // round trips overlap instead of following each other (T = 2048: 14.9 ->
  // 14.2 us)
  const uint4* xr = reinterpret_cast<const uint4*>(x + (size_t)min(t, T - 1) * H);
  uint4 xv[XC];
#pragma unroll
  for (int u = 0; u < XC; ++u) xv[u] = xr[lane + 64 * u];
  const uint4* wg4 = reinterpret_cast<const uint4*>(wg);
  for (int i = threadIdx.x; i < E * nchunk; i += kThreads) s_w[i] = wg4[i];
  tm_lds_barrier();
  if (t >= T) return;
  for (int e = 0; e < E; ++e) {
    const uint4* wr = s_w + e * nchunk;
    float acc = 0.0f;
#pragma unroll
    for (int u = 0; u < XC; ++u) acc = fma8<DT>(xv[u], wr[lane + 64 * u], acc);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc = acc + __shfl_xor(acc, off);
    if (lane == 0) s_logit[wave][e] = Half16<DT>::to_f32(Half16<DT>::round(acc));
  }
  // s_logit[wave] is written and read by this wave only: its LDS operations
  // complete in order
  router_softmax(s_logit[wave], gates, t, E, lane);
}

// Launch the router: the row kernel when W_g fits its LDS copy, H is one of
// its register shapes and there are enough tokens to fill the chip with
// workgroups of kWaves tokens; otherwise one workgroup per token.
template <int DT>
void launch_router_dt(const uint16_t* x, const uint16_t* wg, float* gates, int T, int H, int E,
                      hipStream_t stream) {
  const bool rows_ok = T >= kRowsMinTokens && E * (H / 8) <= kRowsLdsChunks;
  const dim3 rgrid((unsigned)((T + kWaves - 1) / kWaves));
  if (rows_ok && H == 2048) {
    hipLaunchKernelGGL((tm_router_rows_kernel<DT, 4>), rgrid, dim3(kThreads), 0, stream, x, wg,
                       gates, T, H, E);
  } else if (rows_ok && H == 4096) {
    hipLaunchKernelGGL((tm_router_rows_kernel<DT, 8>), rgrid, dim3(kThreads), 0, stream, x, wg,
                       gates, T, H, E);
  } else {
    hipLaunchKernelGGL(tm_router_kernel<DT>, dim3((unsigned)T), dim3(kThreads), 0, stream, x, wg,
                       gates, T, H, E);
  }
}

void launch_router(const uint16_t* x, const uint16_t* wg, float* gates, int T, int H, int E,
                   int dtype, hipStream_t stream) {
  if (dtype == TM_DTYPE_F16)
    launch_router_dt<TM_DTYPE_F16>(x, wg, gates, T, H, E, stream);
  else
    launch_router_dt<TM_DTYPE_BF16>(x, wg, gates, T, H, E, stream);
}

// ------------------------------------------------------- few tokens --
// T <= 64 and E <= 8: one token per lane, no LDS and no barrier between the
// steps (tmb::bucket_wave).  The phases of tm_bucket_kernel are chains of LDS
// round trips behind barriers.  Router and bucketing, E = 8: T = 5 10.7 -> 9.6 us,
// T = 64 10.7 -> 10.3, T = 64 critical path 12.0 -> 11.7; with the 16-expert
// form E = 16 took 17.4 against 14.7 us, so more experts keep the phases.
constexpr int kWaveMaxTokens = 64;
constexpr int kWaveMaxExperts = 8;
constexpr int kWaveThreads = 256;

__global__ void __launch_bounds__(kWaveThreads) tm_bucket_wave_kernel(BucketArgs a) {
  constexpr int EM = kWaveMaxExperts;
  const int lane = threadIdx.x & 63;
  const bool tok = lane < a.T;
  const float a_ld = a.accept[tok ? lane : 0];
  float g[EM];
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    const bool ok = tok && e < a.E;
    const float v = a.gates[ok ? lane * a.E + e : 0];
    g[e] = ok ? v : 0.0f;
  }
  tmb::bucket_wave<kWaveThreads, EM>(a, g, a_ld);
}

// Up to kFusedLogits logits (one or two tokens and 8 experts: an autoregressive
// step): router, softmax and bucketing in one workgroup and one launch; each
// wave computes one logit at a time, so more tokens are faster on more
// workgroups.  T = 1 10.2 -> 8.1 us, T = 2 11.6 -> 10.6; T = 4 this way 11.2 us
// against 9.3 with two launches.
constexpr int kFusedLogits = 16;

template <int DT>
__global__ void __launch_bounds__(kThreads)
tm_route_fused_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg,
                      float* __restrict__ gates, int H, BucketArgs a) {
  constexpr int EM = kWaveMaxExperts;
  __shared__ float s_logit[kFusedLogits];
  __shared__ float s_gate[kFusedLogits];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int T = a.T, E = a.E;
  const bool tok = lane < T;
  const float a_ld = a.accept[tok ? lane : 0];  // requested before the logits
  for (int q = wave; q < T * E; q += kWaves) {
    const int t = q / E, e = q - t * E;
    const float l = router_logit<DT>(x + (size_t)t * H, wg + (size_t)e * H, H, lane);
    if (lane == 0) s_logit[q] = l;
  }
  tm_lds_barrier();
  for (int t = wave; t < T; t += kWaves) {
    const float ex = router_softmax(s_logit + t * E, gates, t, E, lane);
    if (lane < E) s_gate[t * E + lane] = ex;
  }
  tm_lds_barrier();
  float g[EM];
#pragma unroll
  for (int e = 0; e < EM; ++e) {
    const bool ok = tok && e < E;
    const float v = s_gate[ok ? lane * E + e : 0];
    g[e] = ok ? v : 0.0f;
  }
  tmb::bucket_wave<kThreads, EM>(a, g, a_ld);
}

__global__ void __launch_bounds__(kThreads) tm_bucket_kernel(BucketArgs args) {
  __shared__ __attribute__((aligned(16))) BucketShared sh;
  tmb::bucket_phases<kThreads, BucketShared>(args, sh);
}

// ------------------------------------------------------ many tokens --
// The same budget routing and bucketing spread over the chip, in launches whose
// boundaries are the only synchronisation:
//   demand  one workgroup per expert: the demand (and criticality) with the
//           floating-point order of tmb::bucket_phases;
//   top-2   one thread per token: keep set, masked top-2, gates.  With a budget
//           of every expert nothing is dropped whatever the demand, so the
//           demand's workgroups run in this launch;
//   place   per 512 tokens: every workgroup counts each expert's rows before its
//           tokens and in all from the expert ids (ballots over 64 tokens),
//           which is quicker than waiting for a scan of partial counts, and
//           writes its part of every layout.
// Criticalities go through the front of slot_to_row, which `place` overwrites.
// Each launch is bound by latency (loads, then ballots over the experts).
// Router and bucketing, E = 8, same box, budget 8 / budget 4 with the critical
// path, against one workgroup (above 4096 tokens through the output buffers):
// T = 517 17.6 -> 16.6 / 20.5 -> 21.4 us, T = 1000 21.9 -> 18.7 / 21.9 -> 22.0,
// T = 1500 27.4 -> 20.5 / 32.7 -> 25.3, T = 2048 31.7 -> 21.8 / 38.7 -> 26.7, T =
// 6011 113 -> 42 / 148 -> 49; E = 64 T = 1024 97 -> 64 / 125 -> 104, T = 2048 182 -> 89 /
// 235 -> 161; hence kSpreadMinTokens = 1024.  (Device times.  A stand-alone
// route_and_bucket of 8 experts at 1024 .. 1500 tokens is bound by the host, which
// pays 2.3 us per launch: 26.8 -> 28.5-29.8 us with a budget of 8.)
constexpr int kSpreadThreads = 512;
constexpr int kSpreadWaves = kSpreadThreads / 64;
constexpr int kDemandTile = 8192;  // products staged in LDS at a time

// max(crit, accept of the tokens among t0 .. t0 + n that need expert e): e is a
// token's unrestricted top-1, or its top-2 when accept >= tau.  With 8 experts
// the rows of four tokens are requested before the first is compared.
__device__ __forceinline__ float crit_of(const BucketArgs& a, int e, int t0, int n, float crit) {
  const int E = a.E;
  if (E == 8 && (reinterpret_cast<uintptr_t>(a.gates) & 15) == 0) {
    for (int i0 = threadIdx.x; i0 < n; i0 += 4 * kSpreadThreads) {
      float4 lo[4], hi[4];
      float av[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + min(i0 + u * kSpreadThreads, n - 1);
        const float4* g = reinterpret_cast<const float4*>(a.gates + (size_t)t * 8);
        lo[u] = g[0];
        hi[u] = g[1];
        av[u] = a.accept[t];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // past the end: the last token again, same maximum
        Top2 r{-1, -1, 0.0f, 0.0f};
        const float g[8] = {lo[u].x, lo[u].y, lo[u].z, lo[u].w,
                            hi[u].x, hi[u].y, hi[u].z, hi[u].w};
#pragma unroll
        for (int f = 0; f < 8; ++f) r.offer(g[f], f);
        if (r.i1 == e || (r.i2 == e && av[u] >= a.tau)) crit = fmaxf(crit, av[u]);
      }
    }
    return crit;
  }
  for (int i = threadIdx.x; i < n; i += kSpreadThreads) {
    const float av = a.accept[t0 + i];
    const float* g = a.gates + (size_t)(t0 + i) * E;
    Top2 r{-1, -1, 0.0f, 0.0f};
    for (int f = 0; f < E; ++f) r.offer(g[f], f);
    if (r.i1 == e || (r.i2 == e && av >= a.tau)) crit = fmaxf(crit, av);
  }
  return crit;
}

// demand[e] and crit[e]: lane l sums accept[t] gates[t, e] over t = l, l + 64, ..
// in order, then a halving tree.  All threads stage the products, the first
// wave adds them (maxima need no order).
__device__ __forceinline__ void demand_of(const BucketArgs& a, int e, float* __restrict__ crit_out,
                                          float* s_prod, float* s_crit) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int T = a.T, E = a.E;
  const bool critical = a.objective == TM_OBJECTIVE_CRITICAL_PATH;
  float acc = 0.0f, crit = -INFINITY;
  for (int t0 = 0; t0 < T; t0 += kDemandTile) {
    const int n = min(kDemandTile, T - t0);
#pragma unroll 8
    for (int i = tid; i < n; i += kSpreadThreads) {
      const float av = a.accept[t0 + i];
      s_prod[i] = av * a.gates[(size_t)(t0 + i) * E + e];
    }
    if (critical) crit = crit_of(a, e, t0, n, crit);
    __syncthreads();
    if (wave == 0) {
#pragma unroll 8
      for (int i = lane; i < n; i += 64) acc = acc + s_prod[i];
    }
    __syncthreads();
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    acc = acc + __shfl_xor(acc, off);
    crit = fmaxf(crit, __shfl_xor(crit, off));
  }
  if (lane == 0) s_crit[wave] = crit;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kSpreadWaves; ++w) crit = fmaxf(crit, s_crit[w]);
    a.demand_out[e] = acc;
    if (critical) crit_out[e] = crit;
  }
}

__global__ void __launch_bounds__(kSpreadThreads)
tm_bucket_demand_kernel(BucketArgs a, float* __restrict__ crit) {
  __shared__ float s_prod[kDemandTile];
  __shared__ float s_crit[kSpreadWaves];
  demand_of(a, blockIdx.x, crit, s_prod, s_crit);
}

// Workgroups [0, token_groups): one token per thread.  Further workgroups (a
// budget of every expert): the demand of expert blockIdx.x - token_groups.
__global__ void __launch_bounds__(kSpreadThreads)
tm_bucket_top2_kernel(BucketArgs a, float* __restrict__ crit, int token_groups) {
  __shared__ float s_prod[kDemandTile];
  __shared__ float s_crit[kSpreadWaves];
  const int E = a.E;
  if ((int)blockIdx.x >= token_groups) {
    demand_of(a, (int)blockIdx.x - token_groups, crit, s_prod, s_crit);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * kSpreadThreads + threadIdx.x;
  const bool tok = t < a.T;
  unsigned long long keep = E >= 64 ? ~0ull : (1ull << E) - 1ull;
  if (a.budget < E) {  // lane = expert, as in tmb::bucket_phases
    const bool critical = a.objective == TM_OBJECTIVE_CRITICAL_PATH;
    const float d = lane < E ? a.demand_out[lane] : 0.0f;
    const float c = (critical && lane < E) ? crit[lane] : 0.0f;
    int rank = 0;
    for (int f = 0; f < E; ++f) {
      const float df = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d), f));
      const float cf = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), f));
      bool before;
      if (critical && cf != c) {
        before = cf > c;
      } else if (df != d) {
        before = df > d;
      } else {
        before = f < lane;
      }
      rank += before ? 1 : 0;
    }
    keep = __ballot(lane < E && rank < a.budget);
  }
  if (!tok) return;
  const float* g = a.gates + (size_t)t * E;
  Top2 r{-1, -1, 0.0f, 0.0f};
  if ((E & 3) == 0 && (reinterpret_cast<uintptr_t>(a.gates) & 15) == 0) {
#pragma unroll 4
    for (int e = 0; e < E; e += 4) {
      const float4 v = *reinterpret_cast<const float4*>(g + e);
      r.offer(((keep >> e) & 1ull) ? v.x : 0.0f, e);
      r.offer(((keep >> (e + 1)) & 1ull) ? v.y : 0.0f, e + 1);
      r.offer(((keep >> (e + 2)) & 1ull) ? v.z : 0.0f, e + 2);
      r.offer(((keep >> (e + 3)) & 1ull) ? v.w : 0.0f, e + 3);
    }
  } else {
    for (int e = 0; e < E; ++e) r.offer(((keep >> e) & 1ull) ? g[e] : 0.0f, e);
  }
  const float s = r.g1 + r.g2;
  float tg1 = r.g1 / s;
  float tg2 = r.g2 / s;
  if (a.accept[t] < a.tau) { tg1 = 1.0f; tg2 = 0.0f; }
  a.topk_ids[2 * t] = r.i1;
  a.topk_ids[2 * t + 1] = r.i2;
  a.gates_flat[2 * t] = tg1;
  a.gates_flat[2 * t + 1] = tg2;
}

__global__ void __launch_bounds__(kSpreadThreads) tm_bucket_place_kernel(BucketArgs a) {
  __shared__ int s_before[kSpreadWaves][TM_MAX_EXPERTS];  // per wave: rows before this workgroup
  __shared__ int s_after[kSpreadWaves][TM_MAX_EXPERTS];   // per wave: its own and later rows
  __shared__ int s_own[kSpreadWaves][TM_MAX_EXPERTS];     // rows of this workgroup's waves
  __shared__ int s_count[TM_MAX_EXPERTS], s_off[TM_MAX_EXPERTS], s_bs[TM_MAX_EXPERTS],
      s_ts[TM_MAX_EXPERTS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int T = a.T, E = a.E;
  const int first = blockIdx.x * kSpreadThreads;
  // 1. rows per expert before `first` and from it on; lane e keeps expert e.
  //    The ids of four 64-token groups are requested before the first ballot.
  int nb = 0, na = 0;
  constexpr int kBatch = 4;
  for (int t0 = wave * 64; t0 < T; t0 += kBatch * kSpreadThreads) {
    int f1[kBatch], f2[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int t = t0 + u * kSpreadThreads + lane;
      f1[u] = t < T ? (int)a.topk_ids[2 * (size_t)t] : -1;
      f2[u] = t < T ? (int)a.topk_ids[2 * (size_t)t + 1] : -1;
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const bool early = t0 + u * kSpreadThreads < first;  // a group lies on one side of `first`
      for (int e = 0; e < E; ++e) {
        const int c = __popcll(__ballot(f1[u] == e || f2[u] == e));
        if (lane == e) {
          nb += early ? c : 0;
          na += early ? 0 : c;
        }
      }
    }
  }
  if (lane < E) {
    s_before[wave][lane] = nb;
    s_after[wave][lane] = na;
  }
  // 2. this thread's token: ranks within its wave, and the wave's counts
  const int t = first + tid;
  int f1 = -1, f2 = -1, r1 = 0, r2 = 0;
  if (t < T) {
    f1 = (int)a.topk_ids[2 * t];
    f2 = (int)a.topk_ids[2 * t + 1];
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int e = 0; e < E; ++e) {
    const unsigned long long m = __ballot(f1 == e || f2 == e);
    const int rank = __popcll(m & below);
    if (f1 == e) r1 = rank;
    if (f2 == e) r2 = rank;
    if (lane == e) s_own[wave][e] = __popcll(m);
  }
  __syncthreads();
  // 3. totals, offsets, block and tile starts (wave 0, lane = expert); s_own
  //    becomes the rows of the expert before each wave's tokens
  if (wave == 0) {
    int before = 0, total = 0;
    if (lane < E) {
      for (int w = 0; w < kSpreadWaves; ++w) before += s_before[w][lane];
      total = before;
      for (int w = 0; w < kSpreadWaves; ++w) total += s_after[w][lane];
      for (int w = 0; w < kSpreadWaves; ++w) {
        const int c = s_own[w][lane];
        s_own[w][lane] = before;
        before += c;
      }
    }
    int tot_off, tot_blk, tot_tiles;
    const int off = wave_exclusive_scan(total, lane, &tot_off);
    const int bs = wave_exclusive_scan((total + a.BM - 1) / a.BM, lane, &tot_blk);
    const int ts = wave_exclusive_scan((total + TM_GEMM_TILE_M - 1) / TM_GEMM_TILE_M, lane,
                                       &tot_tiles);
    if (lane < E) {
      s_count[lane] = total;
      s_off[lane] = off;
      s_bs[lane] = bs;
      s_ts[lane] = ts;
      if (blockIdx.x == 0) a.expert_offsets[lane] = off;
    }
    if (lane == 0 && blockIdx.x == 0) a.expert_offsets[E] = tot_off;
  }
  __syncthreads();
  const int padded_rows = a.max_blocks * a.BM;
  // 4. this thread's two slots
  if (t < T) {
    const int k1 = s_own[wave][f1] + r1, k2 = s_own[wave][f2] + r2;
    const int p1 = s_off[f1] + k1, p2 = s_off[f2] + k2;
    const int w1 = s_bs[f1] * a.BM + k1, w2 = s_bs[f2] * a.BM + k2;
    a.slot_pos[2 * t] = p1;
    a.slot_pos[2 * t + 1] = p2;
    a.sorted_slots[p1] = 2 * t;
    a.sorted_slots[p2] = 2 * t + 1;
    a.slot_to_row[2 * t] = w1;
    a.slot_to_row[2 * t + 1] = w2;
    if (w1 < padded_rows) a.padded_slots[w1] = 2 * t;
    if (w2 < padded_rows) a.padded_slots[w2] = 2 * t + 1;
  }
  // 5. the entries without a slot, spread over all workgroups (those past the
  //    tokens have nothing else to write): padded rows past an expert's count
  //    or in unused blocks, block owners, the tile list.  Lane e holds expert
  //    e's starts; readlane makes them scalars.
  const int v_cnt = lane < E ? s_count[lane] : 0, v_bs = lane < E ? s_bs[lane] : 0;
  const int v_off = lane < E ? s_off[lane] : 0, v_ts = lane < E ? s_ts[lane] : 0;
  const int bm_shift = a.BM == 32 ? 5 : 4;
  const int g0 = blockIdx.x * kSpreadThreads + tid, step = gridDim.x * kSpreadThreads;
  for (int i0 = g0 - lane; i0 < padded_rows; i0 += step) {  // whole waves: padded_rows % 16 == 0
    const int i = i0 + lane, b = i >> bm_shift;
    int owner = -1;
    bool pad = true;
    for (int e = 0; e < E; ++e) {
      const int cnt = __builtin_amdgcn_readlane(v_cnt, e), bs = __builtin_amdgcn_readlane(v_bs, e);
      const int k = i - (bs << bm_shift);
      if (b >= bs && b < bs + ((cnt + a.BM - 1) >> bm_shift)) owner = e;
      if (k >= 0 && k < cnt) pad = false;
    }
    if (i < padded_rows) {
      if (pad) a.padded_slots[i] = -1;
      if (i == b << bm_shift) a.block_expert_ids[b] = owner;
    }
  }
  for (int j0 = g0 - lane; j0 < a.max_tiles; j0 += step) {
    const int j = j0 + lane;
    int te = -1, r0 = 0, rows = 0;
    for (int e = 0; e < E; ++e) {
      const int cnt = __builtin_amdgcn_readlane(v_cnt, e);
      const int k = j - __builtin_amdgcn_readlane(v_ts, e);
      if (k >= 0 && k * TM_GEMM_TILE_M < cnt) {
        te = e;
        r0 = __builtin_amdgcn_readlane(v_off, e) + k * TM_GEMM_TILE_M;
        rows = min(TM_GEMM_TILE_M, cnt - k * TM_GEMM_TILE_M);
      }
    }
    if (j >= a.max_tiles) continue;
    a.tiles[4 * j] = te;
    a.tiles[4 * j + 1] = r0;
    a.tiles[4 * j + 2] = rows;
    a.tiles[4 * j + 3] = 0;
  }
}

int check_bucket_args(int64_t T, int64_t E, int64_t budget, int objective, int64_t block_m,
                      int64_t max_blocks, int64_t max_tiles) {
  if (T < 1 || T > TM_MAX_TOKENS || E < 2 || E > TM_MAX_EXPERTS) return TM_ERR_SHAPE;
  if (budget < 2 || budget > E) return TM_ERR_ARG;
  if (objective != TM_OBJECTIVE_MASS && objective != TM_OBJECTIVE_CRITICAL_PATH) return TM_ERR_ARG;
  if (block_m != 16 && block_m != 32) return TM_ERR_ARG;
  if (max_blocks < 1 || max_tiles < 1) return TM_ERR_SHAPE;
  if (T <= kFewTokens ? max_blocks * block_m > kMaxPaddedRows
                         : max_blocks * block_m > (int64_t)1 << 30)
    return TM_ERR_SHAPE;
  return TM_OK;
}

// The bucketing launches for T tokens: one token per lane up to 64 tokens and
// 8 experts, one workgroup with every intermediate in LDS, from
// kSpreadMinTokens spread over the chip.
void launch_bucket(const BucketArgs& a, hipStream_t stream) {
  if (a.T <= kWaveMaxTokens && a.E <= kWaveMaxExperts) {
    hipLaunchKernelGGL(tm_bucket_wave_kernel, dim3(1), dim3(kWaveThreads), 0, stream, a);
  } else if (a.T < kSpreadMinTokens) {
    hipLaunchKernelGGL(tm_bucket_kernel, dim3(1), dim3(kThreads), 0, stream, a);
  } else {
    const int groups = (a.T + kSpreadThreads - 1) / kSpreadThreads;
    float* crit = reinterpret_cast<float*>(a.slot_to_row);
    const bool keep_all = a.budget >= a.E;
    if (!keep_all)
      hipLaunchKernelGGL(tm_bucket_demand_kernel, dim3((unsigned)a.E), dim3(kSpreadThreads), 0,
                         stream, a, crit);
    hipLaunchKernelGGL(tm_bucket_top2_kernel, dim3((unsigned)(groups + (keep_all ? a.E : 0))),
                       dim3(kSpreadThreads), 0, stream, a, crit, groups);
    // workgroups past the tokens only fill padded rows: at most one row per thread,
    // up to a workgroup per CU
    const int fill = (a.max_blocks * a.BM + kSpreadThreads - 1) / kSpreadThreads;
    hipLaunchKernelGGL(tm_bucket_place_kernel,
                       dim3((unsigned)std::max(groups, std::min(fill, 256))),
                       dim3(kSpreadThreads), 0, stream, a);
  }
}

// Router and bucketing of one layer.
int launch_route(const uint16_t* x, const uint16_t* wg, float* gates, int H, int dtype,
                 const BucketArgs& a, hipStream_t stream) {
  if (a.T * a.E <= kFusedLogits && a.E <= kWaveMaxExperts) {
    hipLaunchKernelGGL(dtype == TM_DTYPE_F16 ? tm_route_fused_kernel<TM_DTYPE_F16>
                                             : tm_route_fused_kernel<TM_DTYPE_BF16>,
                       dim3(1), dim3(kThreads), 0, stream, x, wg, gates, H, a);
    TM_HIP_CHECK_LAUNCH();
    return TM_OK;
  }
  launch_router(x, wg, gates, a.T, H, a.E, dtype, stream);
  TM_HIP_CHECK_LAUNCH();
  launch_bucket(a, stream);
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}

BucketArgs make_args(const float* gates, const float* accept, int64_t T, int64_t E,
                     int64_t budget, float tau, int objective, int64_t block_m,
                     int64_t max_blocks, int64_t max_tiles, int64_t* topk_ids,
                     float* gates_flat, int64_t* padded_slots, int64_t* block_expert_ids,
                     int64_t* slot_to_row, float* demand, int32_t* expert_offsets,
                     int32_t* sorted_slots, int32_t* slot_pos, int32_t* tiles) {
  BucketArgs a;
  a.gates = gates;
  a.accept = accept;
  a.T = (int)T;
  a.E = (int)E;
  a.budget = (int)budget;
  a.objective = objective;
  a.BM = (int)block_m;
  a.max_blocks = (int)max_blocks;
  a.max_tiles = (int)max_tiles;
  a.tau = tau;
  a.topk_ids = topk_ids;
  a.gates_flat = gates_flat;
  a.padded_slots = padded_slots;
  a.block_expert_ids = block_expert_ids;
  a.slot_to_row = slot_to_row;
  a.demand_out = demand;
  a.expert_offsets = expert_offsets;
  a.sorted_slots = sorted_slots;
  a.slot_pos = slot_pos;
  a.tiles = tiles;
  return a;
}

}  // namespace

extern "C" int tm_op1_router_gates(const void* x, const void* wg, int64_t T, int64_t H,
                                   int64_t E, float* gates, int dtype, void* stream) {
  if (T < 1 || T > TM_MAX_TOKENS || E < 2 || E > TM_MAX_EXPERTS || H < 8 || (H % 8) != 0)
    return TM_ERR_SHAPE;
  if (dtype != TM_DTYPE_BF16 && dtype != TM_DTYPE_F16) return TM_ERR_ARG;
  if (((uintptr_t)x % 16) != 0 || ((uintptr_t)wg % 16) != 0) return TM_ERR_ALIGN;
  launch_router((const uint16_t*)x, (const uint16_t*)wg, gates, (int)T, (int)H, (int)E, dtype,
                (hipStream_t)stream);
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}

extern "C" int tm_op1_route_bucket(const float* gates, const float* accept, int64_t T,
                                   int64_t E, int64_t budget, float tau, int objective,
                                   int64_t block_m, int64_t max_blocks, int64_t max_tiles,
                                   int64_t* topk_ids, float* gates_flat,
                                   int64_t* padded_slots, int64_t* block_expert_ids,
                                   int64_t* slot_to_row, float* demand,
                                   int32_t* expert_offsets, int32_t* sorted_slots,
                                   int32_t* slot_pos, int32_t* tiles, void* stream) {
  const int rc = check_bucket_args(T, E, budget, objective, block_m, max_blocks, max_tiles);
  if (rc != TM_OK) return rc;
  const BucketArgs a = make_args(gates, accept, T, E, budget, tau, objective, block_m, max_blocks,
                                 max_tiles, topk_ids, gates_flat, padded_slots,
                                 block_expert_ids, slot_to_row, demand, expert_offsets,
                                 sorted_slots, slot_pos, tiles);
  launch_bucket(a, (hipStream_t)stream);
  TM_HIP_CHECK_LAUNCH();
  return TM_OK;
}

extern "C" int tm_op1_route(const void* x, const void* wg, const float* accept, int64_t T,
                            int64_t H, int64_t E, int64_t budget, float tau, int objective,
                            int64_t block_m, int64_t max_blocks, int64_t max_tiles,
                            float* gates, int64_t* topk_ids, float* gates_flat,
                            int64_t* padded_slots, int64_t* block_expert_ids,
                            int64_t* slot_to_row, float* demand, int32_t* expert_offsets,
                            int32_t* sorted_slots, int32_t* slot_pos, int32_t* tiles,
                            int dtype, void* stream) {
  const int rc = check_bucket_args(T, E, budget, objective, block_m, max_blocks, max_tiles);
  if (rc != TM_OK) return rc;
  if (H < 8 || (H % 8) != 0) return TM_ERR_SHAPE;
  if (dtype != TM_DTYPE_BF16 && dtype != TM_DTYPE_F16) return TM_ERR_ARG;
  if (((uintptr_t)x % 16) != 0 || ((uintptr_t)wg % 16) != 0) return TM_ERR_ALIGN;
  const BucketArgs a = make_args(gates, accept, T, E, budget, tau, objective, block_m, max_blocks,
                                 max_tiles, topk_ids, gates_flat, padded_slots,
                                 block_expert_ids, slot_to_row, demand, expert_offsets,
                                 sorted_slots, slot_pos, tiles);
  return launch_route((const uint16_t*)x, (const uint16_t*)wg, gates, (int)H, dtype, a,
                      (hipStream_t)stream);
}
