// The router's linear layer and load-balancing statistics around the gate:
// the statistics of MoELayerStats from the logits in one pass, their
// backward, and the linear layer's backward (dx and dW from the gradients of
// the gate path and of the statistics path together).
//
// All of it is small next to the experts, so launches and passes over the
// tokens are what it costs: on MI355X, 16,384 tokens x 512, 16 experts, the
// library's two fp32 dW products alone took 149 us (its tiles hold 16 of
// their output columns) and dx, casts, sums and the second linear pass
// another 80; the linear backward here takes 35 us for the gate path (dx and
// dW) and 20 for the statistics path (dW), and each one's reduce 5. The
// statistics were ten short launches (softmax, mean, sum, divide, ...): a
// four-token forward, bound by the host, went from 194 to 118 us.
#include <algorithm>

#include "common.hpp"

namespace nt {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

// ---------------------------------------------------------------- statistics

// A row's softmax by S = 2^lgS lanes (S >= E, or 64): lane s holds experts
// s, s + 64, ... Returns the lane's probabilities in p (0 past E).
template <int V>
__device__ __forceinline__ void row_softmax(const float* __restrict__ row, int E, int S, int s,
                                            bool live, float (&p)[V]) {
  float m = -INFINITY;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int e = v * kWave + s;
    p[v] = live && e < E ? row[e] : -INFINITY;
    m = fmaxf(m, p[v]);
  }
  for (int o = S / 2; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
  float sum = 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int e = v * kWave + s;
    // a NaN logit stays NaN: fmaxf skipped it, the subtraction does not
    p[v] = live && e < E ? expf(p[v] - m) : 0.f;
    sum += p[v];
  }
  for (int o = S / 2; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, kWave);
#pragma unroll
  for (int v = 0; v < V; ++v) p[v] = live && v * kWave + s < E ? p[v] / sum : 0.f;
}

struct StatsArgs {
  const float* logits;    // [T, E]
  const int32_t* counts;  // [E]
  int64_t T;
  int32_t E;
  float coef;
  int64_t* total;
  float* frac;  // [E]
  float* mean;  // [E]
  float* aux;
  float* partial;  // [blocks][E] when there is more than one block
};

// total, frac, mean and aux from the column sums of the probabilities in
// s_sum[E] (one workgroup).
__device__ void finish_stats(const StatsArgs& a, const float* s_sum, int64_t* s_tot,
                             float* s_part) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  int64_t tot = 0;
  for (int e = threadIdx.x; e < a.E; e += kThreads) tot += a.counts[e];
  for (int o = kWave / 2; o >= 1; o >>= 1) tot += __shfl_xor(tot, o, kWave);
  if (lane == 0) s_tot[wave] = tot;
  __syncthreads();
  tot = 0;
  for (int w = 0; w < kWaves; ++w) tot += s_tot[w];
  float part = 0.f;
  for (int e = threadIdx.x; e < a.E; e += kThreads) {
    const float f = (float)a.counts[e] / (float)tot;
    const float m = s_sum[e] / (float)a.T;
    a.frac[e] = f;
    a.mean[e] = m;
    part += f * m;
  }
  part = wave_sum(part);
  if (lane == 0) s_part[wave] = part;
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = 0.f;
    for (int w = 0; w < kWaves; ++w) sum += s_part[w];
    *a.total = tot;
    *a.aux = a.coef * sum;
  }
}

// Column sums of the row softmaxes; each workgroup takes every gridDim-th
// group of rows and one workgroup alone finishes the statistics.
template <int V>
__global__ void __launch_bounds__(kThreads)
router_stats_kernel(StatsArgs a, int lgS) {
  __shared__ float s_wave[kWaves][NT_MAX_EXPERTS];
  __shared__ int64_t s_tot[kWaves];
  __shared__ float s_part[kWaves];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int S = 1 << lgS, s = lane & (S - 1), rpw = kWave >> lgS;
  float acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.f;
  const int64_t step = (int64_t)gridDim.x * kWaves * rpw;
  for (int64_t r0 = ((int64_t)blockIdx.x * kWaves + wave) * rpw; r0 < a.T; r0 += step) {
    const int64_t r = r0 + (lane >> lgS);
    float p[V];
    row_softmax<V>(a.logits + (r < a.T ? r : 0) * a.E, a.E, S, s, r < a.T, p);
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] += p[v];
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    for (int o = S; o < kWave; o <<= 1) acc[v] += __shfl_xor(acc[v], o, kWave);
    const int e = v * kWave + s;
    if (lane < S && e < a.E) s_wave[wave][e] = acc[v];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < a.E; e += kThreads) {
    float sum = 0.f;
    for (int w = 0; w < kWaves; ++w) sum += s_wave[w][e];
    if (gridDim.x == 1) s_wave[0][e] = sum;
    else a.partial[(int64_t)blockIdx.x * a.E + e] = sum;
  }
  if (gridDim.x > 1) return;
  __syncthreads();
  finish_stats(a, s_wave[0], s_tot, s_part);
}

__global__ void __launch_bounds__(kThreads)
router_stats_finish_kernel(StatsArgs a, int blocks) {
  __shared__ float s_grp[kThreads];
  __shared__ float s_sum[NT_MAX_EXPERTS];
  __shared__ int64_t s_tot[kWaves];
  __shared__ float s_part[kWaves];
  // 256 / per groups of threads sum every (256 / per)-th block's columns
  int per = 1;
  while (per < a.E && per < kThreads) per <<= 1;
  const int c = threadIdx.x & (per - 1), grp = threadIdx.x / per, ngrp = kThreads / per;
  for (int e0 = 0; e0 < a.E; e0 += per) {
    const int e = e0 + c;
    float sum = 0.f;
    if (e < a.E) {
#pragma unroll 8
      for (int b = grp; b < blocks; b += ngrp) sum += a.partial[(int64_t)b * a.E + e];
    }
    s_grp[threadIdx.x] = sum;
    __syncthreads();
    if (grp == 0 && e < a.E) {
      float t = 0.f;
      for (int g = 0; g < ngrp; ++g) t += s_grp[g * per + c];
      s_sum[e] = t;
    }
    __syncthreads();
  }
  finish_stats(a, s_sum, s_tot, s_part);
}

// dlogits = p (v - sum p v), v = (daux coef frac + dmean) / T, p the row's
// softmax (again).
template <int V>
__global__ void __launch_bounds__(kThreads)
router_stats_backward_kernel(const float* __restrict__ logits, const float* __restrict__ frac,
                             const float* __restrict__ daux, const float* __restrict__ dmean,
                             int64_t T, int32_t E, float coef, int lgS,
                             float* __restrict__ dlogits) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int S = 1 << lgS, s = lane & (S - 1), rpw = kWave >> lgS;
  float g[V];
  const float da = daux != nullptr ? *daux * coef : 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int e = v * kWave + s;
    g[v] = e < E ? (da * frac[e] + (dmean != nullptr ? dmean[e] : 0.f)) / (float)T : 0.f;
  }
  const int64_t step = (int64_t)gridDim.x * kWaves * rpw;
  for (int64_t r0 = ((int64_t)blockIdx.x * kWaves + wave) * rpw; r0 < T; r0 += step) {
    const int64_t r = r0 + (lane >> lgS);
    float p[V], dot = 0.f;
    row_softmax<V>(logits + (r < T ? r : 0) * E, E, S, s, r < T, p);
#pragma unroll
    for (int v = 0; v < V; ++v) dot += p[v] * g[v];
    for (int o = S / 2; o >= 1; o >>= 1) dot += __shfl_xor(dot, o, kWave);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int e = v * kWave + s;
      if (r < T && e < E) dlogits[r * E + e] = p[v] * (g[v] - dot);
    }
  }
}

// ------------------------------------------------------------ linear backward

constexpr int kMaxLinearExperts = 32;
constexpr int kBatch = 8;
constexpr int kTok = 64;  // tokens whose gradients a workgroup holds in LDS at a time

// dx[t,:] = dl[t,:] W and partial sums of dW = (dl + da)^T x over this
// workgroup's tokens. A thread owns VEC columns of W (E x VEC registers) and
// of dW; cg column threads side by side, the 256 / cg groups of them take
// every (256 / cg)-th token. x (T) is read once, dx (TD) written once.
template <typename T, typename TD, int EM, int VEC>
__global__ void __launch_bounds__(kThreads)
router_linear_backward_kernel(const typename elem<T>::storage* __restrict__ x,
                              const float* __restrict__ W, const float* __restrict__ dl,
                              const float* __restrict__ da, int64_t T_, int32_t E, int64_t d,
                              int32_t cg, int32_t groups, typename elem<TD>::storage* __restrict__ dx,
                              float* __restrict__ partial) {
  typedef typename elem<T>::storage S;
  typedef typename elem<TD>::storage SD;
  struct alignas(sizeof(S) * VEC) Pack {
    S v[VEC];
  };
  struct alignas(sizeof(SD) * VEC) PackD {
    SD v[VEC];
  };
  __shared__ float s_gx[kTok][EM], s_gw[kTok][EM];
  const int tid = threadIdx.x;
  const int64_t c0 = ((int64_t)blockIdx.y * cg + tid % cg) * VEC;
  const int sub = tid / cg, nsub = kThreads / cg;
  const bool on = c0 < d;
  float w[EM][VEC], acc[EM][VEC];
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      w[e][v] = on && e < E ? W[(int64_t)e * d + c0 + v] : 0.f;
      acc[e][v] = 0.f;
    }
  for (int g = 0; g < groups; ++g) {
    const int64_t t0 = ((int64_t)blockIdx.x * groups + g) * kTok;
    if (t0 >= T_) break;
    const int nt = (int)(T_ - t0 < kTok ? T_ - t0 : kTok);
    __syncthreads();
    for (int i = tid; i < nt * EM; i += kThreads) {
      const int t = i / EM, e = i % EM;
      const float a = dl != nullptr && e < E ? dl[(t0 + t) * E + e] : 0.f;
      const float b = da != nullptr && e < E ? da[(t0 + t) * E + e] : 0.f;
      s_gx[t][e] = a;
      s_gw[t][e] = a + b;
    }
    __syncthreads();
    if (!on) continue;
    // kBatch tokens' loads are issued before the first is used (one wave per
    // SIMD runs here at 16,384 tokens x 512; one token at a time 52 us).
    for (int tb = sub; tb < nt; tb += kBatch * nsub) {
      Pack xp[kBatch];
      if (partial != nullptr) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
          const int t = tb + i * nsub < nt ? tb + i * nsub : tb;
          xp[i] = *reinterpret_cast<const Pack*>(x + (t0 + t) * d + c0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int t = tb + i * nsub;
        if (t >= nt) break;
        if (partial != nullptr) {
#pragma unroll
          for (int v = 0; v < VEC; ++v) {
            const float xv = elem<T>::load(xp[i].v[v]);
#pragma unroll
            for (int e = 0; e < EM; ++e) acc[e][v] = fmaf(s_gw[t][e], xv, acc[e][v]);
          }
        }
        if (dx != nullptr) {
          PackD r;
#pragma unroll
          for (int v = 0; v < VEC; ++v) {
            float z = 0.f;
#pragma unroll
            for (int e = 0; e < EM; ++e) z = fmaf(s_gx[t][e], w[e][v], z);
            r.v[v] = elem<TD>::store(z);
          }
          *reinterpret_cast<PackD*>(dx + (t0 + t) * d + c0) = r;
        }
      }
    }
  }
  if (partial == nullptr || !on) return;
  float* out = partial + ((int64_t)blockIdx.x * nsub + sub) * E * d;
#pragma unroll
  for (int e = 0; e < EM; ++e)
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (e < E) out[(int64_t)e * d + c0 + v] = acc[e][v];
}

// dW = the sum of the partials: 64 elements per workgroup, its four waves
// take every fourth partial, in a fixed order.
__global__ void __launch_bounds__(kThreads)
router_linear_reduce_kernel(const float* __restrict__ partial, int64_t n, int32_t parts,
                            float* __restrict__ dW) {
  __shared__ float s_sum[kWaves][kWave];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t i = (int64_t)blockIdx.x * kWave + lane;
  float sum = 0.f;
  if (i < n) {
#pragma unroll 16
    for (int p = wave; p < parts; p += kWaves) sum += partial[(int64_t)p * n + i];
  }
  s_sum[wave][lane] = sum;
  __syncthreads();
  if (wave == 0 && i < n) dW[i] = (s_sum[0][lane] + s_sum[1][lane]) + (s_sum[2][lane] + s_sum[3][lane]);
}

struct LinearPlan {
  int vec, cg, nsub, groups;
  int64_t blocks, cols;
};
// Up to 512 workgroups along the tokens: enough to fill the chip, and a bound
// on their partial sums. A workgroup of 64 tokens writes nsub E d floats, so
// up to 32,768 tokens the partials are nsub E / 64 of float32 x's bytes (a
// quarter at 16,384 x 512 and 16 experts, all of them at 128 columns, where
// nsub is 4), less above. They are written and read once more; at 32,768 x
// 8,192 and 32 experts they take 512 MiB of workspace.
LinearPlan linear_plan(int64_t T, int64_t d, int vec) {
  LinearPlan p;
  p.vec = vec;
  p.cg = 1;
  while (p.cg < kThreads && (int64_t)p.cg * vec < d) p.cg <<= 1;
  p.nsub = kThreads / p.cg;
  const int64_t toks = ceil_div(std::max<int64_t>(T, 1), kTok);
  p.groups = (int)ceil_div(toks, 512);
  p.blocks = ceil_div(toks, p.groups);
  p.cols = ceil_div(std::max<int64_t>(d, 1), (int64_t)p.cg * vec);
  return p;
}

template <typename T, typename TD>
int run_linear_backward(const void* x, const float* W, const float* dl, const float* da, int64_t T_,
                        int32_t E, int64_t d, void* dx, float* dW, float* ws, hipStream_t s) {
  typedef typename elem<T>::storage S;
  typedef typename elem<TD>::storage SD;
  const bool aligned = reinterpret_cast<uintptr_t>(x) % (2 * sizeof(S)) == 0 &&
                       reinterpret_cast<uintptr_t>(dx) % (2 * sizeof(SD)) == 0;
  const int vec = d % 2 == 0 && aligned ? 2 : 1;
  const LinearPlan p = linear_plan(T_, d, vec);
  if (p.cols > 65535) return NT_ERR_TOO_LARGE;
  const dim3 grid((unsigned)p.blocks, (unsigned)p.cols);
  float* part = dW != nullptr ? ws : nullptr;
#define NT_RLB(EM, VEC)                                                                           \
  hipLaunchKernelGGL((router_linear_backward_kernel<T, TD, EM, VEC>), grid, dim3(kThreads), 0, s,     \
                     static_cast<const S*>(x), W, dl, da, T_, E, d, p.cg, p.groups,               \
                     static_cast<SD*>(dx), part)
#define NT_RLB_V(EM) \
  do {               \
    if (vec == 2) NT_RLB(EM, 2); \
    else NT_RLB(EM, 1);          \
  } while (0)
  if (E <= 8) NT_RLB_V(8);
  else if (E <= 16) NT_RLB_V(16);
  else NT_RLB_V(32);
#undef NT_RLB_V
#undef NT_RLB
  if (dW != nullptr)
    hipLaunchKernelGGL(router_linear_reduce_kernel, dim3((unsigned)ceil_div((int64_t)E * d, kWave)),
                       dim3(kThreads), 0, s, part, (int64_t)E * d, (int32_t)(p.blocks * p.nsub), dW);
  return launch_status();
}

int stats_lg(int32_t E) {
  int lg = 0;
  while (lg < 6 && (1 << lg) < E) ++lg;
  return lg;
}
// Workgroups over the rows: about eight rounds of rows each, at most 256.
int64_t stats_blocks(int64_t T, int32_t E) {
  const int64_t per_round = (int64_t)kWaves * (kWave >> stats_lg(E));
  return std::min<int64_t>(std::max<int64_t>(ceil_div(T, 8 * per_round), 1), 256);
}

template <typename F>
void by_experts(int32_t E, F&& f) {
  const int v = (int)ceil_div(E, kWave);
  if (v <= 1) f(std::integral_constant<int, 1>());
  else if (v <= 2) f(std::integral_constant<int, 2>());
  else if (v <= 4) f(std::integral_constant<int, 4>());
  else f(std::integral_constant<int, 16>());
}

}  // namespace
}  // namespace nt

using namespace nt;

extern "C" {

size_t nt_router_stats_workspace_bytes(int64_t T, int32_t E) {
  if (T < 0 || E < 1 || E > NT_MAX_EXPERTS) return 0;
  const int64_t b = stats_blocks(T, E);
  return b > 1 ? (size_t)(b * E * 4) : 0;
}

int nt_router_stats(const float* logits, const int32_t* counts, int64_t T, int32_t E, float coef,
                    int64_t* total, float* frac, float* mean, float* aux, void* ws, size_t ws_bytes,
                    hipStream_t stream) {
  if (T < 1 || E < 1) return NT_ERR_INVALID_ARG;
  if (E > NT_MAX_EXPERTS) return NT_ERR_TOO_MANY_EXPERTS;
  if (logits == nullptr || counts == nullptr || total == nullptr || frac == nullptr ||
      mean == nullptr || aux == nullptr)
    return NT_ERR_INVALID_ARG;
  const size_t need = nt_router_stats_workspace_bytes(T, E);
  if (need > 0 && (ws == nullptr || ws_bytes < need)) return NT_ERR_WORKSPACE;
  const int blocks = (int)stats_blocks(T, E);
  const StatsArgs a{logits, counts, T, E, coef, total, frac, mean, aux, static_cast<float*>(ws)};
  by_experts(E, [&](auto v) {
    hipLaunchKernelGGL((router_stats_kernel<decltype(v)::value>), dim3(blocks), dim3(kThreads), 0,
                       stream, a, stats_lg(E));
  });
  if (blocks > 1)
    hipLaunchKernelGGL(router_stats_finish_kernel, dim3(1), dim3(kThreads), 0, stream, a, blocks);
  return launch_status();
}

int nt_router_stats_backward(const float* logits, const float* frac, const float* daux,
                             const float* dmean, int64_t T, int32_t E, float coef, float* dlogits,
                             hipStream_t stream) {
  if (T < 1 || E < 1) return NT_ERR_INVALID_ARG;
  if (E > NT_MAX_EXPERTS) return NT_ERR_TOO_MANY_EXPERTS;
  if (logits == nullptr || frac == nullptr || dlogits == nullptr) return NT_ERR_INVALID_ARG;
  const int lg = stats_lg(E);
  const int64_t per_round = (int64_t)kWaves * (kWave >> lg);
  const dim3 grid((unsigned)std::min<int64_t>(ceil_div(T, per_round), 2048));
  by_experts(E, [&](auto v) {
    hipLaunchKernelGGL((router_stats_backward_kernel<decltype(v)::value>), grid, dim3(kThreads), 0,
                       stream, logits, frac, daux, dmean, T, E, coef, lg, dlogits);
  });
  return launch_status();
}

size_t nt_router_linear_backward_workspace_bytes(int64_t T, int32_t E, int64_t d) {
  if (T < 0 || E < 1 || E > kMaxLinearExperts || d < 1) return 0;
  size_t need = 0;
  for (int vec = 1; vec <= 2; ++vec) {
    const LinearPlan p = linear_plan(T, d, vec);
    need = std::max(need, (size_t)(p.blocks * p.nsub * E * d * 4));
  }
  return need;
}

int nt_router_linear_backward_mixed(int x_dtype, int dx_dtype, const void* x, const float* W,
                                    const float* dl, const float* da, int64_t T, int32_t E,
                                    int64_t d, void* dx, float* dW, void* ws, size_t ws_bytes,
                                    hipStream_t stream) {
  if (T < 1 || E < 1 || d < 1) return NT_ERR_INVALID_ARG;
  if (E > kMaxLinearExperts) return NT_ERR_TOO_MANY_EXPERTS;
  if (x == nullptr || W == nullptr) return NT_ERR_INVALID_ARG;
  if (dW != nullptr &&
      (ws == nullptr || ws_bytes < nt_router_linear_backward_workspace_bytes(T, E, d)))
    return NT_ERR_WORKSPACE;
  float* wp = static_cast<float*>(ws);
  auto run = [&](auto tx, auto td) {
    return run_linear_backward<decltype(tx), decltype(td)>(x, W, dl, da, T, E, d, dx, dW, wp,
                                                           stream);
  };
  if (x_dtype == NT_F32) {
    switch (dx_dtype) {
      case NT_F32: return run(float(), float());
      case NT_F16: return run(float(), f16());
      case NT_BF16: return run(float(), bf16());
      default: return NT_ERR_DTYPE;
    }
  }
  if (x_dtype != dx_dtype) return NT_ERR_DTYPE;
  switch (x_dtype) {
    case NT_F16: return run(f16(), f16());
    case NT_BF16: return run(bf16(), bf16());
    default: return NT_ERR_DTYPE;
  }
}

int nt_router_linear_backward(int dtype, const void* x, const float* W, const float* dl,
                              const float* da, int64_t T, int32_t E, int64_t d, void* dx, float* dW,
                              void* ws, size_t ws_bytes, hipStream_t stream) {
  return nt_router_linear_backward_mixed(dtype, dtype, x, W, dl, da, T, E, d, dx, dW, ws, ws_bytes,
                                         stream);
}

}  // extern "C"
