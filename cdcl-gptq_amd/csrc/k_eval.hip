// Evaluation kernels of the synthetic benchmark harness: round-to-nearest quantization
// (engine::rtn_layer), the held-out output error (bench::rel_err) reduction, and the element-wise
// steps of the benchmark's input generator; and the checkpoint-tensor decode and non-finite scan of
// the model pipeline.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "cdclq.h"
#include <algorithm>

#include "cdclq_dev.h"
#include "kernels.h"

namespace cdclq {
namespace {

__device__ __forceinline__ int readlane_int(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// engine::rtn_layer (src/engine.rs:822-838): one wave per (row, group). The group's grid is
// quant::find_params (src/quant.rs:40-83) on the group's values -- min/max from 0, the all-zero
// fallback, the optional 24-step clip search with each lane running one candidate's error sum in
// column order, first minimum wins -- then every value is rounded onto that grid.
__global__ __launch_bounds__(256) void k_rtn(long d_out, int n, int g, int ng, int bits, int mse,
                                             const float* __restrict__ w, float* __restrict__ out) {
  const long wid = ((long)blockIdx.x * 256 + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if (wid >= d_out * ng) return;
  const long r = wid / ng;
  const int gi = (int)(wid - r * ng);
  const int j0 = gi * g, j1 = min(j0 + g, n);
  const float* src = w + r * n;
  const float maxq = (float)((1u << bits) - 1u);
  float lmin = INFINITY, lmax = -INFINITY;
  for (int j = j0 + lane; j < j1; j += 64) {
    lmin = rs_minf(lmin, src[j]);
    lmax = rs_maxf(lmax, src[j]);
  }
  float xmin = rs_minf(0.0f, wave_min(lmin));
  float xmax = rs_maxf(0.0f, wave_max(lmax));
  if (xmin == 0.0f && xmax == 0.0f) {
    xmin = -1.0f;
    xmax = 1.0f;
  }
  float sc, zr;
  grid_mk(xmin, xmax, maxq, &sc, &zr);
  if (mse) {
    const int cand = lane < 24 ? lane : 0;
    const float p = 1.0f - 0.02f * (float)cand;
    float cs, cz;
    grid_mk(p * xmin, p * xmax, maxq, &cs, &cz);
    float errs = 0.0f;
    for (int j = j0; j < j1; ++j) {  // wave-uniform: every lane reads the same value
      const float v = src[j];
      float qq;
      const float e = quant_dq(v, cs, cz, maxq, &qq) - v;
      errs = errs + e * e;
    }
    float be = (lane < 24 && errs == errs) ? errs : INFINITY;
    int bc = lane < 24 ? lane : (1 << 20);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float oe = __shfl_xor(be, o, 64);
      const int oc = __shfl_xor(bc, o, 64);
      if (oe < be || (oe == be && oc < bc)) {
        be = oe;
        bc = oc;
      }
    }
    bc = readlane_int(bc, 0);
    sc = readlane(cs, bc);
    zr = readlane(cz, bc);
  }
  float* dst = out + r * n;
  for (int j = j0 + lane; j < j1; j += 64) {
    float qq;
    dst[j] = quant_dq(src[j], sc, zr, maxq, &qq);
  }
}

// ActGen::sample's per-token step (src/bench.rs:71-78): x = (x + noise) * scale[j] * massive[t],
// with noise = 0.3 * normal drawn on the host in the reference's order.
__global__ __launch_bounds__(256) void k_act_scale(long tokens, int n, const float* __restrict__ noise,
                                                   const float* __restrict__ scale, const float* __restrict__ massive,
                                                   float* __restrict__ x) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= tokens * n) return;
  const long t = i / n;
  const int j = (int)(i - t * n);
  x[i] = (x[i] + noise[i]) * scale[j] * massive[t];
}

// Per-channel RMS of bench::run's asymmetric experiment (src/bench.rs:276-284): f32 sums in token
// order, one thread per channel.
__global__ __launch_bounds__(256) void k_channel_rms(long tokens, int n, const float* __restrict__ x,
                                                     float* __restrict__ rms) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= n) return;
  float s = 0.0f;
  for (long t = 0; t < tokens; ++t) {
    const float v = x[t * n + j];
    s += v * v;
  }
  rms[j] = sqrtf(s / (float)tokens);
}

// xt = x + asym_noise * rms[j] * normal (src/bench.rs:286-292), normals drawn on the host in order.
__global__ __launch_bounds__(256) void k_add_noise(long tokens, int n, float a, const float* __restrict__ rms,
                                                   const float* __restrict__ nrm, const float* __restrict__ x,
                                                   float* __restrict__ xt) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= tokens * n) return;
  const int j = (int)(i % n);
  xt[i] = x[i] + a * rms[j] * nrm[i];
}

unsigned blocks_for(long count) { return (unsigned)((count + 255) / 256); }

}  // namespace

hipError_t rtn_rows(hipStream_t st, long d_out, int n, int g, int bits, int mse, const float* w, float* out) {
  const int ng = (n + g - 1) / g;
  const long waves = d_out * ng;
  if (waves <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rtn, dim3(blocks_for(waves * 64)), dim3(256), 0, st, d_out, n, g, ng, bits, mse, w, out);
  return hipGetLastError();
}

hipError_t act_scale(hipStream_t st, long tokens, int n, const float* noise, const float* scale, const float* massive,
                     float* x) {
  if (tokens * n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_act_scale, dim3(blocks_for(tokens * n)), dim3(256), 0, st, tokens, n, noise, scale, massive, x);
  return hipGetLastError();
}

hipError_t channel_rms(hipStream_t st, long tokens, int n, const float* x, float* rms) {
  hipLaunchKernelGGL(k_channel_rms, dim3(blocks_for(n)), dim3(256), 0, st, tokens, n, x, rms);
  return hipGetLastError();
}

hipError_t add_noise(hipStream_t st, long tokens, int n, float a, const float* rms, const float* nrm, const float* x,
                     float* xt) {
  if (tokens * n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_add_noise, dim3(blocks_for(tokens * n)), dim3(256), 0, st, tokens, n, a, rms, nrm, x, xt);
  return hipGetLastError();
}

}  // namespace cdclq

// ---- checkpoint tensors (src/io.rs:37-45, :205-212)
namespace cdclq {
namespace {

// io::tensor_to_f32: little-endian F32 / F16 / BF16 widened to f32 (exact; NaN payloads keep their
// upper bits with the quiet bit set, as half's to_f32).
__global__ __launch_bounds__(256) void k_decode(long count, int dtype, const uint8_t* __restrict__ src,
                                                float* __restrict__ out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  if (dtype == CDCLQ_DTYPE_F32) {
    out[i] = reinterpret_cast<const float*>(src)[i];
  } else {
    const uint32_t h = reinterpret_cast<const uint16_t*>(src)[i];
    uint32_t u;
    if (dtype == CDCLQ_DTYPE_BF16) {
      u = ((h & 0x7fffu) > 0x7f80u ? (h | 0x0040u) : h) << 16;  // NaN quieted as half::bf16::to_f32
    } else {
      const uint32_t sign = (h & 0x8000u) << 16, exp = (h >> 10) & 0x1fu;
      uint32_t man = h & 0x3ffu;
      if (exp == 0x1fu) {
        u = sign | 0x7f800000u | (man << 13) | (man ? 0x400000u : 0u);
      } else if (exp == 0) {
        if (man == 0) {
          u = sign;
        } else {
          const int lz = __clz((int)man) - 21;
          man = (man << lz) & 0x3ffu;
          u = sign | ((uint32_t)(113 - lz) << 23) | (man << 13);
        }
      } else {
        u = sign | ((exp + 112u) << 23) | (man << 13);
      }
    }
    out[i] = __uint_as_float(u);
  }
}

// Index of the first non-finite element (io.rs first_non_finite): atomicMin over the indices.
__global__ __launch_bounds__(256) void k_first_non_finite(long count, const float* __restrict__ x,
                                                          unsigned long long* __restrict__ first) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const uint32_t u = __float_as_uint(x[i]);
  if ((u & 0x7f800000u) == 0x7f800000u) atomicMin(first, (unsigned long long)i);
}

}  // namespace

hipError_t decode_to_f32(hipStream_t st, long count, int dtype, const void* src, float* out) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_decode, dim3(blocks_for(count)), dim3(256), 0, st, count, dtype,
                     static_cast<const uint8_t*>(src), out);
  return hipGetLastError();
}

hipError_t first_non_finite(hipStream_t st, long count, const float* x, unsigned long long* first) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_first_non_finite, dim3(blocks_for(count)), dim3(256), 0, st, count, x, first);
  return hipGetLastError();
}

}  // namespace cdclq

// ---- calibration capture (scripts/capture_hessians.py:233-245, :266)
namespace cdclq {
namespace {

// xf = x * sqrt(w_t) per token (f32, as `xf * state["w"].sqrt().unsqueeze(1)`)
// 2^lg threads to a row, V columns each (V = 4: 16-byte aligned rows).
template <int V>
__global__ __launch_bounds__(256) void k_token_scale(long t, int n, int lg, const float* __restrict__ x,
                                                     const float* __restrict__ w, float* __restrict__ out) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const int c0 = threadIdx.x & ((1 << lg) - 1), per = 256 >> lg;
  for (long r = (long)blockIdx.x * per + (threadIdx.x >> lg); r < t; r += (long)gridDim.x * per) {
    const float s = sqrtf(w[r]);
    const vec* src = reinterpret_cast<const vec*>(x + r * n);
    vec* dst = reinterpret_cast<vec*>(out + r * n);
    for (int c = c0; c < n / V; c += 1 << lg) dst[c] = src[c] * s;
  }
}

// h = (f32)(acc / count): the 1/N normalisation, rounded once from f64
__global__ __launch_bounds__(256) void k_normalize(long count, const double* __restrict__ acc, double tokens,
                                                   float* __restrict__ h) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i < count) h[i] = (float)(acc[i] / tokens);
}

}  // namespace

hipError_t token_scale(hipStream_t st, long t, int n, const float* x, const float* w, float* out) {
  if (t * n <= 0) return hipSuccess;
  const bool v4 = n % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)out % 16 == 0;
  const int nv = v4 ? n / 4 : n;
  int lg = 8;
  while (lg > 0 && (1 << (lg - 1)) >= nv) --lg;
  // at most 2^20 workgroups, far below 2^32 work-items
  const dim3 grid((unsigned)std::min<long>((t + (256 >> lg) - 1) / (256 >> lg), 1L << 20));
  if (v4)
    hipLaunchKernelGGL(k_token_scale<4>, grid, dim3(256), 0, st, t, n, lg, x, w, out);
  else
    hipLaunchKernelGGL(k_token_scale<1>, grid, dim3(256), 0, st, t, n, lg, x, w, out);
  return hipGetLastError();
}

hipError_t normalize_acc(hipStream_t st, long count, const double* acc, double tokens, float* h) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_normalize, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, count, acc, tokens, h);
  return hipGetLastError();
}

}  // namespace cdclq
