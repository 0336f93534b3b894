// misc.hip - the GEMV's producer and consumers in a decode step: row statistics (the rstd slot an rms prologue reads),
// the split-K sum with the residual RMS update (normadd), and the argmax over the per-tile maxima a softcap GEMV
// writes. rowstats and normadd sum in the reference's order (256 partials, partial t over elements t, t + 256, ... in
// turn, then a halving tree), so the fp32 sums equal the reference's, bit for bit.
//
// Rows of 16-byte aligned values: one wave owns a row, lane l holds the partials 4 l .. 4 l + 3, so 256 consecutive elements
// are one 16-byte load per lane, and the whole tree is lane moves within the wave (no LDS, no barrier). Bound: at a decode
// step's one row, the memory round trips (launch, loads, stores); at thousands of rows, HBM bandwidth. A workgroup of 256
// threads per row with one 4-byte load in flight per thread and nine barriers a tree took, per recorded launch, 24.7 us for
// the statistics of 4608 x 3072 values; this takes 11.7 (4.9 TB/s). Rows that are not aligned, and normadds of lengths that
// suit no form of the wave's, are still a workgroup's.
#include "common.hpp"

// no FMA contraction: every a + b * c rounds the product and the sum separately, as the CPU restatement does, so the
// device sums and the oracle's agree bit for bit
#pragma clang fp contract(off)

namespace p0 {

constexpr int kChunk = 256;   // elements a wave takes per step: 4 consecutive ones per lane

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// the reference's halving tree over 256 partials (engine/ops/misc.js:20-23, engine/llm/lops.js:158-159: level s adds
// red[t + s] to red[t]), partial 4 l + c in component c of lane l; every lane gets the result. Levels 128 and 64 pair
// lanes 32 and 16 apart, 32 .. 4 lanes 8 .. 1 apart (a rotation by s of a row whose values have period 2 s is the
// exchange with lane ^ s), 2 and 1 the components.
__device__ __forceinline__ float tree256(const float (&part)[4]) {
  float v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float t = part[c];
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    t = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    t = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    t = t + dpp_move<0x128>(t);   // row_ror:8
    t = t + dpp_move<0x124>(t);
    t = t + dpp_move<0x122>(t);
    v[c] = t + dpp_move<0x121>(t);
  }
  return (v[0] + v[2]) + (v[1] + v[3]);
}

// the same tree over 256 threads' partials through LDS
constexpr int kRowThreads = 256;
__device__ __forceinline__ float tree256_lds(float v, float* red) {
  const int t = threadIdx.x;
  red[t] = v;
  __syncthreads();
#pragma unroll
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) red[t] = red[t] + red[t + s];
    __syncthreads();
  }
  const float r = red[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ float rsqrt_exact(float v) { return 1.0f / __builtin_sqrtf(v); }

// elements i .. i + 3 of the n at a (0 past their end). VEC: 16-byte aligned rows of a multiple of 4 elements
template <bool VEC>
__device__ __forceinline__ float4 load4(const float* __restrict__ a, int i, int n) {
  if (VEC) return i < n ? *(const float4*)(a + i) : float4{0.0f, 0.0f, 0.0f, 0.0f};
  float4 v;
  v.x = i < n ? a[i] : 0.0f;
  v.y = i + 1 < n ? a[i + 1] : 0.0f;
  v.z = i + 2 < n ? a[i + 2] : 0.0f;
  v.w = i + 3 < n ? a[i + 3] : 0.0f;
  return v;
}
__device__ __forceinline__ float at(const float4& v, int c) { return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w; }

// NB chunks of a row are held in registers (ONCE: a row of at most NB 256 elements, read once); longer rows run in
// batches of NB chunks and are read again in the second pass. An element past the row's end adds 0 to a sum that is
// never -0, which leaves its bits alone; terms that are not plain elements are left out instead.
// engine/ops/misc.js:17-30
template <bool VEC, int NB, bool ONCE>
__global__ __launch_bounds__(256) void rowstats_kernel(const float* __restrict__ x, int64_t ld, int64_t c0,
                                                       int64_t rows, int64_t cols, int mode, float eps,
                                                       float* __restrict__ st, int64_t st_off) {
  const int lane = threadIdx.x & 63;
  const int64_t step = (int64_t)gridDim.x * (blockDim.x >> 6);
  for (int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); row < rows; row += step) {
    const float* xr = x + row * ld + c0;
    float4 v[NB];
    auto load = [&](int64_t b) -> int {   // the batch at b; its length
      const int n = (int)(cols - b < NB * kChunk ? cols - b : NB * kChunk);
#pragma unroll
      for (int k = 0; k < NB; ++k) v[k] = load4<VEC>(xr + b, k * kChunk + 4 * lane, n);
      return n;
    };
    float q[4] = {0.0f, 0.0f, 0.0f, 0.0f}, mean = 0.0f;
    auto sums = [&](float (&s)[4]) {
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) s[c] = s[c] + at(v[k], c);
    };
    auto squares = [&](int n) {
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float d = at(v[k], c) - mean;
          q[c] = k * kChunk + 4 * lane + (VEC ? 0 : c) < n ? q[c] + d * d : q[c];
        }
    };
    if (ONCE) {
      const int n = load(0);
      if (mode == 0) {
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        sums(s);
        mean = tree256(s) / (float)cols;
      }
      squares(n);
    } else {
      if (mode == 0) {
        float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int64_t b = 0; b < cols; b += NB * kChunk) {
          load(b);
          sums(s);
        }
        mean = tree256(s) / (float)cols;
      }
      for (int64_t b = 0; b < cols; b += NB * kChunk) squares(load(b));
    }
    const float var = tree256(q) / (float)cols;
    if (lane == 0) {
      st[(st_off + row) * 2] = mean;
      st[(st_off + row) * 2 + 1] = rsqrt_exact(var + eps);
    }
  }
}

// The same for any row, 256 threads a row, one element each at a time.
__global__ __launch_bounds__(kRowThreads) void rowstats_any_kernel(const float* __restrict__ x, int64_t ld, int64_t c0,
                                                                   int64_t rows, int64_t cols, int mode, float eps,
                                                                   float* __restrict__ st, int64_t st_off) {
  __shared__ float red[kRowThreads];
  const int t = threadIdx.x;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const float* xr = x + row * ld + c0;
    float mean = 0.0f;
    if (mode == 0) {
      float s = 0.0f;
      for (int64_t i = t; i < cols; i += kRowThreads) s = s + xr[i];
      mean = tree256_lds(s, red) / (float)cols;
    }
    float q = 0.0f;
    for (int64_t i = t; i < cols; i += kRowThreads) {
      const float d = xr[i] - mean;
      q = q + d * d;
    }
    const float var = tree256_lds(q, red) / (float)cols;
    if (t == 0) {
      st[(st_off + row) * 2] = mean;
      st[(st_off + row) * 2 + 1] = rsqrt_exact(var + eps);
    }
  }
}

// engine/llm/lops.js:153-170, 16-byte aligned rows, a wave a row. ONCE: the row's partials (four at a time), its residual and
// the norm weights are all in flight together before the first sum; longer rows add the partials again in the second
// pass (the same order, the same bits).
template <int NB, bool ONCE>
__global__ __launch_bounds__(64) void normadd_kernel(const float* __restrict__ T, int64_t nsrc, int64_t ldp,
                                                     const float* __restrict__ W, int64_t woff, float* X,
                                                     float* __restrict__ ST, int64_t stoff, int64_t D, float eps,
                                                     float scale, int mode) {
  const int lane = threadIdx.x;
  const int64_t m = blockIdx.x, xb = m * D;
  float4 t[NB], xv[NB], wv[NB];
  auto length = [&](int64_t b) { return (int)(D - b < NB * kChunk ? D - b : NB * kChunk); };
  auto tsum = [&](int64_t b) {   // the partials in j order
    const int n = length(b);
#pragma unroll
    for (int k = 0; k < NB; ++k) t[k] = float4{0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](const float4 (&v)[NB]) {
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        t[k].x = t[k].x + v[k].x;
        t[k].y = t[k].y + v[k].y;
        t[k].z = t[k].z + v[k].z;
        t[k].w = t[k].w + v[k].w;
      }
    };
    int64_t j = 0;
    for (; j + 4 <= nsrc; j += 4) {
      float4 v[4][NB];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < NB; ++k) v[u][k] = load4<true>(T + (j + u) * ldp + xb + b, k * kChunk + 4 * lane, n);
#pragma unroll
      for (int u = 0; u < 4; ++u) add(v[u]);
    }
    for (; j < nsrc; ++j) {
      float4 v[NB];
#pragma unroll
      for (int k = 0; k < NB; ++k) v[k] = load4<true>(T + j * ldp + xb + b, k * kChunk + 4 * lane, n);
      add(v);
    }
  };
  auto inputs = [&](int64_t b) {
    const int n = length(b);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      xv[k] = wv[k] = float4{0.0f, 0.0f, 0.0f, 0.0f};
      if (mode == 0) {
        xv[k] = load4<true>(X + xb + b, k * kChunk + 4 * lane, n);
        wv[k] = load4<true>(W + woff + b, k * kChunk + 4 * lane, n);
      }
    }
  };
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f}, s2[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  auto squares = [&] {
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] = s[c] + at(t[k], c) * at(t[k], c);
  };
  if (ONCE) {
    inputs(0);
    tsum(0);
    squares();
  } else {
    for (int64_t b = 0; b < D; b += NB * kChunk) {
      tsum(b);
      squares();
    }
  }
  const float rs = rsqrt_exact(tree256(s) / (float)D + eps);
  auto update = [&](int64_t b) {
    const int n = length(b);
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int i = k * kChunk + 4 * lane;
      float y[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        y[c] = mode == 0 ? (at(xv[k], c) + at(t[k], c) * rs * at(wv[k], c)) * scale : at(t[k], c);
        s2[c] = i < n ? s2[c] + y[c] * y[c] : s2[c];
      }
      if (i < n) *(float4*)(X + xb + b + i) = float4{y[0], y[1], y[2], y[3]};
    }
  };
  if (ONCE) {
    update(0);
  } else {
    for (int64_t b = 0; b < D; b += NB * kChunk) {
      inputs(b);
      tsum(b);
      update(b);
    }
  }
  const float r2 = tree256(s2);
  if (lane == 0) ST[stoff + m] = rsqrt_exact(r2 / (float)D + eps);
}

// The same for any row: 256 threads, one element each at a time, the row's sums in LDS between the passes (D floats).
__global__ __launch_bounds__(kRowThreads) void normadd_any_kernel(const float* __restrict__ T, int64_t nsrc, int64_t ldp,
                                                                  const float* __restrict__ W, int64_t woff, float* X,
                                                                  float* __restrict__ ST, int64_t stoff, int64_t D, float eps,
                                                                  float scale, int mode) {
  __shared__ float red[kRowThreads];
  extern __shared__ float tv[];
  const int t = threadIdx.x;
  const int64_t m = blockIdx.x, xb = m * D;
  float s = 0.0f;
  for (int64_t i = t; i < D; i += kRowThreads) {
    float v = 0.0f;
    for (int64_t j = 0; j < nsrc; ++j) v = v + T[j * ldp + xb + i];
    tv[i] = v;
    s = s + v * v;
  }
  const float rs = rsqrt_exact(tree256_lds(s, red) / (float)D + eps);
  float s2 = 0.0f;
  for (int64_t i = t; i < D; i += kRowThreads) {
    float x = X[xb + i];
    if (mode == 0) x = (x + tv[i] * rs * W[woff + i]) * scale;
    else x = tv[i];
    X[xb + i] = x;
    s2 = s2 + x * x;
  }
  const float r2 = tree256_lds(s2, red);
  if (t == 0) ST[stoff + m] = rsqrt_exact(r2 / (float)D + eps);
}

// The same for rows of at most 2048 values, 16-byte aligned, and few of them (a decode step's, a verify pass's): a wave per
// chunk of 256, all of its loads in flight before the first sum; the chunks' squares meet in LDS, where every wave adds
// them in chunk order, which is partial t's order. Per recorded launch 2048 values over 1 or 4 partials take 2.7 us (one
// wave a row: 4.1), 256 rows 3.3; a decode token as a recording, 60 of them, 913 -> 870 us. More rows than CUs: a wave a row.
constexpr int kNaWaves = 8, kNaThreads = 64 * kNaWaves;
__global__ __launch_bounds__(kNaThreads) void normadd_few_kernel(const float* __restrict__ T, int64_t nsrc, int64_t ldp,
                                                                 const float* __restrict__ W, int64_t woff, float* X,
                                                                 float* __restrict__ ST, int64_t stoff, int D, float eps,
                                                                 float scale, int mode) {
  __shared__ __attribute__((aligned(16))) float sq[2][kNaWaves][kChunk];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, i = wv * kChunk + 4 * lane;
  const int64_t m = blockIdx.x, xb = m * D;
  const bool in = i < D;
  const float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float4 xv = zero, w4 = zero;
  if (mode == 0) {
    xv = load4<true>(X + xb, i, D);
    w4 = load4<true>(W + woff, i, D);
  }
  float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t j = 0; j < nsrc; j += 4) {   // four at a time; past the last: the last again, not added
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = load4<true>(T + (j + u < nsrc ? j + u : nsrc - 1) * ldp + xb, i, D);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c) t[c] = j + u < nsrc ? t[c] + at(v[u], c) : t[c];
  }
  auto total = [&](const float (*q)[kChunk]) {
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kNaWaves; ++k) {
      const float4 v = *(const float4*)(q[k] + 4 * lane);
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] = s[c] + at(v, c);
    }
    return tree256(s);
  };
  *(float4*)(sq[0][wv] + 4 * lane) = float4{t[0] * t[0], t[1] * t[1], t[2] * t[2], t[3] * t[3]};
  __syncthreads();
  const float rs = rsqrt_exact(total(sq[0]) / (float)D + eps);
  float y[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) y[c] = mode == 0 ? (at(xv, c) + t[c] * rs * at(w4, c)) * scale : t[c];
  if (in) *(float4*)(X + xb + i) = float4{y[0], y[1], y[2], y[3]};
  *(float4*)(sq[1][wv] + 4 * lane) = in ? float4{y[0] * y[0], y[1] * y[1], y[2] * y[2], y[3] * y[3]} : zero;
  __syncthreads();
  if (wv != 0) return;
  const float r2 = total(sq[1]);
  if (lane == 0) ST[stoff + m] = rsqrt_exact(r2 / (float)D + eps);
}

// engine/llm/lops.js:418-433, engine/llm/lops_spec.js:329-343: (value, index) with ties to the lower index. A running
// best is never NaN, so "better" is a total order on what is combined: any order of the reduction gives its result. A
// workgroup of 16 waves per row, four pairs in flight per thread: a head's 4096 tile maxima in one round, 4.0 us a launch (256
// threads that load 16 pairs one after another: 6.3).
constexpr int kArgThreads = 1024;
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));   // an 8-byte load at 4-byte alignment
__device__ __forceinline__ bool better(float v, uint32_t id, float bv, uint32_t bi) {
  return v > bv || (v == bv && id < bi);
}
__device__ __forceinline__ void wave_best(float& v, uint32_t& id) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const float ov = __shfl_xor(v, s, 64);
    const uint32_t oi = (uint32_t)__shfl_xor((int)id, s, 64);
    if (better(ov, oi, v, id)) { v = ov; id = oi; }
  }
}
__global__ __launch_bounds__(kArgThreads) void argmax_kernel(const float* __restrict__ MX, int64_t n,
                                                            uint32_t* __restrict__ out) {
  __shared__ float rv[kArgThreads / 64];
  __shared__ uint32_t ri[kArgThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const float* row = MX + 2 * (int64_t)blockIdx.x * n;
  float bv = -3.4e38f;
  uint32_t bi = 0xFFFFFFFFu;
  for (int64_t i0 = 0; i0 < n; i0 += 4 * kArgThreads) {
    u32x2a4 p[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t i = i0 + u * kArgThreads + t;
      p[u] = i < n ? *(const u32x2a4*)(row + 2 * i) : u32x2a4{0xFF800000u, 0xFFFFFFFFu};   // -inf: never better
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float v = __uint_as_float(p[u].x);
      if (better(v, p[u].y, bv, bi)) { bv = v; bi = p[u].y; }
    }
  }
  wave_best(bv, bi);
  if (lane == 0) {
    rv[wv] = bv;
    ri[wv] = bi;
  }
  __syncthreads();
  if (wv != 0) return;
  bv = rv[lane & (kArgThreads / 64 - 1)];
  bi = ri[lane & (kArgThreads / 64 - 1)];
  wave_best(bv, bi);
  if (lane == 0) {
    out[2 * blockIdx.x] = bi;
    out[2 * blockIdx.x + 1] = __float_as_uint(bv);
  }
}

// The same with 256 threads, one pair at a time, and a tree through LDS: short rows, or many.
__global__ __launch_bounds__(kRowThreads) void argmax_short_kernel(const float* __restrict__ MX, int64_t n,
                                                                   uint32_t* __restrict__ out) {
  __shared__ float rv[kRowThreads];
  __shared__ uint32_t ri[kRowThreads];
  const int t = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x * n;
  float bv = -3.4e38f;
  uint32_t bi = 0xFFFFFFFFu;
  for (int64_t i = t; i < n; i += kRowThreads) {
    const float v = MX[2 * (b + i)];
    const uint32_t id = __float_as_uint(MX[2 * (b + i) + 1]);
    if (better(v, id, bv, bi)) { bv = v; bi = id; }
  }
  rv[t] = bv;
  ri[t] = bi;
  __syncthreads();
  for (int s = kRowThreads / 2; s > 0; s >>= 1) {
    if (t < s && better(rv[t + s], ri[t + s], rv[t], ri[t])) { rv[t] = rv[t + s]; ri[t] = ri[t + s]; }
    __syncthreads();
  }
  if (t == 0) {
    out[2 * blockIdx.x] = ri[0];
    out[2 * blockIdx.x + 1] = __float_as_uint(rv[0]);
  }
}

// normadd's LDS allowance (one row of up to 150 KB), set once at p0_open
int misc_init() {
  P0_HIP(hipFuncSetAttribute((const void*)normadd_any_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024),
         "p0_open: normadd");
  return P0_OK;
}

static bool vec_ok(const float* p, int64_t a, int64_t b) { return (((uintptr_t)p | (uintptr_t)(a * 4) | (uintptr_t)(b * 4)) & 15) == 0; }

}  // namespace p0

using namespace p0;

extern "C" int p0_rowstats(const p0_rowstats_args_t* a) {
  if (!a) { set_error("rowstats: no arguments"); return P0_EINVAL; }
  if (a->rows < 0 || a->cols <= 0) { set_error("rowstats: rows %lld, cols %lld", (long long)a->rows, (long long)a->cols); return P0_EINVAL; }
  if (a->mode != 0 && a->mode != 1) { set_error("rowstats: mode %d", (int)a->mode); return P0_EINVAL; }
  if (!a->x || !a->st) { set_error("rowstats: missing x or st buffer"); return P0_EINVAL; }
  if (a->x_off % 4) { set_error("rowstats: x offset"); return P0_EINVAL; }
  if (int r = require_open("rowstats")) return r;
  if (a->rows == 0) return P0_OK;
  const int64_t ld = a->x_ld ? a->x_ld : a->cols;
  if (building_chain())   // a chain op (chain_aux.hpp): the same sums in the same order
    return chain_add_rowstats((const float*)((const uint8_t*)a->x + a->x_off), ld, a->x_c0, a->rows, a->cols,
                              (int)a->mode, a->eps, a->st, a->st_off);
  // one row per wave; four waves a workgroup once there are rows for more than the chip holds at one each (1024: the
  // dispatch of thousands of one-wave workgroups is what shows then). 4096 columns stay in registers; a longer row is
  // read again for its variance, 2048 columns at a time.
  const float* x = (const float*)((const uint8_t*)a->x + a->x_off);
  const int wpb = a->rows >= 1024 ? 4 : 1;
  const int64_t blocks = (a->rows + wpb - 1) / wpb;
  const unsigned grid = (unsigned)(blocks < 65536 * 4 ? blocks : 65536 * 4);
  const bool vec = vec_ok(x, ld, a->x_c0) && a->cols % 4 == 0;
  // rows that are not 16-byte aligned are four 4-byte loads a lane and 256 values: a workgroup a row wins from 4096 columns,
  // or 512 once the rows fill the chip (mean and variance, us, a wave / a workgroup a row: one row of 3071 4.9 / 5.0, of 4099
  // 6.7 / 5.7; 1024 rows of 511 3.8 / 4.2, of 2047 6.5 / 5.4; 4608 rows of 2047 20.9 / 16.9)
  if (!vec && a->cols > (a->rows <= 256 ? 4096 : 512)) {
    const unsigned g = (unsigned)(a->rows < 65536 * 4 ? a->rows : 65536 * 4);
    hipLaunchKernelGGL(rowstats_any_kernel, dim3(g), dim3(kRowThreads), 0, ctx().cur, x, ld, a->x_c0, a->rows, a->cols,
                       (int)a->mode, a->eps, a->st, a->st_off);
    P0_LAUNCHED("rowstats");
    return P0_OK;
  }
  auto k = !vec                       ? rowstats_kernel<false, 4, false>
           : a->cols <= 8 * kChunk    ? rowstats_kernel<true, 8, true>
           : a->cols <= 16 * kChunk   ? rowstats_kernel<true, 16, true>
                                      : rowstats_kernel<true, 8, false>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * wpb), 0, ctx().cur, x, ld, a->x_c0, a->rows, a->cols, (int)a->mode, a->eps,
                     a->st, a->st_off);
  P0_LAUNCHED("rowstats");
  return P0_OK;
}

extern "C" int p0_normadd(const p0_normadd_args_t* a) {
  if (!a) { set_error("normadd: no arguments"); return P0_EINVAL; }
  const int64_t D = a->D, M = a->M ? a->M : 1;
  if (D <= 0 || M < 0) { set_error("normadd: D %lld, M %lld", (long long)D, (long long)M); return P0_EINVAL; }
  if (a->mode != 0 && a->mode != 1) { set_error("normadd: mode %d", (int)a->mode); return P0_EINVAL; }
  if (!a->t || !a->x || !a->st || (a->mode == 0 && !a->w)) { set_error("normadd: missing t, w, x or st buffer"); return P0_EINVAL; }
  if (D * (int64_t)sizeof(float) > 150 * 1024) {   // normadd_any_kernel's row in LDS
    set_error("normadd: D %lld exceeds this build's row buffer", (long long)D); return P0_EINVAL;
  }
  if (int r = require_open("normadd")) return r;
  const int64_t nsrc = a->t_n ? a->t_n : 1, ldp = a->t_ld ? a->t_ld : D * M;
  const float eps = a->eps != 0.0f ? a->eps : 1e-6f;
  if (building_chain())
    return chain_add_normadd(a->t, nsrc, ldp, a->w, a->w_off, a->x, a->st, a->st_off, D, M, eps, a->scale, (int)a->mode);
  const bool vec = vec_ok(a->t, ldp, D) && vec_ok(a->x, 0, 0) && (a->mode == 1 || vec_ok(a->w, a->w_off, 0));
  if (vec && D <= kNaWaves * kChunk && M <= 256) {
    hipLaunchKernelGGL(normadd_few_kernel, dim3((unsigned)M), dim3(kNaThreads), 0, ctx().cur, a->t, nsrc, ldp, a->w, a->w_off,
                       a->x, a->st, a->st_off, (int)D, eps, a->scale, (int)a->mode);
    P0_LAUNCHED("normadd");
    return P0_OK;
  }
  // a wave a row where it holds the row and there is enough of it (us, a wave / a workgroup a row: 4608 rows of 512 over one
  // partial 10.1 / 9.8, of 768 10.6 / 12.8, 512 rows of 256 4.5 / 4.1), or in batches of 2048 from 3072 on (one row of 2304
  // 6.6 / 5.8, of 4096 6.8 / 7.9; 4608 rows of 2304 36.0 / 28.7, of 4096 40 / 45); rows that are not 16-byte aligned take a
  // workgroup each (one row of 2048 7.0 / 5.4, 4608 rows 46 / 27)
  if (vec && (D >= 3072 || (D >= 768 && D <= 8 * kChunk))) {
    auto k = D <= 8 * kChunk ? normadd_kernel<8, true> : normadd_kernel<8, false>;
    hipLaunchKernelGGL(k, dim3((unsigned)M), dim3(64), 0, ctx().cur, a->t, nsrc, ldp, a->w, a->w_off, a->x, a->st, a->st_off, D,
                       eps, a->scale, (int)a->mode);
  } else {
    hipLaunchKernelGGL(normadd_any_kernel, dim3((unsigned)M), dim3(kRowThreads), (size_t)D * sizeof(float), ctx().cur, a->t,
                       nsrc, ldp, a->w, a->w_off, a->x, a->st, a->st_off, D, eps, a->scale, (int)a->mode);
  }
  P0_LAUNCHED("normadd");
  return P0_OK;
}

extern "C" int p0_argmaxM(const float* mx, int64_t n, int64_t M, uint32_t* out) {
  if (!mx || !out) { set_error("argmax: missing mx or out buffer"); return P0_EINVAL; }
  if (n < 0 || M < 1) { set_error("argmax: n %lld, M %lld", (long long)n, (long long)M); return P0_EINVAL; }
  if (int r = require_open("argmax")) return r;
  if (building_chain()) return chain_add_argmax(mx, n, M, out);
  // 16 waves pay where one row's pairs are worth them and the rows do not fill the chip by themselves (us, 4 waves / 16: one row
  // of 256 pairs 2.8 / 3.1, of 1536 3.5 / 3.2, 512 rows of 2048 4.1 / 4.3, of 3072 4.7 / 4.3, 2048 rows of 256 3.6 / 9.3)
  const bool wide = n > 1024 && n >= 6 * M;
  auto k = wide ? argmax_kernel : argmax_short_kernel;
  hipLaunchKernelGGL(k, dim3((unsigned)M), dim3(wide ? kArgThreads : kRowThreads), 0, ctx().cur, mx, n, out);
  P0_LAUNCHED("argmax");
  return P0_OK;
}

extern "C" int p0_argmax(const float* mx, int64_t n, uint32_t* out) { return p0_argmaxM(mx, n, 1, out); }
