// gemv1.hip - the standalone GEMV (one row of x, one op per launch), for both weight encodings: q4g32a.t64 and
// q8g64s.t64 (the layouts are in gemv_kernels.hpp and gemv_q8.hip), splits of at most 2048 k.
//
// Replaces the WebGPU dispatch of gemv (engine/llm/lops.js:108-141) where the op is not part of a chain.
//
// Mapping: that of gemvm.hip (16-row blocks, items of NBK blocks, 8 waves each an eighth of K, all of a wave's records in
// flight, one LDS reduction, nothing but outputs leaves the workgroup) with fp32 arithmetic on the VALU, which for one row
// is less work than building matrix-core operands. A lane's 16 record bytes are 32 codes of one (row, group) pair (q4) or
// a quarter of one (q8), so it needs the group's 32 x' (its quarter's 16): the wave loads its 256 x' once (4 a lane),
// applies the prologue, and hands them round through 1 KB of LDS into registers that serve every block.
// Bound: the memory round trips of one launch (arguments, x, records, the stores), about 2.8 us between launches of a
// recording; for the large ops, HBM. Per launch, recorded over a ring of weights (before: gemv.hip's kernel with its 500
// bytes of arguments read in four serial steps, x' staged by every workgroup element by element, K sliced over workgroups
// with partials in uncached memory; q8: gemv_q8.hip's): q4 gate_up 2 x 8192 x 2048 9.6 -> 6.9 us, 3072 x 2048 6.2 -> 3.3,
// 2048 x 2048 5.8 -> 3.2, 2048 x 8192 in 4 splits 7.0 -> 4.9, 256 x 2048 5.2 -> 2.8, 65536 x 2048 20.8 -> 18.9; q8 5120 x
// 1536 6.9 -> 5.0, 1536 x 6144 in 3 splits 7.6 -> 5.4, geglu 6144 x 1536 9.1 -> 7.1 and 12288 x 1536 11.4 -> 10.3, 65536 x
// 1536 30.3 -> 23.8. Relative L2 against float64: q4 1.9e-7 - 2.7e-7 (1.9e-7 - 2.8e-7 before), q8 2.0e-7 (3.8e-7).
// Tried: the partials of a sum or pleg four at a time (q4 over 16 4.3 -> 3.9 us, but every q8 call 0.2 us slower), items of
// 4 blocks (q8 geglu 12288 12.5 us: 192 workgroups of 2 items), 2 workgroups per CU (65536 x 2048 18.6,
// but q8 geglu 6144 8.9), the next item's records loaded block by block as registers come free (262144 x 2048 76 us).
#include "gemvm.hpp"

namespace p0 {

// 2^-24 sum_k q_k x'_k over one row's 32 codes; odd k of x pre-scaled 1/16 (dot32 of gemv_kernels.hpp on registers)
__device__ __forceinline__ float dot32r(const u32x4 q, const float (&x)[32]) {
  const uint32_t u[4] = {q.x, q.y, q.z, q.w};
  float da = 0.0f, db = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t v = u[w], v8 = v >> 8;
    const uint32_t ua = v & 0x000F000Fu, ub = v & 0x00F000F0u, uc = v8 & 0x000F000Fu, ue = v8 & 0x00F000F0u;
    const h2_t a = __builtin_bit_cast(h2_t, ua), b = __builtin_bit_cast(h2_t, ub), c = __builtin_bit_cast(h2_t, uc),
               e = __builtin_bit_cast(h2_t, ue);
    da = __builtin_fmaf((float)a.x, x[8 * w], da);
    db = __builtin_fmaf((float)a.y, x[8 * w + 4], db);
    da = __builtin_fmaf((float)b.x, x[8 * w + 1], da);
    db = __builtin_fmaf((float)b.y, x[8 * w + 5], db);
    da = __builtin_fmaf((float)c.x, x[8 * w + 2], da);
    db = __builtin_fmaf((float)c.y, x[8 * w + 6], db);
    da = __builtin_fmaf((float)e.x, x[8 * w + 3], da);
    db = __builtin_fmaf((float)e.y, x[8 * w + 7], db);
  }
  return da + db;
}
// sum (q_k + 128) x'_k over 16 byte codes
__device__ __forceinline__ float dot16r(const u32x4 q, const float (&x)[32]) {
  const uint32_t u[4] = {q.x ^ 0x80808080u, q.y ^ 0x80808080u, q.z ^ 0x80808080u, q.w ^ 0x80808080u};
  float d = 0.0f, e = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    d = __builtin_fmaf((float)(u[w] & 0xFFu), x[4 * w], d);
    e = __builtin_fmaf((float)((u[w] >> 8) & 0xFFu), x[4 * w + 1], e);
    d = __builtin_fmaf((float)((u[w] >> 16) & 0xFFu), x[4 * w + 2], d);
    e = __builtin_fmaf((float)(u[w] >> 24), x[4 * w + 3], e);
  }
  return d + e;
}

template <int ENC, int NBK, bool GEGLU>
__global__ __launch_bounds__(kGmThreads) void gemv1_kernel(GmP p) {
  constexpr bool Q4 = ENC == P0_ENC_Q4G32A_T64;
  constexpr int GK = Q4 ? 32 : 64, RJ = Q4 ? 2 : 4;   // k per group; record loads per block (quads of groups, groups)
  constexpr int RUN = 256 / RJ, XN = Q4 ? 32 : 16;    // the wave's 256 k are RJ runs, run j at (wv + 8 j) RUN; x' a load needs
  constexpr int U = GEGLU ? NBK / 2 : NBK;            // 16-row blocks of output rows per item
  __shared__ float red[2][kGmWaves][NBK][16];
  __shared__ __attribute__((aligned(16))) float xl[kGmWaves][256], xsl[kGmWaves][8];   // x', and its group sums
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, q = lane >> 4;
  const int pos = stage_pos(blockIdx.x, p.wgs), split = blockIdx.y;
  const int it0 = pos * p.ipw, it1 = min(p.items, it0 + p.ipw);
  if (it0 >= it1) return;
  const int k0 = split * p.kPer, klen = min(p.K, k0 + p.kPer) - k0, ng = klen / GK;

  // ---- x, norm weights (or partials), then the first records: all in flight together
  const int nk = (wv + kGmWaves * (lane * 4 / RUN)) * RUN + lane * 4 % RUN;   // the lane's 4 consecutive k of the split
  const bool xin = nk < klen;
  const int64_t kx = k0 + (xin ? nk : 0);
  const bool plain = p.pro == P0_PRO_RAW || p.pro == P0_PRO_RMS;
  u32x4 xv{}, nv{};
  if (plain || p.nsrc > 0) xv = *P0_GLOBAL(const u32x4, p.X + kx);
  float rstd = 1.0f;
  if (p.pro == P0_PRO_RMS) {
    nv = *P0_GLOBAL(const u32x4, p.NW + kx);
    rstd = *P0_GLOBAL(const float, p.ST);
  } else if (p.pro == P0_PRO_PLEG) {
    nv = *P0_GLOBAL(const u32x4, p.EV + kx);
  }
  __builtin_amdgcn_sched_barrier(0);
  u32x4 rq[NBK][RJ];
  uint32_t rs[NBK][RJ];
  auto load_records = [&](int it) {   // groups past the split: its last one again (scale and min dropped, x' 0)
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      const int row = (it * U + (GEGLU ? b % U : b)) * 16 + (GEGLU && b >= U ? p.N : 0);
      const uint8_t* tb = p.w + ((int64_t)(row >> 6) * p.wG + k0 / GK) * (Q4 ? 1280 : 4224);
      const int r = (row & 63) + l16;
#pragma unroll
      for (int j = 0; j < RJ; ++j) {
        if constexpr (Q4) {
          const int off = min((wv + kGmWaves * j) * 4 + q, ng - 1) * 1280;
          rq[b][j] = *P0_GLOBAL(const u32x4, tb + (unsigned)(off + r * 16));
          rs[b][j] = *P0_GLOBAL(const uint32_t, tb + (unsigned)(off + 1024 + r * 4));
        } else {
          const uint8_t* rec = tb + min(wv + kGmWaves * j, ng - 1) * 4224;
          rq[b][j] = *P0_GLOBAL(const u32x4, rec + (unsigned)(r * 64 + q * 16));
          rs[b][j] = *P0_GLOBAL(const uint16_t, rec + (unsigned)(4096 + r * 2));
        }
      }
    }
  };
  load_records(it0);
  __builtin_amdgcn_sched_barrier(0);

  // ---- x' and its group sums
  float v[4] = {__uint_as_float(xv.x), __uint_as_float(xv.y), __uint_as_float(xv.z), __uint_as_float(xv.w)};
  if (!plain)   // sum, pleg: the other partials, in order (engine/llm/lops.js:50-57)
    for (int j = 1; j < p.nsrc; ++j) {
      const u32x4 t = *P0_GLOBAL(const u32x4, p.X + j * p.ldp + kx);
      v[0] += __uint_as_float(t.x);
      v[1] += __uint_as_float(t.y);
      v[2] += __uint_as_float(t.z);
      v[3] += __uint_as_float(t.w);
    }
  const float n[4] = {__uint_as_float(nv.x), __uint_as_float(nv.y), __uint_as_float(nv.z), __uint_as_float(nv.w)};
  float gs = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (p.pro == P0_PRO_RMS) v[e] = v[e] * rstd * n[e];
    else if (p.pro == P0_PRO_PLEG) v[e] = gelu_tanh(v[e]) * n[e];
    if (!xin) v[e] = 0.0f;
  }
  gs = (v[0] + v[1]) + (v[2] + v[3]);
  gs += dpp_f<0xB1>(gs);    // over the 8 lanes of a 32-k run: quad_perm, quad_perm, row_half_mirror
  gs += dpp_f<0x4E>(gs);
  gs += dpp_f<0x141>(gs);
  if (!Q4) gs += dpp_f<0x140>(gs);   // 16 lanes of a q8 group: row_mirror
  // lanes hand values to other lanes: a wavefront fence on each side keeps the compiler from moving the reads above the
  // writes (the LDS serves one wave's accesses in order)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  *(float4*)(xl[wv] + lane * 4) = float4{v[0], Q4 ? v[1] * 0.0625f : v[1], v[2], Q4 ? v[3] * 0.0625f : v[3]};
  if ((lane & (GK / 4 - 1)) == 0) xsl[wv][lane / (GK / 4)] = gs;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float x[RJ][32], sx[RJ];
#pragma unroll
  for (int j = 0; j < RJ; ++j) {
    const float* xr = xl[wv] + j * RUN + q * XN;
#pragma unroll
    for (int e = 0; e < XN; e += 4) {
      const float4 f = *(const float4*)(xr + e);
      x[j][e] = f.x; x[j][e + 1] = f.y; x[j][e + 2] = f.z; x[j][e + 3] = f.w;
    }
    sx[j] = Q4 ? xsl[wv][j * 4 + q] : xsl[wv][j] * (q == 0 ? 128.0f : 0.0f);   // q8: the bias' share, once a row
  }

  for (int it = it0; it < it1; ++it) {
    float acc[NBK];
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      acc[b] = 0.0f;
#pragma unroll
      for (int j = 0; j < RJ; ++j) {
        if constexpr (Q4) {
          const uint32_t sm = (wv + kGmWaves * j) * 4 + q < ng ? rs[b][j] : 0u;
          acc[b] = __builtin_fmaf(h2f_lo(sm) * 16777216.0f, dot32r(rq[b][j], x[j]), __builtin_fmaf(h2f_hi(sm), sx[j], acc[b]));
        } else {
          const float s = wv + kGmWaves * j < ng ? h2f_lo(rs[b][j]) : 0.0f;
          acc[b] = __builtin_fmaf(s, dot16r(rq[b][j], x[j]) - sx[j], acc[b]);
        }
      }
    }
    if (it + 1 < it1) load_records(it + 1);
    float (*rd)[NBK][16] = red[(it - it0) & 1];   // the other half is still read by slower waves
#pragma unroll
    for (int b = 0; b < NBK; ++b) {   // the quarters of a row are 16 lanes apart
      float t = acc[b];
      const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
      t = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
      const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
      t = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
      if (lane < 16) rd[wv][b][lane] = t;
    }
    __syncthreads();
    // thread -> (block, row), the waves taking turns; a softcap's tile is one wave. The waves' sums in wave order
    const int b = ((tid - 64 * (it - it0)) & (kGmThreads - 1)) >> 4;
    if (b < U) {
      float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
      for (int w = 0; w < kGmWaves; ++w) v0 += rd[w][b][l16];
      if (GEGLU) {
#pragma unroll
        for (int w = 0; w < kGmWaves; ++w) v1 += rd[w][NBK - U + b][l16];
      }
      const int nr = (it * U + b) * 16 + l16;
      epilogue<false>(p, split, 0, nr >> 6, nr & 63, v0, v1);
    }
  }
}

template <int ENC>
static void launch_enc(const GemvP& p, hipStream_t s) {
  const GmPlan pl = gm_plan(p, INT64_MAX);   // items of 4 blocks only for a softcap: 2 ran faster from 512 blocks up too
  auto k = p.epi == P0_EPI_GEGLU ? gemv1_kernel<ENC, 2, true>
           : pl.nbk == 4         ? gemv1_kernel<ENC, 4, false>
           : pl.nbk == 2         ? gemv1_kernel<ENC, 2, false>
                                 : gemv1_kernel<ENC, 1, false>;
  hipLaunchKernelGGL(k, pl.grid, dim3(kGmThreads), 0, s, pl.args);
}

// Splits of at most 2048 k (a wave's records of more do not fit its registers). A q4 op of more than 1024 tiles streams
// from HBM on gemv.hip's kernel: 262144 x 2048 61.2 us there and 61.5 here, with a softcap 66.4 and 70.8; at 65536 rows
// 20.3 and 17.8, 21.7 and 19.9
//
// A short split leaves most of a workgroup's 8 waves without records (a wave takes 128 k of a q4 row at a time, 64 of a
// q8 row), which a call of several items per workgroup, or of a softcap's 4 blocks per item, pays for item by item: such
// calls stay on gemv.hip's and gemv_q8.hip's kernels, from more k the more blocks there are. Per recorded launch, us here /
// there: q4 store 8192 x 320 (512 blocks) 4.0 / 4.6, 16384 x 640 (1024) 5.2 / 5.1, x 960 5.6 / 6.1, 2560 x 10240 in 10 splits
// (1600) 7.9 / 7.5, 8192 x 8192 in 8 (4096) 14.4 / 12.7, 65536 x 1024 14.3 / 12.1, x 1280 14.8 / 14.9; q4 geglu 4096 x 320
// (512) 4.1 / 4.9, 16384 x 960 (2048) 9.5 / 8.4, x 1280 9.6 / 9.9, 32768 x 1280 (4096) 16.5 / 14.3, x 2048 20.5 / 18.6; q4
// softcap 1024 x 320 5.4 / 5.0, 4096 x 704 (256) 5.2 / 5.5, 16384 x 704 (1024) 6.0 / 5.7, x 1024 6.3 / 6.4, 32768 x 704 8.5 /
// 7.4, 65536 x 1024 (4096) 15.0 / 13.5, x 1280 16.1 / 16.3; q8 store 64 x 32768 in 128 splits (512) 4.7 / 4.0, 16384 x 320
// 6.0 / 5.3, x 704 6.1 / 6.5, 32768 x 704 (2048) 10.3 / 8.1, x 1024 11.0 / 12.7; q8 geglu 4096 x 320 4.8 / 6.3, 16384 x 1024
// 11.3 / 11.0; q8 softcap 4096 x 320 7.3 / 5.8, 16384 x 1024 8.9 / 8.7, 1024 x 2048 (64) 7.0 / 6.7, 4096 x 2048 7.2 / 8.2.
bool gemv1_takes(const GemvP& p) {
  const bool q8 = p.enc == P0_ENC_Q8G64S_T64, geglu = p.epi == P0_EPI_GEGLU;
  if (p.kPer > kGmPass || (!q8 && p.NT > 1024)) return false;
  const int64_t blocks = (int64_t)(p.N / 16) * (geglu ? 2 : 1) * p.nsplit;
  if (p.epi == P0_EPI_SOFTCAP)
    return q8 ? p.kPer > 1024 && blocks > 64 : p.kPer > (blocks <= 512 ? 640 : blocks <= 2048 ? 960 : 1152);
  if (q8) {
    // four groups are one each for gemv_q8.hip's four waves, which read the partials as they need them: pleg 64 x 256 over
    // one partial 3.4 / 3.5, over 4 3.9 / 3.7, over 16 5.1 / 4.7
    if (p.kPer <= 256 && p.nsrc > 1 && (p.pro == P0_PRO_SUM || p.pro == P0_PRO_PLEG)) return false;
    if (blocks <= 512) return blocks <= 256 || p.kPer > 256;
    return p.kPer >= (geglu ? 1088 : blocks <= 1024 ? 640 : 1024);
  }
  if (blocks <= 512) return true;
  if (geglu) return blocks <= 2048 && p.kPer >= 1280;
  return p.kPer >= (blocks <= 1024 ? 960 : 1152);
}

void launch_gemv1(const GemvP& p, hipStream_t s) {
  if (p.enc == P0_ENC_Q4G32A_T64) launch_enc<P0_ENC_Q4G32A_T64>(p, s);
  else launch_enc<P0_ENC_Q8G64S_T64>(p, s);
}

}  // namespace p0
