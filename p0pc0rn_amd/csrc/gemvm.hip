// gemvm.hip - the standalone GEMV-M on the matrix cores (2 <= M <= 16 rows of x, one op per launch), for both weight
// encodings: q4g32a.t64 and q8g64s.t64 (the layouts are in gemv_kernels.hpp and gemv_q8.hip).
//
// Replaces the WebGPU dispatch of gemvM (engine/llm/lops_spec.js:159-191) where the op is not part of a chain.
//
// Mapping. The weight rows are cut into blocks of 16 (one v_mfma_f32_16x16x32_f16 operand); a workgroup of 8 waves takes
// an item of NBK blocks (a geglu item: NBK / 2 gate blocks and their up blocks; a softcap item: one 64-row tile) and
// the whole K range of one kPer split (long splits aside, see below), the waves each an eighth of it, so nothing leaves
// the workgroup but outputs: no partials in memory, one barrier per item (the waves' sums meet in LDS).
//  * x' lives in registers. A lane's A operand is 8 consecutive k of one x row: the wave loads its 256 k of every row
//    straight from x (no LDS), scales each row by a power of two so that its largest |x'| lies in [2^14, 2^15), and
//    splits it into fp16 hi + lo, so a value within 2^-18 of its row's largest keeps 22 bits, nothing overflows, and
//    no input needs another path. Infinite and NaN x' stay what they are and keep to their own row.
//  * All of a wave's records of an item are in flight together: a lane's 16-byte load covers 16 rows x 4 groups (q4; a
//    4 x 4 transpose of lane rows and words makes B operands of it, quarter_transpose) or 16 rows x 64 k (q8, whose k
//    order inside a group is chosen so that the lane's 16 bytes are its own two B operands).
//  * Codes become exact fp16 values (q4: q and 16 q; q8: q), scales apply in fp32 to the 16 x 16 results, and the min
//    term's sums of x' come from two MFMAs per group against a constant operand, already in the result layout.
//  * A workgroup with more items than one (a head's 262144 rows) loads the next item's records before it reduces this
//    one's, and keeps x'.
//  * A split of more than 2048 k is taken 2048 at a time; where its items leave CUs idle, those passes are slices of K
//    over workgroups, whose sums meet in the split-K workspace (the GEMV's protocol). 5 rows, one split: 64 x 8192
//    11.3 -> 7.0 us, 512 x 16384 17.0 -> 8.6, geglu 512 x 8192 17.9 -> 9.9 (before: the kernel that cut K over
//    workgroups for every call; without slices 14.5, 27.2 and 22.5).
// Bound: at the E2B shapes, one launch's chain (arguments, x, the split of x', the records, the reduction, the stores);
// for a head, HBM. Per launch, recorded over a ring of weights, 5 rows: q4 gate_up 2 x 8192 x 2048 11.1 us (18.4 before: x'
// staged in LDS by every workgroup, K split over two workgroups with partials in uncached memory), 3072 x 2048 6.7 (11.0),
// 2048 x 8192 in 4 splits 7.4 (13.4), 262144 x 2048 86 us = 3.9 TB/s (95); 16 rows: gate_up 12.2 (38.4). q8, where 4 waves a
// tile took one group after another on the VALU: 5120 x 1536 7.2 (52.4), geglu 6144 x 1536 10.0 (91.5), 16 rows 11.7
// (184). A ring that the last-level cache holds and one far past it read nearly alike: gate_up 11.2 over 168 MB, 11.0 over
// 672; q8 5120 x 1536 7.0 over 194 MB, 7.4 over 584. Relative L2 against float64: 1.2e-7 (q8; 3.8e-7 before), 1.7e-7 (q4;
// 1.9e-7).
// Tried: the min term as a product of its own on the matrix cores (half the fp32 FMAs): 5% faster for the head, 3% slower
// for the small ops, and its fp16 split of the group sums raised the error to 2.2e-7.
#include "gemvm.hpp"

namespace p0 {

typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));

// 8 codes (two words) of a q8 row as exact fp16 values: byte ^ 0x80 = q + 128 under the exponent of 1024, minus 1152
__device__ __forceinline__ half8_t codes_q8(uint32_t w0, uint32_t w1) {
  const h2_t k1152 = {(_Float16)1152.0f, (_Float16)1152.0f};
  const uint32_t w[2] = {w0 ^ 0x80808080u, w1 ^ 0x80808080u};
  u32x4l u;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    u[2 * i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04010400u)) - k1152);
    u[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04030402u)) - k1152);
  }
  return __builtin_bit_cast(half8_t, u);
}

// The arguments of a launch in K slices (a kernel without slices reads GmP alone)
struct GmSliceP : GmP {
  int nks, pps;                // K slices per split, over workgroups, and the passes of a slice
  float* part; unsigned* cnt;  // the slices' sums and the arrival counts (the split-K workspace)
};
template <bool SLICED> struct GmArgs { typedef GmP type; };
template <> struct GmArgs<true> { typedef GmSliceP type; };

// One launch: grid (workgroups, splits x K slices); workgroup pos takes items [pos ipw, (pos + 1) ipw) of its split. SLICED:
// p.nks > 1 slices of a split, one item per workgroup
template <int ENC, int NBK, bool GEGLU, bool PLEG, bool SLICED>
__global__ __launch_bounds__(kGmThreads) void gemvm_kernel(typename GmArgs<SLICED>::type p) {
  constexpr bool Q4 = ENC == P0_ENC_Q4G32A_T64;
  constexpr int GK = Q4 ? 32 : 64;             // k per group
  constexpr int RJ = Q4 ? 2 : 4;               // record loads per block and pass: quads of groups (q4), groups (q8)
  constexpr int U = GEGLU ? NBK / 2 : NBK;     // 16-row blocks of output rows per item
  __shared__ float red[2][kGmWaves][NBK][4][64];
  // per wave, in the order of its k: the norm weights (rms), or x' of four rows (pleg; kPlegRow apart: fewer bank conflicts)
  constexpr int kPlegRow = 256 + 32;
  __shared__ __attribute__((aligned(16))) float nws[kGmWaves][PLEG ? 4 * kPlegRow : 256];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, l16 = lane & 15, q = lane >> 4, m = min(l16, M - 1);
  const int pos = stage_pos(blockIdx.x, p.wgs);
  int split = blockIdx.y, ks = 0;
  if constexpr (SLICED) {
    split = (int)blockIdx.y / p.nks;
    ks = (int)blockIdx.y - split * p.nks;
  }
  const int it0 = pos * p.ipw, it1 = min(p.items, it0 + p.ipw);
  if (it0 >= it1) return;
  // the workgroup's k: its split, or its slice of it (none, for the last slices of a last split shorter than the others)
  int k0s = split * p.kPer, k1s = min(p.K, k0s + p.kPer);
  if constexpr (SLICED) {
    k0s += ks * p.pps * kGmPass;
    k1s = max(k0s, min(k1s, k0s + p.pps * kGmPass));
  }
  const int passes = (k1s - k0s + kGmPass - 1) / kGmPass;

  // weight row of block b of item it (a geglu's blocks U .. NBK - 1: the up rows)
  auto block_row = [&](int it, int b) { return (it * U + (GEGLU ? b % U : b)) * 16 + (GEGLU && b >= U ? p.N : 0); };
  // does this wave have records j of a pass of ng groups, and the groups they hold
  auto has = [&](int j, int ng) { return Q4 ? (wv + kGmWaves * j) * 4 < ng : wv + kGmWaves * j < ng; };

  // every load of a pass is issued whether the pass holds its groups or not (clamped into the split; what lies past it
  // gets scale and min 0, and A operands of 0): no branch keeps them apart, and a wave's loads share one base
  u32x4 rq[NBK][RJ];
  uint32_t rs[NBK][Q4 ? RJ : 1];
  auto load_records = [&](int it, int g0, int ng) {
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      const int row = block_row(it, b);
      const uint8_t* tb = p.w + ((int64_t)(row >> 6) * p.wG + g0) * (Q4 ? 1280 : 4224);
      const int r = (row & 63) + l16;
      if constexpr (Q4) {
#pragma unroll
        for (int j = 0; j < RJ; ++j) {
          const int g = (wv + kGmWaves * j) * 4 + q, off = min(g, ng - 1) * 1280;
          rq[b][j] = *P0_GLOBAL(const u32x4, tb + (unsigned)(off + r * 16));
          rs[b][j] = *P0_GLOBAL(const uint32_t, tb + (unsigned)(off + 1024 + r * 4));
        }
      } else {
#pragma unroll
        for (int j = 0; j < RJ; ++j)
          rq[b][j] = *P0_GLOBAL(const u32x4, tb + min(wv + kGmWaves * j, ng - 1) * 4224 + (unsigned)(r * 64 + q * 16));
        // the lane's quarter q holds the scale of the wave's record q
        rs[b][0] = *P0_GLOBAL(const uint16_t, tb + (unsigned)(min(wv + kGmWaves * q, ng - 1) * 4224 + 4096 + r * 2));
      }
    }
  };

  half8_t ahi[8], alo[8];     // this wave's x' of the pass: chunk c, 8 k of row l16 (q4: group 4 j + b of c = (j, b))
  f4_t sx[Q4 ? 8 : 1];        // q4: the groups' sums of x' in the result layout
  float dsc[4];               // 2^-e of x row 4 q + i, e the row's scale exponent
  // does the pass hold chunk c of this wave (the same for the whole wave: a chunk lies in one group)
  auto in_pass = [&](int c, int ng) {
    return Q4 ? (wv + kGmWaves * (c >> 2)) * 4 + (c & 3) < ng : wv + kGmWaves * (c >> 1) < ng;
  };
  // the wave's 256 k of a pass are RJ runs of RUN, run j at (wv + 8 j) RUN; chunk c holds k at + kl(c) + kq of its run
  constexpr int RUN = 256 / RJ, CR = 8 / RJ;
  const int kq = Q4 ? 8 * q : 16 * q;
  auto kl = [](int c) { return Q4 ? (c % CR) * 32 : 8 * (c % CR); };
  // the k a chunk's loads take (uniform): past the split the wave's first chunk again, whose x' set no other scale for the row
  auto at_k = [&](int c, int ng) {
    return in_pass(c, ng) ? (wv + kGmWaves * (c / CR)) * RUN + kl(c) : in_pass(0, ng) ? wv * RUN : 0;
  };
  u32x4 xv[8][2], nv;
  float rstd = 1.0f;
  const bool rms = p.pro == P0_PRO_RMS;
  // x' in two halves, so that the records' loads go out between them: a wave's loads return in order, and the split of
  // x' overlaps the records' latency
  auto issue_x = [&](int kp, int ng) {
    if constexpr (!PLEG) {
      const float* xr = p.X + m * p.ldx + kp + kq;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        xv[c][0] = *P0_GLOBAL(const u32x4, xr + at_k(c, ng));
        xv[c][1] = *P0_GLOBAL(const u32x4, xr + at_k(c, ng) + 4);
      }
      if (rms) {
        // the lane's 4 of the wave's 256 norm weights (every lane of a quarter needs the same 64: they go through LDS)
        const int nk = (wv + kGmWaves * (lane * 4 / RUN)) * RUN + lane * 4 % RUN;
        rstd = *P0_GLOBAL(const float, p.ST + m * p.statLd);
        nv = *P0_GLOBAL(const u32x4, p.NW + kp + min(nk, ng * GK - 4));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto finish_x = [&](int kp, int ng) {
    float v[8][8];
    if constexpr (PLEG) {
      // Two ways to x' = gelu(sum of partials) ev, whose arithmetic is most of a small call. Few rows: the lanes take 4 of the
      // wave's 256 k each, four rows at a time, and hand x' round through LDS, so that each is worked out once (4 M gelus a
      // lane). Many rows, or few k: each lane its own operands', chunk by chunk (8 per chunk that the pass holds, 16 / M
      // times over). The line is where their counts meet, less the first one's round trips: 2048 x 256 (4 chunks), 16 rows
      // 12.1 us / 7.7, 8 rows 7.9 / 7.5, 3 rows 5.4 / 7.5; 2048 x 2048 (8 chunks), 16 rows 15.3 / 15.1, 8 rows 10.4 / 14.5
      if (M <= 8 && in_pass(M - 1, ng)) {
        const int nk = kp + min((wv + kGmWaves * (lane * 4 / RUN)) * RUN + lane * 4 % RUN, ng * GK - 4);
        for (int r0 = 0; r0 < M; r0 += 4) {
          u32x4 ev[4];
          float t[4][4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            ev[i] = *P0_GLOBAL(const u32x4, p.EV + min(r0 + i, M - 1) * p.evLd + nk);
#pragma unroll
            for (int e = 0; e < 4; ++e) t[i][e] = 0.0f;
          }
          for (int j = 0; j < p.nsrc; ++j) {
            u32x4 y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = *P0_GLOBAL(const u32x4, p.X + j * p.ldp + min(r0 + i, M - 1) * p.ldx + nk);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) t[i][e] += __uint_as_float(y[i][e]);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // as for nws below
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (r0 + i < M) {
              float4 f;
              f.x = gelu_tanh(t[i][0]) * __uint_as_float(ev[i].x);
              f.y = gelu_tanh(t[i][1]) * __uint_as_float(ev[i].y);
              f.z = gelu_tanh(t[i][2]) * __uint_as_float(ev[i].z);
              f.w = gelu_tanh(t[i][3]) * __uint_as_float(ev[i].w);
              *(float4*)(nws[wv] + i * kPlegRow + lane * 4) = f;
            }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
          if (m >= r0 && m < r0 + 4)
#pragma unroll
            for (int c = 0; c < 8; ++c) {
              const float* xr = nws[wv] + (m - r0) * kPlegRow + (in_pass(c, ng) ? (c / CR) * RUN + kl(c) : 0) + kq;
              const float4 x0 = *(const float4*)xr, x1 = *(const float4*)(xr + 4);
              v[c][0] = x0.x; v[c][1] = x0.y; v[c][2] = x0.z; v[c][3] = x0.w;
              v[c][4] = x1.x; v[c][5] = x1.y; v[c][6] = x1.z; v[c][7] = x1.w;
            }
        }
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[c][e] = 0.0f;
          if (!in_pass(c, ng)) continue;
          const int k = kp + at_k(c, ng) + kq;
          for (int j = 0; j < p.nsrc; ++j) {
            const float* xr = p.X + j * p.ldp + m * p.ldx + k;
            const u32x4 x0 = *P0_GLOBAL(const u32x4, xr), x1 = *P0_GLOBAL(const u32x4, xr + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[c][e] += __uint_as_float(x0[e]);
              v[c][e + 4] += __uint_as_float(x1[e]);
            }
          }
          const float* ev = p.EV + m * p.evLd + k;
          const u32x4 e0 = *P0_GLOBAL(const u32x4, ev), e1 = *P0_GLOBAL(const u32x4, ev + 4);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[c][e] = gelu_tanh(v[c][e]) * __uint_as_float(e < 4 ? e0[e & 3] : e1[e & 3]);
        }
      }
    } else {
      if (rms) {
        // a wavefront fence on each side keeps the compiler from moving the reads above other lanes' writes (the LDS
        // serves one wave's accesses in order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        *(u32x4l*)(nws[wv] + lane * 4) = u32x4l(nv);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] = __uint_as_float(xv[c][e >> 2][e & 3]);
        if (rms) {
          const float* nr = nws[wv] + (in_pass(c, ng) ? (c / CR) * RUN + kl(c) : 0) + kq;   // as at_k
          const float4 n0 = *(const float4*)nr, n1 = *(const float4*)(nr + 4);
          const float n[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) v[c][e] = v[c][e] * rstd * n[e];
        }
      }
    }
    // the row's largest |x'| over the wave's k (the lanes of a row are 16 apart): an infinity makes it infinite, a NaN
    // stays out of it
    float big = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int e = 0; e < 8; e += 2) big = fmaxf(fmaxf(big, __builtin_fabsf(v[c][e])), __builtin_fabsf(v[c][e + 1]));
    auto over_row = [](float b) {
      const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(b), __float_as_uint(b), false, false);
      b = fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
      const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(b), __float_as_uint(b), false, false);
      return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
    };
    big = over_row(big);
    const bool inf = __builtin_amdgcn_ballot_w64(big == __builtin_inff()) != 0;
    if (inf) {   // some row holds an infinity: every row's largest finite |x'|
      big = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a = __builtin_fabsf(v[c][e]);
          big = fmaxf(big, a < __builtin_inff() ? a : 0.0f);
        }
      big = over_row(big);
    }
    const int ex = (int)((__float_as_uint(big) >> 23) & 255u) - 127;   // floor(log2 big); -127 for 0 and subnormals
    const int e = min(14 - ex, 126);
    const float sc = __uint_as_float((uint32_t)(e + 127) << 23), sc16 = sc * 0.0625f;
#pragma unroll
    for (int i = 0; i < 4; ++i) dsc[i] = __uint_as_float((uint32_t)(127 - __shfl(e, 4 * q + i, 64)) << 23);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
      for (int e8 = 0; e8 < 8; ++e8) {
        // q4: the code word's nibble order, k 0, 4, 1, 5, 2, 6, 3, 7, odd k scaled 1/16 (their codes come as 16 q).
        // hi and lo are one v_fma_mixlo / mixhi each: fp16(x' 2^e), then fp16 of what that leaves (exact in the fma)
        const int ks = Q4 ? (e8 >> 1) + 4 * (e8 & 1) : e8;
        const float s = Q4 && (ks & 1) ? sc16 : sc;
        const _Float16 hi = (_Float16)__builtin_fmaf(v[c][ks], s, 0.0f);
        ahi[c][e8] = hi;
        alo[c][e8] = (_Float16)__builtin_fmaf(v[c][ks], s, -(float)hi);
      }
      if (!in_pass(c, ng)) ahi[c] = alo[c] = half8_t{};
    }
    if (inf) {   // an infinite x' has no rest (inf - inf would turn it into a NaN)
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int e8 = 0; e8 < 8; ++e8)
          if (__builtin_fabsf((float)ahi[c][e8]) == __builtin_inff()) alo[c][e8] = (_Float16)0.0f;
    }
    if constexpr (Q4) {
      const _Float16 o = (_Float16)1.0f, s = (_Float16)16.0f;
      const half8_t ones = {o, o, s, s, o, o, s, s};
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        sx[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[c], ones, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        sx[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[c], ones, sx[c], 0, 0, 0);
      }
    }
  };
  // the item's sums over this wave's records of a pass, scaled back
  auto consume = [&](int ng, float (&tot)[NBK][4]) {
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if constexpr (Q4) {
#pragma unroll
        for (int j = 0; j < RJ; ++j)
          if (has(j, ng)) {
            const uint32_t sm = (wv + kGmWaves * j) * 4 + q < ng ? rs[b][j] : 0u;   // past the split: contributes 0
            uint32_t qb[4] = {rq[b][j].x, rq[b][j].y, rq[b][j].z, rq[b][j].w};
            uint32_t sb[4] = {sm, sm, sm, sm};
            quarter_transpose(qb);
            quarter_transpose(sb);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              const int c = j * 4 + g;
              const half8_t bq = codes_b(qb[g]);
              f4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[c], bq, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[c], bq, d, 0, 0, 0);
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[i] = __builtin_fmaf(h2f_lo(sb[g]), d[i], __builtin_fmaf(h2f_hi(sb[g]), sx[c][i], acc[i]));
            }
          }
      } else {
        uint32_t sb[4] = {rs[b][0], rs[b][0], rs[b][0], rs[b][0]};
        quarter_transpose(sb);
#pragma unroll
        for (int j = 0; j < RJ; ++j)
          if (has(j, ng)) {
            const half8_t b0 = codes_q8(rq[b][j].x, rq[b][j].y), b1 = codes_q8(rq[b][j].z, rq[b][j].w);
            f4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[2 * j], b0, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[2 * j + 1], b1, d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[2 * j], b0, d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[2 * j + 1], b1, d, 0, 0, 0);
            const float s = h2f_lo(sb[j]);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(s, d[i], acc[i]);
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) tot[b][i] = __builtin_fmaf(acc[i], dsc[i], tot[b][i]);
    }
  };

  // where slice s of this workgroup's item keeps the sum of x row mm, row l16 of block b (h = 1: a geglu's up row)
  auto slice_at = [&](int s, int mm, int b, int h) -> float* {
    if constexpr (SLICED)
      return p.part + ((((int64_t)(split * p.items + it0) * p.nks + s) * (GEGLU ? 2 : 1) + h) * M * U + mm * U + b) * 16 + l16;
    return nullptr;
  };
  auto slice_store = [&](int mm, int b, float v0, float v1) {
    stf<true>(slice_at(ks, mm, b, 0), v0);
    if (GEGLU) stf<true>(slice_at(ks, mm, b, 1), v1);
  };
  auto pass_groups = [&](int ps) { return min(k1s - (k0s + ps * kGmPass), kGmPass) / GK; };
  for (int it = it0; it < it1; ++it) {
    float tot[NBK][4];
#pragma unroll
    for (int b = 0; b < NBK; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) tot[b][i] = 0.0f;
    for (int ps = 0; ps < passes; ++ps) {
      const int g0 = (k0s + ps * kGmPass) / GK;
      // one pass: x' stays for every item, and its records were loaded before the last item's reduction
      if (passes > 1 || it == it0) {
        issue_x(k0s + ps * kGmPass, pass_groups(ps));
        load_records(it, g0, pass_groups(ps));
        __builtin_amdgcn_sched_barrier(0);
        finish_x(k0s + ps * kGmPass, pass_groups(ps));
      }
      consume(pass_groups(ps), tot);
    }
    if (passes == 1 && it + 1 < it1) load_records(it + 1, k0s / GK, pass_groups(0));
    float (*rd)[NBK][4][64] = red[(it - it0) & 1];   // the other half is still read by slower waves
#pragma unroll
    for (int b = 0; b < NBK; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) rd[wv][b][i][lane] = tot[b][i];
    __syncthreads();
    // thread -> (x row, block of output rows, row of 16), 32 / U x rows a round; a softcap's wave takes a whole tile of
    // one x row. The waves' sums are added in wave order
    for (int r = tid >> 4; r < M * U; r += kGmThreads / 16) {
      const int mm = r / U, b = r - mm * U, at = (mm >> 2) * 16 + l16;
      float v0 = 0.0f, v1 = 0.0f;
#pragma unroll
      for (int w = 0; w < kGmWaves; ++w) v0 += rd[w][b][mm & 3][at];
      if (GEGLU) {
#pragma unroll
        for (int w = 0; w < kGmWaves; ++w) v1 += rd[w][NBK - U + b][mm & 3][at];
      }
      const int n = (it * U + b) * 16 + l16;
      if (SLICED) slice_store(mm, b, v0, v1);
      else epilogue<false>(p, split, mm, n >> 6, n & 63, v0, v1);
    }
  }
  if constexpr (SLICED) {
    // the last of an item's slices to arrive adds their sums in slice order. The workspace
    // is uncached memory: a store is in memory once acknowledged, so the arrival count needs no fence
    __shared__ int s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
      auto* c = P0_GLOBAL(unsigned, p.cnt + split * p.items + it0);
      s_last = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(p.nks - 1);
      if (s_last) __hip_atomic_exchange(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // leave it at zero
    }
    __syncthreads();
    if (!s_last) return;
    for (int r = tid >> 4; r < M * U; r += kGmThreads / 16) {
      const int mm = r / U, b = r - mm * U, n = (it0 * U + b) * 16 + l16;
      float v[2] = {0.0f, 0.0f};
      for (int s0 = 0; s0 < p.nks; s0 += 8) {   // 8 slices in flight; past the last: the last again, not added
        float t[8][GEGLU ? 2 : 1];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int h = 0; h < (GEGLU ? 2 : 1); ++h) t[u][h] = ldf<true>(slice_at(min(s0 + u, p.nks - 1), mm, b, h));
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (s0 + u < p.nks)
#pragma unroll
            for (int h = 0; h < (GEGLU ? 2 : 1); ++h) v[h] += t[u][h];
      }
      epilogue<false>(p, split, mm, n >> 6, n & 63, v[0], v[1]);
    }
  }
}

// Splits of several passes: a slice of whole passes per workgroup, as many slices as leave every workgroup one item and a CU
// of its own
static GmSliceP slice_plan(const GemvP& p, const GmPlan& pl) {
  GmSliceP g{};
  (GmP&)g = pl.args;
  const int passes = (min(p.kPer, p.K) + kGmPass - 1) / kGmPass, wgs = g.items * p.nsplit;
  const int most = wgs <= 256 ? 256 / wgs : 1;   // gm_plan gives a workgroup more items than one only past 256
  g.pps = (passes + most - 1) / most;
  g.nks = (passes + g.pps - 1) / g.pps;
  g.part = ctx().part;      // at most 256 workgroups' 16 x 64 sums (a geglu's 16 x 32 twice): 1 MiB of its 64
  g.cnt = ctx().counters;   // nsplit * items <= 256
  return g;
}

template <int ENC, bool SLICED>
static void launch_form(const GemvP& p, const GmPlan& pl, dim3 grid, const typename GmArgs<SLICED>::type& g, hipStream_t s) {
  const bool geglu = p.epi == P0_EPI_GEGLU, pleg = p.pro == P0_PRO_PLEG;
#define P0_GM(NBK, GEGLU) (pleg ? gemvm_kernel<ENC, NBK, GEGLU, true, SLICED> : gemvm_kernel<ENC, NBK, GEGLU, false, SLICED>)
  auto k = geglu ? (pl.nbk == 4 ? P0_GM(4, true) : P0_GM(2, true))
                 : pl.nbk == 4 ? P0_GM(4, false) : pl.nbk == 2 ? P0_GM(2, false) : P0_GM(1, false);
#undef P0_GM
  hipLaunchKernelGGL(k, grid, dim3(kGmThreads), 0, s, g);
}
template <int ENC>
static void launch_enc(const GemvP& p, hipStream_t s) {
  const GmPlan pl = gm_plan(p, 512);
  const GmSliceP g = slice_plan(p, pl);
  if (g.nks > 1) launch_form<ENC, true>(p, pl, dim3(pl.grid.x, pl.grid.y * g.nks), g, s);
  else launch_form<ENC, false>(p, pl, pl.grid, pl.args, s);
}

// q4 calls of few rows that gemv.hip's fp32 kernel (x' staged once a workgroup, K over workgroups) runs faster. The line was
// taken where both were measured; per recorded launch, us here / there:
//  * short splits of many blocks leave most of a workgroup's waves without records. 2 rows: 16384 x 256 6.4 / 5.4, x 512 6.6 /
//    6.1, x 1024 7.4 / 7.4, geglu 16384 x 640 10.6 / 8.7, 2048 x 8192 in splits of 512 8.4 / 7.3, 4096 x 256 (256 blocks) 5.0
//    / 5.0, 64 x 64 4.6 / 4.0; 3 rows: 16384 x 256 6.5 / 6.1, x 512 6.6 / 6.9, geglu 16384 x 640 10.7 / 10.1; 4 rows: 512 x 8192
//    in 64 splits 8.2 / 6.8, 16384 x 256 6.5 / 7.0;
//  * long splits whose passes do not all get a workgroup of their own. 2 rows: 4096 x 8192 16.3 / 12.4, 2048 x 16384 17.6 /
//    12.7, 2048 x 4096 (one pass each) 7.8 / 8.5, 8192 x 8192 20.3 / 19.4, 8192 x 16384 36.6 / 45.1, geglu 8192 x 4096 17.9 /
//    16.8; 3 rows: 4096 x 8192 16.7 / 15.8, 2048 x 4096 7.8 / 9.6; a softcap's items of whole tiles: 2 rows 2048 x 2560 11.5 /
//    9.6, 16384 x 2560 15.2 / 16.3, 3 rows 256 x 2560 10.9 / 9.8.
bool gemvm_takes(const GemvP& p) {
  const int M = p.mrows, geglu = p.epi == P0_EPI_GEGLU;
  if (p.enc == P0_ENC_Q8G64S_T64 || M > 5) return true;
  const int64_t rows = (int64_t)(p.N / 16) * (geglu ? 2 : 1), blocks = rows * p.nsplit;
  if (p.kPer > kGmPass) {
    if (M > 3) return true;
    if (p.epi == P0_EPI_SOFTCAP) return rows > 256;
    if (geglu) return M == 3 || rows > 1024;
    return rows > 256 || blocks * ((p.kPer + kGmPass - 1) / kGmPass) <= 256 || (M == 3 && p.kPer <= 4096);
  }
  if (M == 2) return p.kPer > 64 && (p.kPer > 640 || blocks < 512);
  if (M == 3) return p.kPer > (geglu ? 640 : 256) || blocks < 512;
  return p.kPer > 256 || p.nsplit < 32;
}

void launch_gemvm(const GemvP& p, hipStream_t s) {
  if (p.enc == P0_ENC_Q4G32A_T64) launch_enc<P0_ENC_Q4G32A_T64>(p, s);
  else launch_enc<P0_ENC_Q8G64S_T64>(p, s);
}

}  // namespace p0
