// gemm_n128.hip - the q4g32a.t64 dequant-GEMM in tiles of 128 x 128 outputs (engine/ops/gemm.js:255-322, as gemm.hip),
// for calls whose 256 x 256 tiles would leave most CUs idle: prompt chunks, text streams, small images.
//
//  * K runs in steps of 64 (two q4 groups). X' rows and the raw weight records go to LDS by LDS-DMA, S - 1 steps ahead,
//    written in asm: the compiler, which takes an LDS-DMA load for a pending write of all LDS, would wait for every one in
//    flight before each LDS read. The loads are waited for by count; one barrier a step.
//  * While a step's MFMAs run, the workgroup dequantises the next step's weights from the raw records in LDS into the other
//    of two fp16 tiles, each weight once per workgroup.
//  * When the tiles alone do not fill the chip, K is cut into slices over workgroups: fp32 partial tiles in the uncached
//    split-K workspace, an arrival count per tile, the last workgroup adds the slices in order (the GEMV's protocol).
//  * The epilogue goes through LDS, row by row: 4 consecutive outputs a thread.
// Bound: a step's chain of LDS round trips (records, fragments, the W tile) and its barrier, about 1.0 us for the 0.24 us of
// its MFMAs, with two waves per SIMD to cover for each other; with K slices, the partials through uncached memory.
// Tried on these calls (M = 256, 3072 x 2048; M = 512, 3072 x 9216): weights dequantised straight into the B registers of
// waves that hold all rows of a 64 x 128 tile, no W tile in LDS (19 and 86 us: each weight is dequantised M / 64 times,
// which bounds it from M = 512 on; M = 256, 16384 x 2048 41 against 36); tiles of 256 x 128 (28, 84) and 256 x 256 (44, 76)
// in this form; whole GEMMs at M = 4608 with 256 x 256 tiles in this form (800-890 TFLOP/s) and over a W dequantised
// once (750-960 against 800-990 of gemm.hip, with X' and W by LDS-DMA and two wave groups taking turns).
#include "gemm_common.hpp"

namespace p0 {

// 64 lanes x 16 bytes, buffer resource + lane offset + scalar offset -> LDS at dst + 16 lane
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void dma16(uint32_t dst, int voff, i32x4 rsrc, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(dst), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
__device__ __forceinline__ i32x4 resource(const void* b) {   // raw, no bounds of its own
  const uint64_t a = (uint64_t)(uintptr_t)b;
  return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)a), __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)), -1,
               0x00020000};
}
template <int N>
__device__ __forceinline__ void wait_dma() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

constexpr int kBand = 4;
struct N128P {
  GemmP g;
  int nks, spk;          // K slices, steps per slice
  float* part; unsigned* cnt;
};

template <int WM, int WN, int NT, int S>
struct Shape {
  static constexpr int NW = WM * WN, BMt = 64 * WM, BNt = 32 * WN * NT, Threads = 64 * NW;
  static constexpr int XBytes = BMt * 128, CBytes = 2 * BNt * 16, SBytes = 2 * BNt * 4;   // a step's X', codes, scales
  static constexpr int RBytes = CBytes + SBytes, WBytes = BNt * 128;
  static constexpr int XI = XBytes / 1024 / NW, CL = CBytes / 1024, SL = SBytes / 1024;   // X loads per wave; all code, scale loads
  static constexpr int CI = (CL + NW - 1) / NW, NL = XI + CI + 1;                         // code loads, loads per wave and step
  static constexpr int WPT = 8 * BNt / Threads;                                           // code words a thread dequantises
  static constexpr int Main = S * (XBytes + RBytes) + 2 * WBytes, Pad = BNt + 4;
  static constexpr int Lds = Main > 64 * Pad * 4 ? Main : 64 * Pad * 4;
};

template <int WM, int WN, int NT, int S>
__global__ __launch_bounds__(64 * WM * WN) void n128_kernel(N128P a) {
  using C = Shape<WM, WN, NT, S>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];   // [S] X' | [S] raw records | [2] W tile
  __shared__ int s_last;
  const GemmP& p = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / WN, wn = wv % WN;
  const int nbx = (p.N + C::BNt - 1) / C::BNt, nby = (p.M + C::BMt - 1) / C::BMt, T = nbx * nby * a.nks;
  // consecutive workgroups go to the 8 XCDs in turn: each XCD takes a contiguous run of tiles. The run goes down kBand row
  // tiles, then on to the next column tile (and slice): what an XCD's CUs work on at one time is a block of a few row
  // tiles (X' rows, 2 bytes a value, shared by the block's columns) by many column tiles (weights, 0.625 bytes)
  int t = blockIdx.x;
  if (T % 8 == 0) t = (blockIdx.x % 8) * (T / 8) + blockIdx.x / 8;
  const int per = nbx * a.nks * kBand, band = t / per, rows = min(kBand, nby - band * kBand), in = t - band * per;
  const int mb = band * kBand + in % rows, cs = in / rows, ks = cs % a.nks, nb = cs / a.nks;
  const int m0 = mb * C::BMt, n0 = nb * C::BNt;
  const int nsteps = (p.K + 63) / 64;
  const int s0 = ks * a.spk, s1 = min(nsteps, s0 + a.spk);

  float16v acc[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // ---- sources. Rows of X' and of the W tile are 128 bytes; the 16-byte chunk c of row r sits at position c ^ key(r), so
  // that 16 consecutive rows hold one chunk in 16 different (row parity, position) pairs: no bank conflicts
  auto key = [](int r) { return (r ^ ((r >> 3) & 3)) & 7; };
  const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const i32x4 rx = resource(p.x + (int64_t)m0 * p.ldx);
  int xv[C::XI], xup[C::XI];   // byte offsets; 64 for chunks 4 .. 7
#pragma unroll
  for (int i = 0; i < C::XI; ++i) {
    const int r = (wv * C::XI + i) * 8 + (lane >> 3), c = (lane & 7) ^ key(r);
    xv[i] = min(r, p.M - 1 - m0) * (int)p.ldx * 2 + c * 16;   // rows past M repeat the last one (never stored)
    xup[i] = (c & 4) * 16;
  }
  // W: column slot c of the tile is weight row wr0 + n0 + c; a swiglu's first half of the slots are the gate rows of
  // outputs n0 / 2 + c, the second half their up rows. Every 64 slots are a whole 64-row tile of the weight
  const bool sw = p.epi == P0_GEPI_SWIGLU;
  constexpr int HB = C::BNt / 64;
  auto base64 = [&](int h) {   // records of slots 64 h .. 64 h + 63; columns past N take the weight's last tile
    int64_t tile = sw ? (((h >= HB / 2 ? p.wr1 : p.wr0) + n0 / 2) >> 6) + h % (HB / 2) : ((p.wr0 + n0) >> 6) + h;
    const int64_t last = (p.Nw >> 6) - 1;
    if (tile > last) tile = last;
    return p.w + (tile * p.wG + (p.wk0 >> 5)) * 1280;
  };
  const int odd = p.K & 32;   // the last step has one group
  i32x4 rc[C::CI];
  int cg[C::CI], cd[C::CI];
#pragma unroll
  for (int i = 0; i < C::CI; ++i) {   // codes: a load takes 64 slots of one group; a wave without one repeats another's
    const int q = (wv * C::CI + i) % C::CL;
    cg[i] = q / HB;
    cd[i] = q * 1024;
    rc[i] = resource(base64(q % HB));
  }
  // scales: [group][slot] words, 4 slots a lane; wave wv takes load wv % SL (every wave's loads count alike)
  const int sl = (wv % C::SL) * 256 + lane * 4, sg = sl / C::BNt;
  const uint8_t* const w00 = p.w + (p.wk0 >> 5) * 1280;
  const i32x4 rs = resource(w00);
  const int sv = (int)(base64(sl % C::BNt / 64) - w00) + 1024 + (sl % 64) * 4;
  // steps past the call's last one repeat it (every step's loads count alike; not used), and where the last step has one
  // group only, what belongs to the other re-reads this one
  auto issue_x = [&](int st) {
    const uint32_t d = lbase + (st % S) * C::XBytes + wv * (C::XI * 1024);
    const int sc = min(st, nsteps - 1), so = sc * 128;
    if (odd && sc == nsteps - 1) {
#pragma unroll
      for (int i = 0; i < C::XI; ++i) dma16(d + i * 1024, xv[i] - xup[i], rx, so);
    } else {
#pragma unroll
      for (int i = 0; i < C::XI; ++i) dma16(d + i * 1024, xv[i], rx, so);
    }
  };
  auto issue_w = [&](int st) {
    const uint32_t d = lbase + S * C::XBytes + (st % S) * C::RBytes;
    const int sc = min(st, nsteps - 1);
    const bool one = odd && sc == nsteps - 1;
#pragma unroll
    for (int i = 0; i < C::CI; ++i) dma16(d + cd[i], lane * 16, rc[i], (sc * 2 + (one ? 0 : cg[i])) * 1280);
    dma16(d + C::CBytes + (wv % C::SL) * 1024, sv + (one ? 0 : sg * 1280), rs, sc * 2560);
  };
  // ---- dequant of step st's records into W tile st & 1: thread -> slot tid % BNt, words WPT (tid / BNt) .. of its 8
  const int dslot = tid % C::BNt, dw = tid / C::BNt * C::WPT, dg = dw >> 2;   // two words: one group
  const int dkey = key(dslot);
  uint32_t w[C::WPT], sm;
  auto read_raw = [&](int st) {
    const uint8_t* rw = lds + S * C::XBytes + (st % S) * C::RBytes;
    const uint2 v = *(const uint2*)(rw + dg * (C::BNt * 16) + dslot * 16 + (dw & 3) * 4);
    w[0] = v.x;
    w[1] = v.y;
    sm = *(const uint32_t*)(rw + C::CBytes + dg * (C::BNt * 4) + dslot * 4);
  };
  auto write_w = [&](int st, const u32x4n (&d)[C::WPT]) {
    uint8_t* wt = lds + S * (C::XBytes + C::RBytes) + (st & 1) * C::WBytes + dslot * 128;
#pragma unroll
    for (int i = 0; i < C::WPT; ++i) *(u32x4n*)(wt + (((dw + i) ^ dkey) << 4)) = d[i];
  };
  auto fix = [&](int st) {   // rare: q s + m may round in fp32 already
    if (__builtin_amdgcn_ballot_w64(!pk_exact(sm)) != 0) {
      u32x4n d[C::WPT];
#pragma unroll
      for (int i = 0; i < C::WPT; ++i) d[i] = deq_word(w[i], sm, false);
      if (!pk_exact(sm)) write_w(st, d);
    }
  };
  static_assert(C::WPT == 2, "two code words of one group per thread");

  const int hh = lane >> 5, frow = lane & 31, fkey = key(frow);
  u32x4n av[2][2], bv[2][NT];
  auto frag = [&](int st, int q) {
    const uint8_t* xs = lds + (st % S) * C::XBytes + (wm * 64 + frow) * 128;
    const uint8_t* ws = lds + S * (C::XBytes + C::RBytes) + (st & 1) * C::WBytes + (wn * (32 * NT) + frow) * 128;
    const int c = ((2 * q + hh) ^ fkey) << 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) av[q & 1][i] = *(const u32x4n*)(xs + i * 4096 + c);
#pragma unroll
    for (int j = 0; j < NT; ++j) bv[q & 1][j] = *(const u32x4n*)(ws + j * 4096 + c);
  };
  auto mfma = [&](int q) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, av[q & 1][i]), __builtin_bit_cast(half8, bv[q & 1][j]),
                                                           acc[i][j], 0, 0, 0);
  };
  auto bar = [&] {   // this wave's LDS accesses are done; every wave is here
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // W runs one step ahead of X': step st issues X'(st + S - 1) and W(st + S), reads X'(st) and dequantises W(st + 1)
  issue_w(s0);
#pragma unroll
  for (int j = 0; j < S - 1; ++j) {
    issue_x(s0 + j);
    issue_w(s0 + j + 1);
  }
  wait_dma<(S - 2) * C::NL>();   // X'(s0), W(s0), W(s0 + 1)
  bar();
  {
    read_raw(s0);
    u32x4n d[C::WPT];
#pragma unroll
    for (int i = 0; i < C::WPT; ++i) d[i] = deq_word(w[i], sm, true);
    write_w(s0, d);
    fix(s0);
  }
  bar();
  for (int st = s0; st < s1; ++st) {
    issue_x(st + S - 1);           // into the buffer step st - 1 read
    issue_w(st + S);               // into the one whose records step st - 1 dequantised
    read_raw(st + 1);
    frag(st, 0);
    u32x4n d[C::WPT];
    // the dequant's arithmetic between the MFMAs; its stores last, behind the step's fragment reads
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < 3) frag(st, q + 1);
      if (q < 2 || !odd || st < nsteps - 1) mfma(q);   // K % 64 = 32: the last step has one group
#pragma unroll
      for (int i = q * C::WPT / 4; i < (q + 1) * C::WPT / 4; ++i) d[i] = deq_word(w[i], sm, true);
      __builtin_amdgcn_sched_barrier(0);
    }
    write_w(st + 1, d);
    fix(st + 1);
    wait_dma<(S - 2) * C::NL>();   // X'(st + 1), W(st + 2)
    bar();
  }
  wait_dma<0>();
  bar();

  if (a.nks > 1) {
    // fp32 partials, two registers of a lane at a time (consecutive lanes, consecutive 8 bytes). The workspace is uncached:
    // a store is in memory once acknowledged, and device-scope loads read memory, so the arrival count needs no fence
    typedef unsigned long long u64;
    constexpr int E = C::BMt * C::BNt / 2;
    const int64_t tile = (int64_t)nb * nby + mb;
    u64* mine = (u64*)a.part + (tile * a.nks + ks) * E + wv * (NT * 1024) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float lo = acc[i][j][2 * e], hi = acc[i][j][2 * e + 1];
          const u64 v = (u64)__float_as_uint(lo) | (u64)__float_as_uint(hi) << 32;
          __hip_atomic_store(mine + ((i * NT + j) * 8 + e) * 64, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
      unsigned* c = a.cnt + tile;
      const unsigned prev = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last_in = prev == (unsigned)(a.nks - 1);
      if (last_in) __hip_atomic_exchange(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // leave it at zero
      s_last = last_in;
    }
    __syncthreads();
    if (!s_last) return;
    const u64* all = (const u64*)a.part + tile * a.nks * E + wv * (NT * 1024) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {   // slices in order, 32 loads in flight
        float16v v;
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = 0.0f;
        for (int s = 0; s < a.nks; s += 4) {
          u64 w[4][8];
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e)
              w[u][e] = __hip_atomic_load(all + (int64_t)min(s + u, a.nks - 1) * E + ((i * NT + j) * 8 + e) * 64, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (s + u < a.nks)
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                v[2 * e] += __uint_as_float((uint32_t)w[u][e]);
                v[2 * e + 1] += __uint_as_float((uint32_t)(w[u][e] >> 32));
              }
        }
        acc[i][j] = v;
      }
  }

  // ---- epilogues (engine/ops/gemm.js:187-250), 64 rows (a row of waves) at a time through LDS. acc[i][j][e] is row
  // 32 i + 8 (e / 4) + 4 (lane / 32) + e % 4, column 32 j + lane % 32 of the wave; then a thread takes 4 consecutive columns (a swiglu: 2 outputs) of a row
  float* tl = (float*)lds;   // [64][Pad]
  constexpr int TPR = C::BNt / 4, RPR = C::Threads / TPR;   // threads per row, rows per round
  const int l = tid & (TPR - 1), l32 = l & 31, r0 = tid / TPR;
  const int n = n0 + 4 * l, jn = n0 / 2 + 2 * l;
  const int hd = n >> 7, sec = hd < p.hq ? 0 : hd < p.hq + p.hkv ? 1 : 2;   // heads
  const bool heads = p.epi == P0_GEPI_HEADS;
  const int nc = sw ? min(2, p.N / 2 - jn) : min(4, p.N - n);               // this thread's columns (<= 0: none)
  // per-column vectors. heads: g4 = norm weights; resadd: gate, bias; bias: bias; swiglu: b4 = gate and up biases
  float g4[4] = {1.0f, 1.0f, 1.0f, 1.0f}, b4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (sw) {
      if (p.bv && (c & 1) < nc) b4[c] = p.bv[p.bvOff + (c >> 1) * p.bvUp + jn + (c & 1)];
    } else if (c < nc) {
      if (heads) {
        if (sec < 2) g4[c] = p.ev[p.evOff + (sec ? 128 : 0) + 4 * l32 + c];
      } else if (p.epi == P0_GEPI_RESADD) {
        if (p.ev) g4[c] = p.ev[p.evOff + n + c];
        if (p.bv) b4[c] = p.bv[p.bvOff + n + c];
      } else if (p.epi == P0_GEPI_BIAS) {
        b4[c] = p.ev[p.evOff + n + c];
      }
    }
  }
  const bool f32 = p.epi == P0_GEPI_F32 || p.epi == P0_GEPI_RESADD;
  const bool add = (p.epi == P0_GEPI_RESADD && !p.store) || (p.epi == P0_GEPI_BIAS && p.res);
  for (int ib = 0; ib < WM; ++ib) {
    if (ib) __syncthreads();
    if (wm == ib) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            tl[(32 * i + 8 * (e >> 2) + 4 * hh + (e & 3)) * C::Pad + wn * (32 * NT) + 32 * j + frow] = acc[i][j][e];
    }
    __syncthreads();
    for (int r = r0; r < 64; r += RPR) {
      const int m = m0 + 64 * ib + r;
      if (m >= p.M) break;
      if (nc <= 0) continue;   // whole heads together
      if (sw) {
        const float2 g = *(const float2*)(tl + r * C::Pad + 2 * l), u = *(const float2*)(tl + r * C::Pad + C::BNt / 2 + 2 * l);
        const float y0 = act_f(p, g.x + b4[0]) * (u.x + b4[2]), y1 = act_f(p, g.y + b4[1]) * (u.y + b4[3]);
        _Float16* yp = (_Float16*)p.y + (int64_t)m * p.ldy + p.ny0 + jn;
        if (nc == 2 && ((uintptr_t)yp & 3) == 0) *(uint32_t*)yp = pack_h2(y0, y1);
        else {
          yp[0] = to_h(y0);
          if (nc == 2) yp[1] = to_h(y1);
        }
        continue;
      }
      const float4 f = *(const float4*)(tl + r * C::Pad + 4 * l);
      float v[4] = {f.x, f.y, f.z, f.w};
      if (heads) {   // 32 lanes hold a row of one head
        if (sec < 2) {
          float ss = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
#pragma unroll
          for (int o = 16; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
          const float inv = 1.0f / sqrtf(ss / 128.0f + p.heps);
          float w[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) w[c] = v[c] * inv * g4[c];
          const float* rt = p.rope + (p.hRow0 + m) * 128;
          if (p.hrope == P0_ROPE_HALF) {   // pair (d, d + 64), entry d
            const float* rp = rt + 2 * ((4 * l32) & 63);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              const float o = __shfl_xor(w[c], 16, 64);
              v[c] = l32 >= 16 ? w[c] * rp[2 * c] + o * rp[2 * c + 1] : w[c] * rp[2 * c] - o * rp[2 * c + 1];
            }
          } else {                         // pair (2q, 2q + 1), entry q
            const float* rp = rt + 4 * l32;
#pragma unroll
            for (int c = 0; c < 4; c += 2) {
              v[c] = w[c] * rp[c] - w[c + 1] * rp[c + 1];
              v[c + 1] = w[c] * rp[c + 1] + w[c + 1] * rp[c];
            }
          }
        }
        _Float16* yp = (_Float16*)p.y + (hd * p.hLtot + p.hRow0 + m) * 128 + 4 * l32;
        if (((uintptr_t)yp & 7) == 0) *(uint2*)yp = uint2{pack_h2(v[0], v[1]), pack_h2(v[2], v[3])};
        else {
#pragma unroll
          for (int c = 0; c < 4; ++c) yp[c] = to_h(v[c]);
        }
        continue;
      }
      const int64_t o = (int64_t)m * p.ldy + p.ny0 + n;
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = p.epi == P0_GEPI_RESADD ? g4[c] * (v[c] + b4[c]) : v[c] + b4[c];
      if (f32) {
        float* yp = (float*)p.y + o;
        if (nc == 4 && ((uintptr_t)yp & 15) == 0) {
          if (add) {
            const float4 old = *(const float4*)yp;
            v[0] = old.x + v[0]; v[1] = old.y + v[1]; v[2] = old.z + v[2]; v[3] = old.w + v[3];
          }
          *(float4*)yp = float4{v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c < nc) yp[c] = add ? yp[c] + v[c] : v[c];
        }
      } else {
        _Float16* yp = (_Float16*)p.y + o;
        if (nc == 4 && ((uintptr_t)yp & 7) == 0) {
          if (add) {
            const uint2 old = *(const uint2*)yp;
            const h2 o0 = __builtin_bit_cast(h2, old.x), o1 = __builtin_bit_cast(h2, old.y);
            v[0] += (float)o0.x; v[1] += (float)o0.y; v[2] += (float)o1.x; v[3] += (float)o1.y;
          }
          *(uint2*)yp = uint2{pack_h2(v[0], v[1]), pack_h2(v[2], v[3])};
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (c < nc) yp[c] = to_h(add ? v[c] + (float)yp[c] : v[c]);
        }
      }
    }
  }
}

using Tile = Shape<2, 4, 1, 4>;   // 128 x 128, 8 waves of 64 x 32, four steps' loads in LDS (one workgroup per CU)
static const auto tile_kernel = n128_kernel<2, 4, 1, 4>;

int n128_init() {
  P0_HIP(hipFuncSetAttribute((const void*)tile_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, Tile::Lds), "p0_open: gemm");
  return P0_OK;
}

// K slices: as many as keep one workgroup per CU, each of at least 8 steps, partials within the workspace
static int slices(int64_t tiles, int steps) {
  int nks = (int)(256 / tiles);
  if (nks > steps / 8) nks = steps / 8;
  while (nks > 1 && (size_t)tiles * nks * Tile::BMt * Tile::BNt > ctx().part_floats) --nks;
  return nks < 1 ? 1 : nks;
}
static int64_t tiles_of(const GemmP& p, int bm, int bn) { return ((int64_t)p.N + bn - 1) / bn * (((int64_t)p.M + bm - 1) / bm); }

// Forms: whole 64-row weight tiles (the first weight rows multiples of 64), records 16-byte aligned, X' rows and the weight
// within 32-bit offsets (unsigned ones: rows that go down in memory stay on gemm.hip, which adds 64-bit offsets). Then by
// time: a step of 64 k takes this kernel 1.0 us a round of 256 workgroups, 1.2 us a round, and about 3 us a call, 11 with K
// slices (the partials); the 256 x 256 tiles of gemm.hip 1.4 us while one round holds them all, and 9 us.
// Measured (us, this kernel / gemm.hip): M = 256: 3072 x 2048 21 / 55, 16384 x 2048 swiglu 36 / 62, 2048 x 8192 33 / 179;
// M = 512: 3072 x 3072 35 / 77, 3072 x 9216 75 / 205, 9216 x 3072 95 / 82; M = 1024: 3072 x 9216 128 / 210; M = 2048:
// 3072 x 3072 93 / 82.
bool n128_takes(const GemmP& p) {
  const bool sw = p.epi == P0_GEPI_SWIGLU;
  if (p.wr0 % 64 || (sw && p.wr1 % 64) || ((uintptr_t)p.w & 15)) return false;
  if (p.ldx < 0 || p.ldx >= (1 << 21) || (p.Nw >> 6) * p.wG * 1280 >= (1ll << 31)) return false;
  const int steps = (p.K + 63) / 64;
  const int64_t small = tiles_of(p, Tile::BMt, Tile::BNt), big = tiles_of(p, 256, 256);
  const int nks = slices(small, steps);
  const int64_t rounds = (small * nks + 255) / 256;
  const int64_t here = rounds * ((steps + nks - 1) / nks * 10 + 12) + (nks > 1 ? 108 : 28);   // 0.1 us
  return here < (big + 255) / 256 * steps * 14 + 90;
}

void launch_n128(const GemmP& p, hipStream_t s) {
  N128P a{};
  a.g = p;
  const int steps = (p.K + 63) / 64;
  const int64_t tiles = tiles_of(p, Tile::BMt, Tile::BNt);
  const int nks = slices(tiles, steps);
  a.spk = (steps + nks - 1) / nks;
  a.nks = (steps + a.spk - 1) / a.spk;
  a.part = ctx().part;
  a.cnt = ctx().gemm_counters;   // one per tile where there are slices: at most 128 tiles
  hipLaunchKernelGGL(tile_kernel, dim3((unsigned)(tiles * a.nks)), dim3(Tile::Threads), Tile::Lds, s, a);
}

}  // namespace p0
