// gemvm.hpp - the standalone GEMV launches whose workgroups keep K to themselves: gemvm.hip (2 - 16 rows of x, matrix
// cores) and gemv1.hip (one row). Shared: the weight rows in blocks of 16, items of NBK blocks, 8 waves that each take an
// eighth of a split's K, and the arguments.
#pragma once
#include "gemv_kernels.hpp"

namespace p0 {

constexpr int kGmWaves = 8, kGmThreads = 64 * kGmWaves;
constexpr int kGmPass = 2048;   // k per pass: 8 waves x 8 chunks of 32

// The kernel's arguments, offsets folded into the pointers: three cache lines, read at the start (the whole op
// description, GemvP, is 500 bytes that a cold launch fetches line by line as they come up)
struct GmP {
  const uint8_t* w; const float* X; const float* ST; const float* NW; const float* EV;
  int64_t wG, ldx, statLd, ldp, evLd;
  int N, K, kPer, M, pro, nsrc, items, ipw, wgs;   // wgs: workgroups per split
  int epi, NT; float cap;
  float* Y; float* MX; int64_t ldy, ldm;
};

struct GmPlan {
  GmP args;
  int nbk;      // blocks of 16 weight rows per item
  dim3 grid;    // workgroups, splits
};
inline GmPlan gm_plan(const GemvP& p, int64_t big) {   // big: blocks from which an item takes 4
  // blocks of 16 weight rows over all splits, as many to an item (1, 2 or 4) as keep the items within one per CU (a CU
  // holds one workgroup: the next one starts by splitting x' again); a geglu's gate and up block go together, a softcap
  // needs its tile's 4. q8 5120 x 1536, 5 rows: 320 items of one block 13.5 us, 160 of two 8.8
  GmPlan pl{};
  const int geglu = p.epi == P0_EPI_GEGLU, rows16 = p.N / 16;
  const int64_t blocks = (int64_t)rows16 * (geglu ? 2 : 1) * p.nsplit;
  const int nbk = p.epi == P0_EPI_SOFTCAP || blocks > big ? 4 : blocks > 256 || geglu ? 2 : 1;
  const int items = rows16 / (geglu ? nbk / 2 : nbk);
  const int slots = 256 / (p.nsplit < 256 ? p.nsplit : 256);   // workgroups per split; more items than that are shared out
  const int wgs = items < slots ? items : slots < 1 ? 1 : slots;
  const int ipw = (items + wgs - 1) / wgs;
  pl.nbk = nbk;
  pl.grid = dim3((unsigned)((items + ipw - 1) / ipw), (unsigned)p.nsplit);
  GmP& g = pl.args;
  g.w = p.w;
  g.X = p.X + (p.pro == P0_PRO_RAW || p.pro == P0_PRO_RMS ? p.rowB : 0);   // partials carry no row base
  g.ST = p.ST + p.statOff;
  g.NW = p.NW + p.nOff;
  g.EV = p.EV + p.evOff;
  g.wG = p.wG; g.ldx = p.ldx; g.statLd = p.statLd; g.ldp = p.ldp; g.evLd = p.evLd;
  g.N = p.N; g.K = p.K; g.kPer = p.kPer; g.M = p.mrows; g.pro = p.pro; g.nsrc = p.nsrc;
  g.items = items; g.ipw = ipw; g.wgs = (int)pl.grid.x;
  g.epi = p.epi; g.NT = p.NT; g.cap = p.cap;
  g.Y = p.Y; g.MX = p.MX; g.ldy = p.ldy; g.ldm = p.ldm;
  return pl;
}

bool gemvm_takes(const GemvP& p);                   // do 2..16 rows' op run on gemvm.hip
void launch_gemvm(const GemvP& p, hipStream_t s);   // p.mrows = 2..16 rows, both encodings
bool gemv1_takes(const GemvP& p);                   // does one row's op run on gemv1.hip
void launch_gemv1(const GemvP& p, hipStream_t s);   // one row, both encodings

}  // namespace p0
