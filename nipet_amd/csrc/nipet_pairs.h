// Sinograms that are products of per-(crystal, ring) factors, for gfx950:
//   out[aw][sn] = tw[aw] * sum_{m in members(sn)} w[m] A(aw, r0(m)) B(aw, r1(m)),
//   A(aw, r) = tab[c0(aw) cs + r rs],  B(aw, r) = tab[c1(aw) cs + r rs],
// where members(sn) are the span-1 sinograms (ring pairs r0, r1) of output
// sinogram sn in a fixed order (CSR). Used by the randoms sinogram (singles
// s[c][r], unit weights) and the normalisation sinogram (crystal factors
// E[r][c], axial weights w and transaxial factors tw).
//
// A block has a thread for every sinogram of span 11 (14 waves) and walks groups
// of PAIR_AWB consecutive bins: their 2 x 64 ring factors are in LDS, each
// thread sums its sinogram's members for all bins of the group and writes
// PAIR_AWB coalesced rows. The members of a sinogram are read once for all groups
// (more than 1,024 sinograms: once per group), the next group's factors while
// this one is summed. Bound by the LDS reads of the factors (0.03 ms) and the
// writes (229 MB for span 11: 0.033 ms at the rate of a fill); a block of 256
// threads per group, members one by one: 87 us, now 69. Each
// translation unit that includes this header gets its own copy of the kernel
// (internal linkage).
#pragma once

#include "nipet_common.h"

namespace nipet {
namespace {

constexpr int PAIR_AWB = 8;  // bins per group
constexpr int PAIR_RS = PAIR_AWB + 4;
constexpr int PAIR_MEM = 6;  // members read together (span 11 has at most 6)
constexpr int PAIR_THREADS = 1024;
constexpr int PAIR_BLOCKS = 512;  // two to a CU

struct PairSino {
  const float *tab;      // factor table
  int cs, rs;            // crystal and ring strides of tab
  const short2 *cpair;   // [naw] crystals (c0, c1) of each bin
  const float *tw;       // [naw] per-bin factor, or nullptr (1)
  const int32_t *off;    // [nsn + 1] member ranges
  const short2 *mem_rr;  // [members] ring pair (r0, r1) of each member
  const float *mem_w;    // [members] member weight, or nullptr (1)
  int naw, nsn;
};

__global__ __launch_bounds__(PAIR_THREADS, 8) void k_pair_sino(float *__restrict__ out, PairSino p) {
  // [half of the pair, by turns] ring r's factors of the bins at PAIR_RS r:
  // 16-byte reads without conflicts for consecutive rings
  __shared__ __align__(16) float va[2][64 * PAIR_RS], vb[2][64 * PAIR_RS];
  __shared__ float sw[2][PAIR_AWB];
  const int nthr = blockDim.x, tid = threadIdx.x;
  const int ng = (p.naw + PAIR_AWB - 1) / PAIR_AWB;
  // staging: thread i < 512 has ring i / 8 of bin i % 8; the crystals of a group
  // are read two groups ahead and its factors one ahead
  const int sa = tid & (PAIR_AWB - 1), sr = tid / PAIR_AWB;
  const bool st = sr < 64;
  auto crystals = [&](int g) {
    const int aw = g * PAIR_AWB + sa;
    return st && aw < p.naw ? p.cpair[aw] : make_short2(-1, 0);
  };
  float fx = 0.f, fy = 0.f, ft = 1.f;
  auto factors = [&](int g, short2 cc) {
    fx = fy = 0.f;
    ft = 1.f;
    if (cc.x >= 0) {
      fx = p.tab[cc.x * p.cs + sr * p.rs];
      fy = p.tab[cc.y * p.cs + sr * p.rs];
      if (sr == 0 && p.tw) ft = p.tw[g * PAIR_AWB + sa];
    }
  };
  auto store = [&](int buf) {
    if (!st) return;
    va[buf][sr * PAIR_RS + sa] = fx;
    vb[buf][sr * PAIR_RS + sa] = fy;
    if (sr == 0) sw[buf][sa] = ft;
  };
  short2 rr[PAIR_MEM];
  float w[PAIR_MEM];
  auto members = [&](int m, int m1) {
#pragma unroll
    for (int k = 0; k < PAIR_MEM; k++) {
      const int i = min(m + k, m1 - 1);
      rr[k] = p.mem_rr[max(i, 0)];
      w[k] = p.mem_w ? p.mem_w[max(i, 0)] : 1.f;
    }
  };
  const bool once = p.nsn <= nthr;  // one sinogram a thread
  int o0 = 0, o1 = 0;
  if (tid < p.nsn) {
    o0 = p.off[tid];
    o1 = p.off[tid + 1];
  }
  if (once) members(o0, o1);
  int buf = 0;
  const int dg = gridDim.x;
  factors(blockIdx.x, crystals(blockIdx.x));
  short2 cc = crystals(blockIdx.x + dg);
  store(0);
  for (int g = blockIdx.x; g < ng; g += dg, buf ^= 1) {
    __syncthreads();  // this group's factors written, the other buffer's read
    factors(g + dg, cc);
    cc = crystals(g + 2 * dg);
    const int aw0 = g * PAIR_AWB, na = min(PAIR_AWB, p.naw - aw0);
    for (int sn = tid; sn < p.nsn; sn += nthr) {
      if (!once) {
        o0 = p.off[sn];
        o1 = p.off[sn + 1];
      }
      float acc[PAIR_AWB];
#pragma unroll
      for (int a = 0; a < PAIR_AWB; a++) acc[a] = 0.f;
      for (int m = o0; m < o1; m += PAIR_MEM) {
        if (!once || o1 - o0 > PAIR_MEM) members(m, o1);
#pragma unroll
        for (int k = 0; k < PAIR_MEM; k++) {
          if (m + k >= o1) break;
          const float4 *x = (const float4 *)(va[buf] + rr[k].x * PAIR_RS);
          const float4 *y = (const float4 *)(vb[buf] + rr[k].y * PAIR_RS);
#pragma unroll
          for (int a = 0; a < PAIR_AWB; a += 4) {
            const float4 u = x[a / 4], v = y[a / 4];
            acc[a] += w[k] * (u.x * v.x);
            acc[a + 1] += w[k] * (u.y * v.y);
            acc[a + 2] += w[k] * (u.z * v.z);
            acc[a + 3] += w[k] * (u.w * v.w);
          }
        }
      }
#pragma unroll
      for (int a = 0; a < PAIR_AWB; a++)
        if (a < na) out[(int64_t)(aw0 + a) * p.nsn + sn] = sw[buf][a] * acc[a];
    }
    store(buf ^ 1);
  }
}

inline void launch_pair_sino(float *out, const PairSino &p, hipStream_t st) {
  const int thr = p.nsn > PAIR_THREADS ? PAIR_THREADS : p.nsn < 512 ? 512 : (p.nsn + 63) / 64 * 64;
  const int ng = (p.naw + PAIR_AWB - 1) / PAIR_AWB;
  k_pair_sino<<<ng < PAIR_BLOCKS ? ng : PAIR_BLOCKS, thr, 0, st>>>(out, p);
}

}  // namespace
}  // namespace nipet
