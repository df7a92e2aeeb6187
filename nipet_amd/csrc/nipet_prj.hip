// Siddon forward / back projectors and the fused OSEM subset update for gfx950.
//
// Work decomposition (one workgroup = one transaxial bin of the subset):
//  - the bin's transaxial segment list (FP64-built, device resident) is walked
//    in order; what changes along it for a ring difference are its z crossings
//    (ring centres at z-voxel 2r + 0.5), so the work is per crossing and not per
//    (ring difference, segment);
//  - FP (k_fprj): running sums of the voxel columns along the ray (127 contiguous
//    floats each: coalesced 508-byte reads) in LDS, read once per plane crossing;
//    span-1 -> span-11 sums gathered in a fixed order, one coalesced store per
//    sinogram bin (prj/src/prjf.cu:88-94 uses atomicAdd);
//  - BP (k_bprj): lanes own z-plane pairs and keep the sum of the LORs on each
//    plane; a segment's sums are staged and gathered by voxel column, or one
//    coalesced float atomic per (segment, plane) instead of one per (LOR, piece)
//    (prj/src/prjb.cu:70-82, 153-185).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <utility>

#include "nipet_common.h"

namespace nipet {


static GeomView view(const Geom *g) { return g->view; }

// A sub-batch of NB replicates starting at replicate b0 of a batch of nbt:
// images are [voxel][nbt], sinograms [row][nsn][nbt] (replicate innermost).
struct Batch {
  int nbt, b0;
  // optional per-bin segment window [first, first + count) of the bin's list
  // (nipet_osem_window): the segments whose columns meet the reconstruction
  // mask; the rest carry zero image values (FP) or feed voxels the masked
  // update discards (BP)
  const int32_t *win = nullptr;
};

// The bin's segment list, or its window. A window is clamped into the list
// (nipet_osem_window's always lies inside it), so that the kernels' LDS copy
// of a bin's records (at most MAX_SEG) holds whatever a caller passes.
__device__ inline void seg_range(const GeomView &g, const Batch &bt, int aw, int &beg,
                                 int &nseg) {
  beg = g.off[aw];
  const int n = g.off[aw + 1] - beg;
  nseg = n;
  if (bt.win) {
    const int f = min(max(bt.win[2 * aw], 0), n);
    beg += f;
    nseg = min(max(bt.win[2 * aw + 1], 0), n - f);
  }
}

// The same with wave-uniform results; returns the window's first segment.
__device__ inline int seg_range_u(const int32_t *off, const int32_t *win, int aw, int &beg,
                                  int &nseg) {
  const int o = __builtin_amdgcn_readfirstlane(off[aw]);
  const int n = __builtin_amdgcn_readfirstlane(off[aw + 1]) - o;
  int f = 0;
  nseg = n;
  if (win) {
    f = min(max(__builtin_amdgcn_readfirstlane(win[2 * aw]), 0), n);
    nseg = min(max(__builtin_amdgcn_readfirstlane(win[2 * aw + 1]), 0), n - f);
  }
  beg = o + f;
  return f;
}

template <int NB>
__device__ inline void ldv(float (&r)[NB], const float *p) {
  if constexpr (NB == 1) {
    r[0] = p[0];
  } else if constexpr (NB == 2) {
    float2 t = *reinterpret_cast<const float2 *>(p);
    r[0] = t.x;
    r[1] = t.y;
  } else {
#pragma unroll
    for (int k = 0; k < NB; k += 4) {
      float4 t = *reinterpret_cast<const float4 *>(p + k);
      r[k] = t.x;
      r[k + 1] = t.y;
      r[k + 2] = t.z;
      r[k + 3] = t.w;
    }
  }
}

template <int NB>
__device__ inline void stv(float *p, const float (&r)[NB]) {
  if constexpr (NB == 1) {
    p[0] = r[0];
  } else if constexpr (NB == 2) {
    *reinterpret_cast<float2 *>(p) = make_float2(r[0], r[1]);
  } else {
#pragma unroll
    for (int k = 0; k < NB; k += 4)
      *reinterpret_cast<float4 *>(p + k) = make_float4(r[k], r[k + 1], r[k + 2], r[k + 3]);
  }
}

// Compile-time loop: f(std::integral_constant<int, i>) for i = 0 .. N-1, so
// that register arrays are only ever indexed by constants.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ inline float lor_sfac(float dz, float vox_z, double atn) {
  float az = dz * vox_z;
  float r = az / (float)atn;
  return sqrtf(1.f + r * r);
}

__device__ inline float rdlane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ inline double rdlane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// ---------------------------------------------------------------------------
// Forward projection. MODE 0: emission; 1: attenuation factors;
// 2: OSEM ratio y / (FP + rho) with the 1e-6 guards of prj/src/recon.cu:252-283.
// rho_nb: 0 = one rho shared by all replicates, else rho has the batch layout.
//
// One workgroup per transaxial bin. With C_p(t) the line integral of plane p
// of the bin's voxel columns from the start of the ray to t, the LOR (r0, d)
// (ring centres at zeta = 2 r + 0.5: plane w + 2 r0, w = floor(0.5 + 2 d t /
// atn)) that crosses the z boundary from w to w + 1 at t_w has the value
//   sum_w [C_{w + 2 r0} - C_{w + 1 + 2 r0}](t_w) + C_{w_end + 2 r0}(t_end),
// and its mirror, which runs from plane 2 d + 2 r0 down,
//   C_{2 d - w_end + 2 r0}(t_end) - sum_w [C_p - C_{p + 1}](t_w), p = 2 d - w - 1 + 2 r0.
// The work is therefore one LDS read per z crossing (about 1.8 d per LOR, 37
// on average), not one per voxel segment (272 on average): a subset of 4,894
// bins takes 0.49 ms against 0.95 by segments, all 68,516 bins 6.7 against
// 12.6. VALU, scalar unit and LDS are each at 0.6 of their limits: what is left
// is waves waiting for their turn at all three.
//  - Rows E[j][p] = (C_p - C_{p + 1}) at the start of segment j, a float64
//    prefix sum along the ray, in a ring of FZ_RING rows; a crossing at the
//    fraction f of segment j adds E[j][p] + f (E[j + 1][p] - E[j][p]): one
//    16-byte LDS read. The sums telescope over planes the LOR never enters, so
//    they are kept in float64, which costs no more instructions than float32 on
//    this chip (full-rate FP64); a LOR that misses the object is left with
//    rounding of 1e-16 of the bin's largest line integral (of magnitudes) and is
//    set to 0 (FZ_SNAP).
//  - Two waves stage the rows of a chunk of FZ_CH segments while the others
//    cross the chunk before: one barrier a chunk, and no wave does both. The
//    staging waves wait for memory, so a whole chunk of columns is on its way
//    (one register a row: lane = plane, the next plane from the next lane).
//    All waves staging, then all crossing, with the chunk's totals exchanged:
//    0.56 ms; two planes a lane and half a chunk on its way: 0.55.
//  - Lanes: half a wave is 32 LORs (r0 = lane, lane + 32), the other half
//    their mirrors; the crossing is wave-uniform. Rows hold the even planes
//    and then the odd ones, so the 32 lanes of a half read consecutive
//    words: no bank conflicts at any d.
//  - The crossing waves take the ring differences from the largest down in
//    turns, so that each has about the same number of crossings. From d = 32 on
//    only rings r0 < 32 start a LOR. Where a crossing lies (segment, fraction)
//    is geometry: the table Rays::ev, read through the scalar cache (the vector
//    unit has enough to do).
//  - A LOR below FZ_FAINT of that largest one may be small values beside the
//    rounding of large ones, in a bin that has voxels as small (FZ_SMALL; never
//    mind attenuation factors, which are exp of it, below FZ_MU, and ratios whose
//    additive term is larger or whose LOR is below the guard). The LORs of such a
//    wave and ring difference are walked segment by segment, with the plane
//    changes from the table.
//  - Non-finite voxels: a prefix sum would carry them into LORs that do not
//    touch them. A bin whose line integrals are not finite in float32 is walked
//    segment by segment too.
// Span-1 -> span-N: each output bin sums its LORs in a fixed order from LDS
// (no atomics, bit-reproducible).
constexpr int FZ_THREADS = 1024;
constexpr int FZ_SW = 2;                   // staging waves (planes 0 .. 62, 63 .. 126)
constexpr int FZ_CW = FZ_THREADS / 64 - FZ_SW;  // crossing waves
constexpr int FZ_CH = 30;                  // segments per chunk
constexpr int FZ_PF = FZ_CH;               // columns read ahead by a staging wave
constexpr int FZ_NS = 6;                   // ring differences per crossing wave
constexpr int FZ_RING = 64;                // rows in LDS, by segment modulo FZ_RING
// the ring, its first row again (the row behind the last), and what lanes past
// ring 63 read (the last of it: where a lane without a plane writes)
constexpr int FZ_NE = (FZ_RING + 1) * 128 + 64;
constexpr double FZ_SNAP = 0x1p-44, FZ_FAINT = 0x1p-24;
constexpr float FZ_SMALL = 0x1p-20f, FZ_MU = 0x1p16f;
static_assert(2 * FZ_CH + 1 <= FZ_RING, "a chunk is staged while the one before is read");
static_assert(3 * FZ_CH <= SEG_PAD, "records behind the list are read");
static_assert(FZ_NE * sizeof(double) >= (2 * LI_MAX + 1) * sizeof(float),
              "the per-LOR values reuse the rows' space");

typedef float float2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(8)));
// wave-uniform reads of constant tables (scalar loads)
#define NIPET_CONST __attribute__((address_space(4)))
typedef unsigned int uint2s __attribute__((ext_vector_type(2), aligned(8)));
typedef unsigned int uint16s __attribute__((ext_vector_type(16), aligned(8)));

// VEC: the replicates of a voxel are the sub-batch's (nbt = NB, aligned): one load.
template <int MODE, int NB, bool VEC>
__global__ __launch_bounds__(FZ_THREADS, NB == 1 ? 8 : 4) void k_fprj(
    const GeomView NIPET_CONST *gp, const float *__restrict__ img, float *__restrict__ sino,
    const int32_t *__restrict__ subs, const uint16_t *__restrict__ prompts,
    const float *__restrict__ rho, int rho_nb, Batch bt) {
  __shared__ __align__(16) double E[NB][FZ_NE];
  __shared__ double tot[NB][128];
  __shared__ double cend[NB][128];
  // largest line integral of magnitudes; smallest voxel other than 0, minus 1 (bits
  // without the sign)
  __shared__ unsigned cmax[NB][2], cmin[NB][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = blockIdx.x;
  const int aw = subs ? subs[row] : row;
  const int nbt = VEC ? NB : bt.nbt, b0 = VEC ? 0 : bt.b0, dmax = gp->dmax;
  if (aw < 0 || aw >= gp->naw) {  // invalid bin index: zero row
    const int nsn = gp->nsn;
    float *out = sino + (size_t)row * nsn * nbt + b0;
    for (int i = tid; i < nsn * NB; i += FZ_THREADS) out[(size_t)(i / NB) * nbt + i % NB] = 0.f;
    return;
  }
  int beg, nseg;
  const int first = seg_range_u(gp->off, bt.win, aw, beg, nseg);
  const SegRec NIPET_CONST *seg = (const SegRec NIPET_CONST *)(gp->seg + beg);
  // crossings of ring difference d: ev[ev_off(d) + w]
  const int nev = ev_off(dmax + 1);
  const uint2s NIPET_CONST *ev = (const uint2s NIPET_CONST *)(gp->ev + (size_t)aw * nev);
  // the bin's crossings on their way to L2 (a line per thread)
  float touch = 0.f;
  if (tid * 4 < nev) touch = __uint_as_float(gp->ev[(size_t)aw * nev + tid * 4].y);
  // (finite everywhere: lanes past ring 63 read rows that are not staged yet)
#pragma unroll
  for (int b = 0; b < NB; b++)
    for (int i = tid; i < FZ_NE; i += FZ_THREADS) E[b][i] = 0.0;

  // the crossing waves' ring differences, from dmax down in turns: slots 0 .. 2
  // from 32 up (only rings r0 < 32 start a LOR), 3 .. 5 below; -1: none
  const int cw = wv - FZ_SW, top31 = min(dmax, 31);
  int ds[FZ_NS] = {dmax - cw, dmax - 2 * FZ_CW + 1 + cw, dmax - 2 * FZ_CW - cw,
                   top31 - cw, top31 - 2 * FZ_CW + 1 + cw, top31 - 2 * FZ_CW - cw};
#pragma unroll
  for (int i = 0; i < FZ_NS; i++)
    if (cw < 0 || ds[i] < (i < 3 ? 32 : 0)) ds[i] = -1;
  const bool mir = lane >= 32;  // lanes of the mirrors
  const int sg2 = mir ? -2 : 0;
  double acc[FZ_NS][2][NB];  // ([0 .. 2][1] are not used)
#pragma unroll
  for (int i = 0; i < FZ_NS; i++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[i][0][b] = acc[i][1][b] = 0.0;

  // staging: wave 0 has planes p = lane < 63, wave 1 planes 63 + lane, the next
  // plane's value from the next lane (plane 127: 0). One register a row and
  // replicate, so that a whole chunk is on its way.
  const int pl = min(wv, 1) * 63 + lane;
  const bool own = wv > 0 || lane < 63;
  const int e0 = own ? (pl & 1) * 64 + (pl >> 1) : 127;  // (plane 127 is not used)
  float x0[FZ_PF][NB];
  // lane r: length (bits) of row r of the chunk that is staged, and of the next
  // chunk and its columns, whose values are fetched meanwhile
  int len = 0, len1, col1;
  // (rows past the list have length 0 and some column of the image)
  const char *im = (const char *)(img + b0);
  const unsigned vb = 4 * (VEC ? NB : nbt);  // bytes of a voxel
  auto fetch = [&](auto rc) {
    constexpr int r = decltype(rc)::value;
    // scalar base + 32-bit offset (an image has less than 4 GB)
    const unsigned o = (unsigned)__builtin_amdgcn_readlane(col1, r) * vb + pl * vb;
    if constexpr (VEC && NB == 2) {
      const float2 t = *(const float2 *)(im + o);
      x0[r][0] = t.x;
      x0[r][NB - 1] = t.y;
    } else {
#pragma unroll
      for (int b = 0; b < NB; b++) x0[r][b] = *(const float *)(im + o + 4 * b);
    }
  };
  auto records = [&](int j0) {  // the chunk from segment j0 on
    const int j = j0 + min(lane, FZ_CH - 1);
    const int2 t = *(const int2 *)&gp->seg[beg + j].len;
    len1 = j < nseg ? t.x : 0;
    col1 = t.y;
  };
  double carry[NB];
  float line[NB];    // line integral of the plane's magnitudes so far
  unsigned xmin[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    carry[b] = 0.0;
    line[b] = 0.f;
    xmin[b] = ~0u;
  }
  // rows first + c + 1 .. first + c + FZ_CH, each read again FZ_PF segments on
  auto stage = [&](int c) {
    static_for<FZ_PF>([&](auto rc) {
      constexpr int r = decltype(rc)::value;
      const int slot = (first + c + r + 1) & (FZ_RING - 1);
      const float L = __int_as_float(__builtin_amdgcn_readlane(len, r));
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float x1 = __int_as_float(__builtin_amdgcn_update_dpp(
            0, __float_as_int(x0[r][b]), 0x130 /* wave_shl:1 */, 0xf, 0xf, true));
        carry[b] = fma((double)L, (double)x0[r][b] - (double)x1, carry[b]);
        line[b] = fmaf(L, fabsf(x0[r][b]), line[b]);
        asm volatile("" : "+v"(line[b]));  // (now, not when the later rows are here too)
        if constexpr (MODE != 1) {
          xmin[b] = min(xmin[b], (__float_as_uint(x0[r][b]) << 1) - 1u);
          asm volatile("" : "+v"(xmin[b]));
        }
        E[b][slot * 128 + e0] = carry[b];
        if (slot == 0) E[b][FZ_RING * 128 + e0] = carry[b];
      }
      fetch(rc);
    });
    len = len1;
    records(c + 2 * FZ_CH);
  };
  int wn[FZ_NS] = {0, 0, 0, 0, 0, 0};  // slot i: the next crossing's plane offset
  // the next eight crossings of slot i (a list ends in eight past any segment)
  auto next8 = [&](int i, int w) {
    return *(const uint16s NIPET_CONST *)(ev + ev_off(max(ds[i], 1)) + w);
  };
  auto cross = [&](int c) {
    // crossings in segments below je belong to this chunk (past the list: none)
    const unsigned je = (unsigned)(first + min(c + FZ_CH, nseg)) << 10;
    uint16s nx = next8(0, wn[0]);
    static_for<FZ_NS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      constexpr int NK = i >= 3 ? 2 : 1;  // rings 32 .. 63 start LORs too
      const int d = ds[i];
      uint16s cu = nx;
      if constexpr (i + 1 < FZ_NS) nx = next8(i + 1, wn[i + 1]);
      if (d <= 0) return;
      const int lb = 8 * (lane & 31) + (mir ? 512 + 8 * (d - 1) : 0);
      // N crossings cu[2 q0 ..]: all reads first
      auto some = [&](auto nc, auto qc) {
        constexpr int N = decltype(nc)::value, q0 = decltype(qc)::value;
        double ea[N][NK][NB], eb[N][NK][NB];
#pragma unroll
        for (int n = 0; n < N; n++) {
          const unsigned wd = cu[2 * (q0 + n)];
          const int va = (int)(wd & (FZ_RING * 1024 - 1)) + (lb + sg2 * (int)(wd & 1023));
          const char *pe = (const char *)&E[0][0] + va;
#pragma unroll
          for (int b = 0; b < NB; b++)
#pragma unroll
            for (int k = 0; k < NK; k++) {
              ea[n][k][b] = *(const double *)(pe + b * FZ_NE * 8 + 256 * k);
              eb[n][k][b] = *(const double *)(pe + b * FZ_NE * 8 + 256 * k + 1024);
            }
        }
#pragma unroll
        for (int n = 0; n < N; n++) {
          const double f = __hiloint2double(cu[2 * (q0 + n) + 1], cu[2 * (q0 + n)]);
#pragma unroll
          for (int b = 0; b < NB; b++)
#pragma unroll
            for (int k = 0; k < NK; k++)
              acc[i][k][b] = fma(f, eb[n][k][b] - ea[n][k][b], acc[i][k][b] + ea[n][k][b]);
        }
      };
      using std::integral_constant;
      constexpr int N = NK * NB >= 2 ? 2 : 4;  // crossings read at once (registers)
      integral_constant<int, N> nc;
      int w = wn[i];
      bool full;
      do {
        int done = 0;
        static_for<8 / N>([&](auto qc) {
          constexpr int q = decltype(qc)::value * N;
          if (done == q && (cu[2 * (q + N - 1)] & EV_PLACE) < je) {
            some(nc, integral_constant<int, q>{});
            done = q + N;
          } else if (done == q) {
            static_for<N - 1>([&](auto rc) {
              constexpr int r = decltype(rc)::value;
              if (done == q + r && (cu[2 * (q + r)] & EV_PLACE) < je) {
                some(integral_constant<int, 1>{}, integral_constant<int, q + r>{});
                done = q + r + 1;
              }
            });
            done |= 64;
          }
        });
        full = done == 8;
        w += done & 63;
        if (full) cu = next8(i, w);
      } while (full);
      wn[i] = w;
    });
  };
  // plane offset of ring difference d at the start, rounded down on a tie
  auto start = [&](int d) {
    const double t0 = seg[0].s * (2.0 / gp->atn[aw]);
    return max(__builtin_amdgcn_readfirstlane((int)floor(fma((double)d, t0, 0.5 - 1e-9))), 0);
  };
  // a chunk is staged while the one before it is crossed: as many barriers on
  // both sides (apart, so that neither side's registers burden the other)
  if (wv < FZ_SW) {
    if (nseg > 0) {
      records(0);
      static_for<FZ_PF>([&](auto rc) { fetch(rc); });
      len = len1;
      records(FZ_CH);
    }
    __syncthreads();  // the rows cleared
    for (int c = 0; c < nseg; c += FZ_CH) {
      stage(c);
      __syncthreads();
    }
  } else {
    if (nseg > 0) {
      // plane offset at the start, then past the crossings of earlier segments
      unsigned first_ev[FZ_NS];
#pragma unroll
      for (int i = 0; i < FZ_NS; i++) {
        const int d = max(ds[i], 0);
        wn[i] = start(d);
        first_ev[i] = d > 0 ? ev[ev_off(d) + wn[i]].x : ~0u;
      }
#pragma unroll
      for (int i = 0; i < FZ_NS; i++)
        while ((int)((first_ev[i] & EV_PLACE) >> 10) < first)
          first_ev[i] = ev[ev_off(ds[i]) + ++wn[i]].x;
    }
    __syncthreads();
    for (int c = 0; c < nseg; c += FZ_CH) {
      __syncthreads();  // the chunk staged
      cross(c);
    }
  }
  __syncthreads();  // the last chunk's crossings done (the rows' space is used again)
  asm volatile("" ::"v"(touch));

  // C_p(t_end) = sum of the total differences from plane p up
  if (wv < FZ_SW) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      unsigned m = own ? __float_as_uint(line[b]) : 0u, n = own ? xmin[b] : ~0u;
      for (int o = 32; o > 0; o >>= 1) {
        m = max(m, (unsigned)__shfl_xor((int)m, o));
        n = min(n, (unsigned)__shfl_xor((int)n, o));
      }
      if (lane == 0) {
        cmax[b][wv] = m;
        cmin[b][wv] = n;
      }
      if (own) tot[b][pl] = carry[b];
      if (wv == 0 && lane == 63) tot[b][127] = 0.0;
    }
  }
  __syncthreads();
  if (wv < FZ_SW) {  // wave 0: planes 0 .. 63; wave 1: 64 .. 127; each a suffix sum
#pragma unroll
    for (int b = 0; b < NB; b++) {
      double v = tot[b][wv * 64 + lane];
      for (int o = 1; o < 64; o <<= 1) {
        const double u = __shfl_down(v, o);
        if (lane + o < 64) v += u;
      }
      if (wv == 0) {  // + all of planes 64 .. 127
        double h = tot[b][64 + lane];
        for (int o = 32; o > 0; o >>= 1) h += __shfl_xor(h, o);
        v += h;
      }
      const int p = wv * 64 + lane;
      cend[b][(p & 1) * 64 + (p >> 1)] = v;
    }
  }
  __syncthreads();

  // per-LOR values -> LDS; each output bin then sums its LORs in CSR order
  float *lorv = (float *)&E[0][0];
  static_for<NB>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    const double atn = gp->atn[aw];
    const unsigned um = __builtin_amdgcn_readfirstlane(max(cmax[b][0], cmax[b][1])),
                   un = __builtin_amdgcn_readfirstlane(min(cmin[b][0], cmin[b][1]));
    const float top = __uint_as_float(um), small = __uint_as_float((un + 1u) >> 1);
    const bool slow = !(top < INFINITY);
    // values up to this are walked; in a ratio without a larger additive term, and
    // unless all up to it are below the guard (1e-6, at most six LORs a sinogram)
    const double faint = slow ? INFINITY
                         : MODE == 1 ? (top > FZ_MU ? FZ_FAINT * top : -1.0)
                         : small < FZ_SMALL * top && (MODE == 0 || top > 2.f) ? FZ_FAINT * top
                                                                               : -1.0;
    const double snap = FZ_SNAP * top;
    const float *rh = rho + (size_t)aw * gp->nsn * (rho_nb ? nbt : 1) + (rho_nb ? b0 + b : 0);
    const int rs = rho_nb ? nbt : 1;
    auto put = [&](int li, double v, float sf) {
      float f = (float)v * sf;
      if (MODE == 1) f = expf(-f) * gp->li_nosi[li];
      lorv[2 * li + (mir ? 1 : 0)] = f;
    };
    unsigned redo = 0;  // bit 2 i + k: LORs k of slot i are walked
    if (b > 0) __syncthreads();  // the previous replicate's sums are done
    static_for<FZ_NS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const int d = ds[i];
      if (d < 0) return;
      const float sf = lor_sfac(2.f * d, gp->vox_z, atn);
#pragma unroll
      for (int k = 0; k < (i < 3 ? 1 : 2); k++) {
        const int r0 = (lane & 31) + 32 * k;
        const int li = r0 + d <= 63 ? gp->dr_li[d * 64 + r0] : -1;
        const bool live = li >= 0 && !(mir && d == 0);
        const int pz = (mir ? 2 * d - wn[i] : wn[i]) + 2 * r0;
        const double x = acc[i][k][b];
        double v = live ? cend[b][(pz & 1) * 64 + (pz >> 1)] + (mir ? -x : x) : 0.0;
        bool need = live && !(fabs(v) > faint);
        if (fabs(v) <= snap) v = 0.0;
        if (MODE == 2 && need && !slow) {
          const short2 sn = gp->li_sn[li];
          need = !(fabsf(rh[(size_t)(mir ? sn.y : sn.x) * rs]) > 2.0 * faint);
        }
        if (__builtin_amdgcn_ballot_w64(need)) redo |= 1u << (2 * i + k);
        if (live) put(li, v, sf);
      }
    });
    redo = __builtin_amdgcn_readfirstlane(redo);
    for (; redo; redo &= redo - 1) {
      const int q = __builtin_ctz(redo), i = (q >> 1) % 3, t = q >= 6 ? top31 : dmax;
      const int d = i == 0 ? t - cw : i == 1 ? t - 2 * FZ_CW + 1 + cw : t - 2 * FZ_CW - cw;
      const int r0 = (lane & 31) + 32 * (q & 1);
      const int li = r0 + d <= 63 ? gp->dr_li[d * 64 + r0] : -1;
      if (li < 0 || (mir && d == 0)) continue;
      int w = start(d), j = 0;
      const uint2s NIPET_CONST *e = ev + ev_off(max(d, 1)) + w;
      unsigned at = d > 0 ? e->x : ~0u;
      while ((int)((at & EV_PLACE) >> 10) < first) {
        at = (++e)->x;
        w++;
      }
      unsigned o = ((mir ? 2 * d - w : w) + 2 * r0) * vb + 4 * b;
      auto voxel = [&](int j) { return *(const float *)(im + ((unsigned)seg[j].colz * vb + o)); };
      double v = 0.0, f0 = 0.0;  // f0: the part of segment j that is done
      while (j < nseg) {
        // to the next crossing, or to the end
        const int je = min((int)((at & EV_PLACE) >> 10) - first, nseg);
        if (j < je) {
          if (f0 < 1.0 && seg[j].len > 0.f)
            v += (1.0 - f0) * seg[j].len * (double)voxel(j);
          f0 = 0.0;
#pragma unroll 4
          for (j++; j < je; j++) {
            const float x = voxel(j);
            v += seg[j].len > 0.f ? (double)seg[j].len * (double)x : 0.0;
          }
        }
        if (j >= nseg) break;
        const double f = __hiloint2double(e->y, at & ~EV_PLACE);
        if (f > f0 && seg[j].len > 0.f)
          v += (f - f0) * seg[j].len * (double)voxel(j);
        f0 = fmax(f, f0);
        o += mir ? 0u - vb : vb;
        at = (++e)->x;
      }
      put(li, v, lor_sfac(2.f * d, gp->vox_z, atn));
    }
    // the sinogram's members and, in an OSEM update, its counts and additive
    // term: read before the values are complete
    const int nsn = gp->nsn;
    float *out = sino + (size_t)row * nsn * nbt + b0;
    const uint4 *mem = (const uint4 *)gp->sn_mem;
    const int nm = gp->sn_w / 8;  // 16-byte pieces of 8 members per sinogram
    const uint16_t *pr = prompts + (size_t)aw * nsn * nbt + b0 + b;
    uint4 m4 = make_uint4(0, 0, 0, 0);
    float r = 0.f, y = 0.f;
    auto load = [&](int s) {
      m4 = mem[s * nm];
      if (MODE == 2) {
        r = rh[(size_t)s * rs];
        y = (float)pr[(size_t)s * nbt];
      }
    };
    if (tid < nsn) load(tid);
    if (tid == 0) lorv[2 * LI_MAX] = 0.f;  // absent members
    __syncthreads();
    for (int s = tid; s < nsn; s += FZ_THREADS) {
      float v = 0.f;
      for (int q = 1;; q++) {
        const unsigned int m[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
          v += lorv[m[k] & 0xffff];
          v += lorv[m[k] >> 16];
        }
        if (q == nm) break;
        m4 = mem[s * nm + q];
      }
      if (MODE == 2) {
        const float ee = v + r;
        v = (ee > -EPS && ee < EPS) ? 0.f : y / ee;
      }
      out[(size_t)s * nbt + b] = v;
      if (s + FZ_THREADS < nsn) load(s + FZ_THREADS);
    }
  });
}

// ---------------------------------------------------------------------------
// Forward projection by segments (nipet_fprj_seg; MODE 0: emission, 1:
// attenuation factors): every LOR visits every segment of the bin, in float32.
// The differentiable projectors' forward passes use it: their likelihood is a
// float64 number made of these float32 values, and it stays the same bit for
// bit. (k_fprj takes 0.49 ms a subset instead of 1.04, and differs by 5e-8: 4.9e-8
// from the exact values instead of 5.6e-8.)
//
// Lanes are groups of G LORs of one ring difference.
// LOR (d, r0 + k) lies exactly 2k planes above LOR (d, r0) along the whole ray
// (ring centres at zeta = 2 r + 0.5), so the G LORs of a slot (and their
// mirrors, 2k planes above the mirror of (d, r0)) share the boundary
// positions, the pieces p1 / p2 and the plane steps: per segment a lane
// computes those once and adds 2 (4 across a boundary) products per LOR pair,
// reading the G planes at immediate offsets from one pointer. Slots (d, r0)
// come from the geometry (fp_slot); lanes whose group runs past ring 63 walk phantom LORs
// whose planes lie in zero guard planes and are never written out.
// G = 3 (odd): lanes of one ring difference then sit 6 planes (3 plane pairs)
// apart; in the pair layout (fpg_addr) that is 3 banks, so 32 lanes of one d
// reach 32 distinct banks. Measured on MI355X with a linear plane stride of 17
// floats: G = 3 1.19 ms per subset, G = 5 1.31 ms, G = 4 3.4 ms (bank
// conflicts), one LOR per lane 1.71 ms.
constexpr int SUBSUM = 8;         // float partial sums over 8 segments
constexpr int ZSTRIDE = 128;      // LDS z-column (127 + zero pad)
constexpr int FP_GUARD = 2;       // zero planes below 0 and above 127 (pieces reach ia + 2, ib - 2)
template <int G>
constexpr int fpg_threads() { return FP_G_SLOTS; }  // >= 712 slots of 3 LORs
template <int G>
constexpr int fpg_rounds() { return 1; }
template <int G>
constexpr int fpg_top() { return 2 + 2 * (G - 1); }    // zero planes above 127
template <int G>
constexpr int fpg_planes() { return FP_GUARD + ZSTRIDE + fpg_top<G>(); }

template <int NB, int G>
struct FpSumG {
  float pa[G][NB], pb[G][NB], ta[G][NB], tb[G][NB];
  __device__ void fold() {
    static_for<G>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        ta[k][b] += pa[k][b];
        tb[k][b] += pb[k][b];
        pa[k][b] = 0.f;
        pb[k][b] = 0.f;
      }
    });
  }
};

// Staged chunk of the grouped kernel: planes in pairs, plane p at
// fpg_addr(p) = (p >> 1) * FPG_PP + (p & 1) * CH floats (segment j at + j),
// pair stride FPG_PP = 2 CH + 1. Planes 2k above p stay at the immediate
// offset FPG_PP * k; the next plane up is CH or CH + 1 floats on, by the
// parity of p (kept per lane as oa / ob). Lanes of one ring difference sit 6
// planes (3 pairs) apart at every segment, so their reads step 3 banks and
// reach all 32 banks; a linear plane stride maps 6 planes to an even number of
// banks, 16 of the 32.
constexpr int FPG_CH = 16;
constexpr int FPG_PP = 2 * FPG_CH + 1;
__host__ __device__ constexpr int fpg_addr(int p) { return (p >> 1) * FPG_PP + (p & 1) * FPG_CH; }

struct FpLorG {
  float tbr;   // next z boundary of LOR a relative to the chunk's origin (float)
  float invf;  // boundary spacing (float)
  int ao;      // staged-chunk offset of plane pa = ia + FP_GUARD (LOR a), segment 0
  int bo;      // staged-chunk offset of plane pb = ib - 2 + FP_GUARD (mirror b)
  // fpg_addr(p + 1) - fpg_addr(p) = CH + (p & 1) for p = pa and p = pb:
  // pa + pb = 4 r0 + 2 d + 2 is even, so both planes share their parity (and
  // keep sharing it, since a boundary moves pa up and pb down by one)
  int o;
};

// srx / srl: position and length of the chunk's segment j in lane j (every
// wave holds the chunk's records), broadcast to the scalar unit per segment
template <int G, bool TWO>
__device__ inline void fpg_walk(FpLorG &l, FpSumG<1, G> &acc, float srx, float srl,
                                const float *__restrict__ zs, int nch) {
  constexpr int PP = FPG_PP;
  for (int j8 = 0; j8 < nch; j8 += SUBSUM) {
    const float *za = zs + l.ao + j8;
    const float *zb = zs + l.bo + j8;
    int o = l.o;
#pragma unroll 4
    for (int jj = 0; jj < SUBSUM; jj++) {
      const float2 sl = make_float2(rdlane(srx, j8 + jj), rdlane(srl, j8 + jj));
      if constexpr (!TWO) {
        const float q = l.tbr - sl.x;
        const float p1 = __builtin_amdgcn_fmed3f(q, 0.f, sl.y);
        const bool cr = q <= sl.y;
        static_for<G>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          acc.pa[k][0] = fmaf(p1, za[k * PP + jj], acc.pa[k][0]);       // plane pa + 2k
          acc.pb[k][0] = fmaf(p1, zb[(k + 1) * PP + jj], acc.pb[k][0]);  // plane pb + 2k + 2
        });
        // second piece only where the segment holds a boundary: the same
        // segment for every lane of a ring difference, so whole lane groups
        // skip these reads (and the plane steps) together
        if (cr) {
          const float p2 = sl.y - p1;
          const float *za1 = za + o, *zb1 = zb + o;  // planes pa + 1, pb + 1
          static_for<G>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            acc.pa[k][0] = fmaf(p2, za1[k * PP + jj], acc.pa[k][0]);
            acc.pb[k][0] = fmaf(p2, zb1[k * PP + jj], acc.pb[k][0]);
          });
          za = za1;       // pa + 1
          zb = zb1 - PP;  // pb - 1
          o = PP - o;
          l.tbr += l.invf;
        }
      } else {
        const float q1 = l.tbr - sl.x, q2 = q1 + l.invf;
        const float p1 = __builtin_amdgcn_fmed3f(q1, 0.f, sl.y);
        const float c2 = __builtin_amdgcn_fmed3f(q2, 0.f, sl.y);
        const float p2 = c2 - p1, p3 = sl.y - c2;
        const float *za1 = za + o, *zb1 = zb + o;
        static_for<G>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          const float xa0 = za[k * PP + jj], xa1 = za1[k * PP + jj], xa2 = za[(k + 1) * PP + jj];
          const float xb0 = zb[(k + 1) * PP + jj], xb1 = zb1[k * PP + jj], xb2 = zb[k * PP + jj];
          acc.pa[k][0] = fmaf(p1, xa0, acc.pa[k][0]);
          acc.pa[k][0] = fmaf(p2, xa1, acc.pa[k][0]);
          acc.pa[k][0] = fmaf(p3, xa2, acc.pa[k][0]);
          acc.pb[k][0] = fmaf(p1, xb0, acc.pb[k][0]);
          acc.pb[k][0] = fmaf(p2, xb1, acc.pb[k][0]);
          acc.pb[k][0] = fmaf(p3, xb2, acc.pb[k][0]);
        });
        const int n = (int)(q1 <= sl.y) + (int)(q2 <= sl.y);
        const bool n1 = n == 1, n2 = n == 2;
        za = n1 ? za1 : (n2 ? za + PP : za);
        zb = n1 ? zb1 - PP : (n2 ? zb - PP : zb);
        o = n1 ? PP - o : o;
        l.tbr += (float)n * l.invf;
      }
    }
    l.ao = (int)(za - zs) - j8;
    l.bo = (int)(zb - zs) - j8;
    l.o = o;
    acc.fold();
  }
}

// One bin's segment records [n] copied to LDS with 16-byte loads.
__device__ inline void load_segs(SegRec *dst, const SegRec *__restrict__ src, int n, int tid,
                                 int nthr) {
  const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
  uint4 *d4 = reinterpret_cast<uint4 *>(dst);
  for (int i = tid; i < n; i += nthr) d4[i] = s4[i];
}

// 6 waves per SIMD (two 12-wave workgroups per CU) need <= 80 VGPRs; the
// compiler's own choice for this kernel is 82
template <int MODE, int G>
__global__ __launch_bounds__(fpg_threads<G>()) __attribute__((amdgpu_waves_per_eu(6))) void k_fprj_seg(
    GeomView g, const float *__restrict__ img, float *__restrict__ sino,
    const int32_t *__restrict__ subs) {
  constexpr int NB = 1, nbt = 1, b0 = 0;
  constexpr int CH = FPG_CH;
  constexpr int R = fpg_rounds<G>(), NP = fpg_planes<G>(), FPG_THREADS = fpg_threads<G>();
  static_assert(G == FP_G, "slot tables are built for FP_G LORs per lane");
  constexpr int ZN = fpg_addr(NP), LN = 2 * LI_MAX;  // planes 0 .. NP - 1
  __shared__ __align__(16) float lds[ZN > LN ? ZN : LN];
  __shared__ double inv[R][FPG_THREADS];  // exact boundary spacing (0: direct)
  __shared__ float z0[R][FPG_THREADS];    // zeta of the slot's first LOR at t = 0
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int row = blockIdx.x;
  const int aw = subs ? subs[row] : row;
  const int nsn = g.nsn;
  const int nslot = g.fp_nslot;
  const int16_t *slots = g.fp_slot;
  float *out = sino + (size_t)row * nsn * nbt + b0;
  if (aw < 0 || aw >= g.naw) {  // invalid bin index: zero row
    for (int i = tid; i < nsn * NB; i += FPG_THREADS) out[(i / NB) * nbt + i % NB] = 0.f;
    return;
  }
  int beg, nseg;
  seg_range(g, Batch{1, 0}, aw, beg, nseg);
  const double atn = g.atn[aw];
  const float lmax = g.lmax[aw];
  float *zs = lds;
  // guard planes (never written by the staging loop)
  for (int i = tid; i < fpg_addr(FP_GUARD); i += FPG_THREADS) zs[i] = 0.f;
  for (int i = fpg_addr(FP_GUARD + ZSTRIDE) + tid; i < ZN; i += FPG_THREADS) zs[i] = 0.f;

  FpLorG L[R];
  FpSumG<NB, G> A[R];
  bool two[R], live[R];
  int dr[R];  // d * 64 + r0 of the slot
  const double s0 = nseg > 0 ? g.seg[beg].s : 0.0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int sl = r * FPG_THREADS + tid;
    dr[r] = sl < nslot ? slots[sl] : 0;
    const int d = dr[r] >> 6, r0 = dr[r] & 63;
    const float2 z = make_float2(2.f * r0 + 0.5f, 2.f * d);
    const int wsum = (int)floorf(z.x) + (int)floorf(z.x + z.y);
    int ia;
    double iv = 0.0;
    if (z.y > 0.f) {
      iv = atn / (double)z.y;
      ia = (int)floor((double)z.x + s0 / iv);
    } else {
      ia = (int)floorf(z.x);
    }
    z0[r][tid] = z.x;
    inv[r][tid] = iv;
    const int pa = ia + FP_GUARD, pb = wsum - ia - 2 + FP_GUARD;
    L[r].ao = fpg_addr(pa);
    L[r].bo = fpg_addr(pb);
    L[r].o = CH + (pa & 1);
    L[r].invf = (float)iv;
    static_for<G>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
#pragma unroll
      for (int b = 0; b < NB; b++) A[r].pa[k][b] = A[r].pb[k][b] = A[r].ta[k][b] = A[r].tb[k][b] = 0.f;
    });
    live[r] = r * FPG_THREADS + wave * 64 < nslot;  // wave-uniform
    two[r] = __any(iv > 0.0 && iv < (double)lmax);
  }

  // Software pipeline over chunks of CH segments: while chunk c is walked,
  // each thread has its NST z-column values of chunk c + CH in flight. The
  // bin's segment records sit in LDS (copied once), so neither the column
  // addresses nor a chunk's positions wait on a global load.
  constexpr int NE = CH * ZSTRIDE, NST = (NE + FPG_THREADS - 1) / FPG_THREADS;
  __shared__ SegRec segl[MAX_SEG];
  load_segs(segl, g.seg + beg, nseg, tid, FPG_THREADS);
  float pre[NST];
  auto fetch = [&](int c) {
#pragma unroll
    for (int i = 0; i < NST; i++) {
      const int idx = tid + i * FPG_THREADS;
      const int j = idx / ZSTRIDE, z = idx - j * ZSTRIDE;
      float v = 0.f;
      if (idx < NE && c + j < nseg && z < NZ) v = img[((int64_t)segl[c + j].colz + z) * nbt + b0];
      pre[i] = v;
    }
  };
  __syncthreads();
  if (nseg > 0) fetch(0);
  for (int c = 0; c < nseg; c += CH) {
    const int nch = nseg - c < CH ? nseg - c : CH;
    __syncthreads();
    // positions are relative to the chunk's middle segment: float positions
    // within +-8 segments carry half the rounding of ones within 16
    const double sb = segl[c + (nch >> 1)].s;
    // lanes 0 .. CH-1 of every wave: the chunk's segment positions / lengths
    const int jl = lane < CH ? lane : 0;
    const float srx = c + jl < nseg ? (float)(segl[c + jl].s - sb) : -1e30f;
    const float srl = c + jl < nseg ? segl[c + jl].len : 0.f;
#pragma unroll
    for (int i = 0; i < NST; i++) {
      const int idx = tid + i * FPG_THREADS;
      if (idx < NE) {
        const int j = idx / ZSTRIDE, z = idx - j * ZSTRIDE;
        zs[fpg_addr(z + FP_GUARD) + j] = pre[i];
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      // plane of LOR a: pa = 2 (ao / PP) + (odd plane of its pair)
      const int pq = L[r].ao / FPG_PP;
      const int ia = 2 * pq + (L[r].ao - pq * FPG_PP >= CH ? 1 : 0) - FP_GUARD;
      const double iv = inv[r][tid];
      L[r].tbr = iv > 0.0 ? (float)(((double)(ia + 1) - (double)z0[r][tid]) * iv - sb) : 3e38f;
    }
    __syncthreads();
    if (c + CH < nseg) fetch(c + CH);
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!live[r]) continue;
      if (two[r])
        fpg_walk<G, true>(L[r], A[r], srx, srl, zs, nch);
      else
        fpg_walk<G, false>(L[r], A[r], srx, srl, zs, nch);
    }
  }

  // per-LOR values -> LDS; each output bin then sums its LORs in CSR order
  float *lorv = lds;
  float sf[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int d = dr[r] >> 6;
    sf[r] = lor_sfac(2.f * d, g.vox_z, atn);
    A[r].fold();
  }
  static_for<NB>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (r * FPG_THREADS + tid >= nslot) continue;
      const int d = dr[r] >> 6, r0 = dr[r] & 63;
      static_for<G>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const int li = r0 + k + d <= 63 ? g.dr_li[dr[r] + k] : -1;
        if (li >= 0) {
          float va = A[r].ta[k][b] * sf[r], vb = A[r].tb[k][b] * sf[r];
          if (MODE == 1) {
            const float nosi = g.li_nosi[li];
            va = expf(-va) * nosi;
            vb = expf(-vb) * nosi;
          }
          lorv[2 * li] = va;
          if (d > 0) lorv[2 * li + 1] = vb;
        }
      });
    }
    __syncthreads();
    for (int s = tid; s < nsn; s += FPG_THREADS) {
      float v = 0.f;
      const uint16_t *mem = g.sn_mem + (size_t)s * g.sn_w;
      for (int m = 0; m < g.sn_w && mem[m] < 2 * LI_MAX; m++) v += lorv[mem[m]];
      out[(size_t)s * nbt + b] = v;
    }
  });
}

// Segment windows of the reconstruction mask (nipet_osem_window): m2[c] = 1
// when column c = u + NX v of the mask holds any voxel, optionally dilated by
// a box of half-width r (the resolution model's 17-tap reach); then, one wave
// per bin, the first and last segment of the bin's list whose column is set.
__global__ void k_mask_cols(const uint8_t *__restrict__ mask, uint8_t *__restrict__ m2) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= NX * NY) return;
  const uint8_t *p = mask + (int64_t)c * NZ;
  int any = 0;
  for (int z = 0; z < NZ; z++) any |= p[z];
  m2[c] = any != 0;
}

__global__ void k_mask_dilate(const uint8_t *__restrict__ m2, uint8_t *__restrict__ m2d, int r) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= NX * NY) return;
  const int u = c % NX, v = c / NX;
  int any = 0;
  for (int vv = v - r; vv <= v + r; vv++) {
    if (vv < 0 || vv >= NY) continue;
    for (int uu = u - r; uu <= u + r; uu++)
      if (uu >= 0 && uu < NX) any |= m2[uu + NX * vv];
  }
  m2d[c] = any != 0;
}

__global__ __launch_bounds__(256) void k_seg_window(GeomView g, const uint8_t *__restrict__ m2,
                                                    int32_t *__restrict__ win) {
  const int lane = threadIdx.x & 63;
  const int aw = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (aw >= g.naw) return;  // wave-uniform
  const int beg = g.off[aw], n = g.off[aw + 1] - beg;
  int first = -1, last = -1;
  for (int k0 = 0; k0 < n; k0 += 64) {
    const int k = k0 + lane;
    const bool in = k < n && m2[g.seg[beg + k].colz / NZ] != 0;
    const unsigned long long m = __ballot(in);
    if (m) {
      if (first < 0) first = k0 + __ffsll((long long)m) - 1;
      last = k0 + 63 - __clzll(m);
    }
  }
  if (lane == 0) {
    win[2 * aw] = first < 0 ? 0 : first;
    win[2 * aw + 1] = first < 0 ? 0 : last - first + 1;
  }
}

// ---------------------------------------------------------------------------
// Back projection (adjoint of the emission FP) as a gather, accumulated into img.
//
// One workgroup per transaxial bin; its waves take equal runs of the bin's
// segments. Along a run a wave keeps, for every plane p (lane i: planes 2 i and
// 2 i + 1), S_p = the sum of the LOR values on plane p. LORs change plane only
// at the z crossings of their ring difference d (at t = (w + 1/2) atn / (2 d)
// from plane offset w to w + 1: a LOR (r0, d) from plane w + 2 r0 up, its mirror
// from 2 d - w + 2 r0 down), so a segment costs L S_p plus, for each of the
// crossings inside it (11 of 60 ring differences on average), one look-up of
// the values that come and go:
//   T_p = va[(p - w) >> 1] + vb[((p + w + 1) >> 1) - d],
// which leaves plane p where p + w is even and enters where it is odd; the
// segment gains (rest of the segment behind the crossing) times +-T_p, S_p
// gains +-T_p. (Segment by segment, every ring difference cost about six
// instructions in every segment: 1.24 ms a subset of 4,894 bins.)
//  - What enters leaves again in the same pairs (va, vb), so S_p in float64
//    returns to its former value to 1e-16 of the bin's largest value, and
//    S_p below BP_SNAP of that are set to 0: a plane that no LOR is on gets
//    nothing. The segment's own sum is float64 too (full-rate FP64): a short
//    piece of a segment is a difference here.
//  - A bin with values below BP_FAINT of its largest (zeros aside) may have S_p
//    that small beside the rounding of the large ones. There a wave that meets
//    one sums its run again, segment by segment, from the terms themselves
//    (without a row to overwrite, every run of such a bin is).
//  - S and the segment's sum carry the sign (-1)^p, so that a crossing adds (w
//    even) or subtracts (w odd) one T for all lanes: no per-lane sign.
//  - va / vb (times the 3D length factor of d) sit in LDS, row d at 65 d with
//    the zeros between rows shared, so that every index the gather can form
//    (-d .. 63) stays inside and needs no clamp: 34 KB an image. A plane pair
//    shares va (w even) or vb (w odd): three floats for two planes.
//  - The crossings come from a table in the walk's order (GeomView::bp_ev)
//    through the scalar cache, eight at a time and eight ahead: position, sign
//    and the look-up's two rows need no vector instruction, and a crossing is
//    ten of them and two LDS reads. Finding the crossings with lane d on ring
//    difference d and a ballot per segment, and v_readlane for each: 0.57 ms.
//  - Non-finite sinogram values would stay in S after their LOR has left the
//    plane, and so would the overflow of huge ones: a bin with values from
//    BP_HUGE up is summed segment by segment.
//  - Output: with STAGED every segment's plane sums go to the segment's own row
//    of a scratch buffer (512 bytes an image) and k_bp_gather adds the rows of
//    each voxel column, else float atomics to the image.
// Bound by vector issue (80 % of the cycles, 8 waves per SIMD): 0.40 ms a subset
// for one image, 0.67 for two (with 512 threads, 4 waves per SIMD, 0.82), of which
// the look for small sums is 0.5 %; where every bin has some, 2.7 ms with the
// gather.
template <int NB>
constexpr int bp_threads() {
  return 512 * NB;
}
constexpr float BP_SNAP = 0x1p-45f, BP_FAINT = 0x1p-23f, BP_HUGE = 0x1p120f;

//
// img: the image [voxel][nbt] (atomics, zeroed before), or with STAGED the
// scratch rows [workgroup][rows_per_bin][128][NB].
template <int NB, bool STAGED>
__global__ __launch_bounds__(bp_threads<NB>(), 8) void k_bprj(
    const GeomView NIPET_CONST *gp, float *__restrict__ img, const float *__restrict__ sino,
    const float *__restrict__ sino2, const int32_t *__restrict__ subs, Batch bt, int by_bin,
    int row0) {
  constexpr int THR = bp_threads<NB>(), WAVES = THR / 64, IT = (BP_TN + THR - 1) / THR;
  // vb, an entry that is not used (an odd crossing's va look-up is at lane - 1)
  // and va; first the sinogram row and a zero are staged there
  __shared__ __align__(16) float tab[(2 * BP_TN + 1) * NB];
  // per image: largest magnitude in the row, and smallest other than 0, minus 1
  // (bits without the sign)
  __shared__ unsigned vtop[NB], vlow[NB];
  float *srow = tab;
  static_assert(sizeof(tab) >= 4096 * NB * sizeof(float), "a row of 4095 sinograms");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = row0 + blockIdx.x;
  const int aw = __builtin_amdgcn_readfirstlane(subs ? subs[row] : row);
  if (aw < 0 || aw >= gp->naw) return;
  const int nsn = gp->nsn, nbt = bt.nbt, b0 = bt.b0, dmax = gp->dmax;
  int beg, nseg;
  const int first = seg_range_u(gp->off, bt.win, aw, beg, nseg);
  const SegRec NIPET_CONST *seg = (const SegRec NIPET_CONST *)(gp->seg + beg);
  const double atn = gp->atn[aw];

  // sinogram rows in subset order, or (by_bin) the full [naw][nsn] sinogram
  // read at the bin's own row; sino2: the second of two images, by bin
  unsigned top = 0, low = ~0u;  // of the thread's image
  {
    const int b = tid % NB;
    const bool two = NB == 2 && sino2;
    const float *in = sino + (size_t)(by_bin ? aw : row) * nsn * (two ? 1 : nbt);
    in += two ? 0 : b0 + b;
    if (two && b) in = sino2 + (size_t)aw * nsn;
    const int step = two ? 1 : nbt;
    for (int k = tid / NB; k <= nsn; k += THR / NB) {
      const float x = k < nsn ? in[(size_t)k * step] : 0.f;
      const unsigned u = __float_as_uint(x) << 1;
      top = max(top, u);
      low = min(low, u - 1u);
      srow[k * NB + b] = x;
    }
  }
  if (tid < NB) {
    vtop[tid] = 0;
    vlow[tid] = ~0u;
  }
  __syncthreads();
  for (int o = 32; o >= NB; o >>= 1) {
    top = max(top, (unsigned)__shfl_xor((int)top, o));
    low = min(low, (unsigned)__shfl_xor((int)low, o));
  }
  if (lane < NB) {
    atomicMax(&vtop[lane], top);
    atomicMin(&vlow[lane], low);
  }
  float xa[IT][NB], xb[IT][NB];
#pragma unroll
  for (int k = 0; k < IT; k++) {
    const int i = tid + k * THR;
    if (i < BP_TN) {
      const uint32_t e = gp->bp_tab[i];  // sinograms of LOR and mirror (nsn: none)
      ldv<NB>(xa[k], srow + (e & 0xffff) * NB);
      ldv<NB>(xb[k], srow + (e >> 16) * NB);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < IT; k++) {
    const int i = tid + k * THR;
    if (i >= BP_TN) break;
    const float sf = lor_sfac(2.f * (float)(i / 65), gp->vox_z, atn);  // (padding is 0)
#pragma unroll
    for (int b = 0; b < NB; b++) {
      tab[i * NB + b] = xb[k][b] * sf;
      tab[(BP_TN + 1 + i) * NB + b] = xa[k][b] * sf;
    }
  }
  __syncthreads();
  bool huge = false, faint = false;
  float snap[NB];  // sums that do not count: of empty planes, or (faint) to be summed again
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const unsigned ut = __builtin_amdgcn_readfirstlane(vtop[b]),
                   ul = __builtin_amdgcn_readfirstlane(vlow[b]) + 1u;
    const float t = __uint_as_float(ut >> 1), l = __uint_as_float(ul >> 1);
    huge |= !(t < BP_HUGE);
    const bool f = l < BP_FAINT * t;
    faint |= f;
    snap[b] = (f ? BP_FAINT : BP_SNAP) * t;
  }

  // lane d: crossings of ring difference d
  const bool on = lane >= 1 && lane <= dmax;
  const double m = on ? 2.0 * lane / atn : 0.0;
  // T of planes 2 lane and 2 lane + 1: x = 4 D, y = 516 d - 4 D (bp_event)
  constexpr int Q = 4 * NB;
  int Al = Q * lane, Bl = Q * (lane + BP_TN + 1);
  asm("" : "+v"(Al), "+v"(Bl));  // (kept whole in registers)
  auto lookup = [&](int x, int y, float (&T)[2][NB]) {
    const float *p = (const float *)((const char *)tab + NB * x + Al);
    const float *q = (const float *)((const char *)tab + NB * y + Bl);
    float u[2 * NB], v[NB];
    ldv<NB>(*(float(*)[NB])u, p);
    ldv<NB>(*(float(*)[NB])(u + NB), p + NB);
    ldv<NB>(v, q);
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int b = 0; b < NB; b++) T[k][b] = u[k * NB + b] + v[b];
  };

  const int j0 = nseg * wv / WAVES, j1 = nseg * (wv + 1) / WAVES;
  if (j0 >= j1) return;
  double s = seg[j0].s;
  int w = plane_offset(m, s);

  // the sums of segment j0, j0 + 1, .. (length len) without their signs, to the
  // segment's row or to the image
  float *q = nullptr;
  if constexpr (STAGED)
    q = img + ((size_t)blockIdx.x * gp->maxseg + first + j0) * (128 * NB) + lane * 2 * NB;
  unsigned long long small[2] = {0, 0};  // lanes whose sums were set to 0
  auto put = [&](int colz, float len, const double (&acc)[2][NB]) {
    float v[2 * NB];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int b = 0; b < NB; b++) {
        v[k * NB + b] = (float)(k ? acc[k][b] : -acc[k][b]);
        const bool z = fabsf(v[k * NB + b]) <= snap[b] * len;
        if constexpr (STAGED) small[k] |= __builtin_amdgcn_ballot_w64(z);
        if (z) v[k * NB + b] = 0.f;
      }
    if constexpr (STAGED) {
      stv<2 * NB>(q, v);
      q += 128 * NB;
    } else {
      // atomics to adjacent planes of adjacent lanes: plane lane + 64 h
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const float x0 = __shfl(v[b], 32 * h + (lane >> 1)),
                      x1 = __shfl(v[NB + b], 32 * h + (lane >> 1)), x = lane & 1 ? x1 : x0;
          const int p = lane + 64 * h;
          if (p < NZ && x != 0.f) unsafeAtomicAdd(img + ((int64_t)colz + p) * nbt + b0 + b, x);
        }
    }
  };

  // sum of the LORs of ring differences ds on plane offset w
  auto standing = [&](unsigned long long ds, double (&S)[2][NB]) {
    // LORs of d are on planes of w's parity
    unsigned long long odd = __builtin_amdgcn_ballot_w64(w & 1) & ds, even = ~odd & ds;
    const int x_l = 4 * bp_entry(lane, w);
#pragma unroll
    for (int b = 0; b < NB; b++) S[0][b] = S[1][b] = 0.0;
#pragma unroll 2
    for (; even; even &= even - 1) {
      const int d = __builtin_ctzll(even), x = __builtin_amdgcn_readlane(x_l, d);
      float T[2][NB];
      lookup(x, 516 * d - x, T);
#pragma unroll
      for (int b = 0; b < NB; b++) S[0][b] -= (double)T[0][b];
    }
#pragma unroll 2
    for (; odd; odd &= odd - 1) {
      const int d = __builtin_ctzll(odd), x = __builtin_amdgcn_readlane(x_l, d);
      float T[2][NB];
      lookup(x, 516 * d - x, T);
#pragma unroll
      for (int b = 0; b < NB; b++) S[1][b] += (double)T[1][b];
    }
  };
  const unsigned long long all = ~0ull >> (63 - dmax);

  double acc[2][NB];
  // the run segment by segment, each sum from its own terms
  auto by_segment = [&]() {
    const double inv = on ? atn / (2.0 * lane) : 0.0;
    for (int j = j0; j < j1; j++) {
      const double s1 = j + 1 < nseg ? seg[j + 1].s : s + (double)seg[j].len;
      const int wn = plane_offset(m, s1);
      unsigned long long hit = __builtin_amdgcn_ballot_w64(w < wn);
      double S[2][NB];
      standing(all & ~hit, S);
#pragma unroll
      for (int k = 0; k < 2; k++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[k][b] = s1 > s ? (s1 - s) * S[k][b] : 0.0;
      for (; hit; hit &= hit - 1) {  // pieces of the ring differences that cross
        const int d = __builtin_ctzll(hit), we = __builtin_amdgcn_readlane(wn, d);
        const double step = rdlane(inv, d);
        double pos = s;
        for (int wc = __builtin_amdgcn_readlane(w, d); wc <= we; wc++) {
          const double end = wc < we ? fmin(((double)wc + 0.5) * step, s1) : s1;
          const int x = 4 * bp_entry(d, wc);
          float T[2][NB];
          lookup(x, 516 * d - x, T);
          if (end > pos) {  // (signs as in the walk below)
#pragma unroll
            for (int b = 0; b < NB; b++) {
              if (wc & 1) acc[1][b] += (end - pos) * (double)T[1][b];
              else acc[0][b] -= (end - pos) * (double)T[0][b];
            }
            pos = end;
          }
        }
      }
      put(seg[j].colz, 0.f, acc);
      w = wn;
      s = s1;
    }
  };
  if (huge || (faint && !STAGED)) {
    by_segment();
    return;
  }

  double S[2][NB];
  standing(all, S);
  // lane i: length and column of segment jb + i
  double Ll;
  int Cl = 0, jb;
  auto lengths = [&](int j) {
    jb = j;
    const int i = min(j + lane, nseg - 1);
    const SegRec *sp = gp->seg + beg + i;
    Ll = i + 1 < nseg ? sp[1].s - sp[0].s : (double)sp[0].len;
    if constexpr (!STAGED) Cl = sp[0].colz;
  };
  lengths(j0);
  int j = j0;
  double L = rdlane(Ll, 0);
#pragma unroll
  for (int k = 0; k < 2; k++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[k][b] = L * S[k][b];
  const uint2s NIPET_CONST *ev =
      (const uint2s NIPET_CONST *)(gp->bp_ev + ((const uint32_t NIPET_CONST *)gp->bp_off)[beg + j0]);
  uint32_t live = 1;  // 0 when the run is done (the rest of its last eight is not)
  auto eight = [&](const uint16s &e) {
    if (j - jb >= 56) lengths(j);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const uint32_t lo = e[2 * i], hi = e[2 * i + 1];
      const int x = lo & 0xfffc, y = (int)((lo >> 16) & 0x7f) * 516 - x;
      // T leaves the planes of the offset's parity and enters the others: their
      // signs make it one addition (even offset) or subtraction for all
      const double be = __hiloint2double(hi, lo),
                   sg = __hiloint2double((hi & 0x80000000u) | 0x3ff00000u, 0);
      float T[2][NB];
      lookup(x, y, T);
#pragma unroll
      for (int k = 0; k < 2; k++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
          acc[k][b] = fma(be, (double)T[k][b], acc[k][b]);
          S[k][b] = fma(sg, (double)T[k][b], S[k][b]);
        }
      if (lo & live) {
        put(__builtin_amdgcn_readlane(Cl, j - jb), (float)L, acc);
        live = __builtin_amdgcn_readfirstlane(++j < j1);
        L = rdlane(Ll, j - jb);
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
          for (int b = 0; b < NB; b++) acc[k][b] = L * S[k][b];
      }
    }
  };
  for (uint16s cur = *(const uint16s NIPET_CONST *)ev;; ev += 16) {
    const uint16s nxt = *(const uint16s NIPET_CONST *)(ev + 8);
    eight(cur);
    if (!live) break;
    cur = *(const uint16s NIPET_CONST *)(ev + 16);
    eight(nxt);
    if (!live) break;
  }
  // (lane 63 has no plane 127)
  if (STAGED && faint && (small[0] | (small[1] & (~0ull >> 1)))) {
    q -= (size_t)(j1 - j0) * (128 * NB);
    by_segment();
  }
}

// Most bins of a geometry whose back projections are staged (k_bp_gather keeps a
// bit for each in LDS).
constexpr int BP_NAW = 1 << 17;

// Rows of the launch by transaxial bin, for k_bp_gather. bits: the bins that
// have rows; head[aw].x = last row of bin aw, head[aw].y = its written segments,
// first | count << 16; next[row] = another row of the same bin, or -1 (in no
// fixed order: rows of a bin that is listed more than once are added in any).
__global__ void k_bp_clear(int2 *head, uint32_t *bits, int naw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < naw) head[i].x = -1;
  if (i < BP_NAW / 32) bits[i] = 0;
}
__global__ void k_bp_link(int2 *head, uint32_t *bits, int32_t *next, const int32_t *subs,
                          const int32_t *win, int row0, int n, int naw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int aw = subs ? subs[row0 + i] : row0 + i;
  if (aw < 0 || aw >= naw) return;
  next[i] = atomicExch(&head[aw].x, i);
  head[aw].y = win ? min(max(win[2 * aw], 0), 1024) | min(max(win[2 * aw + 1], 0), 1024) << 16
                   : 1024 << 16;
  atomicOr(&bits[aw >> 5], 1u << (aw & 31));
}

// Sums the staged rows of every voxel column: one wave per column, which walks
// the column's segments of all bins (GeomView::col_ent, ascending, so the order
// of the bins is fixed) and adds the rows of the bins in this launch, 512 bytes an
// image each. add: to the image (later passes) rather than over it.
// A column has a few hundred entries, of which one in 14 (a subset) has a row:
// 64 BP_GE entries are read together and sieved with the bins' bits in LDS;
// what is left is collected there and read eight rows at a time. Bound by
// reading the rows (0.68 GB a subset of 4,894 bins: 0.145 ms at the copy's
// rate). Entries one by one through head[] (a line of L2 each): 0.23 ms.
constexpr int BP_GE = 4, BP_GW = 16;
template <int NB>
__global__ __launch_bounds__(64 * BP_GW) void k_bp_gather(
    const GeomView NIPET_CONST *gp, float *__restrict__ img, const float *__restrict__ stage,
    const int2 *__restrict__ head, const uint32_t *__restrict__ bits,
    const int32_t *__restrict__ next, Batch bt, int add) {
  __shared__ uint32_t has[BP_NAW / 32];
  __shared__ uint32_t list[BP_GW][64 * BP_GE];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.x * BP_GW + wv;
  const int e1 = __builtin_amdgcn_readfirstlane(gp->col_off[c + 1]), maxseg = gp->maxseg;
  int e0 = __builtin_amdgcn_readfirstlane(gp->col_off[c]);
  for (int i = threadIdx.x; i <= (gp->naw - 1) >> 5; i += 64 * BP_GW) has[i] = bits[i];
  __syncthreads();
  float acc[2 * NB];
#pragma unroll
  for (int b = 0; b < 2 * NB; b++) acc[b] = 0.f;
  const float *st = stage + lane * 2 * NB;
  const unsigned long long below = (1ull << lane) - 1;
  for (; e0 < e1; e0 += 64 * BP_GE) {
    uint32_t ent[BP_GE];
#pragma unroll
    for (int u = 0; u < BP_GE; u++) ent[u] = gp->col_ent[min(e0 + 64 * u + lane, e1 - 1)];
    int n = 0;
#pragma unroll
    for (int u = 0; u < BP_GE; u++) {
      const bool hit = (has[ent[u] >> 15] >> ((ent[u] >> 10) & 31) & 1) && e0 + 64 * u + lane < e1;
      const unsigned long long m = __builtin_amdgcn_ballot_w64(hit);
      if (hit) list[wv][n + __popcll(m & below)] = ent[u];
      n += __popcll(m);
    }
    __builtin_amdgcn_wave_barrier();
    for (int i0 = 0; i0 < n; i0 += 64) {
      const uint32_t e = list[wv][min(i0 + lane, n - 1)];
      const int k = e & 1023;
      const int2 hd = head[e >> 10];
      const int ks = k - (hd.y & 0xffff);  // (outside the bin's window: not written)
      int row = i0 + lane < n && ks >= 0 && ks < hd.y >> 16 ? hd.x : -1;
      for (unsigned long long m; (m = __builtin_amdgcn_ballot_w64(row >= 0)) != 0;) {
        const int at = row * maxseg + k;
        do {
          float v[8][2 * NB];
          const unsigned long long m0 = m;
#pragma unroll
          for (int u = 0; u < 8; u++) {
            if (!m) break;
            ldv<2 * NB>(v[u], st + (size_t)__builtin_amdgcn_readlane(at, __builtin_ctzll(m)) *
                                       (128 * NB));
            m &= m - 1;
          }
          const int nv = __popcll(m0) - __popcll(m);
#pragma unroll
          for (int u = 0; u < 8; u++) {
            if (u >= nv) break;
#pragma unroll
            for (int b = 0; b < 2 * NB; b++) acc[b] += v[u][b];
          }
        } while (m);
        row = row >= 0 ? next[row] : -1;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  float *q = img + (int64_t)c * NZ * bt.nbt + bt.b0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int p = 2 * lane + h;
    if (p >= NZ) continue;
#pragma unroll
    for (int b = 0; b < NB; b++) {
      float *o = q + (int64_t)p * bt.nbt + b;
      *o = add ? *o + acc[h * NB + b] : acc[h * NB + b];
    }
  }
}

// ---------------------------------------------------------------------------
// Element-wise kernels.
__global__ void k_fill(float *p, float v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

// rho = (r + s) / (a n) (0 where |a n| < eps), an = a n (prj/src/recon.cu:381-398)
__global__ void k_osem_corr(float *rho, float *an, const float *a, const float *n,
                            const float *r, const float *s, int64_t nel) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < nel; i += stride) {
    float x = a[i] * n[i];
    float rs = (r ? r[i] : 0.f) + (s ? s[i] : 0.f);
    an[i] = x;
    rho[i] = (x > -EPS && x < EPS) ? 0.f : rs / x;
  }
}

// img = mask ? img * (b / sens) : 0 with b/sens = 0 where |sens| < eps
// (prj/src/recon.cu:234-247, 300-315); images [voxel][nb], sens shared
// (sens_nb = 0) or [voxel][nb].
__global__ void k_osem_update(float *img, const float *b, const float *sens, const uint8_t *mask,
                              int64_t nvox, int nb, int sens_nb) {
  const int64_t n = nvox * nb;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) {
    const int64_t v = i / nb;
    float sv = sens_nb ? sens[i] : sens[v];
    float q = (sv > -EPS && sv < EPS) ? 0.f : b[i] / sv;
    img[i] = mask[v] ? img[i] * q : 0.f;
  }
}

// k_osem_update without the per-element index division: one image, four
// voxels per thread (16-byte loads; mask as 4 bytes), or nb = 2 / 4 images of
// one voxel per thread. The same operations per element.
__device__ inline float osem_q(float b, float sv) {
  return (sv > -EPS && sv < EPS) ? 0.f : b / sv;
}
__global__ void k_osem_update_v4(float4 *img, const float4 *b, const float4 *sens,
                                 const uchar4 *mask, int64_t n4) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n4; i += stride) {
    const float4 x = img[i], bb = b[i], sv = sens[i];
    const uchar4 m = mask[i];
    img[i] = make_float4(m.x ? x.x * osem_q(bb.x, sv.x) : 0.f, m.y ? x.y * osem_q(bb.y, sv.y) : 0.f,
                         m.z ? x.z * osem_q(bb.z, sv.z) : 0.f, m.w ? x.w * osem_q(bb.w, sv.w) : 0.f);
  }
}
template <int NB>
__global__ void k_osem_update_w(float *img, const float *b, const float *sens,
                                const uint8_t *mask, int64_t nvox, int sens_nb) {
  int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; v < nvox; v += stride) {
    float x[NB], bb[NB], sv[NB], out[NB];
    ldv<NB>(x, img + v * NB);
    ldv<NB>(bb, b + v * NB);
    if (sens_nb) {
      ldv<NB>(sv, sens + v * NB);
    } else {
#pragma unroll
      for (int k = 0; k < NB; k++) sv[k] = sens[v];
    }
    const bool m = mask[v] != 0;
#pragma unroll
    for (int k = 0; k < NB; k++) out[k] = m ? x[k] * osem_q(bb[k], sv[k]) : 0.f;
    stv<NB>(img + v * NB, out);
  }
}

// k_osem_update (nb = 1) from the two-image back projection b2[v] = (BP(e),
// BP(a n)): the second image is the subset's sensitivity, stored to sens.
__global__ void k_osem_update_pair(float *img, float *sens, const float2 *b2,
                                   const uint8_t *mask, int64_t nvox) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < nvox; i += stride) {
    const float2 bs = b2[i];
    const float sv = bs.y;
    sens[i] = sv;
    float q = (sv > -EPS && sv < EPS) ? 0.f : bs.x / sv;
    img[i] = mask[i] ? img[i] * q : 0.f;
  }
}

// Siemens histogram with replicates innermost, in[(s * nbinang + ali) * nrep + r]
// (uint32 counts) -> device prompts out[(aw * nsn + s) * out_nb + out_b0 + b]
// (uint16, saturating at 65535) for replicates r = r0 + b, b < nb.
__global__ void k_remgaps_u16b(uint16_t *out, const uint32_t *in, const int32_t *aw2ali, int naw,
                               int nsn, int nbinang, int nrep, int r0, int nb, int out_nb,
                               int out_b0) {
  const int64_t n = (int64_t)naw * nsn * nb;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int64_t t = i / nb;
    const int b = (int)(i - t * nb);
    const int aw = (int)(t / nsn), s = (int)(t - (int64_t)aw * nsn);
    const uint32_t v = in[((int64_t)s * nbinang + aw2ali[aw]) * nrep + r0 + b];
    out[t * out_nb + out_b0 + b] = (uint16_t)(v > 65535u ? 65535u : v);
  }
}

// Gap removal / insertion (d_remgaps / d_putgaps, src/scanner_0.cu:94-105,
// 158-166, plus the transpose of mmraux.py:1141): tiled transposes between the
// Siemens layout (nsn, nbinang) and the device layout (naw, nsn): a 64 x 64 tile of (Siemens bin, sinogram) passes through
// LDS, so Siemens rows are read / written along the bin index and device rows
// along the sinogram index, both coalesced. inv[ali] = active bin of Siemens
// bin ali, or -1 in the gaps (zeros on output).
constexpr int GT = 64;

__global__ void k_gap_inv(int32_t *inv, int nbinang) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nbinang) inv[i] = -1;
}

__global__ void k_gap_inv_set(int32_t *inv, const int32_t *aw2ali, int naw, int nbinang) {
  const int aw = blockIdx.x * blockDim.x + threadIdx.x;
  if (aw < naw) {
    const int a = aw2ali[aw];
    if (a >= 0 && a < nbinang) inv[a] = aw;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_remgaps_t(float *__restrict__ out,
                                                   const T *__restrict__ in,
                                                   const int32_t *__restrict__ inv, int nsn,
                                                   int nbinang) {
  __shared__ float tile[GT][GT + 1];
  const int a0 = blockIdx.x * GT, s0 = blockIdx.y * GT;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < GT; r += 4) {  // r: sinogram, tx: Siemens bin
    const int s = s0 + r, a = a0 + tx;
    tile[r][tx] = (s < nsn && a < nbinang) ? (float)in[(int64_t)s * nbinang + a] : 0.f;
  }
  __syncthreads();
  for (int r = ty; r < GT; r += 4) {  // r: Siemens bin, tx: sinogram
    const int a = a0 + r, s = s0 + tx;
    if (a >= nbinang || s >= nsn) continue;
    const int aw = inv[a];
    if (aw >= 0) out[(int64_t)aw * nsn + s] = tile[tx][r];
  }
}

__global__ __launch_bounds__(256) void k_putgaps_t(float *__restrict__ out,
                                                   const float *__restrict__ in,
                                                   const int32_t *__restrict__ inv, int nsn,
                                                   int nbinang) {
  __shared__ float tile[GT][GT + 1];
  const int a0 = blockIdx.x * GT, s0 = blockIdx.y * GT;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < GT; r += 4) {  // r: Siemens bin, tx: sinogram
    const int a = a0 + r, s = s0 + tx;
    float v = 0.f;
    if (a < nbinang && s < nsn) {
      const int aw = inv[a];
      if (aw >= 0) v = in[(int64_t)aw * nsn + s];
    }
    tile[tx][r] = v;
  }
  __syncthreads();
  for (int r = ty; r < GT; r += 4) {  // r: sinogram, tx: Siemens bin (gaps get 0)
    const int s = s0 + r, a = a0 + tx;
    if (s < nsn && a < nbinang) out[(int64_t)s * nbinang + a] = tile[r][tx];
  }
}

static int ew_blocks(int64_t n) {
  int64_t b = (n + 255) / 256;
  return (int)(b < 8192 ? b : 8192);
}

static void launch_osem_update(float *img, const float *b, const float *sens, const uint8_t *mask,
                               int nb, int sens_nb, hipStream_t st) {
  auto al = [](const void *p, size_t a) { return (uintptr_t)p % a == 0; };
  const size_t a = 4 * (size_t)nb;
  if (nb == 1 && NVOX % 4 == 0 && al(img, 16) && al(b, 16) && al(sens, 16) && al(mask, 4))
    k_osem_update_v4<<<ew_blocks(NVOX / 4), 256, 0, st>>>(
        (float4 *)img, (const float4 *)b, (const float4 *)sens, (const uchar4 *)mask, NVOX / 4);
  else if ((nb == 2 || nb == 4) && al(img, a) && al(b, a) && (!sens_nb || al(sens, a)))
    (nb == 2 ? k_osem_update_w<2> : k_osem_update_w<4>)<<<ew_blocks(NVOX), 256, 0, st>>>(
        img, b, sens, mask, NVOX, sens_nb);
  else
    k_osem_update<<<ew_blocks(NVOX * nb), 256, 0, st>>>(img, b, sens, mask, NVOX, nb, sens_nb);
}

}  // namespace nipet

using namespace nipet;

// Replicate sub-batch width (nipet_tune_set): 4 and 2 launch a projector over two
// images at a time, 1 over one; process-wide.
static std::atomic<int> g_width_fp{4}, g_width_bp{4};
// Run lengths of nipet_tune_set_run: kept and reported; the back projector
// now gives every wave one run.
static std::atomic<int> g_run_bp[3] = {{8}, {4}, {6}};
constexpr int BP_RUNS[3][2] = {{8, 6}, {4, 6}, {6, 4}};

// The calling thread's scratch for back projections (nipet_scratch_set).
static thread_local struct {
  char *buf;
  int64_t bytes;
} t_scratch = {nullptr, 0};

// Rows at the largest (bins per pass, 1.7 GB an image at 406 segments), and bins from which
// staging pays: one image's back projection with float atomics / staged took
// 0.204 / 0.222 ms for 1,024 bins, 0.295 / 0.293 for 1,536, 0.359 / 0.350 for
// 2,048 and 0.742 / 0.673 for a subset of 4,893 (the columns' walk costs the same
// for few bins as for many).
constexpr int BP_PASS = 8192, BP_STAGE_MIN = 1536;

static int64_t bp_scratch_bytes(const Geom *g, int rows, int nb) {
  return (int64_t)g->naw * 8 + BP_NAW / 8 + (int64_t)rows * 4 + 256 + (int64_t)rows * g->rays->maxseg * 512 * nb;
}

// One sub-batch of width NB into img (overwritten in its replicates' places).
// bt.win: the bin's segment window, or every segment when NULL; sino2: the
// second of two images (rows by bin), or NULL.
template <int NB>
static void launch_bprj_w(const Geom *g, float *img, const float *sino, const float *sino2,
                          const int32_t *subs, int nprj, Batch bt, int by_bin, hipStream_t st) {
  const auto *gv = (const GeomView NIPET_CONST *)g->dview;
  const int64_t fixed = bp_scratch_bytes(g, 0, NB), per = bp_scratch_bytes(g, 1, NB) - fixed;
  const bool can = t_scratch.buf && nprj >= BP_STAGE_MIN && g->naw <= BP_NAW;
  const int64_t room = can ? (t_scratch.bytes - fixed) / per : 0;
  if (room < BP_STAGE_MIN) {
    if (bt.b0 == 0) k_fill<<<ew_blocks(NVOX * bt.nbt), 256, 0, st>>>(img, 0.f, NVOX * bt.nbt);
    k_bprj<NB, false><<<nprj, bp_threads<NB>(), 0, st>>>(gv, img, sino, sino2, subs, bt, by_bin, 0);
    return;
  }
  const int rows = (int)std::min<int64_t>(std::min(nprj, BP_PASS), room);
  // head, bits, next, rows
  int2 *head = (int2 *)t_scratch.buf;
  uint32_t *bits = (uint32_t *)(head + g->naw);
  int32_t *next = (int32_t *)(bits + BP_NAW / 32);
  float *stage = (float *)(t_scratch.buf + (g->naw * 8 + BP_NAW / 8 + (int64_t)rows * 4 + 255) / 256 * 256);
  for (int r0 = 0; r0 < nprj; r0 += rows) {
    const int n = std::min(rows, nprj - r0);
    k_bp_clear<<<BP_NAW / 256, 256, 0, st>>>(head, bits, g->naw);
    k_bp_link<<<(n + 255) / 256, 256, 0, st>>>(head, bits, next, subs, bt.win, r0, n, g->naw);
    k_bprj<NB, true><<<n, bp_threads<NB>(), 0, st>>>(gv, stage, sino, sino2, subs, bt, by_bin, r0);
    k_bp_gather<NB><<<NX * NY / BP_GW, 64 * BP_GW, 0, st>>>(gv, img, stage, head, bits, next, bt,
                                                            r0 > 0);
  }
}

template <int MODE>
static void launch_fprj(const Geom *g, float *sino, const float *img, const int32_t *subs,
                        int nprj, const uint16_t *prompts, const float *rho, int rho_nb, int nb,
                        hipStream_t st, const int32_t *win = nullptr) {
  const int wmax = g_width_fp.load();
  for (int b0 = 0; b0 < nb;) {
    const int rem = nb - b0;
    const Batch bt{nb, b0, win};
    const auto *gv = (const GeomView NIPET_CONST *)g->dview;
    if (rem >= 2 && wmax >= 2) {
      const bool vec = nb == 2 && (uintptr_t)img % 8 == 0;
      (vec ? k_fprj<MODE, 2, true> : k_fprj<MODE, 2, false>)<<<nprj, FZ_THREADS, 0, st>>>(
          gv, img, sino, subs, prompts, rho, rho_nb, bt);
      b0 += 2;
    } else {
      (nb == 1 ? k_fprj<MODE, 1, true> : k_fprj<MODE, 1, false>)<<<nprj, FZ_THREADS, 0, st>>>(
          gv, img, sino, subs, prompts, rho, rho_nb, bt);
      b0 += 1;
    }
  }
}

// Back projection of nb images into img, which is overwritten.
static void launch_bprj(const Geom *g, float *img, const float *sino, const int32_t *subs,
                        int nprj, int nb, hipStream_t st, int by_bin = 0,
                        const int32_t *win = nullptr) {
  const int wmax = g_width_bp.load();
  for (int b0 = 0; b0 < nb;) {
    const int rem = nb - b0;
    const Batch bt{nb, b0, win};
    if (rem >= 2 && wmax >= 2) {
      launch_bprj_w<2>(g, img, sino, nullptr, subs, nprj, bt, by_bin, st);
      b0 += 2;
    } else {
      launch_bprj_w<1>(g, img, sino, nullptr, subs, nprj, bt, by_bin, st);
      b0 += 1;
    }
  }
}

static int check_geom(const NipetGeom *g, const char *fn) {
  if (!g) {
    set_error("%s: NULL geometry", fn);
    return NIPET_EINVAL;
  }
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev != g->device) {
    set_error("%s: geometry lives on device %d, current device is %d", fn, g->device, dev);
    return NIPET_ESTATE;
  }
  return NIPET_OK;
}

static int check_nprj(const NipetGeom *g, const int32_t *subs, int nprj, int nb, const char *fn) {
  if (nprj <= 0 || (!subs && nprj != g->naw)) {
    set_error("%s: nprj=%d (must be > 0, and = naw=%d when subs is NULL)", fn, nprj, g->naw);
    return NIPET_EINVAL;
  }
  if (nb < 1 || nb > NIPET_MAXBATCH) {
    set_error("%s: batch %d outside 1..%d", fn, nb, NIPET_MAXBATCH);
    return NIPET_EINVAL;
  }
  if (nb > 1 && g->nsn > 837) {
    set_error("%s: batches need at most 837 sinograms (span 11)", fn);
    return NIPET_EINVAL;
  }
  return NIPET_OK;
}

extern "C" {

int64_t nipet_bprj_scratch(const NipetGeom *g, int nprj, int nb) {
  if (!g || nprj < BP_STAGE_MIN || nb < 1 || g->naw > BP_NAW) return 0;
  return bp_scratch_bytes(g, nprj < BP_PASS ? nprj : BP_PASS, nb > 1 ? 2 : 1);
}

int nipet_scratch_set(void *buf, int64_t bytes) {
  if (bytes < 0 || (!buf && bytes) || (uintptr_t)buf % 256) {
    set_error("nipet_scratch_set: bytes < 0, NULL buffer or buffer not aligned to 256 bytes");
    return NIPET_EINVAL;
  }
  t_scratch.buf = (char *)buf;
  t_scratch.bytes = bytes;
  return NIPET_OK;
}

int nipet_fprj_b(const NipetGeom *g, float *sino, const float *img, const int32_t *subs,
                 int nprj, int nb, int att, void *stream) {
  int rc = check_geom(g, "nipet_fprj");
  if (rc) return rc;
  if ((rc = check_nprj(g, subs, nprj, nb, "nipet_fprj"))) return rc;
  if (!sino || !img || (att != 0 && att != 1)) {
    set_error("nipet_fprj: NULL buffer or att not in {0,1}");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_FPRJ, st);
  if (att)
    launch_fprj<1>(g, sino, img, subs, nprj, nullptr, nullptr, 0, nb, st);
  else
    launch_fprj<0>(g, sino, img, subs, nprj, nullptr, nullptr, 0, nb, st);
  prof_end(PK_FPRJ, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_fprj_seg(const NipetGeom *g, float *sino, const float *img, const int32_t *subs,
                   int nprj, int att, void *stream) {
  int rc = check_geom(g, "nipet_fprj_seg");
  if (rc) return rc;
  if ((rc = check_nprj(g, subs, nprj, 1, "nipet_fprj_seg"))) return rc;
  if (!sino || !img || (att != 0 && att != 1)) {
    set_error("nipet_fprj_seg: NULL buffer or att not in {0,1}");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_FPRJ, st);
  (att ? k_fprj_seg<1, FP_G> : k_fprj_seg<0, FP_G>)<<<nprj, fpg_threads<FP_G>(), 0, st>>>(
      view(g), img, sino, subs);
  prof_end(PK_FPRJ, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_fprj(const NipetGeom *g, float *sino, const float *img, const int32_t *subs, int nprj,
               int att, void *stream) {
  return nipet_fprj_b(g, sino, img, subs, nprj, 1, att, stream);
}

int nipet_bprj_b(const NipetGeom *g, float *img, const float *sino, const int32_t *subs,
                 int nprj, int nb, void *stream) {
  int rc = check_geom(g, "nipet_bprj");
  if (rc) return rc;
  if ((rc = check_nprj(g, subs, nprj, nb, "nipet_bprj"))) return rc;
  if (!sino || !img) {
    set_error("nipet_bprj: NULL buffer");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_BPRJ, st);
  launch_bprj(g, img, sino, subs, nprj, nb, st);
  prof_end(PK_BPRJ, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_bprj(const NipetGeom *g, float *img, const float *sino, const int32_t *subs, int nprj,
               void *stream) {
  return nipet_bprj_b(g, img, sino, subs, nprj, 1, stream);
}

int nipet_osem_sens(const NipetGeom *g, float *sens, const float *an, const int32_t *subs,
                    int nprj, void *stream) {
  int rc = check_geom(g, "nipet_osem_sens");
  if (rc) return rc;
  if ((rc = check_nprj(g, subs, nprj, 1, "nipet_osem_sens"))) return rc;
  if (!sens || !an || !subs) {
    set_error("nipet_osem_sens: NULL buffer");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_BPRJ, st);
  launch_bprj(g, sens, an, subs, nprj, 1, st, 1);
  prof_end(PK_BPRJ, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_osem_window(const NipetGeom *g, const uint8_t *mask, int dilate, int32_t *win,
                      void *stream) {
  int rc = check_geom(g, "nipet_osem_window");
  if (rc) return rc;
  if (!mask || !win || dilate < 0 || dilate > 64) {
    set_error("nipet_osem_window: NULL buffer or dilate outside 0 .. 64");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  uint8_t *m2 = nullptr, *m2d = nullptr;
  hipError_t e = hipMallocAsync((void **)&m2, (size_t)NX * NY, st);
  if (e == hipSuccess && dilate > 0) e = hipMallocAsync((void **)&m2d, (size_t)NX * NY, st);
  if (e != hipSuccess) {
    if (m2) (void)hipFreeAsync(m2, st);
    return hip_fail(e, "nipet_osem_window: hipMallocAsync");
  }
  k_mask_cols<<<(NX * NY + 255) / 256, 256, 0, st>>>(mask, m2);
  if (dilate > 0) k_mask_dilate<<<(NX * NY + 255) / 256, 256, 0, st>>>(m2, m2d, dilate);
  k_seg_window<<<(g->naw + 3) / 4, 256, 0, st>>>(view(g), dilate > 0 ? m2d : m2, win);
  (void)hipFreeAsync(m2, st);
  if (m2d) (void)hipFreeAsync(m2d, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_remgaps(float *out, const void *in, int in_dtype, const int32_t *aw2ali, int naw,
                  int nsn, int nbinang, void *stream) {
  if (!out || !in || !aw2ali || naw <= 0 || nsn <= 0 || nbinang < naw ||
      (in_dtype != 0 && in_dtype != 1)) {
    set_error("nipet_remgaps: bad argument");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  int32_t *inv = nullptr;
  NIPET_HIP(hipMallocAsync((void **)&inv, (size_t)nbinang * sizeof(int32_t), st));
  k_gap_inv<<<(nbinang + 255) / 256, 256, 0, st>>>(inv, nbinang);
  k_gap_inv_set<<<(naw + 255) / 256, 256, 0, st>>>(inv, aw2ali, naw, nbinang);
  const dim3 grid((nbinang + GT - 1) / GT, (nsn + GT - 1) / GT);
  if (in_dtype == 0)
    k_remgaps_t<float><<<grid, 256, 0, st>>>(out, (const float *)in, inv, nsn, nbinang);
  else
    k_remgaps_t<uint16_t><<<grid, 256, 0, st>>>(out, (const uint16_t *)in, inv, nsn, nbinang);
  NIPET_HIP(hipGetLastError());
  NIPET_HIP(hipFreeAsync(inv, st));
  return NIPET_OK;
}

// ---- allocation-free gap removal ----
// The inverse bin map of nipet_remgaps lives in a file-scope device array
// instead of stream-ordered scratch. Host code never passes `scratch` itself
// to a kernel (in host code that name is a host-side stand-in, not a device
// address): the address is looked up once per device with
// hipGetSymbolAddress, with that device current, and kept in g_scratch_dev.
static __device__ __align__(256) int32_t scratch[NIPET_NOALLOC_MAXBINANG];

static std::mutex g_scratch_mu;
static int32_t *g_scratch_dev[NIPET_MAXDEVICES] = {};

static int scratch_ptr(int32_t **out, const char *fn) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, fn);
  if (dev < 0 || dev >= NIPET_MAXDEVICES) {
    set_error("%s: device %d beyond the %d devices this library supports", fn, dev,
              NIPET_MAXDEVICES);
    return NIPET_EINVAL;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", fn, dev,
                hipGetErrorString(e));
      return NIPET_EHIP;
    }
    g_scratch_dev[dev] = (int32_t *)p;
  }
  *out = g_scratch_dev[dev];
  return NIPET_OK;
}

int nipet_remgaps_noalloc(float *out, const void *in, int in_dtype, const int32_t *aw2ali,
                          int naw, int nsn, int nbinang, void *stream) {
  if (!out || !in || !aw2ali || naw <= 0 || nsn <= 0 || nbinang < naw ||
      (in_dtype != 0 && in_dtype != 1)) {
    set_error("nipet_remgaps_noalloc: bad argument");
    return NIPET_EINVAL;
  }
  if (nbinang > NIPET_NOALLOC_MAXBINANG) {
    set_error("nipet_remgaps_noalloc: nbinang = %d exceeds the static scratch of %d bins",
              nbinang, NIPET_NOALLOC_MAXBINANG);
    return NIPET_EINVAL;
  }
  int32_t *inv = nullptr;
  int rc = scratch_ptr(&inv, "nipet_remgaps_noalloc");
  if (rc) return rc;
  hipStream_t st = (hipStream_t)stream;
  // the whole map is rewritten by a kernel in every call (no memset node, so
  // the call may be captured into a graph)
  k_gap_inv<<<(nbinang + 255) / 256, 256, 0, st>>>(inv, nbinang);
  k_gap_inv_set<<<(naw + 255) / 256, 256, 0, st>>>(inv, aw2ali, naw, nbinang);
  const dim3 grid((nbinang + GT - 1) / GT, (nsn + GT - 1) / GT);
  if (in_dtype == 0)
    k_remgaps_t<float><<<grid, 256, 0, st>>>(out, (const float *)in, inv, nsn, nbinang);
  else
    k_remgaps_t<uint16_t><<<grid, 256, 0, st>>>(out, (const uint16_t *)in, inv, nsn, nbinang);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_remgaps_u16b(uint16_t *out, const uint32_t *in, const int32_t *aw2ali, int naw,
                       int nsn, int nbinang, int nrep, int r0, int nb, int out_nb, int out_b0,
                       void *stream) {
  if (!out || !in || !aw2ali || naw <= 0 || nsn <= 0 || nbinang <= 0 || nrep < 1 || r0 < 0 ||
      nb < 1 || r0 + nb > nrep || out_b0 < 0 || out_b0 + nb > out_nb) {
    set_error("nipet_remgaps_u16b: bad arguments (naw=%d nsn=%d nrep=%d r0=%d nb=%d out_nb=%d "
              "out_b0=%d)", naw, nsn, nrep, r0, nb, out_nb, out_b0);
    return NIPET_EINVAL;
  }
  const int64_t n = (int64_t)naw * nsn * nb;
  k_remgaps_u16b<<<ew_blocks(n), 256, 0, (hipStream_t)stream>>>(out, in, aw2ali, naw, nsn,
                                                               nbinang, nrep, r0, nb, out_nb,
                                                               out_b0);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_tune_set(int kernel, int width) {
  if ((kernel != NIPET_PROF_FPRJ && kernel != NIPET_PROF_BPRJ) ||
      (width != 1 && width != 2 && width != 4)) {
    set_error("nipet_tune_set: kernel must be FPRJ or BPRJ and width 1, 2 or 4");
    return NIPET_EINVAL;
  }
  (kernel == NIPET_PROF_FPRJ ? g_width_fp : g_width_bp).store(width);
  return NIPET_OK;
}

int nipet_tune_set_run(int width, int spw) {
  const int k = width == 1 ? 0 : (width == 2 ? 1 : (width == 4 ? 2 : -1));
  if (k < 0 || (spw != BP_RUNS[k][0] && spw != BP_RUNS[k][1])) {
    set_error("nipet_tune_set_run: width must be 1, 2 or 4 and the run length 8 or 6 (1), 4 or 6 "
              "(2 and 4)");
    return NIPET_EINVAL;
  }
  g_run_bp[k].store(spw);
  return NIPET_OK;
}

int nipet_tune_get_run(int width, int *spw, int *alt) {
  const int k = width == 1 ? 0 : (width == 2 ? 1 : (width == 4 ? 2 : -1));
  if (k < 0 || !spw) {
    set_error("nipet_tune_get_run: width must be 1, 2 or 4");
    return NIPET_EINVAL;
  }
  *spw = g_run_bp[k].load();
  if (alt) *alt = *spw == BP_RUNS[k][0] ? BP_RUNS[k][1] : BP_RUNS[k][0];
  return NIPET_OK;
}

int nipet_tune_get(int kernel, int *width) {
  if ((kernel != NIPET_PROF_FPRJ && kernel != NIPET_PROF_BPRJ) || !width) {
    set_error("nipet_tune_get: kernel must be FPRJ or BPRJ");
    return NIPET_EINVAL;
  }
  *width = (kernel == NIPET_PROF_FPRJ ? g_width_fp : g_width_bp).load();
  return NIPET_OK;
}

int nipet_putgaps(float *out, const float *in, const int32_t *aw2ali, int naw, int nsn,
                  int nbinang, void *stream) {
  if (!out || !in || !aw2ali || naw <= 0 || nsn <= 0 || nbinang < naw) {
    set_error("nipet_putgaps: bad argument");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  int32_t *inv = nullptr;
  NIPET_HIP(hipMallocAsync((void **)&inv, (size_t)nbinang * sizeof(int32_t), st));
  k_gap_inv<<<(nbinang + 255) / 256, 256, 0, st>>>(inv, nbinang);
  k_gap_inv_set<<<(naw + 255) / 256, 256, 0, st>>>(inv, aw2ali, naw, nbinang);
  const dim3 grid((nbinang + GT - 1) / GT, (nsn + GT - 1) / GT);
  k_putgaps_t<<<grid, 256, 0, st>>>(out, in, inv, nsn, nbinang);
  NIPET_HIP(hipGetLastError());
  NIPET_HIP(hipFreeAsync(inv, st));
  return NIPET_OK;
}

int nipet_osem_corr(float *rho, float *an, const float *a, const float *n, const float *r,
                    const float *s, int64_t nelem, void *stream) {
  if (!rho || !an || !a || !n || nelem <= 0) {
    set_error("nipet_osem_corr: NULL buffer or nelem <= 0");
    return NIPET_EINVAL;
  }
  k_osem_corr<<<ew_blocks(nelem), 256, 0, (hipStream_t)stream>>>(rho, an, a, n, r, s, nelem);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_osem_subset_b(const NipetGeom *g, float *img, const uint16_t *prompts,
                        const float *rho, int rho_per_rep, const float *sens, int sens_per_rep,
                        const uint8_t *mask, const int32_t *win, const int32_t *subs, int nprj,
                        int nb, float *work_sino, float *work_img, void *stream) {
  int rc = check_geom(g, "nipet_osem_subset");
  if (rc) return rc;
  if (!subs || nprj <= 0 || nprj > g->naw) {
    set_error("nipet_osem_subset: subs must be given with 0 < nprj <= naw");
    return NIPET_EINVAL;
  }
  if ((rc = check_nprj(g, subs, nprj, nb, "nipet_osem_subset"))) return rc;
  if (!img || !prompts || !rho || !sens || !mask || !work_sino || !work_img || work_img == img ||
      work_img == sens) {
    set_error("nipet_osem_subset: NULL or aliased buffer");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_FPRJ, st);
  launch_fprj<2>(g, work_sino, img, subs, nprj, prompts, rho, rho_per_rep ? 1 : 0, nb, st, win);
  prof_end(PK_FPRJ, st);
  prof_begin(PK_BPRJ, st);
  launch_bprj(g, work_img, work_sino, subs, nprj, nb, st, 0, win);
  prof_end(PK_BPRJ, st);
  prof_begin(PK_OSEM_UPDATE, st);
  launch_osem_update(img, work_img, sens, mask, nb, sens_per_rep ? 1 : 0, st);
  prof_end(PK_OSEM_UPDATE, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_osem_subset_rm_b(const NipetGeom *g, float *img, const uint16_t *prompts,
                           const float *rho, int rho_per_rep, const float *sens,
                           int sens_per_rep, const uint8_t *mask, const int32_t *win,
                           const int32_t *subs, int nprj, int nb, const float *krnl,
                           float *work_sino, float *work_img, float *work_img2, void *stream) {
  int rc = check_geom(g, "nipet_osem_subset_rm");
  if (rc) return rc;
  if (!subs || nprj <= 0 || nprj > g->naw) {
    set_error("nipet_osem_subset_rm: subs must be given with 0 < nprj <= naw");
    return NIPET_EINVAL;
  }
  if ((rc = check_nprj(g, subs, nprj, nb, "nipet_osem_subset_rm"))) return rc;
  if (!img || !prompts || !rho || !sens || !mask || !krnl || !work_sino || !work_img ||
      !work_img2 || work_img == work_img2 || work_img == img || work_img2 == img ||
      work_img == sens || work_img2 == sens) {
    set_error("nipet_osem_subset_rm: NULL or aliased buffer");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  // resolution-modelled image H x (work_img is the convolution scratch)
  if ((rc = psf_conv(work_img2, img, work_img, krnl, nb, st))) return rc;
  prof_begin(PK_FPRJ, st);
  launch_fprj<2>(g, work_sino, work_img2, subs, nprj, prompts, rho, rho_per_rep ? 1 : 0, nb, st,
                 win);
  prof_end(PK_FPRJ, st);
  prof_begin(PK_BPRJ, st);
  launch_bprj(g, work_img, work_sino, subs, nprj, nb, st, 0, win);
  prof_end(PK_BPRJ, st);
  // H^T of the back projection (symmetric kernels: H), into work_img2
  if ((rc = psf_conv(work_img2, work_img, work_img, krnl, nb, st))) return rc;
  prof_begin(PK_OSEM_UPDATE, st);
  launch_osem_update(img, work_img2, sens, mask, nb, sens_per_rep ? 1 : 0, st);
  prof_end(PK_OSEM_UPDATE, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_osem_subset(const NipetGeom *g, float *img, const uint16_t *prompts, const float *rho,
                      const float *sens, const uint8_t *mask, const int32_t *win,
                      const int32_t *subs, int nprj, float *work_sino, float *work_img,
                      void *stream) {
  return nipet_osem_subset_b(g, img, prompts, rho, 0, sens, 0, mask, win, subs, nprj, 1,
                             work_sino, work_img, stream);
}

int nipet_osem_subset_sens(const NipetGeom *g, float *img, const uint16_t *prompts,
                           const float *rho, const float *an, float *sens, const uint8_t *mask,
                           const int32_t *win, const int32_t *subs, int nprj, float *work_sino,
                           float *work_sino2, float *work_img2, void *stream) {
  int rc = check_geom(g, "nipet_osem_subset_sens");
  if (rc) return rc;
  if (!subs || nprj <= 0 || nprj > g->naw) {
    set_error("nipet_osem_subset_sens: subs must be given with 0 < nprj <= naw");
    return NIPET_EINVAL;
  }
  if ((rc = check_nprj(g, subs, nprj, 2, "nipet_osem_subset_sens"))) return rc;
  if (!img || !prompts || !rho || !an || !sens || !mask || !work_sino || !work_sino2 ||
      !work_img2 || sens == img || work_sino == work_sino2 || work_img2 == img ||
      work_img2 == sens) {
    set_error("nipet_osem_subset_sens: NULL or aliased buffer");
    return NIPET_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  prof_begin(PK_FPRJ, st);
  launch_fprj<2>(g, work_sino, img, subs, nprj, prompts, rho, 0, 1, st, win);
  prof_end(PK_FPRJ, st);
  // both images through one traversal of the rays (independent of the
  // batch autotuner's width)
  prof_begin(PK_BPRJ_PAIR, st);
  launch_bprj_w<2>(g, work_img2, work_sino, an, subs, nprj, Batch{2, 0, win}, 0, st);
  prof_end(PK_BPRJ_PAIR, st);
  prof_begin(PK_OSEM_UPDATE, st);
  k_osem_update_pair<<<ew_blocks(NVOX), 256, 0, st>>>(img, sens, (const float2 *)work_img2, mask,
                                                      NVOX);
  prof_end(PK_OSEM_UPDATE, st);
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

int nipet_osem_iter(const NipetGeom *g, float *img, const uint16_t *prompts, const float *r,
                    const float *s, const float *n, const float *a, const int32_t *subs,
                    int nsub, int stride, const float *sens, const uint8_t *mask,
                    const float *krnl, void *stream) {
  int rc = check_geom(g, "nipet_osem_iter");
  if (rc) return rc;
  if (!img || !prompts || !n || !a || !subs || !sens || !mask || nsub < 1 || stride < 2) {
    set_error("nipet_osem_iter: NULL buffer, nsub < 1 or stride < 2");
    return NIPET_EINVAL;
  }
  int maxc = 0;
  for (int i = 0; i < nsub; i++) {
    const int c = subs[(int64_t)i * stride];
    if (c < 1 || c > stride - 1 || c > g->naw) {
      set_error("nipet_osem_iter: subset %d holds %d bins (must be 1 .. min(stride - 1 = %d, "
                "naw = %d))", i, c, stride - 1, g->naw);
      return NIPET_EINVAL;
    }
    maxc = c > maxc ? c : maxc;
  }
  const bool rm = krnl && krnl[0] >= 0.f;
  hipStream_t st = (hipStream_t)stream;
  const int64_t nel = (int64_t)g->naw * g->nsn;
  // per-call temporaries, stream ordered (the reference allocates and frees
  // its device copies in every call, prj/src/recon.cu:333-419, 511-520)
  float *rho = nullptr, *an = nullptr, *wsino = nullptr, *wimg = nullptr, *wimg2 = nullptr,
        *srm = nullptr;
  int32_t *dsubs = nullptr, *win = nullptr;
  auto release = [&]() {
    void *ps[] = {rho, an, wsino, wimg, wimg2, srm, dsubs, win};
    for (void *q : ps)
      if (q) (void)hipFreeAsync(q, st);
  };
  auto get = [&](void **p, size_t bytes) -> int {
    hipError_t e = hipMallocAsync(p, bytes, st);
    if (e != hipSuccess) {
      *p = nullptr;
      release();
      return hip_fail(e, "nipet_osem_iter: hipMallocAsync");
    }
    return NIPET_OK;
  };
  if ((rc = get((void **)&rho, nel * sizeof(float))) || (rc = get((void **)&an, nel * sizeof(float))) ||
      (rc = get((void **)&wsino, (size_t)maxc * g->nsn * sizeof(float))) ||
      (rc = get((void **)&wimg, NVOX * sizeof(float))) ||
      (rc = get((void **)&dsubs, (size_t)nsub * stride * sizeof(int32_t))) ||
      (rc = get((void **)&win, (size_t)g->naw * 2 * sizeof(int32_t))))
    return rc;
  if (rm && ((rc = get((void **)&wimg2, NVOX * sizeof(float))) ||
             (rc = get((void **)&srm, NVOX * sizeof(float)))))
    return rc;
  hipError_t e = hipMemcpyAsync(dsubs, subs, (size_t)nsub * stride * sizeof(int32_t),
                                hipMemcpyHostToDevice, st);
  if (e != hipSuccess) {
    release();
    return hip_fail(e, "nipet_osem_iter: subset table upload");
  }
  // rho = (r + s) / (a n) once per call (prj/src/recon.cu:381-398)
  k_osem_corr<<<ew_blocks(nel), 256, 0, st>>>(rho, an, a, n, r, s, nel);
  // the mask's segment windows (dilated by the resolution model's reach):
  // after the first update img is zero outside the mask, so the later subsets
  // walk only the segments whose columns meet it
  if ((rc = nipet_osem_window(g, mask, rm ? PSF_R : 0, win, stream))) {
    release();
    return rc;
  }
  for (int i = 0; i < nsub && rc == NIPET_OK; i++) {
    const int c = subs[(int64_t)i * stride];
    const int32_t *rows = dsubs + (int64_t)i * stride + 1;
    const float *si = sens + (int64_t)i * NVOX;
    const int32_t *wi = i > 0 ? win : nullptr;
    if (rm) {
      // the reference convolves the sensitivity images in every call
      // (prj/src/recon.cu:441-445); here one at a time, before its subset
      if ((rc = psf_conv(srm, si, wimg, krnl, 1, st))) break;
      rc = nipet_osem_subset_rm_b(g, img, prompts, rho, 0, srm, 0, mask, wi, rows, c, 1, krnl,
                                  wsino, wimg, wimg2, stream);
    } else {
      rc = nipet_osem_subset_b(g, img, prompts, rho, 0, si, 0, mask, wi, rows, c, 1, wsino, wimg,
                               stream);
    }
  }
  release();
  if (rc) return rc;
  NIPET_HIP(hipGetLastError());
  return NIPET_OK;
}

}  // extern "C"
