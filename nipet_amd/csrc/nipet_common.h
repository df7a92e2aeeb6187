// Shared definitions of the gfx950 NIPET library (device image / sinogram
// geometry, the geometry object, error reporting).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>
#include <vector>

#include "nipet_hip.h"

namespace nipet {

constexpr int NX = 320;   // device image x (u)
constexpr int NY = 320;   // device image y (v)
constexpr int NZ = 127;   // device image z (w), fastest
// segments of one transaxial ray: one per voxel column it crosses, at most
// one more than the grid lines it crosses (checked when the geometry is built)
constexpr int MAX_SEG = NX + NY + 1;
constexpr int SEG_PAD = 128;  // records behind the last list (whole chunks are read)
constexpr int64_t NVOX = (int64_t)NX * NY * NZ;
constexpr int MAXNSN = 4096;  // largest sinogram count handled (span-1: 4084)
constexpr int LI_MAX = 2112;  // largest Michelogram (ring pair) count
constexpr float EPS = 1e-6f;  // OSEM division guard (prj/src/recon.cu:12)
constexpr int PSF_R = 8;      // PSF kernel half-width (17 taps)

// One transaxial segment: start t (cm from the first crystal, double so that
// z-boundary positions along the ray keep sub-nanometre precision), length
// (cm) and the z-column base offset 127*(u + 320 v) of its voxel column.
struct __align__(16) SegRec {
  double s;
  float len;
  int32_t colz;
};

// What the kernels read of a geometry.
struct GeomView {
  const int32_t *off;
  const SegRec *seg;
  const double *atn;
  const uint2 *ev;
  const float *lmax;
  const float2 *li_z;
  const short2 *li_sn;
  const float *li_nosi;
  const int16_t *dr_li;
  const uint16_t *sn_mem;
  const uint32_t *bp_tab;
  const uint2 *bp_ev;
  const uint32_t *bp_off;
  const int32_t *col_off;
  const uint32_t *col_ent;
  const int16_t *fp_slot;
  int naw, nli, ndirect, nsn, dmax, sn_w, fp_nslot, maxseg;
  float vox_z;
};

// The rays of a scanner on one device: transaxial intersection lists in CSR form
// (segments of ray aw are seg[off[aw] .. off[aw+1])) and the z crossings along
// them, 4.3 GB for 68,516 bins of 272 segments. They depend on the crystals, the
// grid and the largest ring difference, not on spans or sinograms: geometries of
// the same rays share them (rays_get).
struct Rays {
  // what they are made of
  int device = 0, naw = 0, dmax = 0;  // dmax: largest ring difference d
  float vox_xy = 0.f, tfov2 = 0.f;
  std::vector<float> crs;
  std::vector<int16_t> s2c;

  int64_t nseg = 0;
  int maxseg = 0;            // longest list
  int32_t *off = nullptr;    // [naw+1]
  SegRec *seg = nullptr;     // [nseg]
  double *atn = nullptr;     // [naw] crystal-to-crystal transaxial distance
  float *lmax = nullptr;     // [naw] longest segment of the ray
  // z crossings of a ray [naw][ev_off(dmax + 1)]: entry ev_off(d) + w is where
  // the LORs of ring difference d pass from plane offset w to w + 1, at t =
  // (w + 1/2) atn / (2 d): how far into its segment, as a fraction in float64,
  // with its low 20 bits (2^-32 of it) replaced by segment << 10 | ev_phi(w);
  // segment 1023 past the end of the list
  uint2 *ev = nullptr;
  // z crossings in the order of the back projector's walk (nseg_ev entries, see
  // bp_event) and the first entry of every segment [nseg + 1]
  uint2 *bp_ev = nullptr;
  uint32_t *bp_off = nullptr;
  // segments by voxel column (CSR): bin << 10 | segment of the bin's list, ascending
  int32_t *col_off = nullptr;   // [NX * NY + 1]
  uint32_t *col_ent = nullptr;  // [nseg]

  Rays() = default;
  Rays(const Rays &) = delete;
  ~Rays();
};

// Geometry resident on one device: rays, and the sinograms their LORs belong to.
struct Geom {
  int device = 0;
  int naw = 0, nli = 0, nsn = 0, ncrs = 0, ndirect = 0;
  std::shared_ptr<const Rays> rays;
  float vox_z = 0.203125f;
  float2 *li_z = nullptr;    // [nli] (zeta_a at t=0, zeta_b - zeta_a) in z-voxel units
  short2 *li_sn = nullptr;   // [nli] output sinogram of LOR a and of its mirror b
  float *li_nosi = nullptr;  // [nli] 1 / (span-1 LORs per output sinogram)
  // ring-difference view of the Michelogram: element li joins ring r0 (LOR a
  // starts there) and ring r0 + d
  int dmax = 0;                // largest ring difference d
  int16_t *dr_li = nullptr;    // [64 * 64] li of (d, r0) at d * 64 + r0, -1 if absent
  // the span-1 LORs of each output sinogram [nsn][sn_w]: 2 li (LOR a) or
  // 2 li + 1 (mirror b), 2 LI_MAX where there are fewer (span 11: at most 6)
  uint16_t *sn_mem = nullptr;
  int sn_w = 8;  // a multiple of 8
  // segment-walking forward projector (k_fprj_seg): slot s walks the LORs
  // (d, r0 + k), k < FP_G, of one ring difference; fp_slot[s] = d * 64 + r0
  int16_t *fp_slot = nullptr;
  int fp_nslot = 0;
  // back-projector LOR table [BP_TN]: at 65 d + r0 the sinograms of LOR (r0, d)
  // and (<< 16) of its mirror; nsn where there is none
  uint32_t *bp_tab = nullptr;
  GeomView view = {};           // the pointers above, and
  GeomView *dview = nullptr;    // its copy on the device
};

// Rows 0 .. 63 of the back projector's LOR table: row d has its 64 - d LORs at
// 65 d, then d + 1 zeros up to row d + 1, so that r0 = -d .. 63 reads zeros
// where there is no LOR; 64 more behind the last row.
constexpr int BP_MAXD = 63;
constexpr int BP_TN = 65 * (BP_MAXD + 1) + 64;

// Plane offset of the LORs of one ring difference at t = s (m = 2 d / atn).
__device__ inline int plane_offset(double m, double s) { return (int)floor(fma(m, s, 0.5)); }

// Entry of Rays::bp_ev: the LORs of ring difference d pass from plane offset w
// to w + 1, beta before the segment's end. A float64 +beta (w even) or -beta
// (odd) with its low 23 bits (2^-30 of beta) replaced by: 1 for the segment's
// last entry, 4 D, and d << 16. The LORs are at entries D + i, D + i + 1 (one
// direction, planes 2 i and 2 i + 1) and BP_TN + 1 + 129 d - D + i (the other,
// both planes) of the kernel's table: vb, one unused entry, va. A segment
// without crossings has one entry of ring difference 64, which has no LORs.
__host__ __device__ constexpr uint32_t bp_entry(int d, int w) {
  return w & 1 ? BP_TN + 65 * d - (w >> 1) : 64 * d + (w >> 1);
}
__device__ inline uint2 bp_event(int d, int w, double beta, bool last) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(w & 1 ? -beta : beta);
  return make_uint2(((uint32_t)b & 0xff800000u) | (uint32_t)d << 16 | bp_entry(d, w) << 2 |
                        (last ? 1u : 0u),
                    (uint32_t)(b >> 32));
}

// Position of plane w in the forward projector's LDS rows (64 even planes, then
// 64 odd ones, of 8 bytes), in bytes.
__host__ __device__ constexpr int ev_phi(int w) { return ((w & 1) << 9) + ((w >> 1) << 3); }
constexpr uint32_t EV_PLACE = 0xfffffu;  // the place in an entry of Rays::ev
static_assert(MAX_SEG < 1023, "segments in 10 bits");
// Crossings of ring difference d in Rays::ev: 2 d, and eight that lie past any
// segment (eight are read at a time).
__host__ __device__ constexpr int ev_off(int d) { return (d - 1) * (d + 8); }

constexpr int FP_G = 3;          // LORs per lane of k_fprj_seg
constexpr int FP_G_SLOTS = 768;  // lanes of that kernel

void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);

// Separable 17-tap convolution of nb replicate-innermost images, kernels
// krnl[3][17] (host) for z, x, y: in -> out, tmp a scratch image (out must
// differ from in and tmp; tmp may be in, which is then overwritten). Launches
// on st only (no synchronisation, no allocation).
int psf_conv(float *out, const float *in, float *tmp, const float *krnl, int nb,
             hipStream_t st);

// Opt-in kernel timing (nipet_prof_*): HIP events recorded around launches on
// the launch stream, resolved when read.
enum ProfKernel {
  PK_FPRJ = 0, PK_BPRJ, PK_OSEM_UPDATE, PK_FILL, PK_HIST, PK_OTHER, PK_BPRJ_PAIR, PK_COUNT
};
void prof_begin(int kernel, hipStream_t st);
void prof_end(int kernel, hipStream_t st);

}  // namespace nipet

struct NipetGeom : nipet::Geom {};

#define NIPET_HIP(call)                                              \
  do {                                                               \
    hipError_t e_ = (call);                                          \
    if (e_ != hipSuccess) return nipet::hip_fail(e_, #call);         \
  } while (0)
