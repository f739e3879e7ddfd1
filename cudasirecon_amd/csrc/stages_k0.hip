// k0 search: overlap construction and inverse FFT, the z-summed overlap
// products, the cross-correlation peak, and the batched modamp reductions.
//
// Reference (src/cudaSirecon/gpuFunctionsImpl.cu): makeoverlaps 497-675 with
// makeOverlaps0Kernel 677-778 / makeOverlaps1Kernel 780-872, aTimesConjB
// 374-414, computeIntensities 416-441, findrealspacemodamp 1074-1148,
// reductionKernel 1150-1220.
//
// Differences in structure (same values up to FP reassociation):
//  * overlaps are generated inside the x-pass of the inverse FFT, only for
//    the 2*zd+1 planes the support can reach; the zero planes are never
//    written;
//  * the fit reads only the per-(x,y) z sums P = sum_z conj(X) Y, SX, SY,
//    which Parseval's identity along z forms from the stored kz planes, so
//    there is no z transform, and the 3D overlap volumes are never re-read:
//    every later line-search step is a 2D reduction of P against a phase ramp;
//  * a whole batch of line-search candidates is reduced in one launch;
//  * every launch covers the overlap pairs (or candidates) of all directions
//    being fitted, one slot per direction, so a launch fills the GPU and the
//    directions share each host read-back.
#include <type_traits>

#include "device_math.hpp"
#include "fft.hpp"
#include "fft2.hpp"
#include "fft_api.hpp"
#include "fft_rp.hpp"
#include "fit_device.hpp"
#include "sizes.hpp"
#include "stages.hpp"

namespace simr {

// Sequential sums in block order, as the host's loops make them, of K
// interleaved components at once: the workgroup stages a chunk of the
// entries in LDS with every thread (coalesced, all loads in flight), then
// lane k adds up component k in order, eight staged values loaded ahead of
// each eight additions.  Returns lane k's sum (k < K).
constexpr int kSeqChunk = 1024;  // entries per LDS chunk

template <typename T, int K, typename Get>
__device__ __forceinline__ T seq_sum_lanes(int n, double* stage, Get get) {
#pragma clang fp contract(off)
  T acc = 0;
  const int lane = threadIdx.x;
  for (int c0 = 0; c0 < n; c0 += kSeqChunk) {
    const int m = n - c0 < kSeqChunk ? n - c0 : kSeqChunk;
    for (int i = threadIdx.x; i < m * K; i += blockDim.x) stage[i] = get(c0 + i / K, i % K);
    __syncthreads();
    if (lane < K) {
      int i = 0;
      for (; i + 8 <= m; i += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = stage[(i + u) * K + lane];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += (T)v[u];
      }
      for (; i < m; ++i) acc += (T)stage[i * K + lane];
    }
    __syncthreads();
  }
  return acc;
}

// Where one element of overlap0 (which == 0) or overlap1 (which == 1) at
// column j, row i, plane z0 comes from, before the inverse transform: its
// band index, the conjugation of the Hermitian mirror, and the OTF factor
// (makeOverlaps0Kernel / makeOverlaps1Kernel).  ok = false: the element is
// zero.  prof1/prof2: radial OTF profiles of order1/order2 at kz = z0.
//
// The reference's tests sqrtf(d) <= rdistcutoff and sqrtf(|otf|^2) * f >
// otfcutoff are made on the squares (sums of squares in fused form), the OTF
// radius index is the hardware square root of d / dkr^2 and the
// normalisation 1/sqrt(|a|^2 + |b|^2) the hardware reciprocal square root:
// within a few ulps of the reference's
// correctly rounded sqrtf and divisions (an element exactly on a cut-off
// circle may land on the other side), far inside the overlap tolerance, at
// a third of the instructions.
struct OvSrc {
  int ind;
  bool ok, conj;
  float2 fact;
};

// Bilinear profile lookup (dev_otfinterpolate's radial interpolation) at a
// radius index that is a square root, so never negative: truncation is the
// floor and the clamp at 0 cannot act; t0 + ar (t1 - t0) in fused form is
// within an ulp of (1 - ar) t0 + ar t1.
__device__ __forceinline__ float2 prof_lerp(const float2* prof, int nxotf, float krindex) {
  int irindex = (int)krindex;
  float ar = __builtin_amdgcn_fractf(krindex);
  if (irindex > nxotf - 2) {
    irindex = nxotf - 2;
    ar = 1.f;
  }
  const float2 t0 = prof[irindex], t1 = prof[irindex + 1];
  return make_float2(__builtin_fmaf(ar, t1.x - t0.x, t0.x), __builtin_fmaf(ar, t1.y - t0.y, t0.y));
}

template <bool RA>
__device__ __forceinline__ OvSrc ov_source(const OvParams& p, float kx, float ky, const float2* prof1,
                                           const float2* prof2, int which, int j, int i, int z0) {
#pragma clang fp contract(off)
  OvSrc o{0, false, false, make_float2(0.f, 0.f)};
  float x1f = (float)j, y1f = (float)i;
  if (x1f > (float)(p.nx / 2)) x1f -= (float)p.nx;
  if (y1f > (float)(p.ny / 2)) y1f -= (float)p.ny;
  x1f *= p.dkx;
  y1f *= p.dky;
  const float d1 = __builtin_fmaf(x1f, x1f, y1f * y1f);
  if (which == 0 ? !(d1 <= p.rc2) : !(d1 < p.rc2)) return o;
  const float x12 = x1f - kx, y12 = y1f - ky;
  const float d12 = __builtin_fmaf(x12, x12, y12 * y12);
  const float x21 = x1f + kx, y21 = y1f + ky;
  const float d21 = __builtin_fmaf(x21, x21, y21 * y21);
  if (!(d12 <= p.rc2 || d21 <= p.rc2)) return o;
  if (z0 == 0 && p.bNoKz0) return o;
  int iin, jin;
  if (j <= p.nx / 2) {
    iin = i;
    jin = j;
  } else {
    jin = p.nx - j;
    iin = i == 0 ? 0 : p.ny - i;
    o.conj = true;
  }
  int zin = o.conj ? -z0 : z0;
  if (zin < 0) zin += p.nz;
  float2 oa, ob;  // own-order OTF at k, other-order OTF at the shifted k
  float sa2, sb2; // their cutoff scales, squared
  if (which == 0) {
    if (!(d12 <= p.rc2)) return o;
    if constexpr (RA) {
      oa = prof_lerp(prof1, p.otf1.nxotf, __builtin_amdgcn_sqrtf(d1 * p.inv_dkr2_1));
      ob = prof_lerp(prof2, p.otf2.nxotf, __builtin_amdgcn_sqrtf(d12 * p.inv_dkr2_2));
    } else {
      oa = otf3d_interp(p.otf1, x1f, y1f, z0, p.kzscale);
      ob = otf3d_interp(p.otf2, x12, y12, z0, p.kzscale);
    }
    sa2 = 1.f;
    sb2 = p.f2;
  } else {
    if (!(d21 <= p.rc2)) return o;
    if constexpr (RA) {
      oa = prof_lerp(prof2, p.otf2.nxotf, __builtin_amdgcn_sqrtf(d1 * p.inv_dkr2_2));
      ob = prof_lerp(prof1, p.otf1.nxotf, __builtin_amdgcn_sqrtf(d21 * p.inv_dkr2_1));
    } else {
      oa = otf3d_interp(p.otf2, x1f, y1f, z0, p.kzscale);
      ob = otf3d_interp(p.otf1, x21, y21, z0, p.kzscale);
    }
    sa2 = p.f2;
    sb2 = 1.f;
  }
  const float ma = __builtin_fmaf(oa.x, oa.x, oa.y * oa.y), mb = __builtin_fmaf(ob.x, ob.x, ob.y * ob.y);
  if (!(ma * sa2 > p.cut2)) return o;
  if (!(mb * sb2 > p.cut2)) return o;
  const float rroot = __builtin_amdgcn_rsqf(ma + mb);
  o.fact = make_float2(ob.x * rroot, ob.y * rroot);
  o.ind = (zin * p.ny + iin) * p.nxh + jin;
  o.ok = true;
  return o;
}

// The overlap element from its source and the two band values read there.
__device__ __forceinline__ float2 ov_combine(const OvSrc& o, float2 vre, float2 vim, bool has_im) {
#pragma clang fp contract(off)
  if (!o.ok) return make_float2(0.f, 0.f);
  if (!has_im) vim = make_float2(0.f, 0.f);
  if (o.conj) {
    vre.y = -vre.y;
    vim.y = -vim.y;
  }
  vre = cmul_nc(vre, o.fact);
  vim = cmul_nc(vim, o.fact);
  return make_float2(vre.x - vim.y, vre.y + vim.x);
}

// Whether row i of overlap `which` can hold a nonzero element: an element at
// lateral frequency (x, y) is nonzero only if |(x, y)| and |(x, y) - s| are
// both within rdistcutoff (s = (kx, ky) for overlap0, -(kx, ky) for overlap1;
// no wrap-around), so the row meets both discs iff |sx| <= a + b with
// a^2 = rc^2 - y^2 and b^2 = rc^2 - (y - sy)^2.  The radii carry a relative
// margin of 1e-4, far beyond the rounding of the per-element tests, so a row
// this rejects is zero.
__device__ __forceinline__ bool ov_row_live(const OvParams& p, float kx, float ky, int which, int i, int z0) {
  if (i >= p.ny || (z0 == 0 && p.bNoKz0)) return false;
  float y = (float)i;
  if (y > (float)(p.ny / 2)) y -= (float)p.ny;
  y *= p.dky;
  const float sx = which == 0 ? kx : -kx, sy = which == 0 ? ky : -ky;
  const float r2 = p.rc2 * 1.0002f;
  const float a2 = r2 - y * y, b2 = r2 - (y - sy) * (y - sy);
  if (a2 < 0.f || b2 < 0.f) return false;
  return fabsf(sx) <= (sqrtf(a2) + sqrtf(b2)) * 1.0001f;
}

// x pass: rows [R*(blockIdx.x/2), +R) of overlap blockIdx.x%2 on plane zb
// (blockIdx.y) of slot blockIdx.z, R = ov_rows(N) (4, fewer when 2R
// transforms would exceed a workgroup or 96 KB of LDS); the plane's two
// radial OTF profiles are built once in LDS.
// A workgroup whose rows all lie outside the overlap's support (about a third
// of them at 3D-SIM geometries) writes zeros and returns.
constexpr int kOvStaticLds = 96 * 1024;
constexpr int ov_rows(int N) {
  int r = 4;
  while (r > 1 && (2 * r * fft_tpt(N) > 1024 || (2 * r * lds_pitch(N) + N) * 8 > kOvStaticLds)) r /= 2;
  return r;
}

template <int N, bool RA>
__global__ __launch_bounds__(ov_rows(N) * fft_tpt(N)) void k_overlaps_x(OvBatch b, const float2* __restrict__ tw) {
  constexpr int kOvRows = ov_rows(N);
  static_assert((kOvRows * lds_pitch(N) + N) * 8 <= kOvStaticLds, "rows and twiddles leave room for the profiles");
  const OvParams& p = b.p[blockIdx.z];
  const int zb = blockIdx.y;
  if (zb > 2 * p.zd) return;  // a slot with a narrower z support (whole block)
  float2* __restrict__ ovx = p.ovx;
  const int nzs = b.nzs_stride;
  constexpr int TPT = fft_tpt(N);
  constexpr int RW = kOvRows;  // rows per workgroup
  constexpr int NT = RW * TPT;
  constexpr int P = lds_pitch(N);
  constexpr int EPT = (RW * N + NT - 1) / NT;
  const int which = blockIdx.x & 1;
  const int i0 = (blockIdx.x >> 1) * RW;
  const int z0 = zb - p.zd;
  float kx = p.kx, ky = p.ky;
  if (p.k0d != nullptr) {
#pragma clang fp contract(off)
    const float2 k = *p.k0d;
    kx = k.x * p.kmul;
    ky = k.y * p.kmul;
  }
  float2* __restrict__ orow = ovx + (((long long)which * nzs + zb) * p.ny + i0) * p.nx;
  {
    bool live = false;
#pragma unroll
    for (int r = 0; r < RW; ++r) live = live || ov_row_live(p, kx, ky, which, i0 + r, z0);
    if (!live) {
#pragma unroll
      for (int q = 0; q < EPT; ++q) {
        const int idx = threadIdx.x + q * NT;
        if (idx < RW * N && i0 + idx / N < p.ny) orow[idx] = make_float2(0.f, 0.f);
      }
      return;  // uniform over the workgroup
    }
  }
  __shared__ float2 lds[RW * P];
  extern __shared__ float2 prof[];  // [2][nxotf]
  FftTw<N> twr;
  __shared__ float2 twstage[N > 1 ? N : 1];
  load_twiddles(twr, twstage, threadIdx.x % TPT, tw, threadIdx.x, blockDim.x);
  const int nxotf = p.otf1.nxotf;
  if constexpr (RA)
    for (int k = threadIdx.x; k < 2 * nxotf; k += NT)
      prof[k] = otf_profile_entry(k < nxotf ? p.otf1 : p.otf2, k < nxotf ? k : k - nxotf, z0, p.kzscale);
  __syncthreads();
  // In chunks of CH elements per thread: the sources of a chunk first, then
  // all its band loads (clamped to a valid index for zero elements) at
  // once, then the products.  Chunks keep the registers (and so the
  // workgroups per CU) within bounds.
  constexpr int CH = EPT < 4 ? EPT : 4;
#pragma unroll
  for (int q0 = 0; q0 < EPT; q0 += CH) {
    OvSrc src[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = threadIdx.x + (q0 + c) * NT;
      const int t = idx / N, j = idx - (idx / N) * N;  // t = row in the workgroup
      const int i = i0 + t;
      src[c] = (q0 + c < EPT && idx < RW * N && i < p.ny)
                   ? ov_source<RA>(p, kx, ky, prof, prof + nxotf, which, j, i, z0)
                   : OvSrc{0, false, false, make_float2(0.f, 0.f)};
    }
    const float2* bre = which == 0 ? p.b1re : p.b2re;
    const float2* bim = which == 0 ? (p.order1 > 0 ? p.b1im : p.b1re) : p.b2im;
    float2 vre[CH], vim[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      vre[c] = bre[src[c].ind];
      vim[c] = bim[src[c].ind];
    }
    const bool has_im = which == 1 || p.order1 > 0;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = threadIdx.x + (q0 + c) * NT;
      if (q0 + c < EPT && idx < RW * N) {
        const int t = idx / N, j = idx - (idx / N) * N;
        lds[t * P + lds_swz<N>(j)] = ov_combine(src[c], vre[c], vim[c], has_im);
      }
    }
  }
  __syncthreads();
  fft_lds<N, true>(lds + (threadIdx.x / TPT) * P, threadIdx.x % TPT, twr);
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    const int idx = threadIdx.x + q * NT;
    if (idx < RW * N) {
      const int t = idx / N, j = idx - (idx / N) * N;
      if (i0 + t < p.ny) orow[idx] = lds[t * P + lds_swz<N>(j)];
    }
  }
}

template <int N>
static void launch_ov_x(const OvBatch& b, int nzs_max, hipStream_t s) {
  const OvParams& p = b.p[0];
  const dim3 grid(2 * ceil_div(p.ny, ov_rows(N)), nzs_max, b.n), block(ov_rows(N) * fft_tpt(N));
  if (p.otf1.ra) {
    const size_t lds = (size_t)2 * p.otf1.nxotf * sizeof(float2);
    if (lds > 160 * 1024 - kOvStaticLds) throw ArgError("OTF table too long for the overlap pass's LDS profiles");
    hipLaunchKernelGGL((k_overlaps_x<N, true>), grid, block, lds, s, b, twiddles(N));
  } else {
    hipLaunchKernelGGL((k_overlaps_x<N, false>), grid, block, 0, s, b, twiddles(N));
  }
  SIMR_LAUNCH_CHECK();
}

void launch_overlaps_x(const OvBatch& b, hipStream_t s) {
  if (b.n < 1 || b.n > kMaxDirs) throw ArgError("overlap batch: 1..8 slots");
  int nzs_max = 0;
  for (int k = 0; k < b.n; ++k) {
    const OvParams& p = b.p[k];
    if (p.nx != b.p[0].nx || p.ny != b.p[0].ny || p.otf1.nxotf != b.p[0].otf1.nxotf ||
        p.otf2.nxotf != b.p[0].otf1.nxotf || p.otf1.ra != b.p[0].otf1.ra || p.otf2.ra != b.p[0].otf1.ra)
      throw ArgError("overlap batch: slots of different geometry");
    if (p.zd < 0 || 2 * p.zd + 1 > b.nzs_stride) throw ArgError("overlap z support wider than its planes");
    nzs_max = std::max(nzs_max, 2 * p.zd + 1);
  }
  switch (b.p[0].nx) {
#define SIMR_CASE(N)                   \
  case N:                              \
    launch_ov_x<N>(b, nzs_max, s);     \
    break;
    SIMR_XY_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      throw ArgError("image width " + std::to_string(b.p[0].nx) + " is not a supported size");
  }
}

// ---------------------------------------------------------------------------
// The overlaps' inverse transforms with the z sums fused, for the FP64 fit:
// the formation runs with the y transform, by columns (k_ovf_cols), and the
// x transform with the z sums, by rows (k_ovf_rows): a workgroup takes row y
// of every stored plane of both overlaps, so P(x, y) and the SX / SY totals
// accumulate in registers plane after plane.  The transformed planes are
// written once and read once (the three-pass form writes them twice and
// reads them twice).  The order of the two 1D transforms is the other one
// than the three-pass form's, so P agrees with it to rounding, not bit for
// bit.

OvSupport ov_support(const OvParams& p) {
  return OvSupport{p.kx, p.ky, p.k0d, p.kmul, p.rc2, p.dkx, p.dky, p.nx, p.ny, p.zd, p.bNoKz0};
}
__device__ __forceinline__ float2 ov_shift(const OvSupport& q) {
#pragma clang fp contract(off)
  if (q.k0d == nullptr) return make_float2(q.kx, q.ky);
  const float2 k = *q.k0d;
  return make_float2(k.x * q.kmul, k.y * q.kmul);
}

// The range of centred columns of overlap `which` (shift k) that can hold a
// nonzero element: those whose frequency lies in the x extent of the lens
// |q| <= rc, |q - s| <= rc (s = k, or -k for overlap1).  Its rightmost point is
// one disc's, if that lies in the other disc, else the discs' right
// intersection; likewise on the left.  The range carries a margin of
// margin * r, far beyond the rounding of the per-element tests; hi < lo: no
// column.  The column pass writes the tiles that meet the range with
// kOvWritten, and the row pass reads the columns in the range with kOvRead:
// the difference is far beyond the rounding of the range in either kernel, so
// no column is read that was not written.  (Plane kz = 0 with bNoKz0 is left
// to the callers.)
constexpr float kOvWritten = 1e-3f, kOvRead = 0.5e-3f;
__device__ __forceinline__ float2 ov_col_range(const OvSupport& p, float2 k, int which, float margin) {
#pragma clang fp contract(off)
  const float sx = which == 0 ? k.x : -k.x, sy = which == 0 ? k.y : -k.y;
  const float r2 = p.rc2 * 1.0002f, r = __builtin_amdgcn_sqrtf(r2);
  const float d2 = sx * sx + sy * sy;
  if (d2 > 4.f * r2) return make_float2(1.f, 0.f);
  // half the chord through the intersections, along x
  const float h = __builtin_amdgcn_sqrtf(fmaxf(r2 - 0.25f * d2, 0.f));
  const float chord = d2 > 0.f ? fabsf(sy) * h * __builtin_amdgcn_rsqf(d2) : r;
  // the right end of the disc further left, if inside the other; else the intersection
  const float e2 = (r - fabsf(sx)) * (r - fabsf(sx)) + sy * sy;  // its squared distance from the other's centre
  const float half = e2 <= r2 ? r - 0.5f * fabsf(sx) : chord;    // the lens is symmetric about s / 2
  const float m = margin * r;
  return make_float2(0.5f * sx - half - m, 0.5f * sx + half + m);
}
__device__ __forceinline__ bool ov_col_live(const OvSupport& p, float2 range, int j) {
#pragma clang fp contract(off)
  const float x = (float)(j > p.nx / 2 ? j - p.nx : j) * p.dkx;
  return x >= range.x && x <= range.y;
}

// The column pass: W adjacent columns of overlap blockIdx.x % 2 on plane
// blockIdx.y of slot blockIdx.z.  Thread (w, j) forms its pass-1 inputs of
// column c0 + w (as k_overlaps_x) straight in registers, transforms them on the
// two-pass register core and stores its outputs; LDS holds one float per
// element.  Tiles without a live column are left unwritten, and the row pass
// does not read them.
// What bounds it is the formation (two radial lookups, square roots and a
// normalisation per element) and its chain of dependent loads, so the plans ask
// for few values a lane (24, else 32) and many wavefronts.  On the radix stages in LDS, every element a trip
// through LDS per stage and dead tiles filled with zeros: 175.6 us in
// a 512x512x48 stack (a launch is three directions), 350 in 1024x1024x16,
// 29.0 in 256x256x32 and 11.2 in one 256x256 plane; now 149, 206, 26.0 and 12.6
// (that one is latency: the shift, the profile, the bands, the twiddles).
// A full OTF (RA = false) is looked up in eight places an element, and the longer
// lengths' kernels keep part of their inputs in scratch (200 to 300 bytes a lane
// at 480, 512 and 1024 rows, none at 64 and 256).
// 480x400x21 and 384x384x26, at three passes before: the row pass's figures.
template <int NY>
constexpr int ovc_want() {
  return rp_ok(NY, 1, kRpWants[1]) ? 1 : rp_ok(NY, 1, kRpWants[2]) ? 2 : 0;
}
template <int NY>
struct OvC {
  static constexpr int WANT = ovc_want<NY>();
  using K = Rp<NY, 1, WANT>;
  static constexpr int span_of(int w) {  // columns offset by 32 / w banks
    const int want = w < 32 ? 32 / w : 1;
    return K::SPAN + ((want - K::SPAN % 32) % 32 + 32) % 32;
  }
  static constexpr int width() {
    int w = NY <= 256 ? 8 : 16;  // (small planes: more workgroups)
    while (w > 4 && (w * K::T > 512 || w * span_of(w) * 4 > 72 * 1024)) w /= 2;
    while (w * K::T % 64) w *= 2;  // whole wavefronts
    return w;
  }
  static constexpr int W = width(), NT = W * K::T;
  static constexpr int LDS = W * span_of(W) * 4;
  static constexpr int VALUES = K::R1 * K::N1 > K::N2 ? K::R1 * K::N1 : K::N2;
  // (128 VGPRs at four wavefronts per SIMD; factors of 5 spill there)
  static constexpr int WAVES = VALUES <= 32 ? (NY % 25 == 0 ? 3 : 4) : VALUES <= 40 ? 2 : 1;
};
template <int NY>
constexpr bool ovf_cols_ok() {
  return OvC<NY>::NT <= 1024 && OvC<NY>::LDS <= 128 * 1024;
}

template <int NY, bool RA>
__global__ __launch_bounds__(OvC<NY>::NT, OvC<NY>::WAVES) void k_ovf_cols(OvBatch b, const float2* __restrict__ tw) {
  using C = OvC<NY>;
  using K = typename C::K;
  constexpr int W = C::W, NT = C::NT, N1 = K::N1, N2 = K::N2;
  // XCD-contiguous tile order: neighbouring column tiles, whose segments of
  // the nx/2+1-element band rows share cache lines, run in one L2
  unsigned bx, by, bz;
  xcd_tile3(bx, by, bz);
  const OvParams& p = b.p[bz];
  const int zb = by;
  if (zb > 2 * p.zd) return;  // a slot with a narrower z support (whole block)
  const int which = bx & 1;
  const int c0 = (bx >> 1) * W;
  const int z0 = zb - p.zd;
  if (z0 == 0 && p.bNoKz0) return;
  const OvSupport sup{p.kx, p.ky, p.k0d, p.kmul, p.rc2, p.dkx, p.dky, p.nx, p.ny, p.zd, p.bNoKz0};
  const float2 k = ov_shift(sup);
  {
    const float2 range = ov_col_range(sup, k, which, kOvWritten);
    bool live = false;
    for (int w = 0; w < W; ++w) live = live || (c0 + w < p.nx && ov_col_live(sup, range, c0 + w));
    if (!live) return;  // uniform over the workgroup
  }
  __shared__ float buf[C::LDS / 4];
  extern __shared__ float2 prof[];  // [2][nxotf]
  const int w = threadIdx.x % W, j = threadIdx.x / W;
  const int nxotf = p.otf1.nxotf;
  if constexpr (RA) {
    for (int i = threadIdx.x; i < 2 * nxotf; i += NT)
      prof[i] = otf_profile_entry(i < nxotf ? p.otf1 : p.otf2, i < nxotf ? i : i - nxotf, z0, p.kzscale);
    __syncthreads();
  }
  const int jc = c0 + w < p.nx ? c0 + w : p.nx - 1;
  const float2* bre = which == 0 ? p.b1re : p.b2re;
  const float2* bim = which == 0 ? (p.order1 > 0 ? p.b1im : p.b1re) : p.b2im;
  const bool has_im = which == 1 || p.order1 > 0;
  float2 in[K::R1 * N1];
  // in chunks: the sources of a chunk first, then all its band loads (clamped
  // to a valid index for zero elements), then the products
  constexpr int E = K::R1 * N1, CH = E <= 16 ? (E < 8 ? E : 8) : 4;
#pragma unroll
  for (int q0 = 0; q0 < E; q0 += CH) {
    OvSrc src[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e = q0 + c < E ? q0 + c : E - 1;
      const int n2 = j + K::T * (e / N1);
      const int i = N2 * (e % N1) + (K::N2 % K::T == 0 || n2 < N2 ? n2 : N2 - 1);
      src[c] = ov_source<RA>(p, k.x, k.y, prof, prof + nxotf, which, jc, i, z0);
    }
    float2 vre[CH], vim[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      vre[c] = bre[src[c].ind];
      vim[c] = bim[src[c].ind];
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (q0 + c < E) in[q0 + c] = ov_combine(src[c], vre[c], vim[c], has_im);
  }
  float2 out[N2];
  rp_transform<NY, 1, true, false, C::WANT>(buf + w * C::span_of(W), j, false, tw, in, out);
  if (c0 + w < p.nx && (K::ROWS == K::T || j < K::ROWS)) {
    float2* col = p.ovx + (((long long)which * b.nzs_stride + zb) * NY + j) * p.nx + c0 + w;
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) col[(long long)(K::OSTEP * k2) * p.nx] = out[k2];
  }
}

// The row pass.  Two groups of T lanes take a plane of row y, one transforming
// X and the other Y on the two-pass register core (wave-private exchange); the
// groups then swap halves of their outputs (lane swaps in registers), so each
// holds X and Y of half the row and adds the products up in its registers, plane
// after plane.  The pairs' sums meet in LDS at the end.
// What bounds it is latency at two to four wavefronts a SIMD: the double sums
// and a row's values fill the registers, so a lane holds half the sums, and
// plans of at most 32 values.  (One group transforming X, then Y, with all the
// sums, spilled at every length above 80.)  Four wavefronts to a workgroup: the
// wavefronts of a SIMD come from several rows.  Live columns only are read.
// Per launch, three directions: 1024x1024x16 224.5 us before (radix stages in
// LDS) and 160 now; 512x512x48 96.9 and 104.5, which the column pass wins back
// (272.5 the pair, now 254).  Sizes that had three passes, both kernels:
// 480x400x21 164.5, now 108; 384x384x26 144.4, now 125; 64x64x9 24.2, now 16.
template <int NX>
constexpr int ovr_want() {
  return NX < 300 && rp_ok(NX, 1, kRpWants[3]) ? 3 : 4;
}
template <int NX>
struct OvR {
  static constexpr int WANT = ovr_want<NX>();
  using K = Rp<NX, 1, WANT>;
  static constexpr int HALF = (K::N2 + 1) / 2;  // outputs a lane accumulates
  static constexpr int SPANP = K::SPAN + ((K::T - K::SPAN % 32) % 32 + 32) % 32;
  static constexpr int MAXP = 256 / (2 * K::T) < 8 ? 256 / (2 * K::T) : 8;  // pairs per workgroup
  static constexpr int threads(int pairs) { return (pairs * 2 * K::T + 63) / 64 * 64; }
  // twiddles; then the exchange buffers, which the pairs' sums reuse
  static constexpr int lds(int pairs) {
    const int ex = threads(pairs) / K::T * SPANP * 4, sums = (pairs + 1) / 2 * NX * 16;
    return K::TABN * 8 + (ex > sums ? ex : sums);
  }
  static constexpr int WAVES = K::N2 > 16 || K::R1 * K::N1 > 24 ? 2 : 3;
  static_assert(K::TABN % 2 == 0, "the double2 sums are 16-byte aligned");
};
template <int NX>
constexpr bool ovf_rows_ok() {
  if constexpr (rp_ok(NX, 1, kRpWants[ovr_want<NX>()]))
    return OvR<NX>::K::T <= 32 && OvR<NX>::lds(OvR<NX>::MAXP) <= 150 * 1024;
  return false;
}

// a of the odd group of T lanes <-> b of the even group next to it
template <int T>
__device__ __forceinline__ void ov_swap(float& a, float& b) {
  if constexpr (T == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else if constexpr (T == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else {
    const bool odd = threadIdx.x & T;
    const float got = __shfl_xor(odd ? a : b, T);
    if (odd)
      a = got;
    else
      b = got;
  }
}

template <int NX>
__global__ __launch_bounds__(OvR<NX>::threads(OvR<NX>::MAXP), OvR<NX>::WAVES) void k_ovf_rows(
    ZsumBatch b, int pairs, const float2* __restrict__ tw) {
#pragma clang fp contract(off)
  using C = OvR<NX>;
  using K = typename C::K;
  constexpr int T = K::T, N1 = K::N1, N2 = K::N2, HALF = C::HALF;
  extern __shared__ float2 twl[];
  __shared__ double red[2][16];
  const int y = blockIdx.x, slot = blockIdx.y;
  const OvSupport& sup = b.sup[slot];
  const float2 k = ov_shift(sup);  // (in flight with the twiddles)
  for (int i = threadIdx.x; i < K::TABN; i += blockDim.x) twl[i] = tw[i];
  __syncthreads();
  const int pair = threadIdx.x / (2 * T), which = threadIdx.x / T % 2, j = threadIdx.x % T;
  float* buf = reinterpret_cast<float*>(twl + K::TABN) + threadIdx.x / T * C::SPANP;
  const int nzs = b.nzs[slot];
  const long long nxy = b.nxy;
  const float2 range = ov_col_range(sup, k, which, kOvRead);
  const int zskip = sup.bNoKz0 ? sup.zd : -1;  // a plane of zeros, not written
  const float2* row = b.ovx[slot] + (long long)which * b.nzs_stride * nxy + (long long)y * NX;
  double pr[HALF], pi[HALF], sx = 0.0, sy = 0.0;
#pragma unroll
  for (int e = 0; e < HALF; ++e) pr[e] = pi[e] = 0.0;
  const bool mine = K::ROWS == T || j < K::ROWS;  // the lane ends with outputs
#pragma unroll 1
  for (int z0 = 0; z0 < nzs; z0 += pairs) {
    const int z = z0 + pair;
    const bool there = pair < pairs && z < nzs && z != zskip;
    const float2* src = row + (long long)(there ? z : 0) * nxy;
    float2 in[K::R1 * N1];
#pragma unroll
    for (int c = 0; c < K::R1; ++c) {
      const int n2 = N2 % T == 0 || j + T * c < N2 ? j + T * c : N2 - 1;
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
        const int x = N2 * n1 + n2;
        in[c * N1 + n1] = make_float2(0.f, 0.f);
        if (there && ov_col_live(sup, range, x)) in[c * N1 + n1] = src[x];
      }
    }
    float2 out[N2], v[2 * HALF];
    rp_transform<NX, 1, true, true, C::WANT>(buf, j, false, twl, in, out);
    rp_sync<true>();
#pragma unroll
    for (int e = 0; e < 2 * HALF; ++e) v[e] = e < N2 ? out[e] : make_float2(0.f, 0.f);
#pragma unroll
    for (int e = 0; e < HALF; ++e) {
      ov_swap<T>(v[e].x, v[e + HALF].x);
      ov_swap<T>(v[e].y, v[e + HALF].y);
    }
    if (mine) {
#pragma unroll
      for (int e = 0; e < HALF; ++e) {
        const double ar = v[e].x, ai = v[e].y, br = v[e + HALF].x, bi = v[e + HALF].y;
        // float x float products are exact in double: a product plus a
        // fused multiply-add is the correctly rounded a*b + c*d
        pr[e] += __builtin_fma(ar, br, ai * bi);
        pi[e] += __builtin_fma(ar, bi, -(ai * br));
        sx += __builtin_fma(ar, ar, ai * ai);
        sy += __builtin_fma(br, br, bi * bi);
      }
    }
  }
  // the pairs' sums, pairwise; entry e of this lane is output x0 + ROWS e
  const int x0 = j + (which ? K::ROWS * HALF : 0);
  double2* const sums = reinterpret_cast<double2*>(twl + K::TABN);
#pragma unroll 1
  for (int n = pairs; n > 1; n = (n + 1) / 2) {
    const int half = (n + 1) / 2;
    __syncthreads();
    if (pair >= half && pair < n && mine) {
#pragma unroll
      for (int e = 0; e < HALF; ++e)
        if (N2 % 2 == 0 || x0 + K::ROWS * e < NX) sums[(pair - half) * NX + x0 + K::ROWS * e] = make_double2(pr[e], pi[e]);
    }
    __syncthreads();
    if (pair + half < n && mine) {
#pragma unroll
      for (int e = 0; e < HALF; ++e)
        if (N2 % 2 == 0 || x0 + K::ROWS * e < NX) {
          const double2 t = sums[pair * NX + x0 + K::ROWS * e];
          pr[e] += t.x;
          pi[e] += t.y;
        }
    }
  }
  const double n = (double)b.nz;
  if (pair == 0 && mine) {
#pragma unroll
    for (int e = 0; e < HALF; ++e) {
      if (N2 % 2 && x0 + K::ROWS * e >= NX) continue;
      const long long at = (long long)y * NX + x0 + K::ROWS * e;
      const double2 pv = make_double2(pr[e] * n, pi[e] * n);
      b.P[slot][at] = pv;
      if (b.cc[slot]) b.cc[slot][at] = make_float2((float)pv.x, -(float)pv.y);
    }
  }
  const double wx = wave_total(sx), wy = wave_total(sy);
  if (threadIdx.x % 64 == 0) {
    red[0][threadIdx.x / 64] = wx;
    red[1][threadIdx.x / 64] = wy;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    for (int w = 0; w < (int)blockDim.x / 64; ++w) t += red[threadIdx.x][w];
    b.totals[slot][threadIdx.x * gridDim.x + y] = t * n;
  }
}

template <int NY>
static bool ovf_cols_launch(const OvBatch& ob, int nzs_max, bool run, hipStream_t s) {
  if constexpr (ovf_cols_ok<NY>()) {
    using C = OvC<NY>;
    const OvParams& p = ob.p[0];
    const size_t lds = p.otf1.ra ? (size_t)2 * p.otf1.nxotf * sizeof(float2) : 0;
    if (lds > 32 * 1024) return false;
    const float2* tw = twiddles_rp(NY, C::K::N2);
    if (!run) return true;
    const dim3 g1(2 * ceil_div(p.nx, C::W), nzs_max, ob.n), b1(C::NT);
    if (p.otf1.ra)
      hipLaunchKernelGGL((k_ovf_cols<NY, true>), g1, b1, lds, s, ob, tw);
    else
      hipLaunchKernelGGL((k_ovf_cols<NY, false>), g1, b1, 0, s, ob, tw);
    SIMR_LAUNCH_CHECK();
    return true;
  } else {
    return false;
  }
}

template <int NX>
static bool ovf_rows_launch(const ZsumBatch& zb, int ny, bool run, hipStream_t s) {
  if constexpr (ovf_rows_ok<NX>()) {
    using C = OvR<NX>;
    const float2* tw = twiddles_rp(NX, C::K::N2);
    if (!run) return true;
    int nzs = 1;
    for (int k = 0; k < zb.n; ++k) nzs = std::max(nzs, zb.nzs[k]);
    // as many pairs as share the planes evenly, at most MAXP
    const int pairs = ceil_div(nzs, ceil_div(nzs, C::MAXP));
    hipLaunchKernelGGL(k_ovf_rows<NX>, dim3(ny, zb.n), dim3(C::threads(pairs)), C::lds(pairs), s, zb, pairs, tw);
    SIMR_LAUNCH_CHECK();
    return true;
  } else {
    return false;
  }
}

static int ovf_nzs_max(const OvBatch& ob) {
  int m = 0;
  for (int k = 0; k < ob.n; ++k) m = std::max(m, 2 * ob.p[k].zd + 1);
  return m;
}

static bool ovf_cols_dispatch(const OvBatch& ob, bool run, hipStream_t s) {
  switch (ob.p[0].ny) {
#define SIMR_CASE(N) \
  case N:            \
    return ovf_cols_launch<N>(ob, ovf_nzs_max(ob), run, s);
    SIMR_XY_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      return false;
  }
}

static bool ovf_rows_dispatch(const ZsumBatch& zb, int nx, int ny, bool run, hipStream_t s) {
  switch (nx) {
#define SIMR_CASE(N) \
  case N:            \
    return ovf_rows_launch<N>(zb, ny, run, s);
    SIMR_XY_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      return false;
  }
}

bool overlaps_fused_ok(const OvBatch& ob, const ZsumBatch& zb) {
  if (ob.n < 1 || ob.n > kMaxDirs || zb.n != ob.n) return false;
  const OvParams& p0 = ob.p[0];
  if (p0.ny > kZsumMaxBlocks) return false;
  for (int k = 0; k < ob.n; ++k) {
    const OvParams& p = ob.p[k];
    if (p.nx != p0.nx || p.ny != p0.ny || p.otf1.nxotf != p0.otf1.nxotf || p.otf2.nxotf != p0.otf1.nxotf ||
        p.otf1.ra != p0.otf1.ra || p.otf2.ra != p0.otf1.ra)
      return false;
    if (p.zd < 0 || 2 * p.zd + 1 > ob.nzs_stride || zb.nzs[k] != 2 * p.zd + 1 || zb.ovx[k] != p.ovx) return false;
  }
  return ovf_cols_dispatch(ob, false, nullptr) && ovf_rows_dispatch(zb, p0.nx, p0.ny, false, nullptr);
}

void overlaps_request_tables(int nx, int ny) {
  OvBatch ob{};
  ZsumBatch zb{};
  ob.n = zb.n = 1;
  ob.p[0].nx = nx;
  ob.p[0].ny = ny;
  (void)ovf_cols_dispatch(ob, false, nullptr);
  (void)ovf_rows_dispatch(zb, nx, ny, false, nullptr);
}

void launch_overlaps_fused_cols(const OvBatch& ob, hipStream_t s) {
  if (!ovf_cols_dispatch(ob, true, s)) throw ArgError("two-pass overlaps: unsupported geometry");
}

void launch_overlaps_fused_rows(const ZsumBatch& zb, int nx, int ny, hipStream_t s) {
  if (!ovf_rows_dispatch(zb, nx, ny, true, s)) throw ArgError("two-pass overlaps: unsupported geometry");
}

// Every reserved plane is transformed (planes beyond a slot's own 2zd+1 hold
// stale values that nothing reads), so the slots form one batch of columns.
void launch_overlaps_y(int nx, int ny, int nzs_stride, float2* ovx, int nslots, hipStream_t s) {
  const long long nxy = (long long)nx * ny;
  fft_cols(ny, ovx, nx, nx, 2LL * nzs_stride * nslots, nxy, true, s);
}

// z pass, reduced to what the fit reads.  The modamp and cross-correlation
// kernels use only the per-(x,y) sums over z of conj(X) Y, |X|^2 and |Y|^2 of
// the inverse-transformed overlaps, and the phase factor they apply depends on
// (x, y) alone (reductionKernel, gpuFunctionsImpl.cu:1150-1190; aTimesConjB
// 391-413).  For the unnormalised inverse DFT along z, Parseval gives
// sum_z conj(x_z) y_z = nz sum_kz conj(X_kz) Y_kz, and only the 2zd+1 stored
// kz planes are nonzero, so the sums are formed from those planes directly
// and the z transform is not needed.  Loads of eight planes of both overlaps
// are in flight at once.
// FP32: float sums, stored per (x, y) in P, SX, SY (k_modamp_fp32 reduces
// them in the reference's blocks).  FP64: double sums; P per (x, y), and of
// SX and SY only what the fit reads, their totals, as one partial per block
// (totals[block], totals[nblocks + block]); ELEM also stores them per (x, y).
int zsum_blocks(long long nxy) { return (int)std::min<long long>(ceil_div(nxy, 256), kZsumMaxBlocks); }

template <bool FP32, bool ELEM>
__global__ __launch_bounds__(256) void k_overlaps_zsum(ZsumBatch b) {
#pragma clang fp contract(off)
  using A = typename std::conditional<FP32, float, double>::type;
  constexpr int KB = 8;
  const int slot = blockIdx.y;
  const float2* __restrict__ ovx = b.ovx[slot];
  double2* __restrict__ P = b.P[slot];
  double* __restrict__ SX = b.SX[slot];
  double* __restrict__ SY = b.SY[slot];
  double* __restrict__ totals = b.totals[slot];
  const int nzs = b.nzs[slot];
  const long long nxy = b.nxy;
  const A n = (A)b.nz;
  double tsx = 0.0, tsy = 0.0;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < nxy; e += (long long)gridDim.x * 256) {
    A sxr = 0, sxi = 0, sx = 0, sy = 0;
    const float2* X = ovx + e;
    const float2* Y = ovx + (long long)b.nzs_stride * nxy + e;
    for (int s = 0; s < nzs; s += KB) {
      const int cnt = nzs - s < KB ? nzs - s : KB;  // uniform
      float2 xa[KB], yb[KB];
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        const long long o = (long long)(k < cnt ? s + k : s) * nxy;
        xa[k] = X[o];
        yb[k] = Y[o];
      }
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        if (k >= cnt) break;
        const A ar = xa[k].x, ai = xa[k].y, br = yb[k].x, bi = yb[k].y;
        if constexpr (FP32) {
          sxr += ar * br + ai * bi;
          sxi += ar * bi - ai * br;
          sx += ar * ar + ai * ai;
          sy += br * br + bi * bi;
        } else {
          // float x float products are exact in double, so a product plus a
          // fused multiply-add gives the correctly rounded a*b + c*d of the
          // plain form
          sxr += __builtin_fma(ar, br, ai * bi);
          sxi += __builtin_fma(ar, bi, -(ai * br));
          sx += __builtin_fma(ar, ar, ai * ai);
          sy += __builtin_fma(br, br, bi * bi);
        }
      }
    }
    const double2 pv = make_double2((double)(sxr * n), (double)(sxi * n));
    P[e] = pv;
    if (b.cc[slot]) b.cc[slot][e] = make_float2((float)pv.x, -(float)pv.y);
    if constexpr (FP32 || ELEM) {
      SX[e] = (double)(sx * n);
      SY[e] = (double)(sy * n);
    }
    if constexpr (!FP32) {
      tsx += sx * n;
      tsy += sy * n;
    }
  }
  if constexpr (!FP32) {
    __shared__ double red[256];
    const double a = block_sum_d<256>(tsx, red);
    const double b = block_sum_d<256>(tsy, red);
    if (threadIdx.x == 0) {
      totals[blockIdx.x] = a;
      totals[gridDim.x + blockIdx.x] = b;
    }
  }
}

void launch_overlaps_z_reduce(const ZsumBatch& b, bool fp32, bool per_elem, hipStream_t s) {
  if (b.n < 1 || b.n > kMaxDirs) throw ArgError("z-sum batch: 1..8 slots");
  for (int k = 0; k < b.n; ++k)
    if (b.nzs[k] < 1 || b.nzs[k] > b.nz || b.nzs[k] > b.nzs_stride)
      throw ArgError("overlap z support wider than the stack");
  const dim3 grid(zsum_blocks(b.nxy), b.n);
  if (fp32)
    hipLaunchKernelGGL((k_overlaps_zsum<true, true>), grid, dim3(256), 0, s, b);
  else if (per_elem)
    hipLaunchKernelGGL((k_overlaps_zsum<false, true>), grid, dim3(256), 0, s, b);
  else
    hipLaunchKernelGGL((k_overlaps_zsum<false, false>), grid, dim3(256), 0, s, b);
  SIMR_LAUNCH_CHECK();
}

// ----------------------------------------------------------------- findk0 peak
__global__ __launch_bounds__(256) void k_argmax_partial(const float2* __restrict__ cc, long long n,
                                                        float* __restrict__ pv, int* __restrict__ pi) {
  cc += (long long)blockIdx.y * n;
  pv += blockIdx.y * gridDim.x;
  pi += blockIdx.y * gridDim.x;
  __shared__ float sv[256];
  __shared__ int si[256];
  const long long chunk = (n + gridDim.x - 1) / gridDim.x;
  const long long b0 = blockIdx.x * chunk;
  const long long b1 = min(n, b0 + chunk);
  float v = -1e30f;
  int idx = 0x7fffffff;
  for (long long e = b0 + threadIdx.x; e < b1; e += 256) better(v, idx, intensity(cc[e]), (int)e);
  sv[threadIdx.x] = v;
  si[threadIdx.x] = idx;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      float a = sv[threadIdx.x];
      int ai = si[threadIdx.x];
      better(a, ai, sv[threadIdx.x + s], si[threadIdx.x + s]);
      sv[threadIdx.x] = a;
      si[threadIdx.x] = ai;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = sv[0];
    pi[blockIdx.x] = si[0];
  }
}

__global__ __launch_bounds__(256) void k_argmax_final(const float2* __restrict__ cc, const float* __restrict__ pv,
                                                      const int* __restrict__ pi, int nparts, int nx, int ny,
                                                      float* __restrict__ vals, int* __restrict__ idx_out) {
  cc += (long long)blockIdx.x * nx * ny;
  pv += blockIdx.x * nparts;
  pi += blockIdx.x * nparts;
  vals += blockIdx.x * 8;
  idx_out += blockIdx.x;
  __shared__ float sv[256];
  __shared__ int si[256];
  float v = -1e30f;
  int idx = 0x7fffffff;
  for (int b = threadIdx.x; b < nparts; b += 256) better(v, idx, pv[b], pi[b]);
  sv[threadIdx.x] = v;
  si[threadIdx.x] = idx;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      float a = sv[threadIdx.x];
      int ai = si[threadIdx.x];
      better(a, ai, sv[threadIdx.x + s], si[threadIdx.x + s]);
      sv[threadIdx.x] = a;
      si[threadIdx.x] = ai;
    }
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  idx = si[0];
  // No element won (every intensity NaN, e.g. from one NaN input pixel spread
  // by the transforms): findpeak keeps its initial centre (0, 0)
  // (gpuFunctionsImpl.cu:443-455).
  if (idx < 0 || idx >= nx * ny) idx = 0;
  const int xc = idx % nx, yc = idx / nx;
  auto I = [&](int y, int x) { return intensity(cc[(long long)y * nx + x]); };
  vals[0] = I(yc, xc);
  vals[1] = I(yc, xc == 0 ? nx - 1 : xc - 1);
  vals[2] = I(yc, xc == nx - 1 ? 0 : xc + 1);
  vals[3] = I(yc == 0 ? ny - 1 : yc - 1, xc);
  vals[4] = I(yc == ny - 1 ? 0 : yc + 1, xc);
  idx_out[0] = idx;
  __threadfence_system();  // the outputs may be host memory
}

void launch_peak_partials(int n, float2* cc, float* partial_val, int* partial_idx, int nx, int ny, hipStream_t s) {
  if (n < 1 || n > kMaxDirs) throw ArgError("peak batch: 1..8 slots");
  const long long nxy = (long long)nx * ny;
  fft_rows(nx, cc, nx, (long long)ny * n, false, s);
  fft_cols(ny, cc, nx, nx, n, nxy, false, s);
  hipLaunchKernelGGL(k_argmax_partial, dim3(kArgBlocks, n), dim3(256), 0, s, cc, nxy, partial_val, partial_idx);
  SIMR_LAUNCH_CHECK();
}

void launch_findpeak(int n, float2* cc, float* partial_val, int* partial_idx, float* peak_vals, int* peak_idx, int nx,
                     int ny, hipStream_t s) {
  launch_peak_partials(n, cc, partial_val, partial_idx, nx, ny, s);
  hipLaunchKernelGGL(k_argmax_final, dim3(n), dim3(256), 0, s, cc, partial_val, partial_idx, kArgBlocks, nx, ny,
                     peak_vals, peak_idx);
  SIMR_LAUNCH_CHECK();
}

// ------------------------------------------------------------ modamp, FP64
// e^{i phi} = e^{i a(x)} e^{i b(y)} with a = 2 pi dxy (x - nx/2) kx and
// b = 2 pi dxy (y - ny/2) ky, so
//   sum P e^{i phi} = sum_x e^{i a(x)} sum_y e^{i b(y)} P(x, y).
// Workgroup (row block, group of up to G candidates of one slot): a thread
// takes columns x, adds the block's rows up with each candidate's row phasors
// (LDS), reading P once for the group, and multiplies by the column phasors.
// Those are products of two table entries, e^{i a(x)} = e^{i a(16 q)}
// e^{i 2 pi dxy kx r}, x = 16 q + r, so a workgroup's few hundred sincos
// (double, some 200 instructions) run once, side by side.
// What bounds it: the latency of that chain at small sizes, the reads of P
// (from the L2, 16 bytes a point for every group) at large ones.  A round of 13
// candidates (of at most kFitReq) for each of three directions: 256^2 7.2 -> 6.0
// us, 512^2 13.7 -> 9.4, 1024^2 38 -> 19.4 against a candidate and four rows per
// workgroup with a sincos per column; 16 rows 14.6 and 30.1 us at the two larger
// sizes (too few workgroups); groups of two the same.
constexpr int kModGroup = 4;
constexpr int kModRows = 8;
int modamp_partials_fp64(int nx, int ny) { return (ny + kModRows - 1) / kModRows; }

__device__ __forceinline__ float2 cand_k(const CandSet& s, int c) { return s.kc ? s.kc[c] : s.k[c]; }
__device__ __forceinline__ int cand_slot(const CandSet& s, int c) {
  return s.nreq ? c / kFitReq : s.ks ? s.ks[c] : s.slot[c];
}
// whether candidate c exists (a device-driven fit's round)
__device__ __forceinline__ bool cand_live(const CandSet& s, int c) {
  return s.nreq == nullptr || c % kFitReq < s.nreq[c / kFitReq];
}

// G > 1: blockIdx.y = direction * groups + group of a device-driven fit's
// round; G = 1: blockIdx.y is the candidate.
template <int G>
__global__ __launch_bounds__(256) void k_modamp_fp64(ModampSlots m, CandSet cs, int nx, int ny, float dxy,
                                                     double2* __restrict__ partials) {
  constexpr int R = kModRows;
  constexpr int kGroups = (kFitReq + G - 1) / G;
  extern __shared__ double2 tab[];  // per candidate: R row phasors, 16 fine and nq coarse column phasors
  __shared__ double red[4][2 * G];
  int c0 = blockIdx.y, nc = 1;
  if (G > 1) {
    const int d = blockIdx.y / kGroups, i0 = (blockIdx.y % kGroups) * G;
    c0 = d * kFitReq + i0;
    nc = min(G, cs.nreq[d] - i0);
    if (nc <= 0) return;  // whole block
  }
  const double2* __restrict__ P = m.P[cand_slot(cs, c0)];
  const double twopi_dxy = 2.0 * 3.14159265358979323846 * (double)dxy;
  const int j0 = blockIdx.x * R;
  const int nrows = min(R, ny - j0);
  P += (long long)j0 * nx;
  const int nq = (nx + 15) / 16, per = R + 16 + nq;
  for (int e = threadIdx.x; e < nc * per; e += 256) {
    const int g = e / per, q = e - g * per;
    const float2 kc = cand_k(cs, c0 + g);
    const double pos = q < R ? (double)(j0 + q) - 0.5 * ny : q < R + 16 ? (double)(q - R) : 16.0 * (q - R - 16) - 0.5 * nx;
    double sn, csn;
    sincos(twopi_dxy * (pos * (q < R ? (double)kc.y : (double)kc.x)), &sn, &csn);
    tab[e] = make_double2(csn, sn);
  }
  __syncthreads();
  double ar[G], ai[G];
#pragma unroll
  for (int g = 0; g < G; ++g) ar[g] = ai[g] = 0.0;
  for (int i = threadIdx.x; i < nx; i += 256) {
    double2 pv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) pv[r] = P[(long long)(r < nrows ? r : 0) * nx + i];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g < nc) {  // uniform
        double tr = 0.0, ti = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const double2 b = r < nrows ? tab[g * per + r] : make_double2(0.0, 0.0);
          tr += pv[r].x * b.x - pv[r].y * b.y;
          ti += pv[r].x * b.y + pv[r].y * b.x;
        }
        const double2 lo = tab[g * per + R + (i & 15)], hi = tab[g * per + R + 16 + (i >> 4)];
        const double er = hi.x * lo.x - hi.y * lo.y, ei = hi.x * lo.y + hi.y * lo.x;
        ar[g] += tr * er - ti * ei;
        ai[g] += tr * ei + ti * er;
      }
    }
  }
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const double x = wave_total(ar[g]), y = wave_total(ai[g]);
    if (lane == 0) {
      red[wave][2 * g] = x;
      red[wave][2 * g + 1] = y;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < nc) {
    const int g = threadIdx.x;
    const double x = (red[0][2 * g] + red[1][2 * g]) + (red[2][2 * g] + red[3][2 * g]);
    const double y = (red[0][2 * g + 1] + red[1][2 * g + 1]) + (red[2][2 * g + 1] + red[3][2 * g + 1]);
    partials[(long long)(c0 + g) * gridDim.x + blockIdx.x] = make_double2(x, y);
  }
}

static void check_cands(const CandSet& c, int ncand) {
  if (ncand < 1 || (c.kc == nullptr && ncand > kArgCand) || ncand > 65535)
    throw ArgError("modamp: 1..128 candidates per launch (by value), 1..65535 from device arrays");
  if (c.nreq != nullptr && (c.kc == nullptr || ncand % kFitReq)) throw ArgError("modamp: a round's candidates come by direction");
  if (c.nreq == nullptr && (c.kc == nullptr) != (c.ks == nullptr)) throw ArgError("modamp: candidates and slots from the same source");
}

// The z-sum totals of a slot that is read must have been queued: zb is 0 until
// its overlaps are.
static void check_totals(const ModampSlots& m, int slot) {
  if (slot < 0 || slot >= kMaxDirs || m.zb[slot] < 1 || m.zb[slot] > kZsumMaxBlocks)
    throw ArgError("modamp: a direction without overlaps");
}

void launch_modamp_fp64(const ModampSlots& m, const CandSet& c, int ncand, int nx, int ny, float dxy,
                        double2* partials, hipStream_t s) {
  check_cands(c, ncand);
  const int nb = modamp_partials_fp64(nx, ny);
  // a device-driven fit's candidates come by direction and share their reads
  // of P; other batches have few candidates, or few of one slot
  const int G = c.nreq != nullptr ? kModGroup : 1;
  const size_t lds = (size_t)G * (kModRows + 16 + (nx + 15) / 16) * sizeof(double2);
  if (c.nreq != nullptr)
    hipLaunchKernelGGL(k_modamp_fp64<kModGroup>, dim3(nb, ncand / kFitReq * ((kFitReq + kModGroup - 1) / kModGroup)),
                       dim3(256), lds, s, m, c, nx, ny, dxy, partials);
  else
    hipLaunchKernelGGL(k_modamp_fp64<1>, dim3(nb, ncand), dim3(256), lds, s, m, c, nx, ny, dxy, partials);
  SIMR_LAUNCH_CHECK();
}

// The result arithmetic of one modamp candidate, in the host's order and
// precision.  fp64: one wavefront per candidate, all in one workgroup, which
// then publishes the fit it completes (pub.out non-null); fp32: one workgroup
// per candidate (float sums in block order).
__global__ __launch_bounds__(64 * kMaxDirs) void k_modamp_finish_fp64(ModampSlots m, const int* __restrict__ kslot,
                                                                      int ncand, const double2* __restrict__ part64,
                                                                      int nparts, float2* amp, float* corr, int stride,
                                                                      int order, const FitState* fit, FitPub pub) {
#pragma clang fp contract(off)
  const int c = threadIdx.x / 64;
  if (c < ncand) {
    const int slot = kslot[c], zb = m.zb[slot];
    const double* __restrict__ totals = m.totals[slot];
    part64 += (long long)c * nparts;
    double xi;
    const double xr = quad_sum(nparts, [&](int i) { return part64[i]; }, &xi);
    const double sx = wave_sum(zb, [&](int i) { return totals[i]; });
    const double sy = wave_sum(zb, [&](int i) { return totals[zb + i]; });
    if (threadIdx.x % 64 == 0) {
      amp[slot * stride + order] = make_float2((float)(xr / sx), (float)(xi / sx));
      corr[slot * stride + order] = (float)sqrt((xr * xr + xi * xi) / (sx * sy));
    }
  }
  if (pub.out != nullptr) {
    __syncthreads();
    fit_publish(fit, pub, amp, corr);
  }
}

__global__ __launch_bounds__(256) void k_modamp_finish_fp32(const int* __restrict__ kslot,
                                                            const float4* __restrict__ part32, int nparts,
                                                            float2* __restrict__ amp, float* __restrict__ corr,
                                                            int stride, int order) {
#pragma clang fp contract(off)
  __shared__ double stage[4 * kSeqChunk];
  __shared__ double sums[4];
  const int c = blockIdx.x, slot = kslot[c];
  part32 += (long long)c * nparts;
  const float v = seq_sum_lanes<float, 4>(nparts, stage, [&](int i, int k) {
    const float4 q = part32[i];
    return (double)(k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w);
  });
  if (threadIdx.x < 4) sums[threadIdx.x] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  const float xr = (float)sums[0], xi = (float)sums[1], sx = (float)sums[2], sy = (float)sums[3];
  const float mx = xr / sx, my = xi / sx;
  amp[slot * stride + order] = make_float2(mx, my);
  corr[slot * stride + order] = sqrtf((xr * xr + xi * xi) / (sx * sy));
}

__global__ void k_fit_publish(const FitState* fit, FitPub pub, const float2* amps, const float* corr) {
  fit_publish(fit, pub, amps, corr);
}

void launch_modamp_finish(bool fp32, const ModampSlots& m, const int* kslot, int ncand, const double2* part64,
                          const float4* part32, int nparts, float2* amp, float* corr, int stride, int order,
                          const FitState* fit, const FitPub& pub, hipStream_t s) {
  if (ncand < 1) return;
  if (ncand > kMaxDirs) throw ArgError("modamp finish: 1..8 candidates");
  if (fp32) {
    hipLaunchKernelGGL(k_modamp_finish_fp32, dim3(ncand), dim3(256), 0, s, kslot, part32, nparts, amp, corr, stride,
                       order);
    if (pub.out != nullptr) hipLaunchKernelGGL(k_fit_publish, dim3(1), dim3(64), 0, s, fit, pub, amp, corr);
  } else {
    for (int k = 0; k < ncand; ++k) check_totals(m, k);  // kslot holds slots 0 .. ncand - 1
    hipLaunchKernelGGL(k_modamp_finish_fp64, dim3(1), dim3(64 * ncand), 0, s, m, kslot, ncand, part64, nparts, amp,
                       corr, stride, order, fit, pub);
  }
  SIMR_LAUNCH_CHECK();
}

__global__ __launch_bounds__(256) void k_modamp_evals(int fp32, ModampSlots m, CandSet cs,
                                                      const double2* __restrict__ part64,
                                                      const float4* __restrict__ part32, int nparts,
                                                      double* __restrict__ out, int host_out) {
#pragma clang fp contract(off)
  __shared__ double stage[4 * kSeqChunk];
  const int c = blockIdx.x;
  if (!cand_live(cs, c)) return;  // whole block
  out += 4LL * c;
  if (fp32) {
    const float4* pp = part32 + (long long)c * nparts;
    const float v = seq_sum_lanes<float, 4>(nparts, stage, [&](int i, int k) {
      const float4 q = pp[i];
      return (double)(k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w);
    });
    if (threadIdx.x < 4) out[threadIdx.x] = v;
  } else {
    // a wavefront for each of xr, xi, sx, sy
    const double2* pp = part64 + (long long)c * nparts;
    const int slot = cand_slot(cs, c), zb = m.zb[slot];
    const double* totals = m.totals[slot];
    const int w = threadIdx.x / 64;
    double v, xi;
    if (w < 2) {
      const double xr = quad_sum(nparts, [&](int i) { return pp[i]; }, &xi);
      v = w == 0 ? xr : xi;
    } else {
      v = wave_sum(zb, [&](int i) { return totals[(w == 2 ? 0 : zb) + i]; });
    }
    if (threadIdx.x % 64 == 0) out[w] = v;
  }
  if (host_out) __threadfence_system();
}

void launch_modamp_evals(bool fp32, const ModampSlots& m, const CandSet& c, int ncand, const double2* part64,
                         const float4* part32, int nparts, double* out, bool host_out, hipStream_t s) {
  check_cands(c, ncand);
  if (!fp32)
    for (int k = 0; k < ncand && c.kc == nullptr; ++k) check_totals(m, c.slot[k]);
  hipLaunchKernelGGL(k_modamp_evals, dim3(ncand), dim3(256), 0, s, fp32 ? 1 : 0, m, c, part64, part32, nparts, out,
                     host_out ? 1 : 0);
  SIMR_LAUNCH_CHECK();
}

__global__ void k_fit_signal(unsigned* flag, unsigned seq) {
  __threadfence_system();
  __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

void launch_fit_signal(unsigned* flag, unsigned seq, hipStream_t s) {
  hipLaunchKernelGGL(k_fit_signal, dim3(1), dim3(1), 0, s, flag, seq);
  SIMR_LAUNCH_CHECK();
}

__device__ __forceinline__ float2 cmul_dev(float2 a, float2 b) {
#pragma clang fp contract(off)
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__global__ void k_amp_policy(AmpPolicy a, float2* __restrict__ amps) {
#pragma clang fp contract(off)
  const int dir = threadIdx.x;
  if (dir >= a.ndirs) return;
  float2* am = amps + dir * a.norders;
  if (a.chain)
    for (int order = 2; order < a.norders; ++order) am[order] = cmul_dev(am[order], am[order - 1]);
  if (a.nforceamp > 0 && a.forceamp[0] > 0.0f) {
    for (int order = 1; order < a.norders; ++order) {
      const float m = sqrtf(am[order].x * am[order].x + am[order].y * am[order].y);
      if (order - 1 < a.nforceamp && m < a.forceamp[order - 1]) {
        const float f = a.forceamp[order - 1] / m;
        am[order].x *= f;
        am[order].y *= f;
      }
    }
  }
  if (!a.fit_all_phases) {
    const float base_phase = atan2f(am[1].y, am[1].x);
    for (int order = 2; order < a.norders; ++order) {
      const float2 amplitude = make_float2(sqrtf(am[order].x * am[order].x + am[order].y * am[order].y), 0.f);
      const float phi = (float)order * base_phase;
      am[order] = cmul_dev(amplitude, make_float2((float)cos((double)phi), (float)sin((double)phi)));
    }
  }
}

void launch_amp_policy(const AmpPolicy& a, float2* amps, hipStream_t s) {
  if (a.ndirs > 64) throw ArgError("amp policy: too many directions");
  hipLaunchKernelGGL(k_amp_policy, dim3(1), dim3(64), 0, s, a, amps);
  SIMR_LAUNCH_CHECK();
}

// ------------------------------------------------------------ modamp, FP32
// reductionKernel on 64x4 blocks, float throughout, the thread z-sums being
// the float P/SX/SY of k_overlaps_zsum; block partials are summed on the host in
// block-index order as cpuReduce does.
int modamp_partials_fp32(int nx, int ny) { return ((nx + 63) / 64) * ((ny + 3) / 4); }

__global__ __launch_bounds__(256) void k_modamp_fp32(ModampSlots m, CandSet cand, int nx, int ny, float dxy,
                                                     float4* __restrict__ partials) {
#pragma clang fp contract(off)
  __shared__ float bx[256], by[256], bs[256], bt[256];
  const int c = blockIdx.z;
  if (!cand_live(cand, c)) return;  // whole block
  const int slot = cand_slot(cand, c);
  const double2* __restrict__ P = m.P[slot];
  const double* __restrict__ SX = m.SX[slot];
  const double* __restrict__ SY = m.SY[slot];
  const float2 kc = cand_k(cand, c);
  const float k0x = kc.x, k0y = kc.y;
  const int i = threadIdx.x + blockIdx.x * 64;
  const int j = threadIdx.y + blockIdx.y * 4;
  const float a = ((float)i - 0.5f * (float)nx) * k0x;
  const float b = ((float)j - 0.5f * (float)ny) * k0y;
  const float angle = (float)(2.0f * 3.14159265358979323846 * (double)(a + b) * (double)dxy);
  float sn, cs;
  sincosf(angle, &sn, &cs);
  float xr = 0.f, xi = 0.f, sx = 0.f, sy = 0.f;
  if (i < nx && j < ny) {
    const long long e = (long long)j * nx + i;
    xr = (float)P[e].x;
    xi = (float)P[e].y;
    sx = (float)SX[e];
    sy = (float)SY[e];
  }
  const float tr = xr * cs - xi * sn;
  const float ti = xr * sn + xi * cs;
  const int lt = threadIdx.y * 64 + threadIdx.x;
  bx[lt] = tr;
  by[lt] = ti;
  bs[lt] = sx;
  bt[lt] = sy;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (lt < s) {
      bx[lt] += bx[lt + s];
      by[lt] += by[lt + s];
      bs[lt] += bs[lt + s];
      bt[lt] += bt[lt + s];
    }
    __syncthreads();
  }
  if (lt == 0) {
    const long long blk = (long long)blockIdx.y * gridDim.x + blockIdx.x;
    partials[(long long)c * gridDim.x * gridDim.y + blk] = make_float4(bx[0], by[0], bs[0], bt[0]);
  }
}

void launch_modamp_fp32(const ModampSlots& m, const CandSet& c, int ncand, int nx, int ny, float dxy,
                        float4* partials, hipStream_t s) {
  check_cands(c, ncand);
  dim3 grid((nx + 63) / 64, (ny + 3) / 4, ncand);
  hipLaunchKernelGGL(k_modamp_fp32, grid, dim3(64, 4), 0, s, m, c, nx, ny, dxy, partials);
  SIMR_LAUNCH_CHECK();
}

// Real-space overlap volumes (the debug dump of the overlap pair,
// cudaSirecon.cpp:330-352,433-445): the inverse DFT along z, unnormalised
// and exp(+i) like the reference's inverse 3D transform, of the 2zd+1 stored
// kz planes (plane j holds kz = j - zd; every other kz is zero) of both
// overlaps: vol[which][z][y][x].  A direct sum over the stored planes; this
// runs once per dumped direction, not in the reconstruction.
__global__ __launch_bounds__(256) void k_overlap_volumes(const float2* __restrict__ ovx, int zd, int nzs_stride, int nz,
                                                         long long nxy, float2* __restrict__ vol) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= nxy) return;
  const int z = blockIdx.y, which = blockIdx.z;
  const int nzs = 2 * zd + 1;
  const float2* src = ovx + (long long)which * nzs_stride * nxy + e;
  float re = 0.f, im = 0.f;
  for (int j = 0; j < nzs; ++j) {
    int m = ((j - zd) * z) % nz;  // exp(2 pi i kz z / nz) depends on kz*z mod nz only
    if (m < 0) m += nz;
    double sd, cd;
    sincospi(2.0 * (double)m / (double)nz, &sd, &cd);
    const float c = (float)cd, sn = (float)sd;
    const float2 v = src[(long long)j * nxy];
    re += v.x * c - v.y * sn;
    im += v.x * sn + v.y * c;
  }
  vol[((long long)which * nz + z) * nxy + e] = make_float2(re, im);
}

void launch_overlap_volumes(const float2* ovx, int zd, int nzs_stride, int nz, long long nxy, float2* vol,
                            hipStream_t s) {
  if (zd < 0 || 2 * zd + 1 > nz || 2 * zd + 1 > nzs_stride) throw ArgError("overlap z support wider than the stack");
  if (nz > 65535) throw ArgError("overlap volumes: too many z planes");
  hipLaunchKernelGGL(k_overlap_volumes, dim3((unsigned)ceil_div(nxy, 256), nz, 2), dim3(256), 0, s, ovx, zd,
                     nzs_stride, nz, nxy, vol);
  SIMR_LAUNCH_CHECK();
}

}  // namespace simr
