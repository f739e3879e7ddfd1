// The k0 search's peak refinement and the k0/modamp line searches on the
// device (findk0, gpuFunctionsImpl.cu:316-370; fitk0andmodamps, 874-1020;
// findrealspacemodamp's result, 1128-1147).  One wavefront per SIM direction
// runs the same walk the host would: each walker step replays a direction's
// walk from its start over the candidates evaluated so far and either
// finishes it (the parabola through its last three points) or asks for the
// next kFitLook steps from the first value it misses.  The float and double
// expressions are the host's, in the same order, and the angles and candidate
// vectors come from the same bit-reproducible cos/sin/atan2 (dtrig.hpp), so
// the device walks evaluate the host walks' candidates.
#include "dtrig.hpp"
#include "fit_device.hpp"

namespace simr {

namespace {

__device__ float fit_parabola(float a1, float a2, float a3) {
#pragma clang fp contract(off)
  const float slope = (float)(0.5 * (double)(a3 - a1));
  const float curve = (a3 + a1) - 2 * a2;
  if (curve == 0) return 0.0f;
  const float peak = -slope / curve;
  if (peak > 1.5f || peak < -1.5f) return 0.0f;
  return peak;
}

template <typename U>
__device__ U fit_xyparabola(U x1, U y1, U x2, U y2, U x3, U y3) {
#pragma clang fp contract(off)
  if (x1 == x2 || x2 == x3 || x3 == x1) return 0;
  const U xbar1 = (U)(0.5 * (double)(x1 + x2));
  const U xbar2 = (U)(0.5 * (double)(x2 + x3));
  const U slope1 = (y2 - y1) / (x2 - x1);
  const U slope2 = (y3 - y2) / (x3 - x2);
  const U curve = (slope2 - slope1) / (xbar2 - xbar1);
  if (curve == 0) return 0;
  return xbar2 - slope2 / curve;
}

// |modamp|^2 of one evaluation (xr, xi, sx, sy), as the host forms it
__device__ double fit_amp2(const double* e, int fp32) {
#pragma clang fp contract(off)
  if (fp32) {
    const float xr = (float)e[0], xi = (float)e[1], sx = (float)e[2];
    const float mx = xr / sx, my = xi / sx;
    const float a2 = mx * mx + my * my;
    return (double)a2;
  }
  const double mx = e[0] / e[2], my = e[1] / e[2];
  return mx * mx + my * my;
}

// One direction's walker state while a walker step runs: one wavefront per
// direction, every lane holding the same scalar state (the logic is
// replicated across the lanes; the cache lookups and the requests are spread
// over them), the evaluated candidates in LDS, private to the wavefront.
struct WalkerLds {
  float ka[kFitCache], km[kFitCache];                            // evaluated (angle, mag) keys
  double amp2[kFitCache], xr[kFitCache], xi[kFitCache];          // their |modamp|^2 and sums
  float ra[kFitReq], rm[kFitReq];                                // this round's requests
};
struct Walker {
  WalkerLds* l;
  int ncache, nreq, lane;
};

__device__ __forceinline__ void walker_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// index of the evaluated key (a, m), or -1: the lanes test 64 keys at a time
__device__ __forceinline__ int walker_find(const Walker& w, float a, float m) {
  const unsigned ua = __float_as_uint(a), um = __float_as_uint(m);
  for (int base = 0; base < w.ncache; base += 64) {
    const int i = base + w.lane;
    const int ic = i < w.ncache ? i : 0;  // an index inside the array for every lane
    const bool hit = i < w.ncache && __float_as_uint(w.l->ka[ic]) == ua && __float_as_uint(w.l->km[ic]) == um;
    const unsigned long long b = __ballot(hit);
    if (b != 0ull) return base + __ffsll((long long)b) - 1;
  }
  return -1;
}

// Requests lane i's (a, m) for every i < n, in lane order, except those that
// are evaluated or already requested (the first request of a step: nreq is
// 0 and n at most kFitReq).
__device__ __forceinline__ void walker_request(Walker& w, int n, float a, float m) {
  const unsigned ua = __float_as_uint(a), um = __float_as_uint(m);
  bool keep = w.lane < n;
  for (int e = 0; e < w.ncache; ++e)
    keep = keep && !(__float_as_uint(w.l->ka[e]) == ua && __float_as_uint(w.l->km[e]) == um);
  for (int e = 0; e < n - 1; ++e) {
    const unsigned va = __shfl(ua, e), vm = __shfl(um, e);
    keep = keep && !(e < w.lane && va == ua && vm == um);
  }
  const unsigned long long mask = __ballot(keep);
  const int at = __popcll(mask & ((1ull << w.lane) - 1ull));
  if (keep && at < kFitReq) {
    w.l->ra[at] = a;
    w.l->rm[at] = m;
  }
  w.nreq = min(__popcll(mask), kFitReq);
  walker_sync();
}

// a after n steps of +-delta, by the float accumulation of the walk
__device__ __forceinline__ float walk_steps(float a, int n, float delta, int sign) {
#pragma clang fp contract(off)
  for (int k = 0; k < kFitLook; ++k)
    if (k < n) a = sign > 0 ? a + delta : a - delta;
  return a;
}

// One walk of fitk0andmodamps (gpuFunctionsImpl.cu:912-983) replayed over the
// cache: from `start` step by `delta` while the modamp magnitude grows, then
// the parabola through the last three points.  true: *out and *nevals set;
// false: the next kFitLook steps from the first missing value are requested.
__device__ __forceinline__ bool walker_replay(Walker& w, bool is_angle, float start, float other, float delta, int fp32,
                                              float* out, int* nevals) {
#pragma clang fp contract(off)
  int n = 0;
  int sign = +1;
  auto val = [&](float a, double* amp) {
    const int i = is_angle ? walker_find(w, a, other) : walker_find(w, other, a);
    if (i < 0) {
      const float q = walk_steps(a, w.lane, delta, sign);
      walker_request(w, kFitLook, is_angle ? q : other, is_angle ? other : q);
      return false;
    }
    *amp = w.l->amp2[i];
    ++n;
    return true;
  };
  float x2 = start;
  double amp2, amp3, amp1 = 0;
  if (!val(start, &amp2)) return false;
  float a = start + delta;
  float x3 = a;
  if (!val(a, &amp3)) return false;
  float x1 = 0;
  if (amp3 > amp2) {
    while (amp3 > amp2) {
      amp1 = amp2;
      x1 = x2;
      amp2 = amp3;
      x2 = x3;
      a += delta;
      x3 = a;
      if (!val(a, &amp3)) return false;
    }
  } else {
    a = start;
    const double t = amp3;
    amp3 = amp2;
    amp2 = t;
    const float tx = x3;
    x3 = x2;
    x2 = tx;
    sign = -1;
    while (amp3 > amp2) {
      amp1 = amp2;
      x1 = x2;
      amp2 = amp3;
      x2 = x3;
      a -= delta;
      x3 = a;
      if (!val(a, &amp3)) return false;
    }
  }
  if (!fp32)
    *out = (float)fit_xyparabola<double>(x1, amp1, x2, amp2, x3, amp3);
  else
    *out = fit_xyparabola<float>(x1, (float)amp1, x2, (float)amp2, x3, (float)amp3);
  *nevals = n;
  return true;
}

// The order-fo2 modamp and correlation of the final evaluation
// (findrealspacemodamp's result, 1128-1147).
__device__ void fit_modamp(const double* e, int fp32, float2* m, float* cc) {
#pragma clang fp contract(off)
  if (fp32) {
    const float xr = (float)e[0], xi = (float)e[1], sx = (float)e[2], sy = (float)e[3];
    const float mx = xr / sx, my = xi / sx;
    *m = make_float2(mx, my);
    *cc = sqrtf((xr * xr + xi * xi) / (sx * sy));
  } else {
    const double mx = e[0] / e[2], my = e[1] / e[2];
    *m = make_float2((float)mx, (float)my);
    *cc = (float)sqrt((e[0] * e[0] + e[1] * e[1]) / (e[2] * e[3]));
  }
}

// What a direction carries from one walker step to the next.
struct DirRun {
  int ncache, nprev, phase, started, nang, nmag, nred, rounds, over, have_totals;
  float angle, mag, k0angle, k0mag;
  float2 kov;
  double sx, sy;
};

// Direction d's start from its cross-correlation's five intensities v around
// the maximum at idx.
__device__ __forceinline__ DirRun fit_start(const FitArgs& a, int d, const float* v, int idx, float2* k0) {
#pragma clang fp contract(off)
  const int xc = idx % a.nx, yc = idx / a.nx;
  float2 pk;
  pk.x = fit_parabola(v[1], v[0], v[2]) + (float)xc;
  pk.y = fit_parabola(v[3], v[0], v[4]) + (float)yc;
  const float2 old = a.guess[d];
  if (old.x / a.dkx < pk.x - (float)(a.nx / 2)) pk.x -= (float)a.nx;
  if (old.x / a.dkx > pk.x + (float)(a.nx / 2)) pk.x += (float)a.nx;
  if (old.y / a.dky < pk.y - (float)(a.ny / 2)) pk.y -= (float)a.ny;
  if (old.y / a.dky > pk.y + (float)(a.ny / 2)) pk.y += (float)a.ny;
  pk.x *= a.dkx / (float)a.fo2;
  pk.y *= a.dky / (float)a.fo2;
  *k0 = pk;
  DirRun r{};
  r.k0mag = sqrtf(pk.x * pk.x + pk.y * pk.y);
  r.k0angle = dtrig::fatan2(pk.y, pk.x);
  r.kov = make_float2(r.k0mag * dtrig::fcos(r.k0angle), r.k0mag * dtrig::fsin(r.k0angle));
  r.phase = kFitAngle;
  return r;
}

// Advances direction d's walks over the cache in w.l (w.ncache entries),
// requests what they need next, and writes the direction's state back (one
// wavefront).
__device__ __forceinline__ void walk_dir(FitState* fs, const FitArgs& a, int d, DirRun r, Walker& w, float2* amps,
                                         float* corr) {
#pragma clang fp contract(off)
  for (int guard = 0; guard < 4; ++guard) {
    if (r.phase == kFitAngle || r.phase == kFitMag) {
      const bool ang = r.phase == kFitAngle;
      const float s0 = ang ? r.k0angle : r.k0mag;
      const float other = ang ? r.k0mag : r.angle;
      const float delta = ang ? a.deltaangle : a.deltamag;
      if (!r.started) {
        // the start (lane 0) and the first kFitLook steps up (lanes 1 ..) and
        // down in one batch
        r.started = 1;
        const int i = w.lane;
        const float q = i == 0            ? s0
                        : i <= kFitLook ? walk_steps(s0 + delta, i - 1, delta, +1)
                                          : walk_steps(s0 - delta, i - 1 - kFitLook, delta, -1);
        walker_request(w, kFitReq, ang ? q : other, ang ? other : q);
        if (w.nreq > 0) break;
      }
      float v;
      int ne = 0;
      if (!walker_replay(w, ang, s0, other, delta, a.fp32, &v, &ne)) break;
      if (ang) {
        r.angle = v;
        r.nang += ne;
      } else {
        r.mag = v;
        r.nmag += ne;
      }
      r.nred += ne;
      r.phase += 1;
      r.started = 0;
    } else if (r.phase == kFitFinal) {
      const int i = walker_find(w, r.angle, r.mag);
      if (i < 0) {
        walker_request(w, 1, r.angle, r.mag);
        break;
      }
      // getmodamp at the fitted angle and magnitude: the fitted k0 and its modamp
      r.kov = make_float2(r.mag * dtrig::fcos(r.angle), r.mag * dtrig::fsin(r.angle));
      const double e[4] = {w.l->xr[i], w.l->xi[i], r.sx, r.sy};
      float2 m;
      float cc;
      fit_modamp(e, a.fp32, &m, &cc);
      if (w.lane == 0) {
        amps[d * a.norders + a.fo2] = m;
        corr[d * a.norders + a.fo2] = cc;
      }
      r.nred += 1;
      r.phase = kFitDone;
    } else {
      break;
    }
  }
  FitDir& f = fs->d[d];
  if (w.lane < w.nreq) {
    // getmodamp's vector at (angle, mag), times order2 - order1 (1093-1094)
    const float ra = w.l->ra[w.lane], rm = w.l->rm[w.lane];
    const float kx = rm * dtrig::fcos(ra), ky = rm * dtrig::fsin(ra);
    fs->kc[d * kFitReq + w.lane] = make_float2(kx * (float)a.fo2, ky * (float)a.fo2);
    f.req_a[w.lane] = ra;
    f.req_m[w.lane] = rm;
  }
  if (w.lane == 0) {
    for (int o = 0; o < a.nothers; ++o) a.kc[o][d] = make_float2(r.kov.x * a.kmul[o], r.kov.y * a.kmul[o]);
    fs->nreq[d] = w.nreq;
    f.ncache = w.ncache;
    f.phase = r.phase;
    f.started = r.started;
    f.angle = r.angle;
    f.mag = r.mag;
    f.kov = r.kov;
    f.n_angle_evals = r.nang;
    f.n_mag_evals = r.nmag;
    f.n_reductions = r.nred;
    f.rounds = r.rounds + (w.nreq > 0 ? 1 : 0);
    f.overflow = r.over;
    f.have_totals = r.have_totals;
    f.sx = r.sx;
    f.sy = r.sy;
  }
}

// The cross-correlations' maxima from their block maxima, the starts, and the
// walks' first requests (one wavefront per direction).
__global__ __launch_bounds__(64 * kMaxDirs) void k_fit_begin(FitState* fs, FitArgs a, const float2* __restrict__ cc,
                                                             const float* __restrict__ pv,
                                                             const int* __restrict__ pi) {
  __shared__ WalkerLds lds[kMaxDirs];
  const int d = threadIdx.x / 64, lane = threadIdx.x % 64;
  if (d >= a.ndirs) return;
  cc += (long long)d * a.nx * a.ny;
  pv += d * kArgBlocks;
  pi += d * kArgBlocks;
  float v = -1e30f;
  int idx = 0x7fffffff;
#pragma unroll
  for (int b = 0; b < kArgBlocks; b += 64) better(v, idx, pv[b + lane], pi[b + lane]);
  for (int off = 32; off > 0; off >>= 1) {
    const float v2 = __shfl_xor(v, off);
    const int i2 = __shfl_xor(idx, off);
    better(v, idx, v2, i2);
  }
  // No element won (every intensity NaN): findpeak keeps its initial centre
  // (gpuFunctionsImpl.cu:443-455).
  if (idx < 0 || idx >= a.nx * a.ny) idx = 0;
  const int xc = idx % a.nx, yc = idx / a.nx;
  // lanes 0..4: centre, x-1, x+1, y-1, y+1, wrapped
  int x = xc, y = yc;
  if (lane == 1) x = xc == 0 ? a.nx - 1 : xc - 1;
  if (lane == 2) x = xc == a.nx - 1 ? 0 : xc + 1;
  if (lane == 3) y = yc == 0 ? a.ny - 1 : yc - 1;
  if (lane == 4) y = yc == a.ny - 1 ? 0 : yc + 1;
  const float in = intensity(cc[(long long)y * a.nx + x]);
  float t[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) t[k] = __shfl(in, k);
  float2 k0;
  const DirRun r = fit_start(a, d, t, idx, &k0);
  if (lane == 0) {
    FitDir& f = fs->d[d];
    f.k0 = k0;
    f.k0mag = r.k0mag;
    f.k0angle = r.k0angle;
  }
  Walker w{&lds[d], 0, 0, lane};
  walk_dir(fs, a, d, r, w, nullptr, nullptr);
}

// One walker step (one wavefront per direction, blockDim = 64 * ndirs).  The
// round's partials are loaded beside the direction's state (a direction's
// candidates always sit at kFitReq d), four lanes to a candidate.
__global__ __launch_bounds__(64 * kMaxDirs) void k_fit_walk(FitState* fs, FitArgs a, ModampSlots m,
                                                            const double2* __restrict__ part64, int nparts,
                                                            float2* amps, float* corr, FitPub pub) {
#pragma clang fp contract(off)
  __shared__ WalkerLds lds[kMaxDirs];
  const int d = threadIdx.x / 64, lane = threadIdx.x % 64;
  if (d < a.ndirs) {  // uniform over each wavefront
    FitDir& f = fs->d[d];
    WalkerLds& l = lds[d];
    const int ci = lane / 4 < kFitReq ? lane / 4 : kFitReq - 1;  // the lane's candidate
    double xr = 0.0, xi = 0.0;
    if (!a.fp32) {
      const double2* p = part64 + (long long)(d * kFitReq + ci) * nparts;
      xr = quad_sum(nparts, [&](int i) { return p[i]; }, &xi);
    }
    DirRun r;
    r.ncache = f.ncache;
    r.nprev = fs->nreq[d];
    r.phase = f.phase;
    r.started = f.started;
    r.nang = f.n_angle_evals;
    r.nmag = f.n_mag_evals;
    r.nred = f.n_reductions;
    r.rounds = f.rounds;
    r.over = f.overflow;
    r.have_totals = f.have_totals;
    r.angle = f.angle;
    r.mag = f.mag;
    r.k0angle = f.k0angle;
    r.k0mag = f.k0mag;
    r.kov = f.kov;
    r.sx = f.sx;
    r.sy = f.sy;
    const int nadd = min(r.nprev, kFitCache - r.ncache);
    if (nadd < r.nprev) r.over = 1;
    // the candidates evaluated so far
    for (int i = lane; i < r.ncache; i += 64) {
      l.ka[i] = f.ca[i];
      l.km[i] = f.cm[i];
      l.amp2[i] = f.camp2[i];
      l.xr[i] = f.cxr[i];
      l.xi[i] = f.cxi[i];
    }
    if (nadd > 0) {
      if (a.fp32) {
        const double* e = fs->ev[d * kFitReq + ci];
        xr = e[0];
        xi = e[1];
        r.sx = fs->ev[d * kFitReq][2];  // the same for every candidate of a direction
        r.sy = fs->ev[d * kFitReq][3];
      } else if (!r.have_totals) {
        const int zb = m.zb[d];
        const double* t = m.totals[d];
        r.sx = wave_sum(zb, [&](int i) { return t[i]; });
        r.sy = wave_sum(zb, [&](int i) { return t[zb + i]; });
        r.have_totals = 1;
      }
      // the round's candidates join them
      if (lane % 4 == 0 && lane / 4 < nadd) {
        const int k = r.ncache + ci;
        const double e[4] = {xr, xi, r.sx, r.sy};
        const double amp2 = fit_amp2(e, a.fp32);
        const float ra = f.req_a[ci], rm = f.req_m[ci];
        l.ka[k] = f.ca[k] = ra;
        l.km[k] = f.cm[k] = rm;
        l.amp2[k] = f.camp2[k] = amp2;
        l.xr[k] = f.cxr[k] = xr;
        l.xi[k] = f.cxi[k] = xi;
      }
    }
    walker_sync();
    Walker w{&l, r.ncache + nadd, 0, lane};
    walk_dir(fs, a, d, r, w, amps, corr);
  }
  if (pub.out != nullptr) {
    __syncthreads();
    fit_publish(fs, pub, amps, corr);
  }
}

void check_fit_args(const FitArgs& a) {
  if (a.ndirs < 1 || a.ndirs > kMaxDirs || a.norders < 1 || a.norders > 5 || a.fo2 < 1 || a.fo2 >= a.norders || a.nothers < 0 ||
      a.nothers > kMaxOrders ||
      kFitReq * a.ndirs > kArgCand)
    throw ArgError("device fit: 1..8 directions, 2..5 orders");
}

}  // namespace

void launch_fit_begin(FitState* fs, const FitArgs& a, const float2* cc, const float* partial_val,
                      const int* partial_idx, hipStream_t s) {
  check_fit_args(a);
  hipLaunchKernelGGL(k_fit_begin, dim3(1), dim3(64 * a.ndirs), 0, s, fs, a, cc, partial_val, partial_idx);
  SIMR_LAUNCH_CHECK();
}

void launch_fit_walk(FitState* fs, const FitArgs& a, const ModampSlots& m, const double2* part64, int nparts,
                     float2* amps, float* corr, const FitPub& pub, hipStream_t s) {
  check_fit_args(a);
  hipLaunchKernelGGL(k_fit_walk, dim3(1), dim3(64 * a.ndirs), 0, s, fs, a, m, part64, nparts, amps, corr, pub);
  SIMR_LAUNCH_CHECK();
}

}  // namespace simr
