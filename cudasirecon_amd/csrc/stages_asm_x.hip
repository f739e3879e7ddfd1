// The x pass of the zoomed band assembly (the passes are laid out in
// stages_asm.hip): inverse x transform of every assembly band's rows,
// modulation and accumulation into the output volume.
#include "device_math.hpp"
#include "fft_api.hpp"
#include "fft_rp.hpp"
#include "sizes.hpp"
#include "stages.hpp"

namespace simr {

// ---- x pass: one output row (plane z, row Y) per slot of T lanes.
// The bands of the row are transformed one after another by the same lanes
// (two-pass register core, wave-private LDS exchange, no workgroup barrier
// after the twiddle table), so lane j always ends with the same output
// columns and the modulated bands add up in its registers; the row is stored
// once.  Rows are numbered plane fastest: the rows that share Y, and with it
// the modulation phasors, run together on one XCD and meet the phasor table
// in its L2.
//
// What bounds it: the loads of the next band (three wavefronts per SIMD, 168
// VGPRs) over vector arithmetic; with every input in cache 512 x 512 x 48
// takes 362 us of the 518.  Prefetching a band ahead spills at 168 VGPRs (and
// then costs more than the wait), and at two wavefronts per SIMD
// it gains 5% at 1024 columns and loses as much at 2048.  Lengths whose plans
// have factors of 5 at 30 to 32 values a lane (200, 400, 480, 720, 800, 1440)
// spill 25 to 42 registers at three wavefronts as it is, the others up to 5.  Planes slowest
// instead of fastest: 575 us (the phasor table then misses the L2).  The
// earlier form, eight bands side by side in a workgroup with the sum through
// LDS, on zero-padded rows (radix-stage core where N = N1 N2, N1 | N2 had no
// solution), against this one, per launch:
//   1024 columns x 1024 x 48 planes  614 -> 518 us   768 x 768 x 26  639 -> 220 us
//   2048 x 2048 x 16                2395 -> 743 us   960 x 800 x 21  745 -> 198 us
//    512 x 512 x 32                  170 -> 107 us   400 x 400 x 32  395 -> 118 us
//    800 x 800 x 26                  894 -> 409 us   480 x 480 x 32  455 -> 153 us

// modulation phasor of assembly band a (>= 1) at output column X of row Y
// (cos_sin_kernel, gpuFunctionsImpl.cu:1942-1954: float angle, then sin/cos):
// 2 (cos, sin) of the modulation phase (the factor 2 of write_outbuffer_kernel2,
// exact in float, folded in)
__device__ __forceinline__ float2 asm_phasor(const AsmParams& p, int a, int X, int Y) {
#pragma clang fp contract(off)
  const int no = p.norders - 1;
  const int dir = (a - 1) / no, order = 1 + (a - 1) % no;
  const float k0x = p.k0[dir].x * (float)order, k0y = p.k0[dir].y * (float)order;
  const float s1 = (float)(X - p.xdim / 2) * k0x;
  const float s2 = (float)(Y - p.ydim / 2) * k0y;
  const float sum = s1 + s2;
  const float angle = (float)((double)p.fact * 3.14159265358979323846 * (double)sum * (double)p.dxyo);
  float sn, cs;
  sincosf(angle, &sn, &cs);
  return make_float2(2.f * cs, 2.f * sn);
}

// The phasors of bands 1 .. nasm-1 at every column of the output rows y0 + Y,
// [band - 1][Y][pos]: pos is the column, or with split halves the even columns
// and then the odd ones (the order in which the x pass's lanes read them).
__global__ __launch_bounds__(256) void k_asm_phasors(AsmParams p, int split, int y0, float2* __restrict__ lut) {
  const int pos = blockIdx.x * 256 + threadIdx.x;
  if (pos >= p.xdim) return;
  const int half = p.xdim / 2;
  const int X = !split ? pos : pos < half ? 2 * pos : 2 * (pos - half) + 1;
  lut[((long long)blockIdx.z * gridDim.y + blockIdx.y) * p.xdim + pos] =
      asm_phasor(p, blockIdx.z + 1, X, y0 + (int)blockIdx.y);
}

template <int N, int HALVES>
struct AsmX {
  static constexpr int LEN = N / HALVES;
  using K = Rp<LEN, HALVES>;
  // floats of one slot's LDS: neighbouring slots of a wavefront offset by T banks
  static constexpr int SPANP = K::SPAN + ((K::T - K::SPAN % 64) % 64 + 64) % 64;
  // Phasors of one band that a lane forms at a time without the table, behind
  // the band's transform.  All of them at once, ahead of it, hold 8 bytes of LDS
  // a value, so that one workgroup fits a CU: one plane of 2560 columns (zoom 2)
  // 228 -> 141 us, 3072 (zoom 3) 382 -> 201.  The transform's outputs live
  // meanwhile, so two wavefronts per SIMD are asked for (at three 50 to 74
  // registers spill).
  static constexpr int PB = K::N2 < 16 ? K::N2 : 16;
  // twiddles, exchange buffers and, without the phasor table, every lane's PB phasors
  static constexpr int lds_bytes(int threads, bool lut) {
    return K::TABN * 8 + threads / K::T * SPANP * 4 + (lut ? 0 : threads * PB * 8);
  }
  static constexpr int MAXT = lds_bytes(256, false) <= 160 * 1024 ? 256 : 128;  // threads per workgroup, at most
  static_assert(lds_bytes(MAXT, false) <= 160 * 1024, "rows, phasors and twiddles fit the LDS");
  static constexpr int MINT = K::SPLIT ? 128 : 64;  // a pair of wavefronts (even, odd half) or one
  // wavefronts per SIMD asked of the register allocator (168 VGPRs each at
  // three, 256 at two)
  static constexpr int waves(bool lut) {
    const int w = rp_waves(rp_values<LEN, HALVES>());
    return lut || w < 3 ? w : 2;
  }
  // rows a workgroup of `threads` takes
  static constexpr int rows(int threads) { return threads / K::T / (K::SPLIT ? 2 : 1); }
};

template <int N, int HALVES, bool PAD>
__device__ __forceinline__ void asm_x_fetch(const AsmParams& p, const float2* src, int j,
                                            float2 (&in)[Rp<N / HALVES, HALVES>::R1 * Rp<N / HALVES, HALVES>::N1]) {
  using K = Rp<N / HALVES, HALVES>;
  constexpr int LEN = N / HALVES, N1 = K::N1, N2 = K::N2;
  const int half = p.nx / 2;
#pragma unroll
  for (int c = 0; c < K::R1; ++c) {
    const int n2 = K::N2 % K::T == 0 || j + K::T * c < N2 ? j + K::T * c : N2 - 1;
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
      const int B = N2 * n1;
      float2& d = in[c * N1 + n1];
      if constexpr (HALVES == 2 && !PAD) {  // source column of frequency n (n <= LEN/2) or n - LEN
        if (B > LEN / 2)
          d = src[B - LEN / 2 - 1 + n2];
        else if (B + N2 - 1 <= LEN / 2)
          d = src[B + LEN / 2 - 1 + n2];
        else
          d = src[B + n2 + (B + n2 > LEN / 2 ? -LEN / 2 - 1 : LEN / 2 - 1)];
      } else {
        const int n = B + n2;
        const bool lo = n <= p.nx - half, hi = n >= LEN - (half - 1);
        const float2 t = src[lo ? n + half - 1 : hi ? n - LEN + half - 1 : 0];
        d = lo || hi ? t : make_float2(0.f, 0.f);
      }
    }
  }
}

// The first ny output rows of every plane at p.stageY and p.out (their planes
// p.ydim rows apart); without the table, all of them.
template <int N, int HALVES, bool PAD, bool LUT>
__global__ __launch_bounds__((AsmX<N, HALVES>::MAXT), (AsmX<N, HALVES>::waves(LUT))) void k_asm_x(
    AsmParams p, int ny, const float2* __restrict__ tw, const float2* __restrict__ lut) {
#pragma clang fp contract(off)
  using C = AsmX<N, HALVES>;
  using K = typename C::K;
  constexpr int T = K::T, N1 = K::N1, N2 = K::N2;
  extern __shared__ float2 twl[];  // twiddles, then the slots' exchange buffers
  for (int i = threadIdx.x; i < K::TABN; i += blockDim.x) twl[i] = tw[i];
  __syncthreads();
  const int slot = threadIdx.x / T, j = threadIdx.x % T;
  float* buf = reinterpret_cast<float*>(twl + K::TABN) + slot * C::SPANP;
  // split halves: wavefront pairs (even, odd) take the same 64 / T rows
  const int wave = threadIdx.x / 64;
  const bool odd = K::SPLIT && (wave & 1);
  const int rslot = K::SPLIT ? (wave >> 1) * (64 / T) + slot % (64 / T) : slot;
  const unsigned q = gridDim.x / 8u, r8 = gridDim.x % 8u, xcd = blockIdx.x % 8u;  // XCD-contiguous rows
  const long long blk = (long long)xcd * q + (xcd < r8 ? xcd : r8) + blockIdx.x / 8u;
  const long long nrows = (long long)ny * p.zdim;
  const long long row = blk * (blockDim.x / T / (K::SPLIT ? 2 : 1)) + rslot;
  const long long rc = row < nrows ? row : nrows - 1;
  const int Y = (int)(rc / p.zdim), z = (int)(rc - (long long)Y * p.zdim);
  const float2* src = p.stageY + ((long long)z * p.ydim + Y) * p.nx;
  const long long band = (long long)p.zdim * p.ydim * p.nx;
  const int jr = K::ROWS == T || j < K::ROWS ? j : K::ROWS - 1;
  const int X0 = K::out0(jr, odd ? 1 : 0);
  // the lane's phasors: entry pos0 + PSTEP k2 of each band's row
  constexpr int PSTEP = K::SPLIT ? N1 : K::ROWS;
  const float2* ph = LUT ? lut + (long long)Y * N + (K::SPLIT && odd ? N / 2 : 0) + jr : nullptr;
  float2* phl = reinterpret_cast<float2*>(reinterpret_cast<float*>(twl + K::TABN) + blockDim.x / T * C::SPANP);
  float acc[N2];
#pragma unroll 1
  for (int a = 0; a < p.nasm; ++a, src += band) {
    float2 in[K::R1 * N1], v[N2];
    int jo = j;
    // keeps the general zoom's per-element offsets from being hoisted out of
    // the band loop into registers
    if (HALVES == 1 || PAD) asm volatile("" : "+v"(jo));
    asm_x_fetch<N, HALVES, PAD>(p, src, jo, in);
    rp_transform<C::LEN, HALVES, true, true>(buf, j, odd, twl, in, v);
    rp_sync<true>();
    // write_outbuffer_kernel1/2, gpuFunctionsImpl.cu:1956-1991: band 0 adds
    // its real part, side bands Re(2 v phasor).  2 v.x cos - 2 v.y sin, ph =
    // 2 (cos, sin): a product and a fused multiply-add in float.  The
    // reference forms this term in double and rounds once when adding it to
    // the float output; here the term itself carries up to an ulp of its
    // larger product, a few 1e-8 of the output, for a third of the
    // instructions.
    if (a == 0) {
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) acc[k2] = 0.f + v[k2].x;
    } else if constexpr (LUT) {
      const float2* pa = ph + (long long)(a - 1) * ny * N;
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) {
        const float2 f = pa[PSTEP * k2];
        acc[k2] += __builtin_fmaf(v[k2].x, f.x, -(v[k2].y * f.y));
        if (k2 % 8 == 7) __builtin_amdgcn_sched_barrier(0);  // bounds the phasors in flight
      }
    } else {
      constexpr int PB = C::PB;
#pragma unroll
      for (int k0 = 0; k0 < N2; k0 += PB) {
        const int n = N2 - k0 < PB ? N2 - k0 : PB;
#pragma unroll 1
        for (int i = 0; i < n; ++i)
          phl[i * blockDim.x + threadIdx.x] = asm_phasor(p, a, X0 + K::OSTEP * (k0 + i), Y);
#pragma unroll
        for (int i = 0; i < PB; ++i) {
          if (k0 + i >= N2) break;
          const float2 f = phl[i * blockDim.x + threadIdx.x];
          acc[k0 + i] += __builtin_fmaf(v[k0 + i].x, f.x, -(v[k0 + i].y * f.y));
        }
      }
    }
  }
  if (row < nrows && (K::ROWS == T || j < K::ROWS)) {
    float* orow = p.out + ((long long)z * p.ydim + Y) * N + X0;
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) orow[K::OSTEP * k2] = acc[k2];
  }
}

// The x pass of a stack too small to fill the device with one wavefront per
// 64 / T rows: the bands of those rows go to different wavefronts of a
// workgroup, the modulated terms meet in LDS and are added up there in band
// order (the same sum, term by term, as k_asm_x's).  The phasors are formed
// in the kernel, one LDS slot per output between the two steps.  Against
// one wavefront walking the bands of its rows: 128 columns x 128 x 9 planes
// 24 -> 14 us, 512 x 512 (one plane, 4 bands) 28 -> 13 us.
template <int N, int HALVES>
struct AsmXW {
  static constexpr int LEN = N / HALVES;
  using K = Rp<LEN, HALVES>;
  static constexpr int EXCH = 64 / K::T * AsmX<N, HALVES>::SPANP;          // floats, the exchange
  static constexpr int REGION = EXCH > 128 * K::N2 ? EXCH : 128 * K::N2;  // of one wavefront
  static constexpr int rows() { return 64 / K::T; }
  static int waves(int nasm) { return nasm * (K::SPLIT ? 2 : 1); }
  static size_t lds_bytes(int nasm) { return (size_t)K::TABN * 8 + (size_t)waves(nasm) * REGION * 4; }
};

template <int N, int HALVES, bool PAD>
__global__ __launch_bounds__(1024) void k_asm_x_wide(AsmParams p, const float2* __restrict__ tw) {
#pragma clang fp contract(off)
  using C = AsmXW<N, HALVES>;
  using K = typename C::K;
  constexpr int T = K::T, N2 = K::N2, NH = K::SPLIT ? 2 : 1;
  extern __shared__ float2 twl[];  // twiddles, then the wavefronts' regions
  for (int i = threadIdx.x; i < K::TABN; i += blockDim.x) twl[i] = tw[i];
  __syncthreads();
  float* const regions = reinterpret_cast<float*>(twl + K::TABN);
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int a = wave / NH, h = wave % NH;
  const int slot = lane / T, j = lane % T;
  float* const reg = regions + wave * C::REGION;
  const long long nrows = (long long)p.ydim * p.zdim;
  const long long row0 = (long long)blockIdx.x * C::rows();
  {
    const long long row = row0 + slot < nrows ? row0 + slot : nrows - 1;
    const int Y = (int)(row / p.zdim), z = (int)(row - (long long)Y * p.zdim);
    const float2* src = p.stageY + (((long long)a * p.zdim + z) * p.ydim + Y) * p.nx;
    float2 in[K::R1 * K::N1], v[N2];
    asm_x_fetch<N, HALVES, PAD>(p, src, j, in);
    rp_transform<C::LEN, HALVES, true, true>(reg + slot * AsmX<N, HALVES>::SPANP, j, h != 0, twl, in, v);
    rp_sync<true>();
    // the lane's outputs, read back by the same lane
    float2* const own = reinterpret_cast<float2*>(reg) + lane;
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) own[k2 * 64] = v[k2];
    if (a > 0) {
      const int X0 = K::out0(K::ROWS == T || j < K::ROWS ? j : K::ROWS - 1, h);
#pragma unroll 2
      for (int k2 = 0; k2 < N2; ++k2) {
        const float2 f = asm_phasor(p, a, X0 + K::OSTEP * k2, Y), w = own[k2 * 64];
        own[k2 * 64].x = __builtin_fmaf(w.x, f.x, -(w.y * f.y));
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * N2 * NH; i += blockDim.x) {
    const int ln = i % 64, k2 = i / 64 % N2, hh = i / (64 * N2);
    const float2* t = reinterpret_cast<const float2*>(regions + hh * C::REGION) + k2 * 64 + ln;
    float acc = 0.f + t->x;
    for (int b = 1; b < p.nasm; ++b) acc += t[(long long)b * NH * (C::REGION / 2)].x;
    const long long row = row0 + ln / T;
    const int jj = ln % T;
    if (row < nrows && (K::ROWS == T || jj < K::ROWS)) {
      const int Y = (int)(row / p.zdim), z = (int)(row - (long long)Y * p.zdim);
      p.out[((long long)z * p.ydim + Y) * N + K::out0(jj, hh) + K::OSTEP * k2] = acc;
    }
  }
}

// The x pass at zoomed width N.  The phasor table pays where several planes
// read each of its rows (1, 2 and 3 planes: slower).  It lies in the idle z-pass
// staging; where that holds some of the output rows only (zoom^2 above the number
// of planes, about), the pass goes over the rows in parts, if a part fills the
// device twice over (two of the smallest workgroups per SIMD).  Elsewhere the
// phasors are formed in the kernel.  1536 columns, zoom 3, 6 planes: 301 us
// without the table, 238 in parts; 2048, zoom 4: 728 and 392; 120 columns at zoom
// 8, 9 planes: 187, and 329 in parts of a quarter of that bound.
constexpr long long kAsmPartGroups = 2048;
template <int N, int HALVES, bool PAD>
static void launch_asm_x_n(const AsmParams& p, bool run, hipStream_t s) {
  using C = AsmX<N, HALVES>;
  const float2* tw = twiddles_rp(N, C::K::N2);
  if (!run) return;
  const long long nrows = (long long)p.ydim * p.zdim;
  if constexpr (N <= 1024) {
    using W = AsmXW<N, HALVES>;
    // At most one wavefront per SIMD in the other form: the bands side by
    // side.  (Above that the other form's wavefronts already fill the SIMDs
    // and share the phasor table.)
    if (ceil_div(nrows, W::rows()) * (C::K::SPLIT ? 2 : 1) <= 1024 && p.nasm > 1 && W::waves(p.nasm) <= 16 &&
        W::lds_bytes(p.nasm) <= 160 * 1024) {
      hipLaunchKernelGGL((k_asm_x_wide<N, HALVES, PAD>), dim3(ceil_div(nrows, W::rows())), dim3(64 * W::waves(p.nasm)),
                         W::lds_bytes(p.nasm), s, p, tw);
      SIMR_LAUNCH_CHECK();
      return;
    }
  }
  // small stacks: smaller workgroups, so that the rows spread over the CUs
  const auto threads_for = [](long long rows) {
    int t = C::MAXT;
    while (t > C::MINT && rows < 1024LL * C::rows(t)) t /= 2;
    return t;
  };
  // the output rows whose phasors the table's place holds at a time
  const long long per_row = (long long)(p.nasm - 1) * N, room = (long long)p.nasm * p.zdim * p.ny * p.nx;
  const int parts = p.zdim >= 4 && p.nasm > 1 && per_row <= room ? ceil_div(p.ydim, room / per_row) : 0;
  const int step = parts > 0 ? ceil_div(p.ydim, parts) : 0;
  if (parts == 1 || (long long)step * p.zdim >= kAsmPartGroups * C::rows(C::MINT)) {
    for (int y0 = 0; y0 < p.ydim; y0 += step) {
      const int ny = p.ydim - y0 < step ? p.ydim - y0 : step;
      const int threads = threads_for((long long)ny * p.zdim);
      AsmParams q = p;
      q.stageY += (long long)y0 * p.nx;
      q.out += (long long)y0 * N;
      hipLaunchKernelGGL(k_asm_phasors, dim3(ceil_div(N, 256), ny, p.nasm - 1), dim3(256), 0, s, p,
                         C::K::SPLIT ? 1 : 0, y0, p.stageZ);
      SIMR_LAUNCH_CHECK();
      hipLaunchKernelGGL((k_asm_x<N, HALVES, PAD, true>), dim3(ceil_div((long long)ny * p.zdim, C::rows(threads))),
                         dim3(threads), C::lds_bytes(threads, true), s, q, ny, tw, p.stageZ);
      SIMR_LAUNCH_CHECK();
    }
    return;
  }
  const int threads = threads_for(nrows);
  hipLaunchKernelGGL((k_asm_x<N, HALVES, PAD, false>), dim3(ceil_div(nrows, C::rows(threads))), dim3(threads),
                     C::lds_bytes(threads, false), s, p, p.ydim, tw, (const float2*)nullptr);
  SIMR_LAUNCH_CHECK();
}

static void asm_x_dispatch(const AsmParams& p, bool run, hipStream_t s) {
  switch (p.xdim) {
#define SIMR_CASE(N)                            \
  case N:                                       \
    if (2 * p.nx == N)                          \
      launch_asm_x_n<N, 2, false>(p, run, s);   \
    else if (2 * p.nx < N && rp_halves_pay<N>()) \
      launch_asm_x_n<N, 2, rp_halves_pay<N>()>(p, run, s); \
    else                                        \
      launch_asm_x_n<N, 1, false>(p, run, s);   \
    return;
    SIMR_ZOOM_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      throw ArgError("zoomed width " + std::to_string(p.xdim) + " is not a supported size");
  }
}

void asm_x_request_tables(const AsmParams& p) { asm_x_dispatch(p, false, nullptr); }
void launch_asm_x(const AsmParams& p, hipStream_t s) { asm_x_dispatch(p, true, s); }

}  // namespace simr
