// Zoomed band assembly (reference: assemblerealspacebands,
// src/cudaSirecon/gpuFunctionsImpl.cu:1741-1851; move_kernel 1853-1913;
// write_outbuffer_kernel1/2 1914-1940; cos_sin_kernel 1942-1954).
//
// The reference, per direction and order, zero-fills a (zoom nx)(zoom ny)(z_zoom nz)
// complex volume, scatters the half-complex band into it (move_kernel),
// inverse-transforms the whole volume and accumulates Re(.) or
// 2 Re(. e^{i phi}) into the output.  Here the inverse transform is split into
// its three 1D passes and pruned to where data can be non-zero:
//   z pass  : reads the band through move_kernel's index map, only for the
//             nx*ny columns the band occupies;
//   y pass  : zero-padded to zoom*ny, only for the nx occupied x columns;
//   x pass  : zero-padded to zoom*nx, all bands of a row at once, with the
//             modulation and the accumulation into the output fused in, so the
//             output is written once per stack instead of read-modified-written
//             per band.
// The order-0 bands of all directions share one transform (linearity).
#include "device_math.hpp"
#include "fft.hpp"
#include "fft_api.hpp"
#include "fft_rp.hpp"
#include "sizes.hpp"
#include "stages.hpp"

namespace simr {

// Whether centred column xc (lateral frequency (xc - (nx/2 - 1)) dkx) lies
// beyond the filter's support for every y, so that every value of it, in
// every stage of the assembly, is zero.  The y pass writes zeros for tiles of
// such columns without reading or transforming them.
__device__ __forceinline__ bool asm_col_dead(const AsmParams& p, int xc) {
  const float kx = (float)(xc - (p.nx / 2 - 1)) * p.dkx;
  return p.rc2_zero > 0.f && kx * kx > p.rc2_zero;
}

// move_kernel's map: occupied output coordinate x = xc - (nx/2 - 1), xc < nx.
__device__ __forceinline__ int z_of_zout(int zout, int nz, int zdim, bool& valid) {
  valid = true;
  if (nz == 1) {
    valid = zout == 0;
    return 0;
  }
  if (zout <= nz - nz / 2) return zout;
  if (zout >= zdim - (nz / 2 - 1)) return zout - zdim;
  valid = false;
  return 0;
}

// ---- z pass: W adjacent xc columns of row yc (blockIdx.y) of band a (blockIdx.z)
template <int N>
__global__ __launch_bounds__(256) void k_asm_z(AsmParams p, const float2* __restrict__ tw) {
  constexpr int TPT = fft_tpt(N);
  constexpr int W = (256 / TPT) > 0 ? 256 / TPT : 1;
  constexpr int NT = W * TPT;
  constexpr int LP = lds_pitch(N);
  __shared__ float2 lds[W * LP];
  FftTw<N> twr;
  __shared__ float2 twstage[N > 1 ? N : 1];
  load_twiddles(twr, twstage, threadIdx.x % TPT, tw, threadIdx.x, blockDim.x);
  const int a = blockIdx.z, yc = blockIdx.y;
  const int xc0 = blockIdx.x * W;
  const int y = yc - (p.ny / 2 - 1);
  // Band value that move_kernel places at lateral (x, y) and axial z (centred
  // coordinates; x < 0 reads the Hermitian mirror, conjugated).  Every
  // address is computed first (invalid elements point at element 0 and are
  // zeroed afterwards), so all loads of a thread are in flight together.
  constexpr int B = (N * W + NT - 1) / NT;
  long long ind[B];
  unsigned okmask = 0, cjmask = 0;
  static_assert(B <= 32, "per-thread element masks hold 32 bits");
#pragma unroll
  for (int k = 0; k < B; ++k) {
    const int idx = threadIdx.x + k * NT;
    const int zout = idx / W, w = idx - (idx / W) * W;
    const int xc = xc0 + w;
    bool valid;
    int z = z_of_zout(zout, p.nz, N, valid);
    valid = valid && xc < p.nx && idx < N * W;
    int x = xc - (p.nx / 2 - 1), yy = y;
    const bool cj = x < 0;
    if (cj) {
      x = -x;
      yy = -yy;
      z = -z;
    }
    if (yy < 0) yy += p.ny;
    if (z < 0) z += p.nz;
    ind[k] = valid ? ((long long)z * p.ny + yy) * p.nxh + x : 0;
    okmask |= (valid ? 1u : 0u) << k;
    cjmask |= (cj ? 1u : 0u) << k;
  }
  float2 v[B];
  const long long dirstride = (long long)p.nbands * p.band_stride;
  if (a == 0) {  // band 0: sum over directions (move_kernel adds the order-0 bands)
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = make_float2(0.f, 0.f);
    for (int d = 0; d < p.ndirs; ++d) {
      const float2* bd = p.bands + d * dirstride;
#pragma unroll
      for (int k = 0; k < B; ++k) {
        const float2 b = bd[ind[k]];
        v[k].x += b.x;
        v[k].y += b.y;
      }
    }
#pragma unroll
    for (int k = 0; k < B; ++k)
      if ((cjmask >> k) & 1u) v[k].y = -v[k].y;
  } else {  // side band: re + i im of the order's two real-space bands
    const int no = p.norders - 1;
    const int dir = (a - 1) / no, order = 1 + (a - 1) % no;
    const float2* bre = p.bands + dir * dirstride + (2 * order - 1) * p.band_stride;
    const float2* bim = p.bands + dir * dirstride + (2 * order) * p.band_stride;
#pragma unroll
    for (int k = 0; k < B; ++k) {
      float2 re = bre[ind[k]], im = bim[ind[k]];
      if ((cjmask >> k) & 1u) {
        re.y = -re.y;
        im.y = -im.y;
      }
      v[k] = make_float2(re.x - im.y, re.y + im.x);
    }
  }
#pragma unroll
  for (int k = 0; k < B; ++k) {
    const int idx = threadIdx.x + k * NT;
    const int zout = idx / W, w = idx - (idx / W) * W;
    if (idx < N * W) lds[w * LP + lds_swz<N>(zout)] = ((okmask >> k) & 1u) ? v[k] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft_lds<N, true>(lds + (threadIdx.x / TPT) * LP, threadIdx.x % TPT, twr);
  for (int idx = threadIdx.x; idx < N * W; idx += NT) {
    const int zout = idx / W, w = idx - (idx / W) * W;
    const int xc = xc0 + w;
    if (xc < p.nx) p.stageZ[(((long long)a * N + zout) * p.ny + yc) * p.nx + xc] = lds[w * LP + lds_swz<N>(zout)];
  }
}

// ---- z pass, Hermitian-paired (zdim == nz, even nx and ny).
// An output column with x < 0 holds conj(B(-x, -y, -z)), and with zdim == nz
// the z map is the identity mod nz, so its inverse transform is the conjugate
// of the stored column's: one transform of stored column (x, s) gives output
// (x, s) and, conjugated, output (-x, -s).  A workgroup therefore reads the
// stored columns x in [x0, x0+W) of stored rows s and -s once (the other
// kernel reads every mirrored element a second time) and writes the four
// output columns they feed.  Side band a: value re + i im, so re and im are
// transformed separately: direct R + iI, mirror conj(R) + i conj(I).
// Band 0 (sum over directions): direct B, mirror conj(B).
// threads per workgroup of the paired z pass: W = threads / (slots * TPT)
// stored columns, so each plane's read of a stored row is W * 8 bytes.
// Side bands (four slots) take 512 threads, eight columns; band 0 (two
// slots) 256 threads, also eight columns.
template <bool B0>
constexpr int asm_zp_threads() {
  return B0 ? 256 : 512;
}
template <int N, bool B0>
constexpr int asm_zp_slots() {
  return B0 ? 2 : 4;  // transforms per stored column: rows s, -s (x re, im)
}
template <int N, bool B0>
constexpr int asm_zp_w() {
  return asm_zp_threads<B0>() / (asm_zp_slots<N, B0>() * fft_tpt(N));
}
template <int N>
constexpr bool asm_zp_ok() {
  return N > kAsmZRegMax && 4 * fft_tpt(N) <= 256;
}

template <int N, bool B0>
__global__ __launch_bounds__(asm_zp_threads<B0>()) void k_asm_z_pair(AsmParams p, const float2* __restrict__ tw) {
  constexpr int TPT = fft_tpt(N);
  constexpr int S = asm_zp_slots<N, B0>();
  constexpr int W = asm_zp_w<N, B0>();
  constexpr int NT = S * W * TPT;
  static_assert(NT == asm_zp_threads<B0>(), "one transform slot per TPT threads");
  constexpr int LP = lds_pitch(N);
  __shared__ float2 lds[S * W * LP];
  FftTw<N> twr;
  __shared__ float2 twstage[N > 1 ? N : 1];
  unsigned bx, by, bz;
  xcd_tile3(bx, by, bz);
  const int a = B0 ? 0 : 1 + (int)bz;
  const int s = (int)by, sp = s == 0 ? 0 : p.ny - s;  // stored rows s and -s
  const int x0 = (int)bx * W;
  const int xmax = p.nx / 2;  // stored columns 0 .. nx/2 feed the output
  const int ycs = s + p.ny / 2 - 1;                  // output row of centred y = s
  const int ycp = (s == 0 ? 0 : -s) + p.ny / 2 - 1;  // output row of centred y = -s
  const int ycp2 = s == p.ny / 2 ? ycs : ycp;        // s = ny/2 is its own mirror
  {
    // The tile's columns lie at |kx| >= x0 dkx on rows |ky| = s dky: when
    // even the nearest is beyond the filter's support, every output is zero,
    // and the y pass does not read it.
    const float kx = (float)x0 * p.dkx, ky = (float)s * p.dky;
    if (p.rc2_zero > 0.f && kx * kx + ky * ky > p.rc2_zero) return;  // uniform over the workgroup
  }
  load_twiddles(twr, twstage, threadIdx.x % TPT, tw, threadIdx.x, blockDim.x);
  const long long dirstride = (long long)p.nbands * p.band_stride;
  const float2* b0;
  const float2* b1;
  if (B0) {
    b0 = p.bands;
    b1 = nullptr;
  } else {
    const int no = p.norders - 1;
    const int dir = (a - 1) / no, order = 1 + (a - 1) % no;
    b0 = p.bands + dir * dirstride + (2 * order - 1) * p.band_stride;
    b1 = b0 + p.band_stride;
  }
  // element e = (j * N + z) * W + w: slot j (B0: row s, row -s; else re s,
  // im s, re -s, im -s), plane z, column x0 + w (clamped: the columns past
  // nx/2 are transformed but never written)
  constexpr int E = S * N * W;
  constexpr int B = (E + NT - 1) / NT;
  long long off[B];
  int slot[B];
#pragma unroll
  for (int k = 0; k < B; ++k) {
    const int e = threadIdx.x + k * NT < E ? threadIdx.x + k * NT : E - 1;  // past E: a valid address, not stored
    const int w = e % W, jz = e / W;
    const int j = jz / N, z = jz - j * N;
    const int row = (B0 ? j : j >> 1) == 0 ? s : sp;
    const int x = x0 + w <= xmax ? x0 + w : xmax;
    off[k] = ((long long)z * p.ny + row) * p.nxh + x;
    slot[k] = (j * W + w) * LP + lds_swz<N>(z);
  }
  float2 v[B];
  if (B0) {
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = make_float2(0.f, 0.f);
    for (int d = 0; d < p.ndirs; ++d) {
      const float2* bd = b0 + d * dirstride;
#pragma unroll
      for (int k = 0; k < B; ++k) {
        const float2 t = bd[off[k]];
        v[k].x += t.x;
        v[k].y += t.y;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const int e = threadIdx.x + k * NT < E ? threadIdx.x + k * NT : E - 1;
      const int j = (e / W) / N;
      v[k] = ((j & 1) ? b1 : b0)[off[k]];
    }
  }
#pragma unroll
  for (int k = 0; k < B; ++k)
    if (threadIdx.x + k * NT < E) lds[slot[k]] = v[k];
  __syncthreads();
  fft_lds<N, true>(lds + (threadIdx.x / TPT) * LP, threadIdx.x % TPT, twr);
  for (int idx = threadIdx.x; idx < W * N; idx += NT) {
    const int w = idx % W, zout = idx / W;
    const int xs = x0 + w;
    if (xs > xmax) continue;
    const int zp = lds_swz<N>(zout);
    float2 ds, dp, ms, mp;
    if (B0) {
      const float2 bs = lds[w * LP + zp], bp = lds[(W + w) * LP + zp];
      ds = bs;
      dp = bp;
      ms = make_float2(bs.x, -bs.y);
      mp = make_float2(bp.x, -bp.y);
    } else {
      const float2 rs = lds[w * LP + zp], is = lds[(W + w) * LP + zp];
      const float2 rp = lds[(2 * W + w) * LP + zp], ip = lds[(3 * W + w) * LP + zp];
      ds = make_float2(rs.x - is.y, rs.y + is.x);
      dp = make_float2(rp.x - ip.y, rp.y + ip.x);
      ms = make_float2(rs.x + is.y, is.x - rs.y);
      mp = make_float2(rp.x + ip.y, ip.x - rp.y);
    }
    float2* plane = p.stageZ + ((long long)a * N + zout) * p.ny * p.nx;
    const int xd = xs + p.nx / 2 - 1;
    plane[(long long)ycs * p.nx + xd] = ds;
    plane[(long long)ycp2 * p.nx + xd] = dp;
    if (xs >= 1 && xs <= xmax - 1) {
      const int xm = p.nx / 2 - 1 - xs;
      plane[(long long)ycp2 * p.nx + xm] = ms;  // mirror of row s lands in row -s
      plane[(long long)ycs * p.nx + xm] = mp;   // and that of row -s in row s
    }
  }
}

// ---- y pass: W adjacent xc columns of plane zout (blockIdx.y) of band a (blockIdx.z)
// Two-pass register core (fft_rp.hpp): every lane loads its pass-1 inputs
// straight from global memory, the intermediate goes through LDS, and the
// outputs leave from registers.  HALVES = 2 (exact 2x zoom): the zero-padded
// transform of N = 2 ny points as the two ny-point halves.
// Thread (w, j, h): column xc0 + w, lane j of its transform, half h (plans
// that split the halves); every row access of a wavefront is a W-column
// segment.  16 columns (whole 128-byte lines) where the workgroup then has
// at most 512 threads and 80 KB of LDS, so that two share a CU.
template <int N, int HALVES>
struct AsmY {
  static constexpr int LEN = N / HALVES;
  using K = Rp<LEN, HALVES>;
  static constexpr int GROUPS = K::T * (K::SPLIT ? 2 : 1);  // lanes of one column
  static constexpr int span_of(int w) {                     // floats of one transform's LDS
    const int want = w < 32 ? 32 / w : 1;                   // columns offset by 32 / w banks: conflict-free
    return K::SPAN + ((want - K::SPAN % 32) % 32 + 32) % 32;
  }
  static constexpr int lds_of(int w) { return w * (K::SPLIT ? 2 : 1) * span_of(w) * 4; }
  static constexpr int width() {
    int w = 16;
    while (w > 4 && (w * GROUPS > 512 || lds_of(w) > 80 * 1024)) w /= 2;
    while (w * K::T < 64) w *= 2;  // whole wavefronts, each within one half
    return w;
  }
  static constexpr int W = width();
  static constexpr int VALUES = K::R1 * K::HL * K::N1 > K::N2 ? K::R1 * K::HL * K::N1 : K::N2;
  // wavefronts per SIMD asked of the register allocator (128 VGPRs each at
  // four, 168 at three): four where that does not spill.  Split halves and
  // factors of 5 do (800 rows: 29 registers, 243 us against 142 us at three).
  // A workgroup of 512 threads is two wavefronts per SIMD whatever is asked for:
  // 2304 and 4096 rows spill about 40 registers there (4096 x 2048 columns x 6
  // planes 2.55 ms, on the radix stages before 2.33, the one length that lost).
  static constexpr int WAVES = VALUES <= 32 ? (K::SPLIT || LEN % 5 == 0 ? 3 : 4) : VALUES <= 40 ? 2 : 1;
  static constexpr int NT = W * GROUPS;
  static constexpr int LDS = lds_of(W);
};

template <int N, int HALVES, bool PAD>
__global__ __launch_bounds__((AsmY<N, HALVES>::NT), (AsmY<N, HALVES>::WAVES)) void k_asm_y(AsmParams p, const float2* __restrict__ tw) {
  using C = AsmY<N, HALVES>;
  using K = typename C::K;
  constexpr int W = C::W, LEN = C::LEN, N1 = K::N1, N2 = K::N2;
  static_assert(C::NT <= 1024 && C::LDS <= 160 * 1024, "the tile fits a workgroup");
  __shared__ float buf[C::LDS / 4];
  unsigned bx, by, bz;
  xcd_tile3(bx, by, bz);
  const int a = (int)bz, zout = (int)by;
  const int xc0 = (int)bx * W;
  float2* const dst = p.stageY + ((long long)a * p.zdim + zout) * (long long)N * p.nx;
  {
    // the tile's column nearest to the centre decides: the dead columns lie
    // at both ends of the row (uniform over the workgroup)
    const int c = p.nx / 2 - 1 < xc0 ? xc0 : (p.nx / 2 - 1 > xc0 + W - 1 ? xc0 + W - 1 : p.nx / 2 - 1);
    if (asm_col_dead(p, c)) {
      for (int idx = threadIdx.x; idx < N * W; idx += C::NT) {
        const int Y = idx / W, w = idx - (idx / W) * W;
        if (xc0 + w < p.nx) dst[(long long)Y * p.nx + xc0 + w] = make_float2(0.f, 0.f);
      }
      return;
    }
  }
  const int w = threadIdx.x % W, g = threadIdx.x / W;
  const int j = K::SPLIT ? g % K::T : g;
  const bool odd = K::SPLIT && g >= K::T;
  const int xc = xc0 + w < p.nx ? xc0 + w : p.nx - 1;
  const float2* const src = p.stageZ + ((long long)a * p.zdim + zout) * p.ny * p.nx + xc;
  // Rows beyond the filter's support in this column are zero; the z pass
  // does not write them.  The bound is taken a little inside the z pass's
  // (rc2_zero), so rounding never reads an element that was not written.
  const int hy = p.ny / 2 - 1;
  float2 in[K::R1 * N1];
#pragma unroll
  for (int c = 0; c < K::R1; ++c) {
    const int n2 = K::N2 % K::T == 0 || j + K::T * c < N2 ? j + K::T * c : N2 - 1;
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) {
      const int n = N2 * n1 + n2;
      // frequency of element n, and its source row (centred: row y + hy)
      int y;
      bool live = true;
      if (HALVES == 2 && !PAD) {
        y = n > LEN / 2 ? n - LEN : n;
      } else {
        const bool lo = n <= p.ny - p.ny / 2, hi = n >= LEN - hy;
        y = lo ? n : n - LEN;
        live = lo || hi;
      }
      live = live && !asm_dead(p, xc - (p.nx / 2 - 1), y, p.rc2_zero * 0.9999f);
      const float2 t = src[(long long)(live ? y + hy : hy) * p.nx];
      in[c * N1 + n1] = live ? t : make_float2(0.f, 0.f);
    }
  }
  float2 out[N2];
  rp_transform<LEN, HALVES, true, false>(buf + (w + (odd ? W : 0)) * C::span_of(W), j, odd, tw, in, out);
  if (xc0 + w < p.nx && (K::ROWS == K::T || j < K::ROWS)) {
    float2* dcol = dst + (long long)K::out0(j, odd ? 1 : 0) * p.nx + xc0 + w;
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) dcol[(long long)(K::OSTEP * k2) * p.nx] = out[k2];
  }
}

template <int N>
static bool launch_asm_z_pair(const AsmParams& p, hipStream_t s) {
  if constexpr (asm_zp_ok<N>()) {
    if (p.zdim != p.nz || p.nz == 1 || (p.nx & 1) || (p.ny & 1)) return false;
    const int nstored = p.nx / 2 + 1;
    hipLaunchKernelGGL((k_asm_z_pair<N, true>), dim3(ceil_div(nstored, asm_zp_w<N, true>()), p.ny / 2 + 1, 1),
                       dim3(asm_zp_threads<true>()), 0, s, p, twiddles(N));
    SIMR_LAUNCH_CHECK();
    if (p.nasm > 1) {
      hipLaunchKernelGGL((k_asm_z_pair<N, false>),
                         dim3(ceil_div(nstored, asm_zp_w<N, false>()), p.ny / 2 + 1, p.nasm - 1), dim3(asm_zp_threads<false>()), 0, s, p,
                         twiddles(N));
      SIMR_LAUNCH_CHECK();
    }
    return true;
  }
  return false;
}

// ---- z pass for depths without a transform kernel (any zdim): the
// move_kernel gather of k_asm_z, one element per thread, into dst
// [a][zout][y][x] (the y-pass staging buffer, idle until the y pass), then a
// direct inverse DFT along z (dft_cols) from dst into stageZ.
__global__ __launch_bounds__(256) void k_asm_z_gather(AsmParams p, int N, float2* __restrict__ dst) {
#pragma clang fp contract(off)
  const long long nxy = (long long)p.nx * p.ny;
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long long)N * nxy) return;
  const int a = blockIdx.y;
  const int zout = (int)(e / nxy);
  const long long r = e - (long long)zout * nxy;
  const int yc = (int)(r / p.nx), xc = (int)(r - (long long)yc * p.nx);
  bool valid;
  int z = z_of_zout(zout, p.nz, N, valid);
  int x = xc - (p.nx / 2 - 1), yy = yc - (p.ny / 2 - 1);
  const bool cj = x < 0;
  if (cj) {
    x = -x;
    yy = -yy;
    z = -z;
  }
  if (yy < 0) yy += p.ny;
  if (z < 0) z += p.nz;
  float2 v = make_float2(0.f, 0.f);
  if (valid) {
    const long long ind = ((long long)z * p.ny + yy) * p.nxh + x;
    const long long dirstride = (long long)p.nbands * p.band_stride;
    if (a == 0) {  // band 0: sum over directions
      for (int d = 0; d < p.ndirs; ++d) {
        const float2 b = p.bands[d * dirstride + ind];
        v.x += b.x;
        v.y += b.y;
      }
      if (cj) v.y = -v.y;
    } else {  // side band: re + i im of the order's two real-space bands
      const int no = p.norders - 1;
      const int dir = (a - 1) / no, order = 1 + (a - 1) % no;
      float2 re = p.bands[dir * dirstride + (2 * order - 1) * p.band_stride + ind];
      float2 im = p.bands[dir * dirstride + (2 * order) * p.band_stride + ind];
      if (cj) {
        re.y = -re.y;
        im.y = -im.y;
      }
      v = make_float2(re.x - im.y, re.y + im.x);
    }
  }
  dst[((long long)a * N + zout) * nxy + r] = v;
}

static void launch_asm_z_any(const AsmParams& p, hipStream_t s) {
  const long long nxy = (long long)p.nx * p.ny;
  const long long n = (long long)p.zdim * nxy;
  if (ceil_div(n, 256) > 2147483647LL || p.nasm > 65535) throw ArgError("assembly z pass: stack too large");
  hipLaunchKernelGGL(k_asm_z_gather, dim3((unsigned)ceil_div(n, 256), p.nasm), dim3(256), 0, s, p, p.zdim, p.stageY);
  SIMR_LAUNCH_CHECK();
  dft_cols(p.stageY, p.stageZ, p.zdim, nxy, nxy, n, p.nasm, true, s);
}

void launch_asm_z(const AsmParams& p, hipStream_t s) {
  if (asm_z_in_registers(p)) {
    launch_asm_z_reg(p, s);
    return;
  }
  switch (p.zdim) {
#define SIMR_CASE(N)                                                                              \
  case N: {                                                                                       \
    if (launch_asm_z_pair<N>(p, s)) return;                                                       \
    constexpr int W = (256 / fft_tpt(N)) > 0 ? 256 / fft_tpt(N) : 1;                              \
    hipLaunchKernelGGL(k_asm_z<N>, dim3(ceil_div(p.nx, W), p.ny, p.nasm), dim3(256), 0, s, p,     \
                       twiddles(N));                                                              \
    SIMR_LAUNCH_CHECK();                                                                          \
    return;                                                                                       \
  }
    SIMR_Z_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      launch_asm_z_any(p, s);
  }
}

// The y pass at zoomed height N; run = false only requests its twiddle table.
template <int N, int HALVES, bool PAD>
static void launch_asm_y_n(const AsmParams& p, bool run, hipStream_t s) {
  using C = AsmY<N, HALVES>;
  const float2* tw = twiddles_rp(N, C::K::N2);
  if (!run) return;
  hipLaunchKernelGGL((k_asm_y<N, HALVES, PAD>), dim3(ceil_div(p.nx, C::W), p.zdim, p.nasm), dim3(C::NT), 0, s, p, tw);
  SIMR_LAUNCH_CHECK();
}

static void asm_y_dispatch(const AsmParams& p, bool run, hipStream_t s) {
  switch (p.ydim) {
#define SIMR_CASE(N)                            \
  case N:                                       \
    if (2 * p.ny == N)                          \
      launch_asm_y_n<N, 2, false>(p, run, s);   \
    else if (2 * p.ny < N && rp_halves_pay<N>()) \
      launch_asm_y_n<N, 2, rp_halves_pay<N>()>(p, run, s); \
    else                                        \
      launch_asm_y_n<N, 1, false>(p, run, s);   \
    return;
    SIMR_ZOOM_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      throw ArgError("zoomed height " + std::to_string(p.ydim) + " is not a supported size");
  }
}

void asm_y_request_tables(const AsmParams& p) { asm_y_dispatch(p, false, nullptr); }
void launch_asm_y(const AsmParams& p, hipStream_t s) { asm_y_dispatch(p, true, s); }

}  // namespace simr
