// The z transforms of stacks up to 64 planes deep: a thread owns one (x, y)
// column and transforms it in its registers (reg_dft, constants only).  The
// loads and stores of a wavefront are 64 neighbouring columns of one plane
// each, all planes' loads in flight at once, and nothing goes through LDS.
// Depths with prime factors up to 31 all have such a transform (a prime's
// costs about as many operations per point as its value), so a stack may be as
// deep as the sample asks for.
//
// What bounds them: HBM.
#include "fft2.hpp"
#include "sizes.hpp"
#include "stages.hpp"

namespace simr {

bool z_in_registers(int n) {
  switch (n) {
#define SIMR_CASE(N) case N:
    SIMR_REG_SIZES(SIMR_CASE)
#undef SIMR_CASE
    return true;
    default:
      return false;
  }
}

// ---- forward: columns (x, ky) of every [z][ny][nxh] volume, in place.
// Only columns that something reads are transformed: inside the filter's and
// the overlaps' lateral support (ZColumns::rc2).  DEAD: only the others.
// blockIdx = (64 columns of x, 4 rows, volume); the wavefronts of a row whose
// first column is outside have nothing to do.
// Per launch, against LDS transforms of every column: 15 volumes of 512 x 512
// x 48 334 -> 235 us (0.93 GB, 4.0 TB/s), 1024 x 1024 x 16 384 -> 266 us
// (4.6 TB/s), 256 x 256 x 32 39 -> 33 us, 480 x 400 x 21 75 -> 69 us; 384 x
// 384 x 26 302 us of direct DFT and copy -> 71 us.
template <int N>
__global__ __launch_bounds__(256, N <= 24 ? 4 : N <= 40 ? 3 : N <= 56 ? 2 : 1) void k_zcols(float2* __restrict__ data, ZColumns c, int dead) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), row = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= c.nxh || row >= c.ny || z_column_dead(c, x, row) != (dead != 0)) return;
  const long long plane = (long long)c.nxh * c.ny;
  float2* col = data + (long long)blockIdx.z * plane * N + (long long)row * c.nxh + x;
  float2 v[N];
#pragma unroll
  for (int z = 0; z < N; ++z) v[z] = col[z * plane];
  reg_dft<N, false>(v);
#pragma unroll
  for (int z = 0; z < N; ++z) col[z * plane] = v[z];
}

void launch_zcols(int n, float2* data, const ZColumns& c, int volumes, bool dead, hipStream_t s) {
  const dim3 grid(ceil_div(c.nxh, 64), ceil_div(c.ny, 4), volumes);
  switch (n) {
#define SIMR_CASE(N)                                                                     \
  case N:                                                                                \
    hipLaunchKernelGGL(k_zcols<N>, grid, dim3(256), 0, s, data, c, dead ? 1 : 0);        \
    SIMR_LAUNCH_CHECK();                                                                 \
    return;
    SIMR_REG_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      throw ArgError("z transform of length " + std::to_string(n) + " is not done in registers");
  }
}

// ---- assembly: the inverse z transform of one band's column, zero-padded to
// zdim planes (move_kernel's placement, z_of_zout).  A stored column (x, s),
// 0 <= x <= nx/2, feeds two output columns: its own, and for 0 < x < nx/2
// column -x of the row of -s, which reads the Hermitian mirror: element z
// there is conj of the stored element -z.  A side band is re + i im of its
// order's two real-space bands, so with zdim == nz the mirror's transform is the
// conjugate of the transform of re - i im: the thread reads the planes once and
// transforms both (PAD = false, up to 32 planes).  With zero padding, or more
// planes than two transforms' registers hold, the mirror's planes are placed
// anew and read a second time (PAD = true).  Band 0 sums the directions' order-0 bands; its mirror is
// the conjugate.  Columns beyond the filter's support are not written (the y
// pass does not read them).
template <int N>
__device__ __forceinline__ int asm_zin(const AsmParams& p, int zo, bool mirror) {  // the stored plane, or -1
  int z = zo;
  if (p.nz == 1) return zo == 0 ? 0 : -1;
  if (zo > p.nz - p.nz / 2) {
    if (zo < N - (p.nz / 2 - 1)) return -1;
    z = zo - N;
  }
  if (mirror) z = -z;
  return z < 0 ? z + p.nz : (z >= p.nz ? z - p.nz : z);
}

template <int N>
__device__ __forceinline__ void asm_z_store(float2* dst, long long nxy, const float2* v, bool cj) {
#pragma unroll
  for (int z = 0; z < N; ++z) dst[z * nxy] = cj ? make_float2(v[z].x, -v[z].y) : v[z];
}

template <int N, bool PAD>
__global__ __launch_bounds__(256, PAD || N <= 21 ? (N <= 32 ? 3 : N <= 50 ? 2 : 1) : 2) void k_asm_z_reg(AsmParams p) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63), s = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x > p.nx / 2 || s >= p.ny) return;
  const int a = blockIdx.z;
  const long long off = (long long)s * p.nxh + x, plane = (long long)p.nxh * p.ny, nxy = (long long)p.nx * p.ny;
  const long long dirstride = (long long)p.nbands * p.band_stride;
  float2* out = p.stageZ + (long long)a * N * nxy;
  const int top = p.ny - p.ny / 2, c0 = p.ny / 2 - 1;  // the largest centred row, the row of y = 0
  const int y = s <= top ? s : s - p.ny;
  const int sm = s == 0 ? 0 : p.ny - s;
  const int ym = sm <= top ? sm : sm - p.ny;
  const bool direct = !asm_dead(p, x, y, p.rc2_zero);
  const bool mirror = x >= 1 && x <= p.nx / 2 - 1 && !asm_dead(p, -x, ym, p.rc2_zero);
  if (!direct && !mirror) return;
  float2* dd = out + (long long)(y + c0) * p.nx + x + p.nx / 2 - 1;
  float2* dm = out + (long long)(ym + c0) * p.nx - x + p.nx / 2 - 1;
  const int no = p.norders - 1;
  const int dir = a == 0 ? 0 : (a - 1) / no, order = a == 0 ? 0 : 1 + (a - 1) % no;
  const float2* bre = p.bands + dir * dirstride + (order == 0 ? 0 : 2 * order - 1) * p.band_stride + off;
  const float2* bim = bre + p.band_stride;
  auto load0 = [&](float2 (&v)[N], bool mir) {  // band 0: the directions' sum
#pragma unroll
    for (int z = 0; z < N; ++z) v[z] = make_float2(0.f, 0.f);
    for (int d = 0; d < p.ndirs; ++d) {
#pragma unroll
      for (int z = 0; z < N; ++z) {
        const int zi = PAD ? asm_zin<N>(p, z, mir) : z;  // uniform; a valid address for the padding, dropped below
        const float2 t = (bre + d * dirstride)[(zi < 0 ? 0 : zi) * plane];
        v[z].x += t.x;
        v[z].y += t.y;
      }
    }
    if (PAD) {
#pragma unroll
      for (int z = 0; z < N; ++z)
        if (asm_zin<N>(p, z, mir) < 0) v[z] = make_float2(0.f, 0.f);
    }
  };
  if constexpr (!PAD) {
    float2 v[N];
    if (a == 0) {
      load0(v, false);
      reg_dft<N, true>(v);
      if (direct) asm_z_store<N>(dd, nxy, v, false);
      if (mirror) asm_z_store<N>(dm, nxy, v, true);
    } else {
      float2 u[N];
#pragma unroll
      for (int z = 0; z < N; ++z) {
        const float2 re = bre[z * plane], im = bim[z * plane];
        v[z] = make_float2(re.x - im.y, re.y + im.x);
        u[z] = make_float2(re.x + im.y, re.y - im.x);
      }
      reg_dft<N, true>(v);
      if (direct) asm_z_store<N>(dd, nxy, v, false);
      __builtin_amdgcn_sched_barrier(0);
      reg_dft<N, true>(u);
      if (mirror) asm_z_store<N>(dm, nxy, u, true);
    }
  } else {
#pragma unroll 1
    for (int m = 0; m < 2; ++m) {
      const bool mir = m != 0;
      if (!(mir ? mirror : direct)) continue;
      float2 v[N];
      if (a == 0) {
        load0(v, mir);
#pragma unroll
        for (int z = 0; z < N; ++z) v[z].y = mir ? -v[z].y : v[z].y;
      } else {
#pragma unroll
        for (int z = 0; z < N; ++z) {
          const int zi = asm_zin<N>(p, z, mir), za = zi < 0 ? 0 : zi;
          const float2 re = bre[za * plane], im = bim[za * plane];
          const float2 t = mir ? make_float2(re.x + im.y, im.x - re.y) : make_float2(re.x - im.y, re.y + im.x);
          v[z] = zi < 0 ? make_float2(0.f, 0.f) : t;
        }
      }
      reg_dft<N, true>(v);
      asm_z_store<N>(mir ? dm : dd, nxy, v, false);
    }
  }
}

// Where it is taken.  Unpadded depths up to 21 keep both transforms of a side
// band in registers without spilling: 9 planes of 64 x 64 9.9 -> 5.0 us, 21 of
// 480 x 400 94 -> 70 us, 16 of 1024 x 1024 the same 307 us as the paired LDS
// kernel; from there on that kernel is faster (32 of 256 x 256 44 us against
// 88, 48 of 512 x 512 257 us against 408: two wavefronts per SIMD, or
// spills) and this one serves the depths that it has no transform for (26 of
// 384 x 384: 105 us, against 322 us of gather and direct DFT).
bool asm_z_in_registers(const AsmParams& p) {
  if (!z_in_registers(p.zdim)) return false;
  bool only = false;  // no LDS transform of this length
  switch (p.zdim) {
#define SIMR_CASE(N) case N:
    SIMR_REG_ONLY_SIZES(SIMR_CASE)
#undef SIMR_CASE
    only = true;
  }
  return only || (p.zdim == p.nz && p.zdim <= kAsmZRegMax);
}

void launch_asm_z_reg(const AsmParams& p, hipStream_t s) {
  const dim3 grid(ceil_div(p.nx / 2 + 1, 64), ceil_div(p.ny, 4), p.nasm);
  if (p.zdim == p.nz && p.zdim <= 32) {
    switch (p.zdim) {
#define SIMR_CASE(N)                                                         \
  case N:                                                                    \
    hipLaunchKernelGGL((k_asm_z_reg<N, false>), grid, dim3(256), 0, s, p);   \
    SIMR_LAUNCH_CHECK();                                                     \
    return;
      SIMR_REG_PAIR_SIZES(SIMR_CASE)
#undef SIMR_CASE
    }
  }
  switch (p.zdim) {
#define SIMR_CASE(N)                                                         \
  case N:                                                                    \
    hipLaunchKernelGGL((k_asm_z_reg<N, true>), grid, dim3(256), 0, s, p);    \
    SIMR_LAUNCH_CHECK();                                                     \
    return;
    SIMR_REG_ONLY_SIZES(SIMR_CASE)
#undef SIMR_CASE
    default:
      throw ArgError("z transform of length " + std::to_string(p.zdim) + " is not done in registers");
  }
}

}  // namespace simr
