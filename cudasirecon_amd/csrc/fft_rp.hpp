// Two-pass register FFT core for any factorisation N = N1 N2 (no N1 | N2
// condition, unlike fft2.hpp), register in and register out, with the
// transposed intermediate exchanged through LDS one float component at a
// time (4 bytes per element, so twice the transforms fit a CU).
//
//   X[k1 + N1 k2] = sum_{n2} W_N2^{n2 k2} W_N^{n2 k1} sum_{n1} W_N1^{n1 k1} x[N2 n1 + n2]
//
// T lanes (at least the rows of the intermediate; a power of two unless the
// plan's RpWant says otherwise) work on one
// transform: pass 1, lane j takes columns n2 = j, j + T, ...; pass 2, lane j
// takes row j and ends with X[j + rows k2].
//
// Zero padding by exactly two (the zoomed transforms at zoom 2) is done
// without the zeros: of the inverse transform of length 2M with M occupied
// frequencies k in [-(M/2-1), M/2], the even outputs are the M-point
// transform of the input and the odd outputs the M-point transform of the
// input times exp(2 pi i k / 2M).  In the split N = N1 N2 of the M-point
// transform that ramp is exp(i pi n1 / N1) (compile-time constants, applied
// to the pass-1 inputs), exp(i pi n2 / M) (merged into the pass-1 twiddles,
// W_2M^{n2 (2 k1 + 1)}) and a sign for the negative frequencies.
// HL = 2: one lane computes both halves of its columns, rows 2 k1 + h, and
// lane j ends with X[j + 2 N1 k2].  HL = 1 with the odd flag given: the even
// and the odd half are two transforms, X[2 (j + N1 k2) + h].
#pragma once
#include "fft2.hpp"

namespace simr {

struct RpPlan {
  int n1, n2, hl, lanes;
};

// instructions per point of an in-register transform, roughly
constexpr int rp_dft_cost(int n) {
  if (n == 1) return 0;
  const Radices rd = make_radices(n);
  if (rd.n < 0) return 1000;
  int c = 0;
  for (int i = 0; i < rd.n; ++i) c += rd.r[i] == 8 ? 8 : rd.r[i] == 4 ? 4 : rd.r[i] == 2 ? 2 : rd.r[i] == 3 ? 5 : rd.r[i] == 5 ? 8 : 5 + rd.r[i];
  return c + 3 * (rd.n - 1);
}
constexpr int rp_pow2(int n) {
  int t = 1;
  while (t < n) t *= 2;
  return t;
}

// The plan of a length: HALVES = 2 for a transform of M = len points used as
// the two halves of a 2M-point one, else 1.  Lane-instructions per output
// decide; more than 40 values per lane cost occupancy and are taken only
// where nothing else divides the length.
// RpWant bounds the values a lane holds in each pass (kernels with a short
// chain per thread, or with other registers to keep; taken only if a split
// within the bounds exists, else rp_plan is empty), and lets T be any multiple
// of 4 where the lanes of a transform need not share a wavefront.
struct RpWant {
  int max1 = 100, max2 = 80;
  bool any_t = false;
};
constexpr RpPlan rp_plan(int len, int halves, RpWant want = RpWant()) {
  RpPlan best{0, 0, 0, 0};
  long long best_cost = 0;
  for (int n1 = 2; n1 <= 64; ++n1) {
    if (len % n1) continue;
    const int n2 = len / n1;
    if (n2 < 2 || n2 > 80 || make_radices(n1).n < 0 || make_radices(n2).n < 0) continue;
    for (int hl = 1; hl <= halves; ++hl) {
      const int rows = hl * n1;
      if (rows > 64) continue;
      const int t = want.any_t ? (rows + 3) / 4 * 4 : rp_pow2(rows);
      const int r1 = (n2 + t - 1) / t;
      if (r1 * hl * n1 > want.max1 || n2 > want.max2) continue;
      // per value: input loads (6), twiddle and exchange (7); the odd half's ramp
      long long c = (long long)r1 * n1 * (hl * (rp_dft_cost(n1) + 7) + 6);
      if (halves == 2) c += (hl == 2 ? 4 : 2) * r1 * n1;
      c += (long long)n2 * (rp_dft_cost(n2) + 7);
      if (n2 > 32) c = c * (n2 > 40 ? 20 : 11) / 10;
      if (r1 * hl * n1 > 40) c = c * (r1 * hl * n1 > 64 ? 20 : 13) / 10;
      c = c * t * (halves == 2 && hl == 1 ? 2 : 1);
      if (best.n1 == 0 || c < best_cost) {
        best = RpPlan{n1, n2, hl, t};
        best_cost = c;
      }
    }
  }
  return best;
}
constexpr bool rp_ok(int len, int halves, RpWant want = RpWant()) { return rp_plan(len, halves, want).n1 > 0; }

// HALVES as in rp_plan; NT2 = HALVES * LEN is the length of the twiddle table.
// WANT: the index of the kernel's RpWant in kRpWants.
constexpr RpWant kRpWants[] = {
    RpWant(),
    RpWant{24, 24, true},   // 1: short columns of workgroup-wide tiles
    RpWant{32, 32, true},   // 2: the same, longer columns
    RpWant{32, 20, false},  // 3: rows whose products are summed in doubles beside them
    RpWant{32, 32, false},  // 4: the same, longer rows
};
template <int LEN, int HALVES, int WANT = 0>
struct Rp {
  static constexpr RpPlan P = rp_plan(LEN, HALVES, kRpWants[WANT]);
  static_assert(P.n1 > 0, "no plan for this length");
  static constexpr int N1 = P.n1, N2 = P.n2, HL = P.hl, T = P.lanes;
  static constexpr int ROWS = HL * N1;                  // rows of one transform's intermediate
  static constexpr int R1 = (N2 + T - 1) / T;           // pass-1 columns per lane
  static constexpr int RP = N2 | 1;                     // row pitch, floats: odd, free of conflicts
  static constexpr int SPAN = ROWS * RP;                // floats of one transform's intermediate
  static constexpr int NT2 = HALVES * LEN;
  static constexpr int TABN = HALVES * N1 * N2;         // entries of the arranged twiddle table
  static constexpr bool SPLIT = HALVES == 2 && HL == 1; // even and odd half are separate transforms
  // first output of lane j (row j) and the step between its outputs
  __device__ static __forceinline__ int out0(int j, int h) { return SPLIT ? 2 * j + h : j; }
  static constexpr int OSTEP = SPLIT ? 2 * N1 : ROWS;
};

// Wavefronts per SIMD that a lane's values (a pass's inputs or outputs) leave
// room for beside the sums and addresses of the assembly passes.
constexpr int rp_waves(int values) { return values <= 32 ? 3 : values <= 40 ? 2 : 1; }
template <int LEN, int HALVES>
constexpr int rp_values() {
  using K = Rp<LEN, HALVES>;
  return K::R1 * K::HL * K::N1 > K::N2 ? K::R1 * K::HL * K::N1 : K::N2;
}
// Whether a transform of N points with fewer than N/2 of them occupied (a zoom
// above two) is better done as the halves of an N/2-point one, with the empty
// frequencies as zeros in its input, than whole: where the halves' plan leaves
// room for more wavefronts, and for long ones where a lane forms both halves.
// Assembly x pass, whole and as halves, 6 planes: 1536 points (384 columns) 490
// and 297 us, 1920 (480) 807 and 414, 2048 (512) 910 and 392, 2304 (576) 1086 and
// 985, 2880 (720) 1677 and 1263; without more room 3072 points (768) take 1746
// and 2115, 4096 (1024) 2824 and 3662.
template <int N>
constexpr bool rp_halves_pay() {
  return rp_waves(rp_values<N / 2, 2>()) > rp_waves(rp_values<N, 1>()) || (N > 1024 && Rp<N / 2, 2>::HL == 2);
}

// o[n1] = v[n1] exp(+-i pi n1 / N1), negated where the frequency of element
// N2 n1 + n2 of the M-point input is negative (index above M/2)
template <int LEN, bool INV, int N1I = 0>
__device__ __forceinline__ void rp_ramp(float2* o, const float2* v, int n2) {
  using K = Rp<LEN, 2>;
  if constexpr (N1I < K::N1) {
    float2 a = ctw_mul<N1I, 2 * K::N1, INV>(v[N1I]);
    constexpr int B = K::N2 * N1I;
    if constexpr (B > LEN / 2) {
      a = make_float2(-a.x, -a.y);
    } else if constexpr (B + K::N2 - 1 > LEN / 2) {
      const float s = B + n2 > LEN / 2 ? -1.f : 1.f;
      a = make_float2(a.x * s, a.y * s);
    }
    o[N1I] = a;
    rp_ramp<LEN, INV, N1I + 1>(o, v, n2);
  }
}

template <bool WAVE>
__device__ __forceinline__ void rp_sync() {
  fft2_sync<WAVE>();
}

// One transform (or one half, or both halves of a doubled one) by lanes
// j < T.  in[c N1 + n1]: element N2 n1 + j + T c of the LEN-point input
// (columns j + T c >= N2: anything finite or not, never used).  odd: the
// half, for SPLIT plans (uniform over the wavefront).  buf: SPAN floats of
// this transform.  tw: twiddles_rp(HALVES LEN, N2), rows HALVES k1 + h.  out[k2] = X[out0 + OSTEP k2] (lanes
// j >= ROWS: nothing useful).  buf is free again after the caller's next
// rp_sync.  WAVE: the T lanes lie in one wavefront and no other touches buf;
// otherwise workgroup barriers, and every thread of the workgroup calls it.
template <int LEN, int HALVES, bool INV, bool WAVE, int WANT = 0>
__device__ __forceinline__ void rp_transform(float* buf, int j, bool odd, const float2* tw,
                                             const float2 (&in)[Rp<LEN, HALVES, WANT>::R1 * Rp<LEN, HALVES, WANT>::N1],
                                             float2 (&out)[Rp<LEN, HALVES, WANT>::N2]) {
  using K = Rp<LEN, HALVES, WANT>;
  constexpr int N1 = K::N1, N2 = K::N2, HL = K::HL, R1 = K::R1;
  float2 v[R1 * HL * N1];
#pragma unroll
  for (int c = 0; c < R1; ++c) {
    const int n2 = j + K::T * c;
    float2* a = v + c * HL * N1;
    if constexpr (K::SPLIT) {
      if (odd) {
        rp_ramp<LEN, INV>(a, &in[c * N1], n2);
      } else {
#pragma unroll
        for (int i = 0; i < N1; ++i) a[i] = in[c * N1 + i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < N1; ++i) a[i] = in[c * N1 + i];
      if constexpr (HL == 2) rp_ramp<LEN, INV>(a + N1, &in[c * N1], n2);
    }
    const int n2c = (K::N2 % K::T == 0 || n2 < N2) ? n2 : N2 - 1;  // a valid table entry
#pragma unroll
    for (int h = 0; h < HL; ++h) {
      reg_dft<N1, INV>(a + h * N1);
      const float2* wr = tw + (K::SPLIT && odd ? N2 : 0) + n2c;
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
        const int row = HALVES * k1 + h;
        if (row > 0 || K::SPLIT) {
          float2 w = wr[row * N2];
          if (INV) w.y = -w.y;
          a[h * N1 + k1] = cmul(a[h * N1 + k1], w);
        }
        // bounds the table entries in flight (registers)
        if (k1 % 8 == 7) __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  const float* rowp = buf + (K::ROWS < K::T && j >= K::ROWS ? K::ROWS - 1 : j) * K::RP;
#pragma unroll
  for (int part = 0; part < 2; ++part) {
#pragma unroll
    for (int c = 0; c < R1; ++c) {
      const int n2 = j + K::T * c;
      if (K::N2 % K::T == 0 || n2 < N2) {
#pragma unroll
        for (int h = 0; h < HL; ++h)
#pragma unroll
          for (int k1 = 0; k1 < N1; ++k1) {
            const float2 a = v[(c * HL + h) * N1 + k1];
            buf[(HL * k1 + h) * K::RP + n2] = part ? a.y : a.x;
          }
      }
    }
    rp_sync<WAVE>();
#pragma unroll
    for (int i = 0; i < N2; ++i) {
      if (part)
        out[i].y = rowp[i];
      else
        out[i].x = rowp[i];
    }
    if (part == 0) rp_sync<WAVE>();
  }
  __builtin_amdgcn_sched_barrier(0);
  reg_dft<N2, INV>(out);
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace simr
