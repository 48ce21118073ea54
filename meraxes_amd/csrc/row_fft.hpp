// row_fft.hpp - inverse real transforms (C2R) of contiguous packed rows.
//
// A workgroup of NT threads brings P packed rows ("pencils") of NH = N / 2
// complex back to real cells: the untwist E + i O of each pair (k, NH - k), then
// the Stockham stages of SchedV<NH, 0>, on the same values in the same order
// as a transform staged in LDS (fft_lds) would.  What is different is where
// the values live:
//   * the first stage runs on registers straight from global memory.  The
//     untwist pairs point k with NH - k; a thread takes the radix-R1
//     butterflies u and Q - u (Q = NH / R1), which hold each other's partners
//     (unit 0 takes 0 and Q / 2, each its own partner), so no point is
//     exchanged before the first LDS write;
//   * the middle stages run in LDS (stockham_stage);
//   * the last stage's outputs stay in registers: a thread takes butterfly j
//     of a row for every field, so the fields of a cell meet in one thread.
// The rows go through LDS nradix - 1 times instead of nradix + 3, with three
// barriers for two radices and five for three.  Staged in LDS the ladder's last
// pass had 7 to 12 waves per CU at the lengths with a factor 3 or 5; per step
// it went from 336 to 146 us (320^3, four fields, now at its vector
// instructions: about 80 per complex point, 130 us), from 77 to 35 us (160^3,
// five fields), from 65 to 32 us (192^3) and from 13.9 to 9.1 us (128^3).
#pragma once
#include "fft_lds.hpp"

namespace mrx {

template <int N>
struct RowCfg {
  static constexpr int NH = N / 2;
  using S = SchedV<NH, 0>;
  static constexpr int NR = S::nradix;
  static constexpr int R1 = S::radix[0], RL = S::radix[NR - 1];
  static_assert(R1 % 2 == 0 && NR >= 2, "the untwist pairs points over an even first radix");
  static constexpr int Q = NH / R1;        // first-stage butterflies of a row
  static constexpr int U = (Q + 1) / 2;    // units: two butterflies each (unit 0 one, if Q is odd)
  static constexpr int NBL = NH / RL;      // last-stage butterflies of a row
  // Two-wave workgroups (three waves where 128 is not a multiple of NBL: 40 at
  // N = 320, four rows): small ones, so that many hide each other's barriers.
  // Their rows give every thread one last-stage butterfly of all fields when
  // its outputs fit the registers (RL <= 5); a radix-8 last stage of four
  // fields would take 64 registers and 16 KiB of LDS per wave, so those rows
  // are half as many and their results go through LDS once more.
  static constexpr bool kViaLds = RL > 5;
  static constexpr int NT = (128 % NBL == 0) ? 128 : 192;
  static constexpr int pow2_below(int v) { return v >= 2 ? 2 * pow2_below(v / 2) : 1; }
  static constexpr int ROWS = pow2_below(NT / NBL / (kViaLds ? 2 : 1));
  static_assert((N * N) % ROWS == 0, "workgroups must tile the rows");
};

// LDS float2 of P rows
template <int N>
constexpr int row_lds(int P)
{
  return P * RowCfg<N>::NH + (P * RowCfg<N>::NH) / 32 + 1;
}

// E + i O and conj(E) + i conj(O) of the pair (k, NH - k), w = conj(tw[k])
__device__ __forceinline__ void untwist_pair(float2 xk, float2 xnk, float2 w, float2& yk, float2& ynk)
{
  const float2 xm = cconj(xnk);
  const float2 E = cadd(xk, xm);
  const float2 O = cmul(csub(xk, xm), w);
  yk = make_float2(E.x - O.y, E.y + O.x);
  ynk = make_float2(E.x + O.y, -E.y + O.x);
}

// z ? p : q by value (a conditional between array elements would select their
// addresses and move the arrays to scratch memory)
__device__ __forceinline__ float2 csel(bool z, float2 p, float2 q)
{
  return make_float2(z ? p.x : q.x, z ? p.y : q.y);
}

// Untwists the two butterflies of a unit: a[m] is point ja + m Q, b[m] point jb
// + m Q, with (ja, jb) = (u, Q - u), or (0, Q / 2) for unit 0.
template <int N>
__device__ __forceinline__ void untwist_unit(float2* a, float2* b, const float2* tw, int u, int ja, int jb)
{
  using C = RowCfg<N>;
  constexpr int R1 = C::R1, Q = C::Q, H = R1 / 2;
  const bool z = (u == 0);
  float2 a2[H], b2[H];  // the second results: of a[m] and of b[m]
  const float2 a0 = a[0], ah = a[H];
#pragma unroll
  for (int m = 0; m < H; ++m) {
    // partners: b[R1 - 1 - m] of a[m] and a[R1 - 1 - m] of b[m]; in unit 0
    // a[R1 - m] and b[R1 - 1 - m]
    const float2 pa = csel(z, a[(R1 - m) % R1], b[R1 - 1 - m]);
    const float2 pb = csel(z, b[R1 - 1 - m], a[R1 - 1 - m]);
    float2 ya, yb;
    untwist_pair(a[m], pa, cconj(tw[ja + m * Q]), ya, a2[m]);
    untwist_pair(b[m], pb, cconj(tw[jb + m * Q]), yb, b2[m]);
    a[m] = ya;
    b[m] = yb;
  }
#pragma unroll
  for (int m = 0; m < H; ++m) {
    const float2 to_b = csel(z, b2[m], a2[m]);  // lands in b[R1 - 1 - m]
    // a[R1 - 1 - m] takes b2[m]; in unit 0 a2[m + 1] (the point R1 - (m + 1)),
    // m + 1 = H being the self-paired point NH / 2
    const float2 to_a = csel(z, a2[(m + 1) % H], b2[m]);
    b[R1 - 1 - m] = to_b;
    a[R1 - 1 - m] = to_a;
  }
  float2 yh, unused;
  untwist_pair(ah, ah, cconj(tw[C::NH / 2]), yh, unused);
  a[0] = csel(z, make_float2(a0.x + a0.y, a0.x - a0.y), a[0]);  // the packed DC and Nyquist values
  a[H] = csel(z, yh, a[H]);
}

// Loads, untwists and first stage of P rows into s; load(pencil, k) returns
// point k of a row.  INPLACE: load reads s itself, so every point is loaded
// before the first is overwritten.  Ends with a barrier.
template <int N, int P, int NT = RowCfg<N>::NT, bool INPLACE = false, class Load>
__device__ __forceinline__ void rows_first(float2* s, const float2* tw, int tid, Load load)
{
  using C = RowCfg<N>;
  constexpr int NH = C::NH, R1 = C::R1, Q = C::Q, U = C::U;
  constexpr int NU = P * U, PT = (NU + NT - 1) / NT;
  float2 a[PT][R1], b[PT][R1];
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const int e = tid + p * NT;
    if ((NU % NT == 0) || e < NU) {
      const int c = e / U, u = e % U;
      const int jb = u ? Q - u : Q / 2;
#pragma unroll
      for (int m = 0; m < R1; ++m) {
        a[p][m] = load(c, u + m * Q);
        b[p][m] = load(c, jb + m * Q);
      }
    }
  }
  if (INPLACE) __syncthreads();
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const int e = tid + p * NT;
    if ((NU % NT == 0) || e < NU) {
      const int c = e / U, u = e % U;
      const int jb = u ? Q - u : Q / 2;
      untwist_unit<N>(a[p], b[p], tw, u, u, jb);
      Bfly<R1, true>::run(a[p]);
      Bfly<R1, true>::run(b[p]);
#pragma unroll
      for (int m = 0; m < R1; ++m) s[lds_addr<true>(c * NH + u * R1 + m)] = a[p][m];
      if ((Q % 2 == 0) || u != 0) {
#pragma unroll
        for (int m = 0; m < R1; ++m) s[lds_addr<true>(c * NH + jb * R1 + m)] = b[p][m];
      }
    }
  }
  __syncthreads();
}

template <int N, int P, int I, int NS, int NT = RowCfg<N>::NT>
__device__ __forceinline__ void rows_middle(float2* s, const float2* tw, int tid)
{
  using C = RowCfg<N>;
  if constexpr (I + 1 < C::NR) {
    constexpr int R = C::S::radix[I];
    stockham_stage<C::NH, R, NS, P, NT, true, 1, C::NH, false, 2, true>(s, tw, tid);
    rows_middle<N, P, I + 1, NS * R, NT>(s, tw, tid);
  }
}

// Last-stage butterfly j of row c: v[m] = point j + m NBL of the complex
// result (real cells 2n and 2n + 1).
template <int N>
__device__ __forceinline__ void rows_last(const float2* s, const float2* tw, int c, int j, float2* v)
{
  using C = RowCfg<N>;
  constexpr int NH = C::NH, RL = C::RL, NBL = C::NBL;
#pragma unroll
  for (int m = 0; m < RL; ++m) v[m] = s[lds_addr<true>(c * NH + j + m * NBL)];
#pragma unroll
  for (int m = 1; m < RL; ++m) v[m] = cmul(v[m], cconj(tw[m * j * 2]));
  Bfly<RL, true>::run(v);
}

// The last stage of P rows in place (a butterfly's outputs replace its
// inputs): real cells 2n, 2n + 1 of row c are float2 lds_addr(c NH + n).  Ends
// with a barrier.
template <int N, int P, int NT = RowCfg<N>::NT>
__device__ __forceinline__ void rows_last_lds(float2* s, const float2* tw, int tid)
{
  using C = RowCfg<N>;
  constexpr int NB = P * C::NBL, PT = (NB + NT - 1) / NT;
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const int e = tid + p * NT;
    if ((NB % NT == 0) || e < NB) {
      const int c = e / C::NBL, j = e % C::NBL;
      float2 v[C::RL];
      rows_last<N>(s, tw, c, j, v);
#pragma unroll
      for (int m = 0; m < C::RL; ++m) s[lds_addr<true>(c * C::NH + j + m * C::NBL)] = v[m];
    }
  }
  __syncthreads();
}

}  // namespace mrx
