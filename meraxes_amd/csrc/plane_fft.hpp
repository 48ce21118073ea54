// plane_fft.hpp - the ladder's inverse y pass and its last pass in one kernel,
// for grids whose x planes fit in LDS (N <= 128).
//
// The y pass reads and writes every spectrum only for the z pass to read it
// again.  A plane (fixed x) of all fields is 4 N^2 bytes per field, 64 KiB at
// 128^3; a workgroup that held it all would leave half the chip idle there, so
// a plane is split by output row: the first radix-8 stage of the y transform
// sends output m of every butterfly to the rows y = m mod 8, which no later
// stage mixes.  PARTS workgroups read the plane (dealt to one XCD back to back,
// so all but the first read its L2) and form 8 / PARTS of the outputs each, m
// apart by PARTS (such outputs share most of their additions): N / PARTS rows
// of every field in LDS, where the remaining y stages, the row transforms
// (row_fft.hpp) and the per-cell test follow.  Operations and values are
// k_colpass's and c2r_threshold_rows', so the results are the same bits.
//
// The ladder's steps of a group run side by side (blockIdx.y): a cell's outcome
// at a step depends on the earlier ones only through "crossed before", so each
// step writes its crossings (a byte per cell pair) and its J_21 where the
// group's first crossing may be, and k_ladder_combine folds them into the
// state in order.  One step at a time (DIRECT, the batch) updates the state
// itself.
//
// Bound by the LDS stages and their barriers: a group of four radii of four
// fields at 128^3 takes 64 us, 134 MB at 2 TB/s, and forming a part's outputs
// alone instead of all eight gave nothing.  Whole bubble finder, y pass and
// threshold apart and now: 318 to 207 us (64^3), 1417 to 1273 us (128^3, four
// fields); 24 boxes of 64^3 to 128^3 in cohorts 9510 to 7930 us.
#pragma once
#include "reion_kernels.hpp"

namespace mrx {

// kernels exist for N <= 128 with a first y radix of eight; planes are dealt to 8 XCDs
template <int N>
constexpr bool plane_ok()
{
  return N <= 128 && SchedV<N, 0>::radix[0] == 8 && N % 8 == 0;
}

template <int N, int NF>
struct PlaneCfg {
  // Two parts while two workgroups' rows (2 NF N^2 bytes each) fit in a CU's
  // LDS, else four: 56 and 67 us with 2 and 4 for eight boxes of two fields at
  // 128^3, but 73 and 64 us for four fields.  One part, the whole plane, was no
  // faster at 64^3 and 96^3 (11.4 and 9.9 us, 32.5 and 31.7 us) and slower at
  // 128^3 (77 us).
  static constexpr int PARTS = NF * N * N * 2 <= 72 * 1024 ? 2 : 4;
  // threads by the rows there are: 1024 against 512 at 128^3 64 and 70 us, 512
  // against 256 at 96^3 32 and 38 us, against 1024 34 us
  static constexpr int NT = N >= 128 ? 1024 : N >= 96 ? 512 : 256;
  static constexpr int CH = 2;  // first-stage butterflies a thread loads at once
  static constexpr int NH = N / 2, NB1 = N / 8, MR = 8 / PARTS, ROWS = MR * NB1;
};

// A y stage of radix R after the first, on the NF * MR sub-transforms of length
// NB1 = N / 8 (rows pm NB1 + j, residue part + PARTS (pm mod MR)) of every
// kz column.
// Stockham index p of the whole transform is 8 j + m: strides are multiples of
// 8, so a stage of size NS = 8 NSC works on j alone, with twiddle index k = 8 (j
// mod NSC) + m.
template <int N, int NF, int R, int NSC>
__device__ __forceinline__ void plane_stage(float2* s, const float2* tw, int tid, int part)
{
  using C = PlaneCfg<N, NF>;
  constexpr int NH = C::NH, NB1 = C::NB1, MR = C::MR, NT = C::NT;
  constexpr int NB = NB1 / R, NU = NF * MR * NB * NH, PT = (NU + NT - 1) / NT;
  float2 v[PT][R];
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const int e = tid + p * NT;
    if ((NU % NT == 0) || e < NU) {
      const int c = e % NH, j = e / NH % NB, pm = e / (NH * NB);
#pragma unroll
      for (int i = 0; i < R; ++i) v[p][i] = s[lds_addr<true>((pm * NB1 + j + i * NB) * NH + c)];
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PT; ++p) {
    const int e = tid + p * NT;
    if ((NU % NT == 0) || e < NU) {
      const int c = e % NH, j = e / NH % NB, pm = e / (NH * NB);
      const int k = 8 * (j % NSC) + part + C::PARTS * (pm % MR);
#pragma unroll
      for (int i = 1; i < R; ++i) v[p][i] = cmul(v[p][i], cconj(tw[i * k * (N / (8 * NSC * R))]));
      Bfly<R, true>::run(v[p]);
      const int row = pm * NB1 + (j / NSC) * NSC * R + j % NSC;
#pragma unroll
      for (int i = 0; i < R; ++i) s[lds_addr<true>((row + i * NSC) * NH + c)] = v[p][i];
    }
  }
  __syncthreads();
}

template <int N, int NF, int I, int NSC>
__device__ __forceinline__ void plane_stages(float2* s, const float2* tw, int tid, int part)
{
  using S = SchedV<N, 0>;
  if constexpr (I < S::nradix) {
    constexpr int R = S::radix[I];
    plane_stage<N, NF, R, NSC>(s, tw, tid, part);
    plane_stages<N, NF, I + 1, NSC * R>(s, tw, tid, part);
  }
}

// The rows y = 8 j + part + PARTS m, m < MR, of plane x of every field, x
// and y transformed, into s: row f ROWS + m NB1 + j.  Ends with a barrier.
template <int N, int NF>
__device__ __forceinline__ void plane_rows(float2* s, const float2* tw, int tid, const float2* __restrict__ T,
                                           long fstride, int x, int part)
{
  using C = PlaneCfg<N, NF>;
  constexpr int NH = C::NH, NB1 = C::NB1, MR = C::MR, ROWS = C::ROWS, NT = C::NT;
  constexpr int NU = NF * NB1 * NH;  // first-stage butterflies
  constexpr int CH = C::CH;
  const float2* src = T + (long)x * N * NH;
  for (int e0 = 0; e0 < NU; e0 += CH * NT) {
    float2 a[CH][8];
#pragma unroll
    for (int p = 0; p < CH; ++p) {
      const int e = e0 + tid + p * NT;
      if (e < NU) {
        const int c = e % NH, j = e / NH % NB1, f = e / (NH * NB1);
        const float2* g = src + f * fstride + j * NH + c;
#pragma unroll
        for (int i = 0; i < 8; ++i) a[p][i] = g[i * NB1 * NH];
      }
    }
#pragma unroll
    for (int p = 0; p < CH; ++p) {
      const int e = e0 + tid + p * NT;
      if (e < NU) {
        const int c = e % NH, j = e / NH % NB1, f = e / (NH * NB1);
        // uniform branches, so that only a part's own outputs are formed
#pragma unroll
        for (int q = 0; q < C::PARTS; ++q)
          if (part == q) {
            Bfly<8, true>::run(a[p]);
#pragma unroll
            for (int m = 0; m < MR; ++m)
              s[lds_addr<true>((f * ROWS + m * NB1 + j) * NH + c)] = a[p][q + C::PARTS * m];
          }
      }
    }
  }
  __syncthreads();
  plane_stages<N, NF, 1, 1>(s, tw, tid, part);
}

// One step (T: its spectra after the x pass) for one part of plane x.  DIRECT:
// the state and J_21 are updated; otherwise the crossings of cell pair i go to
// cross[i] and J_21 of those never crossed before the group to cand (two floats
// per pair, null without the UVB).
template <int N, class FS, bool DIRECT>
__device__ __forceinline__ void plane_threshold(const float2* __restrict__ T, long fstride,
                                                const float2* __restrict__ twN, const ThrGrids& g,
                                                uint8_t* __restrict__ cross, float2* __restrict__ cand, bool fresh,
                                                StepArgs a)
{
  a.last = 0;  // the unfiltered last step takes the plain y and last passes
  using C = PlaneCfg<N, FS::N>;
  constexpr int NF = FS::N, NH = C::NH, NB1 = C::NB1, ROWS = C::ROWS, NT = C::NT, P = NF * ROWS;
  constexpr int NPAIR = ROWS * NH;
  __shared__ float2 s[row_lds<N>(P)];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x;
  // workgroup g: part and plane such that a plane's parts follow each other on XCD g mod 8
  const int slot = blockIdx.x / 8, part = slot % C::PARTS, x = slot / C::PARTS * 8 + blockIdx.x % 8;
  for (int i = tid; i < N; i += NT) tw[i] = twN[i];
  plane_rows<N, NF>(s, tw, tid, T, fstride, x, part);
  rows_first<N, P, NT, true>(s, tw, tid, [&](int c, int k) { return s[lds_addr<true>(c * NH + k)]; });
  rows_middle<N, P, 1, RowCfg<N>::R1, NT>(s, tw, tid);
  rows_last_lds<N, P, NT>(s, tw, tid);
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
  for (int e = tid; e < NPAIR; e += NT) {
    const int r = e / NH, n = e % NH;
    const long row = (long)x * N + 8 * (r % NB1) + part + C::PARTS * (r / NB1);
    const long pair = row * NH + n;
    uint16_t* sp = reinterpret_cast<uint16_t*>(g.state) + pair;
    const uint32_t st = fresh ? 0xFFFFu : *sp;
    float c[2][NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const float2 v = s[lds_addr<true>((f * ROWS + r) * NH + n)];
      c[0][f] = clamp_field<FS>(v.x, f);
      c[1][f] = clamp_field<FS>(v.y, f);
    }
    if constexpr (DIRECT) {
      const uint32_t sn = threshold_pair<N, FS>(c, st, row, 2 * n, a, g, sum);
      if (fresh || sn != st) *sp = (uint16_t)sn;
    } else {
      const CellTest<FS> t0{c[0], a}, t1{c[1], a};
      const bool c0 = t0.cross(), c1 = t1.cross();
      cross[pair] = (uint8_t)((c0 ? 1 : 0) | (c1 ? 2 : 0));
      if (FS::SFR && ((c0 && (st & 0xFFu) == 0xFFu) || (c1 && (st >> 8) == 0xFFu)))
        cand[pair] = make_float2(t0.j21(), t1.j21());
    }
  }
}

// K = gridDim.y steps from a.step on; step k's spectra at T + k kstride, its
// crossings at cross + k N^3 / 2 and candidates at cand + k N^3 / 2.
template <int N, class FS>
__global__ __launch_bounds__((PlaneCfg<N, FS::N>::NT)) void k_plane_threshold(const float2* __restrict__ T, long fstride,
                                                                     long kstride,
                                                                     const float2* __restrict__ twN,
                                                                     const StepDev* __restrict__ steps, ThrGrids g,
                                                                     uint8_t* __restrict__ cross,
                                                                     float2* __restrict__ cand, StepArgs a)
{
  const bool fresh = a.step == 0;
  const long k = blockIdx.y, npair = (long)N * N * (N / 2);
  a.step += (int)k;
  step_load(a, steps);
  plane_threshold<N, FS, false>(T + k * kstride, fstride, twN, g, cross + k * npair, cand + k * npair, fresh, a);
}

// Folds K steps' crossings into the state, in step order, eight cells (four
// pairs) per thread: a cell's first crossing takes that step's J_21, its latest
// is its state.
__global__ __launch_bounds__(kNT) void k_ladder_combine(const uint32_t* __restrict__ cross,
                                                       const float* __restrict__ cand, uint64_t* __restrict__ state,
                                                       float* __restrict__ J21, long npair, int K, int step0, int uvb)
{
  const long q = (long)blockIdx.x * kNT + threadIdx.x;  // of npair / 4
  if (4 * q >= npair) return;
  const uint64_t old = step0 == 0 ? ~0ull : state[q];
  uint64_t st = old;
  constexpr int CH = 8;  // steps loaded at once: the loop is a chain of load latencies otherwise
  for (int k0 = 0; k0 < K; k0 += CH) {
    uint32_t m[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) m[i] = k0 + i < K ? cross[(k0 + i) * (npair / 4) + q] : 0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (!m[i]) continue;
      const int k = k0 + i;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (!((m[i] >> (8 * (c / 2) + c % 2)) & 1)) continue;
        if (uvb && ((st >> (8 * c)) & 0xFFu) == 0xFFu)
          J21[8 * q + c] = cand[2 * (k * npair + 4 * q) + c];
        st = (st & ~(0xFFull << (8 * c))) | ((uint64_t)(step0 + k) << (8 * c));
      }
    }
  }
  if (st != old || step0 == 0) state[q] = st;
}

// One step of every box of a cohort (blockIdx.y is the box; the arguments are
// k_c2r_threshold_batch's, T before the y pass).
template <int N, class FS>
__global__ __launch_bounds__((PlaneCfg<N, FS::N>::NT)) void k_plane_threshold_batch(
  const float2* __restrict__ T, long fstride, long bstride, const float2* __restrict__ twN,
  const BoxDev* __restrict__ boxes, uint8_t* __restrict__ state, const float* __restrict__ Rtab,
  const StepDev* __restrict__ steps, const double* __restrict__ J21c_tab, int nstep, StepArgs a)
{
  const int box = blockIdx.y;
  const BoxDev bx = boxes[box];
  step_load(a, steps);
  a.eff = bx.eff;
  a.redshift = bx.redshift;
  a.bias = bx.bias;
  a.J21c = J21c_tab[(long)box * nstep + a.step];
  const ThrGrids g{bx.deltax, state + (long)box * N * N * N, bx.xH, bx.r_bubble, bx.J21, bx.z_in, bx.J21_ion, nullptr,
                   Rtab};
  plane_threshold<N, FS, true>(T + box * bstride, fstride, twN, g, nullptr, nullptr, a.step == 0, a);
}

}  // namespace mrx
