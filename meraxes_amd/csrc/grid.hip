// grid.hip - galaxy gridding on the device: construct_baryon_grids
// (src/core/reionization.c:1353-1615) for one process holding the whole box.
//
// The reference walks the galaxies in order and adds each one's value to a
// float buffer cell, `buffer[ind] += v` with v double, so every cell's value is
// a sequence of float roundings in galaxy order.  Here each galaxy gets its
// cell as a key (pos_to_ngp of its position, misc_tools.c:163-173), the (key,
// galaxy index) pairs are sorted by key with a stable radix sort (rocPRIM), and
// the first galaxy of every run of equal keys sums its run in galaxy order with
// the reference's roundings and writes the cell's final values into the padded
// grids (the reference's final pass, :1530-1600).  Dead galaxies are dealt over
// the cells with a mark in their index that the sums skip: a key of their own
// past the last cell would cost a sort pass where N^3 is a power of 256 and put
// them all in one run.  The grids are therefore identical to the reference's,
// bit for bit, whatever the number of galaxies per cell.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>

#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../include/mrx_reion.h"
#include "ctx.hpp"

namespace mrx {
namespace {

constexpr int kGT = 256;

struct GridArgs {
  int N;
  int bh;    // Flag_BHFeedback
  int spin;  // Flag_IncludeSpinTemp
  unsigned ncell;  // N^3
  double box_size;
  double bh_limit;  // BlackHoleMassLimitReion
  double a_bh, a_uv;  // ReionAlphaUVBH, ReionAlphaUV
  double ts;  // sfr_timescale
};

#pragma clang fp contract(off)
// pos_to_ngp (misc_tools.c:163-173): nearbyint in the default rounding mode
// (ties to even), an index above N-1 wraps to 0; -1 for an index the
// reference's assert rejects (negative, or not a number).
__device__ __forceinline__ int ngp(float x, double side, int nx)
{
  const double v = rint((double)x / side * (double)nx);
  if (!(v > -1.0)) return -1;
  if (v > (double)(nx - 1)) return 0;
  return (int)v;
}

constexpr unsigned kDead = 0x80000000u;  // mark of a dead galaxy in its index (n < 2^31)

// The values of one galaxy, side by side: the sums read them in cell order,
// one 32-byte access per galaxy instead of four scattered ones.
struct alignas(32) GalVal {
  double fesc, gross, bhm, ebhm;
};

// Keys, values and counts: counts[0] dead galaxies, counts[1] galaxies below the black
// hole mass limit (N_BlackHoleMassLimitReion, :1473-1478); *bad = the lowest
// index of a galaxy whose grid index is negative.  Grid-stride over at most
// 1024 workgroups, with the counts reduced per workgroup (one atomic per
// workgroup and counter: the atomics of 4096 workgroups on one line took most
// of 117 us for 2e6 galaxies).
__global__ __launch_bounds__(kGT) void k_grid_keys(const float* __restrict__ pos, const int* __restrict__ type,
                                                   const double* __restrict__ fesc,
                                                   const double* __restrict__ gross,
                                                   const double* __restrict__ bhm,
                                                   const double* __restrict__ ebhm, GridArgs a, long n,
                                                   unsigned* __restrict__ keys, unsigned* __restrict__ vals,
                                                   GalVal* __restrict__ gal,
                                                   unsigned long long* __restrict__ counts, int* __restrict__ bad)
{
  __shared__ unsigned red[2][kGT / 64];
  unsigned n_dead = 0, n_below = 0;
  for (long g = (long)blockIdx.x * kGT + threadIdx.x; g < n; g += (long)gridDim.x * kGT) {
    unsigned key = (unsigned)g % a.ncell, val = (unsigned)g;
    const double m = a.bh ? bhm[g] : 0.0;
    if (type[g] > 2) {
      ++n_dead;
      val |= kDead;
    } else {
      const int ix = ngp(pos[3 * g], a.box_size, a.N);
      const int iy = ngp(pos[3 * g + 1], a.box_size, a.N);
      const int iz = ngp(pos[3 * g + 2], a.box_size, a.N);
      if (ix < 0 || iy < 0 || iz < 0)
        atomicMin(bad, (int)g);
      else
        key = (unsigned)iz + (unsigned)a.N * ((unsigned)iy + (unsigned)a.N * (unsigned)ix);
      if (a.bh && !(m >= a.bh_limit)) ++n_below;
    }
    keys[g] = key;
    vals[g] = val;
    gal[g] = GalVal{fesc[g], a.spin ? gross[g] : 0.0, m, a.bh ? ebhm[g] : 0.0};
  }
  for (int o = 32; o > 0; o >>= 1) {
    n_dead += __shfl_xor(n_dead, o);
    n_below += __shfl_xor(n_below, o);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][w] = n_dead;
    red[1][w] = n_below;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned d = 0, b = 0;
    for (int k = 0; k < kGT / 64; ++k) {
      d += red[0][k];
      b += red[1][k];
    }
    if (d) atomicAdd(&counts[0], (unsigned long long)d);
    if (b) atomicAdd(&counts[1], (unsigned long long)b);
  }
}

// The grids before the sums, in one pass: stars, weighted_sfr and (spin) sfr
// zeroed, the SFR history ring moved by one slot (:1376-1398, :1580-1600), its
// slot 0 zeroed at the real cells, its padding kept.  V floats per access: 4
// when every grid is 16-byte aligned (a grid of N N (N + 2) floats, N even, is a
// whole number of them, so every slot is aligned as the first), else 1.  A
// launch per copied slot and per zeroed grid took 370 us for the 1.2 GB of
// 256^3 grids and 8 slots.
constexpr int kShift = 4;  // slots in flight per thread
template <int V>
struct alignas(4 * V) Floats {
  float v[V];
};
template <int V>
__global__ __launch_bounds__(kGT) void k_grid_init(float* __restrict__ stars, float* __restrict__ wsfr,
                                                   float* __restrict__ sfr, float* hist, int nstore, unsigned n,
                                                   int N)
{
  using P = Floats<V>;
  const unsigned i = blockIdx.x * kGT + threadIdx.x;  // of n accesses per grid
  if (i >= n) return;
  const P zero = {};
  reinterpret_cast<P*>(stars)[i] = zero;
  reinterpret_cast<P*>(wsfr)[i] = zero;
  if (!nstore) return;
  reinterpret_cast<P*>(sfr)[i] = zero;
  P* h = reinterpret_cast<P*>(hist) + i;
  P first = h[0];
  // slots from the last down, kShift of them loaded before the first is stored
  for (int s = nstore - 1; s >= 1; s -= kShift) {
    P v[kShift];
#pragma unroll
    for (int u = 0; u < kShift; ++u)
      if (s - u >= 1) v[u] = h[(size_t)(s - u - 1) * n];
#pragma unroll
    for (int u = 0; u < kShift; ++u)
      if (s - u >= 1) h[(size_t)(s - u) * n] = v[u];
  }
  const unsigned z0 = (unsigned)((unsigned long long)i * V % (unsigned)(N + 2));
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const unsigned z = z0 + k, zr = z >= (unsigned)(N + 2) ? z - (N + 2) : z;
    if (zr < (unsigned)N) first.v[k] = 0.0f;
  }
  h[0] = first;
}

// The first galaxy of each run of equal keys sums the run in galaxy order and
// writes the cell (reionization.c:1436-1515 accumulation, :1530-1600 final
// pass).  The next kAhead entries of the run are loaded before the first is
// added: a crowded cell's run is one thread's serial chain (128 us of 2e6
// galaxies on 256^3 went to runs of about a hundred, one load after another).
constexpr int kAhead = 4;
__global__ __launch_bounds__(kGT) void k_grid_accumulate(const unsigned* __restrict__ skey,
                                                         const unsigned* __restrict__ sval, long n,
                                                         const GalVal* __restrict__ gal, GridArgs a,
                                                         float* __restrict__ stars, float* __restrict__ wsfr,
                                                         float* __restrict__ sfr, float* __restrict__ hist0)
{
  const long p = (long)blockIdx.x * kGT + threadIdx.x;
  if (p >= n) return;
  const unsigned key = skey[p];
  if (p > 0 && skey[p - 1] == key) return;
  float st = 0.0f, ws = 0.0f, sf = 0.0f;
  bool more = true;
  for (long q = p; more; q += kAhead) {
    bool in[kAhead], alive[kAhead];
    GalVal g[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      in[u] = q + u < n && skey[q + u] == key;
      const unsigned v = in[u] ? sval[q + u] : kDead;
      alive[u] = !(v & kDead);
      if (alive[u]) g[u] = gal[v];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      more = more && in[u];
      if (!alive[u]) continue;
      const double f = g[u].fesc;
      st = (float)((double)st + f);  // prop_stellar
      ws = (float)((double)ws + f);  // prop_weighted_sfr
      if (a.bh) {
        if (g[u].bhm >= a.bh_limit) {
          const double e = g[u].ebhm;
          st = (float)((double)st + e);
          ws = (float)((double)ws + e * a.a_bh / a.a_uv);
        }
      }
      if (a.spin) sf = (float)((double)sf + g[u].gross);  // prop_sfr
    }
  }
  const unsigned N = (unsigned)a.N;
  const long pad = (long)(key / N) * (N + 2) + key % N;  // INDEX_PADDED of the INDEX_REAL key
  stars[pad] = (st < 0) ? 0.0f : st;
  double v = (double)ws;
  v = (v > 0) ? v / a.ts : 0;
  wsfr[pad] = (float)v;
  if (a.spin) {
    double u = (double)sf;
    u = (u > 0) ? u / a.ts : 0;
    sfr[pad] = (float)u;
    hist0[pad] = (float)u;
  }
}
#pragma clang fp contract(on)

#define G_TRY(call)                                                                                   \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess)                                                                             \
      return ctx_fail(ctx, MRX_EDEVICE, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, \
                      __LINE__);                                                                      \
  } while (0)

// device buffer slots of ctx_buffer used here
enum { S_KEY, S_VAL, S_KEY2, S_VAL2, S_SORT, S_CNT, S_POS, S_TYPE, S_FESC, S_GROSS, S_BHM, S_EBHM, S_STARS,
       S_WSFR, S_SFR, S_HIST, S_GAL };

template <class T>
int stage_in(mrx_ctx* ctx, int slot, const T* host, size_t n, const T** dev)
{
  T* d = static_cast<T*>(ctx_buffer(ctx, slot, sizeof(T) * n));
  if (!d) return MRX_ENOMEM;
  if (n) G_TRY(hipMemcpyAsync(d, host, sizeof(T) * n, hipMemcpyHostToDevice, ctx_stream(ctx)));
  *dev = d;
  return MRX_OK;
}

}  // namespace
}  // namespace mrx

using namespace mrx;

extern "C" int mrx_construct_baryon_grids(mrx_ctx* ctx, const mrx_grid_params* p, long n_gal, const float* pos,
                                          const int* type, const double* fesc_weighted_gsm,
                                          const double* gross_stellar_mass, const double* black_hole_mass,
                                          const double* effective_bhm, float* stars, float* weighted_sfr, float* sfr,
                                          float* sfr_histories, mrx_grid_stats* stats)
{
  if (!ctx) return MRX_EINVAL;
  if (!p) return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: null params");
  const int N = p->grid_dim;
  if (N < 2 || (N & 1) || N > 1600)
    return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: grid_dim %d must be even, 2..1600", N);
  if (n_gal < 0 || n_gal >= (1L << 31))
    return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: n_gal %ld outside [0, 2^31)", n_gal);
  if (!(p->box_size > 0)) return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: box_size must be > 0");
  if (n_gal > 0 && (!pos || !type || !fesc_weighted_gsm))
    return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: pos, type and fesc_weighted_gsm are required");
  if (p->include_spin_temp && ((n_gal > 0 && !gross_stellar_mass) || !sfr || !sfr_histories || p->n_store_sfr < 1))
    return ctx_fail(ctx, MRX_EINVAL,
                    "construct_baryon_grids: include_spin_temp needs gross_stellar_mass, sfr, sfr_histories and "
                    "n_store_sfr >= 1");
  if (p->bh_feedback && n_gal > 0 && (!black_hole_mass || !effective_bhm))
    return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: bh_feedback needs black_hole_mass and effective_bhm");
  if (!stars || !weighted_sfr) return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: null output grid");
  if (hipSetDevice(ctx_device(ctx)) != hipSuccess) return ctx_fail(ctx, MRX_EDEVICE, "hipSetDevice failed");
  hipStream_t st = ctx_stream(ctx);
  const bool spin = p->include_spin_temp != 0, bh = p->bh_feedback != 0;
  const size_t np = (size_t)2 * N * N * (N / 2 + 1);
  const size_t ng = (size_t)n_gal;

  // sfr_timescale = ReionSfrTimescale * hubble_time(snapshot) (virial_properties.c:79-93)
  const double zplus1 = p->redshift + 1;
  const double H = p->hubble * sqrt(p->omega_m * zplus1 * zplus1 * zplus1 + p->omega_k * zplus1 * zplus1 +
                                    p->omega_lambda);
  GridArgs a;
  a.N = N;
  a.bh = bh ? 1 : 0;
  a.spin = spin ? 1 : 0;
  a.ncell = (unsigned)N * N * N;
  a.box_size = p->box_size;
  a.bh_limit = p->bh_mass_limit_reion;
  a.a_bh = p->alpha_uv_bh;
  a.a_uv = p->alpha_uv;
  a.ts = p->reion_sfr_timescale * (1.0 / H);

  // inputs where they lie, or staged
  const float* dpos = pos;
  const int* dtype = type;
  const double *dfesc = fesc_weighted_gsm, *dgross = gross_stellar_mass, *dbhm = black_hole_mass,
               *debhm = effective_bhm;
  float *dstars = stars, *dwsfr = weighted_sfr, *dsfr = sfr, *dhist = sfr_histories;
  const bool host = !p->pointers_on_device;
  const size_t nstore = spin ? (size_t)p->n_store_sfr : 0;
  if (host) {
    int rc;
    if ((rc = stage_in(ctx, S_POS, pos, 3 * ng, &dpos)) || (rc = stage_in(ctx, S_TYPE, type, ng, &dtype)) ||
        (rc = stage_in(ctx, S_FESC, fesc_weighted_gsm, ng, &dfesc)))
      return rc;
    if (spin && (rc = stage_in(ctx, S_GROSS, gross_stellar_mass, ng, &dgross))) return rc;
    if (bh && ((rc = stage_in(ctx, S_BHM, black_hole_mass, ng, &dbhm)) ||
               (rc = stage_in(ctx, S_EBHM, effective_bhm, ng, &debhm))))
      return rc;
    dstars = static_cast<float*>(ctx_buffer(ctx, S_STARS, sizeof(float) * np));
    dwsfr = static_cast<float*>(ctx_buffer(ctx, S_WSFR, sizeof(float) * np));
    if (!dstars || !dwsfr) return MRX_ENOMEM;
    if (spin) {
      dsfr = static_cast<float*>(ctx_buffer(ctx, S_SFR, sizeof(float) * np));
      dhist = static_cast<float*>(ctx_buffer(ctx, S_HIST, sizeof(float) * np * nstore));
      if (!dsfr || !dhist) return MRX_ENOMEM;
      G_TRY(hipMemcpyAsync(dhist, sfr_histories, sizeof(float) * np * nstore, hipMemcpyHostToDevice, st));
    }
  } else if ((reinterpret_cast<uintptr_t>(dpos) | reinterpret_cast<uintptr_t>(dfesc)) & 7) {
    return ctx_fail(ctx, MRX_EINVAL, "construct_baryon_grids: device arrays must be naturally aligned");
  }

  // keys, counts and the validity check before any output is touched
  unsigned* keys = static_cast<unsigned*>(ctx_buffer(ctx, S_KEY, sizeof(unsigned) * (ng + 1)));
  unsigned* vals = static_cast<unsigned*>(ctx_buffer(ctx, S_VAL, sizeof(unsigned) * (ng + 1)));
  unsigned* keys2 = static_cast<unsigned*>(ctx_buffer(ctx, S_KEY2, sizeof(unsigned) * (ng + 1)));
  unsigned* vals2 = static_cast<unsigned*>(ctx_buffer(ctx, S_VAL2, sizeof(unsigned) * (ng + 1)));
  unsigned long long* cnt = static_cast<unsigned long long*>(ctx_buffer(ctx, S_CNT, 64));
  GalVal* gal = static_cast<GalVal*>(ctx_buffer(ctx, S_GAL, sizeof(GalVal) * ng));
  if (!keys || !vals || !keys2 || !vals2 || !cnt || !gal) return MRX_ENOMEM;
  int* bad = reinterpret_cast<int*>(cnt + 2);
  const unsigned long long init[3] = {0ull, 0ull, 0x7fffffffull};
  G_TRY(hipMemcpyAsync(cnt, init, sizeof init, hipMemcpyHostToDevice, st));
  const unsigned nb = (unsigned)((ng + kGT - 1) / kGT);
  if (ng) {
    k_grid_keys<<<nb < 1024 ? nb : 1024, kGT, 0, st>>>(dpos, dtype, dfesc, dgross, dbhm, debhm, a, n_gal, keys,
                                                       vals, gal, cnt, bad);
    G_TRY(hipGetLastError());
  }
  unsigned long long h[3];
  G_TRY(hipMemcpyAsync(h, cnt, sizeof h, hipMemcpyDeviceToHost, st));
  G_TRY(hipStreamSynchronize(st));
  const int first_bad = (int)(h[2] & 0xffffffffull);
  if (first_bad != 0x7fffffff)
    return ctx_fail(ctx, MRX_EINVAL,
                    "construct_baryon_grids: galaxy %d has a negative grid index (pos_to_ngp asserts, "
                    "misc_tools.c:170)",
                    first_bad);

  {
    const uintptr_t align = reinterpret_cast<uintptr_t>(dstars) | reinterpret_cast<uintptr_t>(dwsfr) |
                            (spin ? reinterpret_cast<uintptr_t>(dsfr) | reinterpret_cast<uintptr_t>(dhist) : 0);
    const unsigned n4 = (unsigned)(np / 4), n1 = (unsigned)np;
    if ((align & 15) == 0)
      k_grid_init<4><<<(n4 + kGT - 1) / kGT, kGT, 0, st>>>(dstars, dwsfr, dsfr, dhist, (int)nstore, n4, N);
    else
      k_grid_init<1><<<(unsigned)((np + kGT - 1) / kGT), kGT, 0, st>>>(dstars, dwsfr, dsfr, dhist, (int)nstore, n1, N);
    G_TRY(hipGetLastError());
  }

  if (ng) {
    // stable sort of (cell, galaxy) by cell
    unsigned bits = 1;
    while (bits < 32 && ((unsigned long long)(a.ncell - 1) >> bits) != 0) ++bits;
    size_t tmp_bytes = 0;
    G_TRY(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys, keys2, vals, vals2, (unsigned)ng, 0, bits, st));
    void* tmp = ctx_buffer(ctx, S_SORT, tmp_bytes);
    if (!tmp) return MRX_ENOMEM;
    G_TRY(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys, keys2, vals, vals2, (unsigned)ng, 0, bits, st));
    k_grid_accumulate<<<nb, kGT, 0, st>>>(keys2, vals2, n_gal, gal, a, dstars, dwsfr, dsfr, dhist);
    G_TRY(hipGetLastError());
  }

  if (host) {
    G_TRY(hipMemcpyAsync(stars, dstars, sizeof(float) * np, hipMemcpyDeviceToHost, st));
    G_TRY(hipMemcpyAsync(weighted_sfr, dwsfr, sizeof(float) * np, hipMemcpyDeviceToHost, st));
    if (spin) {
      G_TRY(hipMemcpyAsync(sfr, dsfr, sizeof(float) * np, hipMemcpyDeviceToHost, st));
      G_TRY(hipMemcpyAsync(sfr_histories, dhist, sizeof(float) * np * nstore, hipMemcpyDeviceToHost, st));
    }
    G_TRY(hipStreamSynchronize(st));
  }
  if (stats) {
    stats->n_dead = (long)h[0];
    stats->n_gridded = n_gal - (long)h[0];
    stats->n_bh_below_limit = (long)h[1];
    stats->sfr_timescale = a.ts;
  }
  return ctx_finish(ctx);
}
