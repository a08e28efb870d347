// efdc_cgp.hip -- CONGRAD as one persistent launch per solve.
//
// The multi-kernel solve (efdc_puv.hip) pays two launches and two grid
// reductions per iteration; at the sizes of a real lake (10^4 .. 10^6 wet
// cells, a working set that lives in the 256 MB MALL) that is latency, not
// bandwidth.  Here every workgroup owns one contiguous range of wet cells
// (L order) and keeps the rows of its cells -- coefficients, neighbour
// indices and all CG vectors -- in registers for the whole solve.  Each
// exchange between iterations moves only
//   * the workgroup's own vector values, through an LDS window that also
//     holds the cells just outside the range that its rows reference, and
//   * the values that the neighbouring workgroups need (cells with a
//     neighbour outside the range) and the dot-product partials, as
//     tagged words in memory.
//
// Exchange protocol.  Every word that crosses workgroups is 64 bits: 32
// bits of data and, above them, the number of the exchange (a double is two
// such words).  The writer stores them with agent-scope atomic stores, which
// are written through to the coherent memory side, and waits for nothing; a
// reader polls the words that it needs themselves until every one carries
// the number.  So an exchange is one trip through memory: with flag words,
// the writer waited for its stores before raising its flag and the reader
// fetched the data after seeing it, three trips (us a solve, flags : tagged
// words; FP64, 29 iterations, 5 k cells 178 : 105, 79 k 216 : 131; mixed, 17
// to 20 inner iterations, 79 k 126 : 103, 696 k 161 : 151).  A slot of
// partials is 48 bytes a workgroup: packed closer, the workgroups' stores to
// one 128-byte line delay each other (79 k FP64 160 : 194), spread over a line
// each, every poll reads more lines (169).
// Two slot parities suffice: a workgroup can only write exchange T+2 after
// it has read every workgroup's sums of T+1, and every workgroup posts those
// only after it has consumed T.  Exchange numbers grow across launches (the
// host numbers launches), so a slot never holds a number yet to come; when
// the numbering wraps the host clears the slots.
//
// FP64 (the reference's Jacobi-PCG, EFDC/congrad.f90:52-187): the same
// recurrences and stop test as the reference, two exchanges per iteration
// (alpha needs p.Ap, beta needs r.z).
//
// Mixed: the inner FP32 CG on the Jacobi-scaled unit-diagonal operator is
// written in the Chronopoulos-Gear form (one exchange per iteration
// carries (r,r), (Ar,r) and the halo triples r, w = Ar, s = Ap); FP64 dot
// products, FP64 alpha/beta, FP64 residual refinement of P inside the
// same launch.
//
// Every wait is bounded: a workgroup that waits too long raises the abort
// flag and leaves, the others see the flag and leave too, and the host
// reports the failure.  All workgroups compute the same sums from the
// same partials in the same order, so they take the same branches.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "efdc_internal.h"

namespace {

constexpr int PB = 512;           // threads per workgroup
constexpr int PW = PB / 64;       // waves per workgroup
constexpr unsigned SPIN_MAX = 1u << 21;
// An inner (FP32) solve stops at the smaller of two reductions of its
// residual: the set one (rtol), or what the outer FP64 test still needs,
// with a margin of 10 in the norm (squared here), so that a round that only
// has to finish the solve is not carried past the target.  The outer test
// is always made on the FP64 residual.
constexpr double INNER_MARGIN2 = 1e-2;
constexpr int WIN = 2048;         // LDS window reach beyond the own range
constexpr int HMAX = 2 * WIN;     // outside cells of one workgroup, at most
constexpr int NVMAX = 3;          // partials per exchange, at most
constexpr int PCG64_CPT_MAX = 6;     // cells per thread, FP64
constexpr int PSLOTS = PB * PCG64_CPT_MAX;  // slots of partials: a workgroup's or a basin tile's
constexpr int PCGMX_CPT_SMALL = 8;  // cells per thread of every mixed form
constexpr int PCGMX_CPT_MAX = 16;   // of the pipelined form alone

typedef unsigned long long u64;

struct Bar {
  unsigned *ctr;                  // 9 counters, TICKET_PAD apart
  int *abort;
  unsigned spin_max;              // polling rounds before a wait gives up
};

// An index the compiler must treat as unknown at this point: keeps it from
// hoisting the 64-bit addresses of every neighbour access out of the
// iteration loop (which would pin two VGPRs per address for the whole
// solve and spill); the address is recomputed where it is used.
__device__ __forceinline__ int opaque(int v) {
  __asm__ volatile("" : "+v"(v));
  return v;
}

// Tagged words: data below, the exchange's number above.
__device__ __forceinline__ void put_word(u64 *p, unsigned tag, unsigned v) {
  __hip_atomic_store(p, (u64)tag << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get_word(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool has_tag(u64 w, unsigned tag) { return (unsigned)(w >> 32) == tag; }
__device__ __forceinline__ void put_f64(u64 *p, unsigned tag, double v) {
  const u64 b = (u64)__double_as_longlong(v);
  put_word(p, tag, (unsigned)b);
  put_word(p + 1, tag, (unsigned)(b >> 32));
}
__device__ __forceinline__ double f64_of(u64 lo, u64 hi) {
  return __longlong_as_double((long long)(hi << 32 | (lo & 0xffffffffull)));
}

// Grid barrier number `gen` (1, 2, ...) with counters, for the few places
// where a plain FP64 array (P) must become visible to every workgroup.
// Returns false if the barrier was abandoned.
__device__ bool grid_barrier(const Bar &b, unsigned gen) {
  __shared__ int s_ok;
  __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have completed
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nb = (int)gridDim.x;
    const int x = blockIdx.x & 7;
    const unsigned nx = (unsigned)((nb >> 3) + (x < (nb & 7) ? 1 : 0));
    const unsigned ng = nb < 8 ? (unsigned)nb : 8u;
    unsigned *gx = b.ctr + x * TICKET_PAD, *gg = b.ctr + 8 * TICKET_PAD;
    if (atomic_inc(gx) == gen * nx - 1u) atomic_inc(gg);
    const unsigned target = gen * ng;
    int ok = 1;
    unsigned spins = 0;
    while (__hip_atomic_load(gg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
      if (++spins > b.spin_max ||
          ((spins & 255u) == 0u &&
           __hip_atomic_load(b.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        __hip_atomic_store(b.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(2);
    }
    s_ok = ok;
  }
  __syncthreads();
  return s_ok != 0;
}

struct Xch {
  u64 *ps;             // partials: [parity][slot][NVMAX][2 words]
  u64 *hx;             // halo slots: [parity][cell], one word (FP32) or two (FP64) each
  int ncell;
  int w0, nb;          // the slots that take part: w0 .. w0+nb-1
};

__device__ __forceinline__ u64 *pslot(const Xch &x, unsigned tag, int slot) {
  return x.ps + ((size_t)(tag & 1u) * PSLOTS + slot) * (2 * NVMAX);
}
__device__ __forceinline__ u64 *hslot32(const Xch &x, unsigned tag) {
  return x.hx + (size_t)(tag & 1u) * x.ncell;
}
__device__ __forceinline__ u64 *hslot64(const Xch &x, unsigned tag) {
  return x.hx + (size_t)(tag & 1u) * x.ncell * 2;
}

// Set by a wave whose wait was abandoned; the workgroup leaves after its
// next barrier.  Cleared before the kernel's first barrier.
__device__ __forceinline__ int &bad() {
  __shared__ int s_bad;
  return s_bad;
}
// One more polling round of a wave: true when it has to give up.
__device__ __forceinline__ bool give_up(const Bar &b, unsigned &spins) {
  ++spins;
  const int ab = (spins & 255u) == 0u
                     ? __builtin_amdgcn_readfirstlane(__hip_atomic_load(
                           b.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                     : 0;
  if (spins > b.spin_max || ab) {
    __hip_atomic_store(b.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bad() = 1;
    return true;
  }
  __builtin_amdgcn_s_sleep(1);
  return false;
}

// Block sum of NV partials into this workgroup's slots of exchange `tag`
// (lane j of wave 0 adds value j in the order of the waves).
template <int NV>
__device__ void post(double (&v)[NV], const Xch &x, unsigned tag) {
  __shared__ double sh[NV][PW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; ++j) v[j] = wave_sum_dpp(v[j]);
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) sh[j][w] = v[j];
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double pv[PW];
#pragma unroll
    for (int q = 0; q < PW; ++q) pv[q] = sh[threadIdx.x][q];
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < PW; ++q) s += pv[q];
    put_f64(pslot(x, tag, (int)blockIdx.x) + 2 * threadIdx.x, tag, s);
  }
}

// Outside cells' words of exchange `tag`, by the calling threads t = 0 ..
// nt-1 (whole waves): cell(h) is entry h's cell, put(h, value) takes its
// value.  Every lane loads (past the list's end, its last cell again) and the
// loads of a batch are in flight together; a vote ends the wave's loop.
// False if the wait was abandoned.
template <int HB, typename CellF, typename PutF>
__device__ __forceinline__ bool halo32(const Xch &x, unsigned tag, int nhalo, int t, int nt,
                                       const Bar &b, CellF cell, PutF put) {
  const u64 *base = hslot32(x, tag);
  const int lane = t & 63;
  for (int h0 = __builtin_amdgcn_readfirstlane(t - lane); h0 < nhalo; h0 += HB * nt) {
    int c[HB];
    u64 v[HB];
#pragma unroll
    for (int u = 0; u < HB; ++u) c[u] = cell(min(h0 + lane + u * nt, nhalo - 1));
    unsigned spins = 0;
    for (;;) {
      bool ready = true;
#pragma unroll
      for (int u = 0; u < HB; ++u) v[u] = get_word(base + (size_t)c[u]);
#pragma unroll
      for (int u = 0; u < HB; ++u) ready = ready && has_tag(v[u], tag);
      if (__all(ready)) break;
      if (give_up(b, spins)) return false;
    }
#pragma unroll
    for (int u = 0; u < HB; ++u)
      if (h0 + lane + u * nt < nhalo) put(h0 + lane + u * nt, __uint_as_float((unsigned)v[u]));
  }
  return true;
}
template <int HB, typename CellF, typename PutF>
__device__ __forceinline__ bool halo64(const Xch &x, unsigned tag, int nhalo, int t, int nt,
                                       const Bar &b, CellF cell, PutF put) {
  const u64 *base = hslot64(x, tag);
  const int lane = t & 63;
  for (int h0 = __builtin_amdgcn_readfirstlane(t - lane); h0 < nhalo; h0 += HB * nt) {
    int c[HB];
    u64 lo[HB], hi[HB];
#pragma unroll
    for (int u = 0; u < HB; ++u) c[u] = cell(min(h0 + lane + u * nt, nhalo - 1));
    unsigned spins = 0;
    for (;;) {
      bool ready = true;
#pragma unroll
      for (int u = 0; u < HB; ++u) {
        lo[u] = get_word(base + 2 * (size_t)c[u]);
        hi[u] = get_word(base + 2 * (size_t)c[u] + 1);
      }
#pragma unroll
      for (int u = 0; u < HB; ++u) ready = ready && has_tag(lo[u], tag) && has_tag(hi[u], tag);
      if (__all(ready)) break;
      if (give_up(b, spins)) return false;
    }
#pragma unroll
    for (int u = 0; u < HB; ++u)
      if (h0 + lane + u * nt < nhalo) put(h0 + lane + u * nt, f64_of(lo[u], hi[u]));
  }
  return true;
}

// The sums of exchange `tag`: wave 0 polls the partials of every workgroup
// (lane l those of workgroups l, l+64, ..., UG at a time) and adds them in
// that order, then a DPP wave sum; the other waves meanwhile run halo(t, nt)
// as threads t = 0 .. nt-1.  Returns the sums (same bits in every workgroup)
// after one workgroup barrier, or false if a wait was abandoned.
template <int NV, int UG, typename HaloF>
__device__ __forceinline__ bool exchange(const Xch &x, unsigned tag, const Bar &b,
                                         double (&sum)[NV], HaloF halo) {
  __shared__ double shs[NV];
  const int t = threadIdx.x, lane = t & 63;
  const int nb = x.nb;
  if (t < 64) {
    double v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = 0.0;
    bool ok = true;
    for (int u0 = 0; 64 * u0 < nb && ok; u0 += UG) {
      u64 lo[UG][NV], hi[UG][NV];
      unsigned spins = 0;
      for (;;) {
        // the lane number made opaque: the addresses are formed here, not
        // held in registers across the caller's loops
        const int ln = opaque(lane);
        bool ready = true;
#pragma unroll
        for (int u = 0; u < UG; ++u) {
          const u64 *q = pslot(x, tag, x.w0 + min(ln + 64 * (u0 + u), nb - 1));  // every lane loads
#pragma unroll
          for (int j = 0; j < NV; ++j) {
            lo[u][j] = get_word(q + 2 * j);
            hi[u][j] = get_word(q + 2 * j + 1);
          }
        }
#pragma unroll
        for (int u = 0; u < UG; ++u)
#pragma unroll
          for (int j = 0; j < NV; ++j)
            ready = ready && has_tag(lo[u][j], tag) && has_tag(hi[u][j], tag);
        if (__all(ready)) break;
        if (give_up(b, spins)) { ok = false; break; }
      }
#pragma unroll
      for (int u = 0; u < UG; ++u)
#pragma unroll
        for (int j = 0; j < NV; ++j)
          v[j] += lane + 64 * (u0 + u) < nb ? f64_of(lo[u][j], hi[u][j]) : 0.0;
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = wave_sum_dpp(v[j]);
    if (lane == 0) {
#pragma unroll
      for (int j = 0; j < NV; ++j) shs[j] = v[j];
    }
  } else {
    halo(t - 64, PB - 64);
  }
  // shs is written again only after every wave has passed the next post()
  __syncthreads();
  if (bad()) return false;
#pragma unroll
  for (int j = 0; j < NV; ++j) sum[j] = shs[j];
  return true;
}
struct NoHalo {
  __device__ void operator()(int, int) const {}
};

// The same sums with nothing to fetch beside them and a large state in
// registers: wave g < 4 polls the partials of workgroups 64 g .. 64 g + 63
// (and 256 further on), one group of words in its registers.  Four in wave 0,
// as exchange holds them, are registers that every wave is allotted (FP64
// pipelined solve, 6 cells per thread: 106 spilled).
template <int NV>
__device__ __forceinline__ bool exchange_waves(const Xch &x, unsigned tag, const Bar &b,
                                               double (&sum)[NV]) {
  constexpr int G = 4;
  __shared__ double shw[G][NV];
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (g < G) {
    double v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = 0.0;
    bool ok = true;
    for (int q0 = 64 * g; q0 < x.nb && ok; q0 += 64 * G) {
      u64 lo[NV], hi[NV];
      unsigned spins = 0;
      for (;;) {
        const int ln = opaque(lane);  // as in exchange
        const u64 *q = pslot(x, tag, x.w0 + min(q0 + ln, x.nb - 1));  // every lane loads
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          lo[j] = get_word(q + 2 * j);
          hi[j] = get_word(q + 2 * j + 1);
        }
        bool ready = true;
#pragma unroll
        for (int j = 0; j < NV; ++j) ready = ready && has_tag(lo[j], tag) && has_tag(hi[j], tag);
        if (__all(ready)) break;
        if (give_up(b, spins)) { ok = false; break; }
      }
#pragma unroll
      for (int j = 0; j < NV; ++j) v[j] += q0 + lane < x.nb ? f64_of(lo[j], hi[j]) : 0.0;
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = wave_sum_dpp(v[j]);
    if (lane == 0) {
#pragma unroll
      for (int j = 0; j < NV; ++j) shw[g][j] = v[j];
    }
  }
  // shw is written again only after every wave has passed the next post()
  __syncthreads();
  if (bad()) return false;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < G; ++q) s += shw[q][j];
    sum[j] = s;
  }
  return true;
}

// ---- sums of a basin, in the order of the per-basin launches (k_scg_*):
// 512-cell tiles from the basin's first cell, 256 threads of two cells each;
// waves, then the four waves of a tile, then the tiles as sum_parts adds them.

// wave_sum's tree for M values of each lane together, without LDS: the lanes
// 32 apart by exchanging register halves, where a pair of values shares the
// halves from then on, those 16 apart by exchanging rows, where two pairs share
// the rows; after that a row's values repeat every 8 lanes, then every 4, so a
// rotation within the row brings the partner's.  r[i] holds value 4 i + (0, 2,
// 1, 3) in the rows 0 to 3 (M <= 2: value 0 in rows 0 and 1, value 1 in 2 and 3).
__device__ __forceinline__ double fold32(double x, double y) {
  const u64 a = (u64)__double_as_longlong(x), b = (u64)__double_as_longlong(y);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
  const auto hi =
      __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
  return f64_of(lo[0], hi[0]) + f64_of(lo[1], hi[1]);
}
__device__ __forceinline__ double fold16(double x, double y) {
  const u64 a = (u64)__double_as_longlong(x), b = (u64)__double_as_longlong(y);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
  const auto hi =
      __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
  return f64_of(lo[0], hi[0]) + f64_of(lo[1], hi[1]);
}
template <int M>
__device__ __forceinline__ void wave_sums_tree(const double (&v)[M], double (&r)[(M + 3) / 4]) {
  constexpr int P = (M + 1) / 2;
  double w[P];
#pragma unroll
  for (int i = 0; i < P; ++i) w[i] = fold32(v[2 * i], v[2 * i + 1 < M ? 2 * i + 1 : 2 * i]);
#pragma unroll
  for (int i = 0; i < (M + 3) / 4; ++i) {
    double s = fold16(w[2 * i], w[2 * i + 1 < P ? 2 * i + 1 : 2 * i]);
    s += dpp_move<0x128, 0xf>(s);  // row_ror:8
    s += dpp_move<0x124, 0xf>(s);  // row_ror:4
    s += dpp_move<0x4e, 0xf>(s);   // quad_perm [2,3,0,1]
    s += dpp_move<0xb1, 0xf>(s);   // quad_perm [1,0,3,2]
    r[i] = s;
  }
}

// The partials of this workgroup's tiles (v[m]: tile 2 m + half, half 1 the
// upper four waves) into their slots; ntile of them exist.
template <int NV, int NT>
__device__ __forceinline__ void post_tiles(double (&v)[NT][NV], const Xch &x, unsigned tag,
                                           int ntile) {
  constexpr int M = NT * NV, R = (M + 3) / 4;
  __shared__ double sh[4 * R][PW];  // value m NV + j of every wave
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double u[M], r[R];
#pragma unroll
  for (int q = 0; q < M; ++q) u[q] = v[q / NV][q % NV];
  wave_sums_tree<M>(u, r);
  if ((lane & 15) == 0) {
    const int row = lane >> 4, q = M <= 2 ? row >> 1 : (row & 1) * 2 + (row >> 1);
#pragma unroll
    for (int i = 0; i < R; ++i) sh[4 * i + q][w] = r[i];
  }
  __syncthreads();
  if (threadIdx.x < 2 * NT * NV) {
    const int tile = (int)threadIdx.x / NV, j = (int)threadIdx.x % NV;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < PW / 2; ++q) s += sh[(tile >> 1) * NV + j][(tile & 1) * (PW / 2) + q];
    if (tile < ntile)
      put_f64(pslot(x, tag, (int)blockIdx.x * 2 * NT + tile) + 2 * j, tag, s);
  }
}

// exchange over the tiles of a basin in sum_parts' order: thread t of 256
// adds tiles t, t + 256, .., then its tree.  As many of the first four waves as the
// tiles need poll (wave 0 alone up to 64 tiles); the others run halo(t, nt).
template <int NV, typename HaloF>
__device__ __forceinline__ bool exchange_tiles(const Xch &x, unsigned tag, const Bar &b,
                                               double (&sum)[NV], HaloF halo) {
  constexpr int W = EFDC_BLOCK / 64;  // sum_parts' waves
  static_assert(NV <= 2, "value j of the sums lies in the rows 2 j and 2 j + 1");
  __shared__ double shs[W][2];
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int nw = min(W, (x.nb + 63) >> 6);
  if (g < nw) {
    double v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = 0.0;
    bool ok = true;
    for (int h0 = 64 * g; h0 < x.nb && ok; h0 += 64 * W) {
      u64 lo[NV], hi[NV];
      unsigned spins = 0;
      for (;;) {
        const int ln = opaque(lane);  // as in exchange
        const u64 *p = pslot(x, tag, x.w0 + min(h0 + ln, x.nb - 1));  // every lane loads
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          lo[j] = get_word(p + 2 * j);
          hi[j] = get_word(p + 2 * j + 1);
        }
        bool ready = true;
#pragma unroll
        for (int j = 0; j < NV; ++j)
          ready = ready && has_tag(lo[j], tag) && has_tag(hi[j], tag);
        if (__all(ready)) break;
        if (give_up(b, spins)) { ok = false; break; }
      }
#pragma unroll
      for (int j = 0; j < NV; ++j) v[j] += h0 + lane < x.nb ? f64_of(lo[j], hi[j]) : 0.0;
    }
    double r[1];
    wave_sums_tree<NV>(v, r);
    if ((lane & 31) == 0) shs[g][lane >> 5] = r[0];
  } else {
    halo((int)threadIdx.x - 64 * nw, PB - 64 * nw);
  }
  // shs is written again only after every wave has passed the next post_tiles()
  __syncthreads();
  if (bad()) return false;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    double s = 0.0;
    for (int q = 0; q < nw; ++q) s += shs[q][j];
    sum[j] = s;
  }
  return true;
}

// neighbour slots of a row
enum { NS = 0, NN = 1, NW = 2, NE = 3 };


// Compact list of the outside cells a workgroup's rows reference (sorted
// by index).  `mark` holds 2*WIN flags on entry (slot g: cell b0-WIN+g for
// g < WIN, cell b1+g-WIN above) and the list on return; returns its length.
__device__ int compact_halo(int *mark, int b0, int b1) {
  __shared__ int wtot[PW];
  __shared__ int total;
  constexpr int PER = 2 * WIN / PB;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int f[PER];
  int cnt = 0;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    f[u] = mark[t * PER + u];
    cnt += f[u] ? 1 : 0;
  }
  int inc = cnt;  // inclusive scan over the workgroup
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(inc, off, 64);
    if (lane >= off) inc += v;
  }
  if (lane == 63) wtot[w] = inc;
  __syncthreads();
  int base = 0;
  for (int q = 0; q < w; ++q) base += wtot[q];
  if (t == PB - 1) total = base + inc;
  int pos = base + inc - cnt;
  __syncthreads();   // every flag has been read
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if (f[u]) {
      const int g = t * PER + u;
      mark[pos++] = g < WIN ? b0 - WIN + g : b1 + (g - WIN);
    }
  }
  __syncthreads();
  return total;
}

__device__ __forceinline__ int ghost_of(int j, int b0, int b1) {
  return j < b0 ? WIN - (b0 - j) : WIN + (j - b1);
}

// ---------------------------------------------------------------------
// FP64 Jacobi-PCG (EFDC/congrad.f90)
// ---------------------------------------------------------------------
struct P64Args {
  const double *ccc, *ccs, *ccw, *ccn, *cce, *ccci, *fptmp;
  double *x;                 // P, in/out
  const int *lw, *le, *ls, *ln;
  int nwet, lc0, rowmajor, mutual;
  Xch xc;
  unsigned tag0;
  Bar bar;
  CgState *st;
  double rsqm, rel_tol;
  int iterm;
  // basins: {first cell, end of the basin, first workgroup, tiles} and the
  // basin of every workgroup, the basins' states, a copy of x
  const int4 *wg;
  const int *wgseg;
  CgState *segst;
  double *xsave;
};

// SEG: every basin of an ensemble is a solve of its own, by the workgroups of
// its cells: sums, stop test and iteration count are the basin's, and a basin
// that has stopped frees its workgroups while the others go on.  Its sums are
// taken over the tiles and in the order of the per-basin launches, so a
// basin's bits are those of the basin alone with those launches, whatever
// basins share the context and however many cells a thread has: a half of
// the workgroup owns a tile, a thread two cells of it 256 apart (CPT is even).
// Against two launches over all basins per iteration, whose vectors go through
// memory (40 basins of 16000 cells, FP64, 15 iterations): 4 steps 3460 -> 1960 us.
template <int CPT, bool SEG>
__global__ __launch_bounds__(PB) void k_pcg64(P64Args a) {
  // the window, then one word that stays zero (read in place of a
  // neighbour that is not a cell, so that every lane loads)
  __shared__ double lds[2 * WIN + CPT * PB + 1];
  __shared__ int hl[2 * WIN];
  __shared__ double zh[HMAX];  // z of the outside cells
  constexpr int ZS = 2 * WIN + CPT * PB;
  // Groups of 64 slots in flight.  Below the most cells per thread there are at
  // most PCG64_NB workgroups, one group: the second one's loads repeat its last
  // slot, and without them a solve is no faster (us, 2 : 1; 21 k cells 73.8 :
  // 75.0, 79 k 86.7 : 87.9, 276 k 117.7 : 118.5).
  constexpr int UG = CPT < PCG64_CPT_MAX ? 2 : 4;
  static_assert(!SEG || CPT % 2 == 0, "a tile is two cells a thread of half a workgroup");
  constexpr int NT = SEG ? CPT / 2 : 1;
  int b0 = 1 + (int)blockIdx.x * CPT * PB, b1 = min(b0 + CPT * PB, a.nwet + 1);
  Xch xc = a.xc;
  // the cells of this solve: in the row-major form the first cell of a basin
  // has the last one of the basin before it for i-1, uncoupled
  int c0 = 1, c1 = a.lc0;
  if (SEG) {
    const int4 q = a.wg[blockIdx.x];
    b0 = q.x;
    b1 = min(b0 + CPT * PB, q.y);
    c0 = a.wg[q.z].x;
    c1 = q.y;
    xc.w0 = q.z * CPT;
    xc.nb = q.w;
  }
  const int ntile = (b1 - b0 + PB - 1) / PB;
  // the cell of row k
  auto cell = [&](int k) {
    const int t = (int)threadIdx.x;
    return SEG ? b0 + ((k & ~1) + (t >> 8)) * PB + (k & 1) * (PB / 2) + (t & (PB / 2 - 1))
               : b0 + k * PB + t;
  };
  const bool fast = a.rowmajor && (a.st->symok == 0);
  const int lc0 = a.lc0;

  double ccc[CPT], cs[CPT], cn[CPT], cw[CPT], ce[CPT], cci[CPT];
  double x[CPT], r[CPT], p[CPT], ap[CPT];
  int nb[CPT][4];
  unsigned expo = 0u;        // bit k: another workgroup reads cell k

  auto inside = [&](int j) { return j >= b0 && j < b1; };
  auto real = [&](int j) { return j >= c0 && j < c1; };
  auto slot = [&](int j) { return j - b0 + WIN; };
  auto publish_z = [&](int i, unsigned tag, double z) {
    put_f64(hslot64(xc, tag) + 2 * (size_t)opaque(i), tag, z);
  };

  for (int g = threadIdx.x; g < 2 * WIN; g += PB) hl[g] = 0;
  if (threadIdx.x == 0) { lds[ZS] = 0.0; bad() = 0; }
  __syncthreads();
  // partials: the thread's, or (SEG) those of its cells in each of its tiles
  double v2[NT][2] = {};
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = cell(k);
    x[k] = r[k] = p[k] = ap[k] = 0.0;
    ccc[k] = 1.0; cs[k] = cn[k] = cw[k] = ce[k] = cci[k] = 0.0;
    nb[k][NS] = nb[k][NN] = nb[k][NW] = nb[k][NE] = lc0;
    if (i < b1) {
      // the row as in the multi-kernel solve (row_of)
      const int js = a.ls[i], jn = a.ln[i];
      int jw, je;
      double s_ = a.ccs[i], w_ = a.ccw[i], n_, e_;
      if (fast) {
        jw = i - 1;
        je = i + 1;
        n_ = (jn != lc0) ? a.ccs[jn] : 0.0;
        e_ = (je != lc0) ? a.ccw[je] : 0.0;
      } else {
        jw = a.lw[i];
        je = a.le[i];
        n_ = (jn != lc0) ? a.ccn[i] : 0.0;
        e_ = (je != lc0) ? a.cce[i] : 0.0;
        if (jw == lc0) w_ = 0.0;
      }
      if (js == lc0) s_ = 0.0;
      nb[k][NS] = js; nb[k][NN] = jn; nb[k][NW] = jw; nb[k][NE] = je;
      ccc[k] = a.ccc[i]; cs[k] = s_; cn[k] = n_; cw[k] = w_; ce[k] = e_;
      cci[k] = a.ccci[i];
      bool out = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = nb[k][q];
        if (real(j) && !inside(j)) {
          out = true;
          hl[ghost_of(j, b0, b1)] = 1;
        }
      }
      if (out || !a.mutual) expo |= 1u << k;
      const double *P = a.x;
      x[k] = P[i];
      if (SEG) a.xsave[i] = x[k];
      // RCG = FPTMP - CCC*P - CCN*PN - CCS*PS - CCW*PW - CCE*PE (:73)
      const double rr = a.fptmp[i] - ccc[k] * x[k] - n_ * P[jn] - s_ * P[js] -
                        w_ * P[jw] - e_ * P[je];
      r[k] = rr;
      v2[SEG ? k >> 1 : 0][0] += rr * (rr * cci[k]);   // RPCG = sum RCG*PCG (:80-85)
      v2[SEG ? k >> 1 : 0][1] += a.fptmp[i] * a.fptmp[i];
    }
  }
  __syncthreads();
  const int nhalo = compact_halo(hl, b0, b1);

  // the window keeps p of the outside cells, formed here by their owner's
  // operations from their published z = CCCI*r
  for (int h = threadIdx.x; h < nhalo; h += PB) lds[slot(hl[h])] = 0.0;

  unsigned tag = a.tag0;
  auto halo = [&](int t, int nt) {
    halo64<2>(xc, tag, nhalo, t, nt, a.bar, [&](int h) { return hl[h]; },
              [&](int h, double z) { zh[h] = z; });
  };
  // exchange: z of the outside cells (the owner forms it, so they load no
  // CCCI of an outside cell), RPCG and |FPTMP|^2
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    if (expo & (1u << k)) publish_z(cell(k), tag, cci[k] * r[k]);
  double s2[2];
  if constexpr (SEG) {
    post_tiles<2, NT>(v2, xc, tag, ntile);
    if (!exchange_tiles<2>(xc, tag, a.bar, s2, halo)) return;
  } else {
    post<2>(v2[0], xc, tag);
    if (!exchange<2, UG>(xc, tag, a.bar, s2, halo)) return;
  }
  double rpcg = s2[0];
  const double bnorm2 = s2[1];
  const double rsqm = a.rel_tol > 0.0 ? a.rel_tol * a.rel_tol * bnorm2 : a.rsqm;
  double beta = 0.0, alpha = 0.0, rsq = 0.0, papcg = 0.0;
  int iter = 0, status = 0;
  bool done = (rpcg == 0.0);  // :88

  while (!done) {
    // p = CCCI*r + beta*p (:134,158) on the own rows ...  (no branch per
    // row: the lanes past b1, the last workgroup's, hold zero vectors and
    // zero couplings to lc0, so their rows stay zero; their slots are read
    // by no row)
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      p[k] = cci[k] * r[k] + beta * p[k];
      lds[slot(cell(k))] = p[k];
    }
    // ... and on the outside cells
    for (int h = threadIdx.x; h < nhalo; h += PB) {
      double &pj = lds[slot(hl[h])];
      pj = zh[h] + beta * pj;
    }
    __syncthreads();
    double v1[NT][1] = {};
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      double pq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = nb[k][q];
        pq[q] = lds[real(j) ? slot(j) : ZS];
      }
      // APCG = CCC*PCG + CCS*PS + CCN*PN + CCW*PW + CCE*PE (:113)
      ap[k] = ccc[k] * p[k] + cs[k] * pq[NS] + cn[k] * pq[NN] + cw[k] * pq[NW] +
              ce[k] * pq[NE];
      v1[SEG ? k >> 1 : 0][0] += ap[k] * p[k];
    }
    ++tag;
    double s1[1];
    if constexpr (SEG) {
      post_tiles<1, NT>(v1, xc, tag, ntile);
      if (!exchange_tiles<1>(xc, tag, a.bar, s1, NoHalo())) return;
    } else {
      post<1>(v1[0], xc, tag);
      if (!exchange<1, UG>(xc, tag, a.bar, s1, NoHalo())) return;
    }
    papcg = s1[0];
    alpha = rpcg / papcg;  // :124
    double v[NT][2] = {};
    ++tag;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = cell(k);
      x[k] = x[k] + alpha * p[k];        // :132
      const double rr = r[k] - alpha * ap[k];  // :133
      r[k] = rr;
      const double z = cci[k] * rr;      // :134
      v[SEG ? k >> 1 : 0][0] += rr * z;
      v[SEG ? k >> 1 : 0][1] += rr * rr;
      if (expo & (1u << k)) publish_z(i, tag, z);
    }
    if constexpr (SEG) {
      post_tiles<2, NT>(v, xc, tag, ntile);
      if (!exchange_tiles<2>(xc, tag, a.bar, s2, halo)) return;
    } else {
      post<2>(v[0], xc, tag);
      if (!exchange<2, UG>(xc, tag, a.bar, s2, halo)) return;
    }
    beta = s2[0] / rpcg;  // :147-148
    rpcg = s2[0];
    rsq = s2[1];
    iter += 1;
    if (rsq <= rsqm) done = true;  // :165
    else if (iter >= a.iterm) { done = true; status = 1; }
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = cell(k);
    if (i < b1) a.x[opaque(i)] = x[k];
  }
  if ((SEG ? (int)blockIdx.x * CPT == xc.w0 : blockIdx.x == 0) && threadIdx.x == 0) {
    CgState *st = SEG ? a.segst + a.wgseg[blockIdx.x] : a.st;
    st->rpcg = rpcg;
    st->papcg = papcg;
    st->alpha = alpha;
    st->beta = beta;
    st->rsq = rsq;
    st->rsqm = rsqm;
    st->bnorm2 = bnorm2;
    st->iter = iter;
    st->done = 1;
    st->status = status;
  }
}

// ---------------------------------------------------------------------
// Mixed: FP32 Chronopoulos-Gear CG on A' = D^-1/2 A D^-1/2, FP64
// refinement (same operator and scaling as the multi-kernel mixed solve)
// ---------------------------------------------------------------------
struct PMxArgs {
  const double *ccc, *ccs, *ccw, *fptmp;
  const double *dis;         // 1/sqrt(CCC)
  const float *as, *aw;      // A'(i,S), A'(i,W) in FP32
  double *x;                 // P, in/out
  const int *ls, *ln;
  int nwet, lc0;
  Xch xc;
  unsigned tag0;
  Bar bar;
  CgState *st;
  double rsqm, rel_tol, rtol2;
  int iterm, max_outer;
  int pdeg;                  // terms of the workgroup-local Neumann preconditioner
};

template <int CPT>
__global__ __launch_bounds__(PB) void k_pcgmx(PMxArgs a) {
  // the window, then one word that stays zero: a row reads it in place of
  // a neighbour it does not couple to, so that every lane loads
  __shared__ float lds[2 * WIN + CPT * PB + 1];
  __shared__ int hl[2 * WIN];
  __shared__ float zh[HMAX], qh[HMAX];  // u or z, and q, of the outside cells
  constexpr int ZS = 2 * WIN + CPT * PB;
  // y (the inner solution) and z = M^-1 w of the own rows live in LDS:
  // with them in registers the 6..8-cells-per-thread shapes would spill
  __shared__ float lys[CPT * PB], lzs[CPT * PB];
  const int b0 = 1 + (int)blockIdx.x * CPT * PB;
  const int b1 = min(b0 + CPT * PB, a.nwet + 1);
  const int lc0 = a.lc0;

  float as_[CPT], an_[CPT], aw_[CPT], ae_[CPT];
  float r[CPT], w[CPT], s[CPT], p[CPT];
  float u[CPT], q[CPT];  // M^-1 r, M^-1 s
  auto Y = [&](int k) -> float & { return lys[k * PB + threadIdx.x]; };
  auto Z = [&](int k) -> float & { return lzs[k * PB + threadIdx.x]; };
  int js[CPT], jn[CPT];
  unsigned expo = 0u;

  auto inside = [&](int j) { return j >= b0 && j < b1; };
  auto real = [&](int j) { return j > 0 && j < lc0; };
  auto slot = [&](int j) { return j - b0 + WIN; };
  auto rval = [&](int j) { return lds[real(j) ? slot(j) : ZS]; };
  auto publish_w = [&](int i, unsigned tag, float v) {
    put_word(hslot32(a.xc, tag) + (size_t)opaque(i), tag, __float_as_uint(v));
  };

  // M^-1 v: the first pdeg terms of the Neumann series of A' restricted to
  // the workgroup's own cells, sum_j N^j v with N = I - A' (couplings to
  // cells of other workgroups dropped), by Horner's rule t <- v + N t.  M^-1
  // is a polynomial in the symmetric local block whose eigenvalues lie in
  // (-1, 1), so it is symmetric positive definite and CG stays CG; it needs
  // no exchange between workgroups.  The own slots of the LDS window carry t.
  // No branch per row: the lanes past b1 (the last workgroup's) hold zero
  // coefficients and zero vectors, so their rows stay zero, and their
  // slots, which no row reads, hold those zeros.
  auto precond = [&](const float (&v)[CPT], float (&t)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) t[k] = v[k];
    for (int d = 1; d < a.pdeg; ++d) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < CPT; ++k) lds[slot(b0 + k * PB + (int)threadIdx.x)] = t[k];
      __syncthreads();
      float tn[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        // indices made opaque: the slot addresses are formed at each use
        // rather than held in registers across the whole solve
        const int i = opaque(b0 + k * PB + (int)threadIdx.x);
        const int jsk = opaque(js[k]), jnk = opaque(jn[k]);
        const float ts = lds[inside(jsk) ? slot(jsk) : ZS];
        const float tnn = lds[inside(jnk) ? slot(jnk) : ZS];
        const float tw = lds[i - 1 >= b0 ? slot(i - 1) : ZS];
        const float te = lds[i + 1 < b1 ? slot(i + 1) : ZS];
        tn[k] = v[k] - (as_[k] * ts + an_[k] * tnn + aw_[k] * tw + ae_[k] * te);
      }
#pragma unroll
      for (int k = 0; k < CPT; ++k) t[k] = tn[k];
    }
    __syncthreads();  // every read of the own slots is done
  };

  for (int g = threadIdx.x; g < 2 * WIN; g += PB) hl[g] = 0;
  if (threadIdx.x == 0) { lds[ZS] = 0.0f; bad() = 0; }
  __syncthreads();
  double fp2 = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = b0 + k * PB + (int)threadIdx.x;
    as_[k] = an_[k] = aw_[k] = ae_[k] = 0.0f;
    r[k] = w[k] = s[k] = p[k] = 0.0f;
    u[k] = q[k] = 0.0f;
    Y(k) = 0.0f;
    Z(k) = 0.0f;
    js[k] = jn[k] = lc0;
    if (i < b1) {
      const int s_ = a.ls[i], n_ = a.ln[i];
      js[k] = s_;
      jn[k] = n_;
      // A'(i,S) = CCS(i) d(i) d(S), A'(i,W) = CCW(i) d(i) d(i-1), formed
      // once per solve by the scaling pass; the north and east entries are
      // the south / west entries of the neighbour
      as_[k] = a.as[i];
      aw_[k] = a.aw[i];
      if (n_ != lc0) an_[k] = a.as[n_];
      if (i + 1 != lc0) ae_[k] = a.aw[i + 1];
      const int nbq[4] = {s_, n_, i - 1, i + 1};
      bool out = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = nbq[q];
        if (real(j) && !inside(j)) {
          out = true;
          hl[ghost_of(j, b0, b1)] = 1;
        }
      }
      if (out) expo |= 1u << k;
      fp2 += a.fptmp[i] * a.fptmp[i];
    }
  }
  __syncthreads();
  const int nhalo = compact_halo(hl, b0, b1);

  unsigned tag = a.tag0, gen = 0;
  auto halo = [&](int t, int nt) {
    halo32<4>(a.xc, tag, nhalo, t, nt, a.bar, [&](int h) { return hl[h]; },
              [&](int h, float v) { zh[h] = v; });
  };
  double rsqm = a.rsqm, bnorm2 = 0.0, rsq64 = 0.0, bn_in = 0.0;
  int total = 0, outer = 0, status = 0, inner = 0;

  for (;;) {
    // ---- FP64 residual r = FPTMP - A P, scaled to r' = D^-1/2 r (FP32)
    double v3[3] = {0.0, 0.0, fp2};
    // every lane loads (a lane past b1 from the last own cell; its js, jn
    // are lc0) and the own rows are selected
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const bool own = i < b1;
      const int s_ = opaque(js[k]), n_ = opaque(jn[k]);
      const int io = opaque(own ? i : b1 - 1);
      const int ie = io + 1;  // <= lc0
      const double *P = a.x;
      const double ccs_i = a.ccs[io], ccs_n = a.ccs[n_], ccw_i = a.ccw[io];
      const double ccw_e = a.ccw[ie], fpt = a.fptmp[io], cci = a.ccc[io], di = a.dis[io];
      const double p_i = fetch(&P[io]), p_n = fetch(&P[n_]), p_s = fetch(&P[s_]);
      const double p_w = fetch(&P[io - 1]), p_e = fetch(&P[ie]);
      const double cs = (s_ != lc0) ? ccs_i : 0.0;
      const double cn = (n_ != lc0) ? ccs_n : 0.0;
      const double cw = ccw_i;
      const double ce = (ie != lc0) ? ccw_e : 0.0;
      const double rr = fpt - cci * p_i - cn * p_n - cs * p_s - cw * p_w - ce * p_e;
      const float rs = (float)(di * rr);
      r[k] = own ? rs : 0.0f;
      Y(k) = 0.0f;
      v3[0] += own ? rr * rr : 0.0;
      v3[1] += own ? (double)rs * (double)rs : 0.0;
    }
    // the partials go out while the preconditioner runs
    post<3>(v3, a.xc, tag);
    // u0 = M^-1 r0, exported for the neighbours' A u0
    precond(r, u);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      lds[slot(i)] = u[k];
      if (expo & (1u << k)) publish_w(i, tag, u[k]);
    }
    fp2 = 0.0;
    {
      double s3[3];
      if (!exchange<3, 4>(a.xc, tag, a.bar, s3, halo)) return;
      if (outer == 0) {
        bnorm2 = s3[2];
        rsqm = a.rel_tol > 0.0 ? a.rel_tol * a.rel_tol * bnorm2 : a.rsqm;
      }
      rsq64 = s3[0];
      bn_in = s3[1];
    }
    if (rsq64 <= rsqm) break;
    if (outer >= a.max_outer || bn_in == 0.0) { status = 1; break; }
    const double rt2 = fmax(a.rtol2, INNER_MARGIN2 * rsqm / rsq64);

    // ---- w0 = A' u0, z0 = M^-1 w0; gamma0 = (r,u), delta0 = (w,u),
    // rho0 = (r,r); s_-1 = p_-1 = q_-1 = 0.  From here on the window holds u
    // of the outside cells and qh their q, formed by their owner's operations
    // from their published z.
    for (int h = threadIdx.x; h < nhalo; h += PB) {
      lds[slot(hl[h])] = zh[h];
      qh[h] = 0.0f;
    }
    __syncthreads();
    ++tag;
    double v2[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      s[k] = 0.0f;
      p[k] = 0.0f;
      q[k] = 0.0f;
      // a lane past b1 may read a slot no one wrote: its row is zero
      const float wk = u[k] + as_[k] * rval(js[k]) + an_[k] * rval(jn[k]) +
                       aw_[k] * rval(i - 1) + ae_[k] * rval(i + 1);
      w[k] = i < b1 ? wk : 0.0f;
      v2[0] += (double)r[k] * (double)u[k];
      v2[1] += (double)w[k] * (double)u[k];
      v2[2] += (double)r[k] * (double)r[k];
    }
    post<3>(v2, a.xc, tag);
    {
      float zt[CPT];
      precond(w, zt);
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int i = b0 + k * PB + (int)threadIdx.x;
        Z(k) = zt[k];
        if (expo & (1u << k)) publish_w(i, tag, zt[k]);
      }
    }
    double gam, del;
    {
      double s3[3];
      if (!exchange<3, 4>(a.xc, tag, a.bar, s3, halo)) return;
      gam = s3[0];
      del = s3[1];
    }
    double gam_prev = 0.0, alpha_prev = 1.0;
    inner = 0;
    for (;;) {
      double beta, alpha;
      if (inner == 0) {
        beta = 0.0;
        alpha = gam / del;
      } else {
        beta = gam / gam_prev;
        alpha = gam / (del - beta * gam / alpha_prev);
      }
      // own rows: p = u + beta p, s = w + beta s, q = z + beta q,
      // y += alpha p, r -= alpha s, u -= alpha q
      // the vector updates in FP32 (one rounding each, fused multiply-add),
      // the same operations as a neighbour's recomputation below
      const float bf = (float)beta, af = (float)alpha;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int i = b0 + k * PB + (int)threadIdx.x;
        p[k] = fmaf(bf, p[k], u[k]);
        s[k] = fmaf(bf, s[k], w[k]);
        q[k] = fmaf(bf, q[k], Z(k));
        Y(k) = fmaf(af, p[k], Y(k));
        r[k] = fmaf(-af, s[k], r[k]);
        u[k] = fmaf(-af, q[k], u[k]);
        lds[slot(i)] = u[k];
      }
      // the outside cells' u
      for (int h = threadIdx.x; h < nhalo; h += PB) {
        const float qj = fmaf(bf, qh[h], zh[h]);
        qh[h] = qj;
        float &uj = lds[slot(hl[h])];
        uj = fmaf(-af, qj, uj);
      }
      __syncthreads();
      ++tag;
      double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int i = b0 + k * PB + (int)threadIdx.x;
        const float wk = u[k] + as_[k] * rval(js[k]) + an_[k] * rval(jn[k]) +
                         aw_[k] * rval(i - 1) + ae_[k] * rval(i + 1);
        w[k] = i < b1 ? wk : 0.0f;
        v[0] += (double)r[k] * (double)u[k];
        v[1] += (double)w[k] * (double)u[k];
        v[2] += (double)r[k] * (double)r[k];
      }
      post<3>(v, a.xc, tag);
      {
        float zt[CPT];
        precond(w, zt);
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          const int i = b0 + k * PB + (int)threadIdx.x;
          Z(k) = zt[k];
          if (expo & (1u << k)) publish_w(i, tag, zt[k]);
        }
      }
      double s3[3];
      if (!exchange<3, 4>(a.xc, tag, a.bar, s3, halo)) return;
      inner += 1;
      gam_prev = gam;
      alpha_prev = alpha;
      gam = s3[0];
      del = s3[1];
      if (s3[2] <= rt2 * bn_in || inner >= a.iterm) break;
    }
    total += inner;
    ++tag;
    // ---- P += D^-1/2 y (FP64), visible to every workgroup for the
    // next residual
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const bool own = i < b1;
      const int io = opaque(own ? i : b1 - 1);  // every lane loads
      double *P = a.x;
      const double pn = fetch(&P[io]) + a.dis[io] * (double)Y(k);
      if (own) publish(&P[io], pn);
    }
    ++outer;
    if (!grid_barrier(a.bar, ++gen)) return;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    CgState *st = a.st;
    st->rsq64 = rsq64;
    st->rsq = rsq64;
    st->rsqm = rsqm;
    st->bnorm2 = bnorm2;
    st->bnorm2_in = bn_in;
    st->iter = total;
    st->inner_iter = inner;
    st->outer = outer;
    st->done = 1;
    st->status = status;
  }
}

// ---------------------------------------------------------------------
// Mixed, pipelined: the same FP32 inner solve in the pipelined form of the
// preconditioned Chronopoulos-Gear CG (Ghysels and Vanroose, 2014): each
// iteration posts the partial sums of (r,u), (w,u), (r,r) and one halo word
// (m = M^-1 w), waits only for the workgroups that own its outside cells,
// forms n = A' m, and then waits for the sums of every workgroup -- which
// were posted one SpMV earlier -- to take alpha and beta:
//   z = n + beta z, q = m + beta q, s = w + beta s, p = u + beta p,
//   y += alpha p, r -= alpha s, u -= alpha q, w -= alpha z.
// The iterates are those of k_pcgmx in exact arithmetic; the outer FP64
// refinement is the same.
// ---------------------------------------------------------------------
template <int CPT>
__global__ __launch_bounds__(PB) void k_pcgmx_pl(PMxArgs a) {
  // the window, then one word that stays zero: a row reads it in place of
  // a neighbour it does not couple to, so that every lane loads
  __shared__ float lds[2 * WIN + CPT * PB + 1];
  // More than 8 cells per thread (BIG): to stay within 160 KiB of LDS the
  // outside cells are a list of 16-bit window slots and their values go
  // straight to the window; towards 256 VGPRs, a row keeps the window slots
  // of its south and north neighbours in one word, M^-1 v stays in the window,
  // and the rows' addresses are formed where they are used.  Bound by the
  // exchanges and, at 12, 14 and 16 cells per thread, by 30, 91 and 157 spilled
  // registers.  Against two launches per iteration of the multi-kernel solve
  // (31 inner iterations, this one 17; lakes, event-timed): 1.10 M cells 1024 -> 233
  // us, 1.37 M 1108 -> 269, 2.02 M 1320 -> 525.  Up to 8 the plain form is the
  // faster one for all its spills (30 at 7, 69 at 8; us a solve of 13
  // iterations, plain : BIG; 6 cells 134 : 155, 7 156 : 168, 8 172 : 178).
  constexpr bool BIG = CPT > PCGMX_CPT_SMALL;
  static_assert(!BIG || 3 * CPT * PB >= 2 * WIN, "the list of outside cells is formed there");
  __shared__ int hl[BIG ? 1 : 2 * WIN];
  __shared__ unsigned short hs[BIG ? 2 * WIN : 1];
  constexpr int ZS = 2 * WIN + CPT * PB;
  // y, q = M^-1 s and z = A' q of the own rows live in LDS
  __shared__ float lyqz[3 * CPT * PB];
  const int b0 = 1 + (int)blockIdx.x * CPT * PB;
  const int b1 = min(b0 + CPT * PB, a.nwet + 1);
  const int lc0 = a.lc0;

  float as_[CPT], an_[CPT], aw_[CPT], ae_[CPT];
  float r[CPT], u[CPT], w[CPT], s[CPT], p[CPT];
  auto Y = [&](int k) -> float & { return lyqz[k * PB + threadIdx.x]; };
  auto Q = [&](int k) -> float & { return lyqz[(CPT + k) * PB + threadIdx.x]; };
  auto Z = [&](int k) -> float & { return lyqz[(2 * CPT + k) * PB + threadIdx.x]; };
  int js[BIG ? 1 : CPT], jn[BIG ? 1 : CPT];
  unsigned jj[BIG ? CPT : 1];
  unsigned expo = 0u;

  // BIG: the compiler works on a few rows at a time (loads of all sixteen in
  // flight would spill the solve's state)
  auto fence = [](int k_) {
    if (BIG && k_ % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  };
  auto inside = [&](int j) { return j >= b0 && j < b1; };
  auto real = [&](int j) { return j > 0 && j < lc0; };
  auto slot = [&](int j) { return j - b0 + WIN; };
  // the cell of a window slot (ZS: none), and a slot where it is an own cell's
  auto cellof = [&](int sl) { return sl == ZS ? lc0 : sl - WIN + b0; };
  auto ownslot = [&](int sl) { return sl >= WIN && sl < b1 - b0 + WIN ? sl : ZS; };
  auto publish_w = [&](int i, unsigned tag, float v) {
    put_word(hslot32(a.xc, tag) + (size_t)opaque(i), tag, __float_as_uint(v));
  };
  // BIG: the outside-read rows' slots, one base per call and no address kept
  auto post_rows = [&](unsigned tag) {
    u64 *h = hslot32(a.xc, tag) + (size_t)opaque(b0 + (int)threadIdx.x);
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (expo & (1u << k))
        put_word(h + k * PB, tag, __float_as_uint(lds[WIN + k * PB + (int)threadIdx.x]));
  };
  // M^-1 v by the local Neumann polynomial, as in k_pcgmx.  No branch per
  // row: the lanes past b1 (the last workgroup's) hold zero coefficients
  // and zero vectors, so their rows stay zero, and their slots, which no
  // row reads, hold those zeros.
  auto precond = [&](const float (&v)[CPT], float (&t)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) t[k] = v[k];
    for (int d = 1; d < a.pdeg; ++d) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < CPT; ++k) lds[slot(b0 + k * PB + (int)threadIdx.x)] = t[k];
      __syncthreads();
      float tn[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int i = b0 + k * PB + (int)threadIdx.x;
        const float ts = lds[inside(js[k]) ? slot(js[k]) : ZS];
        const float tnn = lds[inside(jn[k]) ? slot(jn[k]) : ZS];
        const float tw = lds[i - 1 >= b0 ? slot(i - 1) : ZS];
        const float te = lds[i + 1 < b1 ? slot(i + 1) : ZS];
        tn[k] = v[k] - (as_[k] * ts + an_[k] * tnn + aw_[k] * tw + ae_[k] * te);
      }
#pragma unroll
      for (int k = 0; k < CPT; ++k) t[k] = tn[k];
    }
    __syncthreads();
  };
  // BIG: the same with the result (and every step's values) in the own slots
  // of the window, one register per row instead of two
  auto precond_lds = [&](const float (&v)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) lds[WIN + k * PB + (int)threadIdx.x] = v[k];
    for (int d = 1; d < a.pdeg; ++d) {
      __syncthreads();
      float tn[CPT];
      const int tt = opaque((int)threadIdx.x);
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const unsigned q = (unsigned)opaque((int)jj[k]);
        const float ts = lds[ownslot((int)(q & 0xffffu))];
        const float tnn = lds[ownslot((int)(q >> 16))];
        const float tw = lds[k == 0 && tt == 0 ? ZS : WIN + k * PB + tt - 1];
        const float te = lds[k * PB + tt + 1 < b1 - b0 ? WIN + k * PB + tt + 1 : ZS];
        tn[k] = v[k] - (as_[k] * ts + an_[k] * tnn + aw_[k] * tw + ae_[k] * te);
        fence(k);
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < CPT; ++k) lds[WIN + k * PB + (int)threadIdx.x] = tn[k];
    }
  };
  // y = A' x with x in the window (own slots and outside cells)
  auto spmv_lds = [&](float (&y)[CPT]) {
    const int tt = opaque((int)threadIdx.x);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + tt;
      const unsigned q = (unsigned)opaque((int)jj[k]);
      const float vs = lds[q & 0xffffu], vn = lds[q >> 16];
      const float vw = lds[real(i - 1) ? slot(i - 1) : ZS];
      const float ve = lds[real(i + 1) ? slot(i + 1) : ZS];
      const float yk = lds[slot(i)] + as_[k] * vs + an_[k] * vn + aw_[k] * vw + ae_[k] * ve;
      y[k] = i < b1 ? yk : 0.0f;
      fence(k);
    }
  };
  // y = A' x on the own rows from the LDS window (own slots and outside
  // cells); a lane past b1 may read a slot no one wrote, so its row is
  // replaced by zero
  auto spmv = [&](const float (&x)[CPT], float (&y)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const float vs = lds[real(js[k]) ? slot(js[k]) : ZS];
      const float vn = lds[real(jn[k]) ? slot(jn[k]) : ZS];
      const float vw = lds[real(i - 1) ? slot(i - 1) : ZS];
      const float ve = lds[real(i + 1) ? slot(i + 1) : ZS];
      const float yk = x[k] + as_[k] * vs + an_[k] * vn + aw_[k] * vw + ae_[k] * ve;
      y[k] = i < b1 ? yk : 0.0f;
    }
  };

  int *mark = BIG ? (int *)lyqz : hl;  // the list is formed where Y, Q, Z will be
  for (int g = threadIdx.x; g < 2 * WIN; g += PB) mark[g] = 0;
  if (threadIdx.x == 0) { lds[ZS] = 0.0f; bad() = 0; }
  __syncthreads();
  double fp2 = 0.0;
  // every lane loads (a lane past b1 from the last own cell) and keeps the
  // values of an own row only
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = b0 + k * PB + (int)threadIdx.x;
    const bool own = i < b1;
    const int ic = own ? i : b1 - 1;
    r[k] = u[k] = w[k] = s[k] = p[k] = 0.0f;
    const int s_ = a.ls[ic], n_ = a.ln[ic];
    const float as_i = a.as[ic], aw_i = a.aw[ic], as_n = a.as[n_], aw_e = a.aw[ic + 1];
    const double fpt = a.fptmp[ic];
    if constexpr (BIG) {
      const unsigned sl = own && real(s_) ? slot(s_) : ZS, nl = own && real(n_) ? slot(n_) : ZS;
      jj[k] = sl | nl << 16;
    } else {
      js[k] = own ? s_ : lc0;
      jn[k] = own ? n_ : lc0;
    }
    as_[k] = own ? as_i : 0.0f;
    aw_[k] = own ? aw_i : 0.0f;
    an_[k] = (own && n_ != lc0) ? as_n : 0.0f;
    ae_[k] = (own && ic + 1 != lc0) ? aw_e : 0.0f;
    if (own) {
      const int nbq[4] = {s_, n_, i - 1, i + 1};
      bool out = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = nbq[q];
        if (real(j) && !inside(j)) {
          out = true;
          mark[ghost_of(j, b0, b1)] = 1;
        }
      }
      if (out) expo |= 1u << k;
    }
    fp2 += own ? fpt * fpt : 0.0;
    fence(k);
  }
  __syncthreads();
  const int nhalo = compact_halo(mark, b0, b1);
  if constexpr (BIG) {
    for (int h = threadIdx.x; h < nhalo; h += PB) hs[h] = (unsigned short)slot(mark[h]);
    __syncthreads();  // the list is read before Y takes its place
  }

  unsigned tag = a.tag0, gen = 0;
  // the outside cells' words of exchange `tag` into the window, by every wave
  // (a wave of the workgroup may still read own slots only)
  auto halo = [&]() {
    halo32<4>(a.xc, tag, nhalo, (int)threadIdx.x, PB, a.bar,
              [&](int h) { return BIG ? (int)hs[h] + b0 - WIN : hl[h]; },
              [&](int h, float v) { lds[BIG ? (int)hs[h] : slot(hl[h])] = v; });
    __syncthreads();  // (an abandoned wait: the next exchange leaves)
  };
  double rsqm = a.rsqm, bnorm2 = 0.0, rsq64 = 0.0, bn_in = 0.0;
  int total = 0, outer = 0, status = 0, inner = 0;

  for (;;) {
    // ---- FP64 residual r = FPTMP - A P, scaled to r' = D^-1/2 r (FP32)
    double v3[3] = {0.0, 0.0, fp2};
    // every lane loads (a lane past b1 from the last own cell; its js, jn
    // are lc0) and the own rows are selected, so the loads of all the
    // thread's rows are in flight together
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const bool own = i < b1;
      int s_, n_;
      if constexpr (BIG) {
        const unsigned q = (unsigned)opaque((int)jj[k]);
        s_ = cellof((int)(q & 0xffffu));
        n_ = cellof((int)(q >> 16));
      } else {
        s_ = opaque(js[k]);
        n_ = opaque(jn[k]);
      }
      const int io = opaque(own ? i : b1 - 1);
      const int ie = io + 1;  // <= lc0
      const double *P = a.x;
      const double ccs_i = a.ccs[io], ccs_n = a.ccs[n_], ccw_i = a.ccw[io];
      const double ccw_e = a.ccw[ie], fpt = a.fptmp[io], cci = a.ccc[io], di = a.dis[io];
      const double p_i = fetch(&P[io]), p_n = fetch(&P[n_]), p_s = fetch(&P[s_]);
      const double p_w = fetch(&P[io - 1]), p_e = fetch(&P[ie]);
      const double cs = (s_ != lc0) ? ccs_i : 0.0;
      const double cn = (n_ != lc0) ? ccs_n : 0.0;
      const double cw = ccw_i;
      const double ce = (ie != lc0) ? ccw_e : 0.0;
      const double rr = fpt - cci * p_i - cn * p_n - cs * p_s - cw * p_w - ce * p_e;
      const float rs = (float)(di * rr);
      r[k] = own ? rs : 0.0f;
      Y(k) = 0.0f;
      v3[0] += own ? rr * rr : 0.0;
      v3[1] += own ? (double)rs * (double)rs : 0.0;
      fence(k);
    }
    post<3>(v3, a.xc, tag);
    if constexpr (BIG) {
      precond_lds(r);
#pragma unroll
      for (int k = 0; k < CPT; ++k) u[k] = lds[WIN + k * PB + (int)threadIdx.x];
      post_rows(tag);
    } else {
      precond(r, u);
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const int i = b0 + k * PB + (int)threadIdx.x;
        lds[slot(i)] = u[k];
        if (expo & (1u << k)) publish_w(i, tag, u[k]);
      }
    }
    fp2 = 0.0;
    halo();
    {
      double s3[3];
      if (!exchange<3, BIG ? 2 : 4>(a.xc, tag, a.bar, s3, NoHalo())) return;
      if (outer == 0) {
        bnorm2 = s3[2];
        rsqm = a.rel_tol > 0.0 ? a.rel_tol * a.rel_tol * bnorm2 : a.rsqm;
      }
      rsq64 = s3[0];
      bn_in = s3[1];
    }
    if (rsq64 <= rsqm) break;
    if (outer >= a.max_outer || bn_in == 0.0) { status = 1; break; }
    const double rt2 = fmax(a.rtol2, INNER_MARGIN2 * rsqm / rsq64);

    // ---- w0 = A' u0; s, p, q, z start at 0
    if constexpr (BIG) spmv_lds(w);
    else spmv(u, w);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      s[k] = p[k] = 0.0f;
      Q(k) = Z(k) = 0.0f;
    }
    double gam_prev = 0.0, alpha_prev = 1.0;
    inner = 0;
    for (;;) {
      ++tag;
      // the sums of this iteration go out first ...
      // (the lanes past b1 add zeros)
      double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        v[0] += (double)r[k] * (double)u[k];
        v[1] += (double)w[k] * (double)u[k];
        v[2] += (double)r[k] * (double)r[k];
        fence(k);
      }
      post<3>(v, a.xc, tag);
      // ... then m = M^-1 w and its outside values
      float m[BIG ? 1 : CPT];
      if constexpr (BIG) {
        precond_lds(w);
        post_rows(tag);
      } else {
        precond(w, m);
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          const int i = b0 + k * PB + (int)threadIdx.x;
          lds[slot(i)] = m[k];
          if (expo & (1u << k)) publish_w(i, tag, m[k]);
        }
      }
      // n = A' m once the neighbouring workgroups' m has arrived
      halo();
      float n[CPT];
      if constexpr (BIG) spmv_lds(n);
      else spmv(m, n);
      // the sums of every workgroup
      double s3[3];
      if (!exchange<3, BIG ? 2 : 4>(a.xc, tag, a.bar, s3, NoHalo())) return;
      const double gam = s3[0], del = s3[1];
      if (s3[2] <= rt2 * bn_in || inner >= a.iterm) break;
      double beta, alpha;
      if (inner == 0) {
        beta = 0.0;
        alpha = gam / del;
      } else {
        beta = gam / gam_prev;
        alpha = gam / (del - beta * gam / alpha_prev);
      }
      // the vector updates in FP32 (one rounding each, fused multiply-add);
      // the sums, alpha and beta stay FP64 and the outer FP64 residual
      // decides convergence
      const float bf = (float)beta, af = (float)alpha;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const float zk = fmaf(bf, Z(k), n[k]);
        const float mk = BIG ? lds[WIN + k * PB + (int)threadIdx.x] : m[BIG ? 0 : k];
        const float qk = fmaf(bf, Q(k), mk);
        s[k] = fmaf(bf, s[k], w[k]);
        p[k] = fmaf(bf, p[k], u[k]);
        Y(k) = fmaf(af, p[k], Y(k));
        r[k] = fmaf(-af, s[k], r[k]);
        u[k] = fmaf(-af, qk, u[k]);
        w[k] = fmaf(-af, zk, w[k]);
        Z(k) = zk;
        Q(k) = qk;
        fence(k);
      }
      inner += 1;
      gam_prev = gam;
      alpha_prev = alpha;
    }
    total += inner;
    ++tag;
    // ---- P += D^-1/2 y (FP64), visible to every workgroup for the next
    // residual
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const bool own = i < b1;
      const int io = opaque(own ? i : b1 - 1);  // every lane loads
      double *P = a.x;
      const double pn = fetch(&P[io]) + a.dis[io] * (double)Y(k);
      if (own) publish(&P[io], pn);
      fence(k);
    }
    ++outer;
    if (!grid_barrier(a.bar, ++gen)) return;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    CgState *st = a.st;
    st->rsq64 = rsq64;
    st->rsq = rsq64;
    st->rsqm = rsqm;
    st->bnorm2 = bnorm2;
    st->bnorm2_in = bn_in;
    st->iter = total;
    st->inner_iter = inner;
    st->outer = outer;
    st->done = 1;
    st->status = status;
  }
}

// ---------------------------------------------------------------------
// FP64 Jacobi-PCG, pipelined (opt-in: efdc_set_cg64_pipeline).  The
// reference's PCG (EFDC/congrad.f90:91-169) rewritten in the pipelined order
// of Ghysels and Vanroose (2014), as k_pcgmx_pl does for the mixed inner
// solve: an iteration posts its sums (r,u), (w,u), (r,r) and the m = CCCI w
// of its outside-read cells; it waits only for the workgroups
// that own its outside cells, forms n = A m, and only then waits for every
// workgroup's sums to take alpha and beta.  The Jacobi preconditioner is
// diagonal, so u = CCCI r, m = CCCI w and q = CCCI s are formed where they
// are used; the state is x, r, w, s, p (registers) and z = A q (LDS):
//   z = n + beta z, s = w + beta s, p = u + beta p,
//   x += alpha p, r -= alpha s, w -= alpha z.
// Same iterates as the reference's recurrences in exact arithmetic, one
// exchange per iteration instead of two.  The stop test is the
// reference's, (r,r) <= RSQM (:165), made on the sums of the iteration
// that would update from r.
// Bound by the exchange, and at 6 cells per thread by 256 registers: x in LDS
// and the neighbours' window slots in 16 bits each leave 12 spilled (us a
// solve of 18 to 19 iterations, this form : the default one; 79 k cells 74 : 85,
// 276 k 105 : 118, 483 k 133 : 153, 696 k 174 : 190).
// ---------------------------------------------------------------------
template <int CPT>
__global__ __launch_bounds__(PB) void k_pcg64_pl(P64Args a) {
  // the window, then one word that stays zero (read in place of a
  // neighbour that is not a cell, so that every lane loads)
  __shared__ double lds[2 * WIN + CPT * PB + 1];
  __shared__ int hl[2 * WIN];
  __shared__ double lzs[CPT * PB], lxs[CPT * PB];
  constexpr int ZS = 2 * WIN + CPT * PB;
  const int b0 = 1 + (int)blockIdx.x * CPT * PB;
  const int b1 = min(b0 + CPT * PB, a.nwet + 1);
  const bool fast = a.rowmajor && (a.st->symok == 0);
  const int lc0 = a.lc0;

  double ccc[CPT], cs[CPT], cn[CPT], cw[CPT], ce[CPT], cci[CPT];
  double r[CPT], w[CPT], s[CPT], p[CPT];
  unsigned nj[CPT][2];       // window slots of S | N << 16 and W | E << 16
  unsigned expo = 0u;        // bit k: another workgroup reads cell k
  auto Z = [&](int k) -> double & { return lzs[k * PB + threadIdx.x]; };

  auto X = [&](int k) -> double & { return lxs[k * PB + threadIdx.x]; };
  auto inside = [&](int j) { return j >= b0 && j < b1; };
  auto real = [&](int j) { return j > 0 && j < lc0; };
  auto slot = [&](int j) { return j - b0 + WIN; };
  auto publish_m = [&](int i, unsigned tag, double v) {
    put_f64(hslot64(a.xc, tag) + 2 * (size_t)opaque(i), tag, v);
  };
  // y = A v on the own rows from the window (own slots and outside cells);
  // the lanes past b1 have ccc = 1, zero couplings and v = 0
  auto spmv = [&](const double (&v)[CPT], double (&y)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      double pq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const unsigned u = (unsigned)opaque((int)nj[k][q >> 1]);
        pq[q] = lds[q & 1 ? u >> 16 : u & 0xffffu];
      }
      // APCG = CCC*PCG + CCS*PS + CCN*PN + CCW*PW + CCE*PE (:113)
      y[k] = ccc[k] * v[k] + cs[k] * pq[NS] + cn[k] * pq[NN] + cw[k] * pq[NW] +
             ce[k] * pq[NE];
    }
  };

  for (int g = threadIdx.x; g < 2 * WIN; g += PB) hl[g] = 0;
  if (threadIdx.x == 0) { lds[ZS] = 0.0; bad() = 0; }
  __syncthreads();
  double fp2 = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = b0 + k * PB + (int)threadIdx.x;
    X(k) = r[k] = w[k] = s[k] = p[k] = 0.0;
    Z(k) = 0.0;
    ccc[k] = 1.0; cs[k] = cn[k] = cw[k] = ce[k] = cci[k] = 0.0;
    nj[k][0] = nj[k][1] = ZS | (unsigned)ZS << 16;
    if (i < b1) {
      // the row as in the multi-kernel solve (row_of)
      const int js = a.ls[i], jn = a.ln[i];
      int jw, je;
      double s_ = a.ccs[i], w_ = a.ccw[i], n_, e_;
      if (fast) {
        jw = i - 1;
        je = i + 1;
        n_ = (jn != lc0) ? a.ccs[jn] : 0.0;
        e_ = (je != lc0) ? a.ccw[je] : 0.0;
      } else {
        jw = a.lw[i];
        je = a.le[i];
        n_ = (jn != lc0) ? a.ccn[i] : 0.0;
        e_ = (je != lc0) ? a.cce[i] : 0.0;
        if (jw == lc0) w_ = 0.0;
      }
      if (js == lc0) s_ = 0.0;
      const int nb[4] = {js, jn, jw, je};
      ccc[k] = a.ccc[i]; cs[k] = s_; cn[k] = n_; cw[k] = w_; ce[k] = e_;
      cci[k] = a.ccci[i];
      bool out = false;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = nb[q];
        if (real(j) && !inside(j)) {
          out = true;
          hl[ghost_of(j, b0, b1)] = 1;
        }
      }
      auto ws = [&](int j) { return real(j) ? (unsigned)slot(j) : (unsigned)ZS; };
      nj[k][0] = ws(js) | ws(jn) << 16;
      nj[k][1] = ws(jw) | ws(je) << 16;
      if (out || !a.mutual) expo |= 1u << k;
      const double *P = a.x;
      const double x0 = P[i];
      X(k) = x0;
      // RCG = FPTMP - CCC*P - CCN*PN - CCS*PS - CCW*PW - CCE*PE (:73)
      r[k] = a.fptmp[i] - ccc[k] * x0 - n_ * P[jn] - s_ * P[js] - w_ * P[jw] - e_ * P[je];
      fp2 += a.fptmp[i] * a.fptmp[i];
    }
  }
  __syncthreads();
  const int nhalo = compact_halo(hl, b0, b1);

  // set-up exchange: u = CCCI r of the outside-read cells and |FPTMP|^2;
  // then w = A u (the owners publish u, so no CCCI of an outside cell is
  // loaded)
  unsigned tag = a.tag0;
  // the outside cells' values of exchange `tag` into the window, by every wave
  auto halo = [&]() {
    halo64<2>(a.xc, tag, nhalo, (int)threadIdx.x, PB, a.bar, [&](int h) { return hl[h]; },
              [&](int h, double v) { lds[slot(hl[h])] = v; });
    __syncthreads();  // (an abandoned wait: the next exchange leaves)
  };
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = b0 + k * PB + (int)threadIdx.x;
    const double uk = cci[k] * r[k];
    lds[slot(i)] = uk;
    if (expo & (1u << k)) publish_m(i, tag, uk);
  }
  {
    double v1[1] = {fp2};
    post<1>(v1, a.xc, tag);
  }
  double s1[1];
  halo();
  if (!exchange_waves<1>(a.xc, tag, a.bar, s1)) return;
  const double bnorm2 = s1[0];
  const double rsqm = a.rel_tol > 0.0 ? a.rel_tol * a.rel_tol * bnorm2 : a.rsqm;
  {
    double u0[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) u0[k] = cci[k] * r[k];
    spmv(u0, w);
  }

  double gam_prev = 0.0, alpha_prev = 1.0, gam = 0.0, alpha = 0.0, beta = 0.0, rsq = 0.0;
  int iter = 0, status = 0;
  for (;;) {
    ++tag;
    // the sums of this iteration go out first (the lanes past b1 add zeros) ...
    double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double uk = cci[k] * r[k];
      v[0] += r[k] * uk;
      v[1] += w[k] * uk;
      v[2] += r[k] * r[k];
    }
    post<3>(v, a.xc, tag);
    // ... then m = CCCI w on the window (every wave is past its reads of the
    // last SpMV: post's barrier) and m of the outside-read cells
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = b0 + k * PB + (int)threadIdx.x;
      const double mk = cci[k] * w[k];
      lds[slot(i)] = mk;
      if (expo & (1u << k)) publish_m(i, tag, mk);
    }
    // n = A m once the neighbouring workgroups' m has arrived
    halo();
    double m[CPT], n[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) m[k] = cci[k] * w[k];
    spmv(m, n);
    // the sums of every workgroup
    double s3[3];
    if (!exchange_waves<3>(a.xc, tag, a.bar, s3)) return;
    gam = s3[0];
    const double del = s3[1];
    rsq = s3[2];
    if (rsq <= rsqm || gam == 0.0) break;  // :165 (and RPCG = 0, :88)
    if (iter >= a.iterm) { status = 1; break; }
    if (iter == 0) {
      beta = 0.0;
      alpha = gam / del;
    } else {
      beta = gam / gam_prev;
      alpha = gam / (del - beta * gam / alpha_prev);
    }
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double zk = n[k] + beta * Z(k);
      s[k] = w[k] + beta * s[k];
      p[k] = cci[k] * r[k] + beta * p[k];
      X(k) = X(k) + alpha * p[k];
      r[k] = r[k] - alpha * s[k];
      w[k] = w[k] - alpha * zk;
      Z(k) = zk;
    }
    iter += 1;
    gam_prev = gam;
    alpha_prev = alpha;
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = b0 + k * PB + (int)threadIdx.x;
    if (i < b1) a.x[opaque(i)] = X(k);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    CgState *st = a.st;
    st->rpcg = gam;
    st->papcg = 0.0;
    st->alpha = alpha;
    st->beta = beta;
    st->rsq = rsq;
    st->rsqm = rsqm;
    st->bnorm2 = bnorm2;
    st->iter = iter;
    st->done = 1;
    st->status = status;
  }
}

// Jacobi scaling of the mixed solve from a scaled system (CCC, CCS, CCW)
// given directly: dis = 1/sqrt(CCC), A'(i,S), A'(i,W) in FP32.
__global__ __launch_bounds__(256) void k_mx_coef(const double *ccc, const double *ccs,
                                                 const double *ccw, const int *ls, int nwet,
                                                 int lc0, double *dis, float *as, float *aw) {
  const int i = 1 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i > nwet) return;
  const int js = ls[i];
  const double di = 1.0 / sqrt(ccc[i]);
  const double ds = (js != lc0) ? 1.0 / sqrt(ccc[js]) : 0.0;
  const double dw = (i - 1 > 0) ? 1.0 / sqrt(ccc[i - 1]) : 0.0;
  const double cs = (js != lc0) ? ccs[i] : 0.0;
  dis[i] = di;
  as[i] = (float)(cs * di * ds);
  aw[i] = (float)(ccw[i] * di * dw);
}

// Slots that carry no exchange's number.
__global__ __launch_bounds__(256) void k_pcg_clear(u64 *ps, long nps, u64 *hx, long nhx) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < nps + nhx; i += gridDim.x * 256L)
    (i < nps ? ps[i] : hx[i - nps]) = 0;
}

__global__ void k_pcg_reset(unsigned *ctr, int *abort) {
  const int t = threadIdx.x;
  if (t < PCG_NCTR) ctr[t] = 0u;
  if (t == 0) *abort = 0;
}

template <typename K>
int occupancy(K kern) {
  int nbpc = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nbpc, kern, PB, 0) != hipSuccess)
    return 0;
  return nbpc;
}

}  // namespace

// Terms of the workgroup-local preconditioner of the mixed persistent solve
// when the caller leaves the choice to the library.
constexpr int PCG_PDEG_DEFAULT = 3;
// Exchange numbers: launch number (1 .. 4095) in the top 12 bits, exchange
// within the launch in the low 20 bits.
constexpr int PCG_TAG_BITS = 20;
constexpr long PCG_TAGS_PER_LAUNCH = 1L << PCG_TAG_BITS;
constexpr unsigned PCG_LAUNCH_CYCLE = (1u << (32 - PCG_TAG_BITS)) - 1u;

int pcg_prepare(efdc_ctx *c) {
  if (c->pcg_ready) return EFDC_OK;
  int dev = c->device, ncu = 0;
  HIP_TRY(c, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  int coop = 0;
  HIP_TRY(c, hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
  c->pcg_ncu = coop ? ncu : 0;
  const int occ64[PCG64_CPT_MAX + 1] = {
      0, occupancy(k_pcg64<1, false>), occupancy(k_pcg64<2, false>), occupancy(k_pcg64<3, false>),
      occupancy(k_pcg64<4, false>), occupancy(k_pcg64<5, false>), occupancy(k_pcg64<6, false>)};
  const int occmx[PCGMX_CPT_SMALL + 1] = {
      0, occupancy(k_pcgmx<1>), occupancy(k_pcgmx<2>), occupancy(k_pcgmx<3>),
      occupancy(k_pcgmx<4>), occupancy(k_pcgmx<5>), occupancy(k_pcgmx<6>),
      occupancy(k_pcgmx<7>), occupancy(k_pcgmx<8>)};
  // 10, 12, 14 and 16 cells per thread in the pipelined form alone
  const int occpl[PCGMX_CPT_MAX + 1] = {
      0, occupancy(k_pcgmx_pl<1>), occupancy(k_pcgmx_pl<2>), occupancy(k_pcgmx_pl<3>),
      occupancy(k_pcgmx_pl<4>), occupancy(k_pcgmx_pl<5>), occupancy(k_pcgmx_pl<6>),
      occupancy(k_pcgmx_pl<7>), occupancy(k_pcgmx_pl<8>), 0, occupancy(k_pcgmx_pl<10>), 0,
      occupancy(k_pcgmx_pl<12>), 0, occupancy(k_pcgmx_pl<14>), 0, occupancy(k_pcgmx_pl<16>)};
  const int occ64p[PCG64_CPT_MAX + 1] = {
      0, occupancy(k_pcg64_pl<1>), occupancy(k_pcg64_pl<2>), occupancy(k_pcg64_pl<3>),
      occupancy(k_pcg64_pl<4>), occupancy(k_pcg64_pl<5>), occupancy(k_pcg64_pl<6>)};
  // 2, 4 and 6 cells per thread for basins
  const int occ64s[PCG64_CPT_MAX + 1] = {
      0, 0, occupancy(k_pcg64<2, true>), 0, occupancy(k_pcg64<4, true>), 0,
      occupancy(k_pcg64<6, true>)};
  for (int k = 0; k <= PCG64_CPT_MAX; ++k) {
    c->pcg_occ64[k] = std::min(occ64[k], occ64p[k]);
    c->pcg_occseg[k] = occ64s[k];
  }
  for (int k = 0; k <= PCGMX_CPT_MAX; ++k)
    c->pcg_occmx[k] = k <= PCGMX_CPT_SMALL ? std::min(occmx[k], occpl[k]) : occpl[k];
  c->pcg_ncell = c->n_wet() + 2;
  int s;
  // two parities of two words a cell, and of NVMAX doubles a workgroup
  if ((s = dev_alloc(c, &c->pcg_hx, sizeof(u64) * 4 * (size_t)c->pcg_ncell))) return s;
  if ((s = dev_alloc(c, &c->pcg_ps, sizeof(u64) * 2 * PSLOTS * 2 * NVMAX))) return s;
  if ((s = dev_alloc(c, (void **)&c->pcg_ctr, sizeof(unsigned) * PCG_NCTR))) return s;
  c->pcg_abort = &c->st->pabort;
  c->pcg_launch = 0;
  c->pcg_ready = true;
  return EFDC_OK;
}

// Cells per thread and workgroup count of a persistent solve, or 0 when
// the problem does not fit in one co-resident grid: the fewest cells per
// thread that need at most nb_want workgroups, else the most that fit.
static int pcg_shape(const efdc_ctx *c, const int *occ, int cpt_max, int &nb,
                     int nb_want = PB) {
  const int n = c->n_wet();
  int best = 0;
  for (int cpt = 1; cpt <= cpt_max; ++cpt) {
    const int need = (n + cpt * PB - 1) / (cpt * PB);
    const int cap = occ[cpt] * c->pcg_ncu;
    if (occ[cpt] > 0 && need <= cap && need <= PB) {
      best = cpt;
      nb = need;
      if (need <= nb_want) break;
    }
  }
  return best;
}

// FP64: every workgroup reads the partials of all of them, twice an
// iteration, which beyond about 64 costs more than a further row per thread
// (us a solve of 29 iterations, workgroups : cells per thread; 79 k cells 155 :
// 1 160, 78 : 2 150, 52 : 3 137, 26 : 6 153; 276 k cells 180 : 3 213, 135 : 4
// 197, 90 : 6 181; 22 k cells 43 : 1 126, 22 : 2 131).  The mixed solve, one
// exchange per iteration with the preconditioner behind it, gains nothing
// (169 k cells 166 : 2 109, 111 : 3 114, 83 : 4 117).
constexpr int PCG64_NB = 64;
// The pipelined form reads them once, behind the SpMV, so it takes more
// workgroups before a row more (us a solve of 18 iterations, workgroups : cells
// per thread; 156 k cells 153 : 2 85, 102 : 3 82, 61 : 5 86; 276 k 180 : 3 105,
// 108 : 5 104, 90 : 6 114; 483 k 236 : 4 139, 189 : 5 133, 158 : 6 141).
constexpr int PCG64_PIPE_NB = 192;
static int pcg_shape64(const efdc_ctx *c, int &nb) {
  return pcg_shape(c, c->pcg_occ64, PCG64_CPT_MAX, nb, c->pcg64_pipe ? PCG64_PIPE_NB : PCG64_NB);
}

// The form of the mixed persistent solve, and its shape: more than 8 cells
// per thread (1.05 to 2.1 million cells on 256 CUs) in the pipelined form
// alone, which also runs there while the tuner has found the other faster.
static bool pcg_pipelined(const efdc_ctx *c) {
  return c->pcg_pipe_mode == 2 || (c->pcg_pipe_mode == 0 && c->pcg_pipe_tuned);
}
static int pcg_shape_mx(const efdc_ctx *c, int &nb) {
  const int cpt = pcg_shape(c, c->pcg_occmx, PCGMX_CPT_SMALL, nb);
  if (cpt || c->pcg_pipe_mode == 1) return cpt;
  return pcg_shape(c, c->pcg_occmx, PCGMX_CPT_MAX, nb);
}

bool pcg_applicable(efdc_ctx *c, bool mixed) {
  if (c->prm.cg_kernel == EFDC_CG_KERNEL_MULTI) return false;
  if (c->band > WIN) return false;  // a neighbour beyond the LDS window
  // the exchanges of one solve must fit one launch's tag range
  const long per_outer = 3L + c->prm.ITERM;
  const long outers = mixed ? (long)c->prm.mixed_max_outer + 1 : 1;
  if ((mixed ? per_outer * outers : 1L + 2L * c->prm.ITERM) >= PCG_TAGS_PER_LAUNCH)
    return false;
  if (pcg_prepare(c) != EFDC_OK || c->pcg_ncu == 0) return false;
  int nb = 0;
  return mixed ? pcg_shape_mx(c, nb) > 0
               : pcg_shape64(c, nb) > 0;
}

// The persistent grid is sized to be co-resident (the occupancy table times
// the CUs).  A cooperative launch guarantees it, at the price of the
// runtime's cooperative dispatch (about 15 us per solve on MI355X); a plain
// launch of the same grid is co-resident whenever no other work holds the
// CUs, and otherwise every bounded wait gives up and the solve reports an
// abort, after which it is solved again with the cooperative launch
// (pcg_solve, pcg_retry_deferred).  pcg_launch_mode 1 always uses the
// cooperative launch.
template <typename Args>
static int coop_launch(efdc_ctx *c, const void *fn, int nb, Args &args) {
  void *kargs[] = {&args};
  if (c->pcg_launch_mode == 0 && !c->pcg_force_coop) {
    HIP_TRY(c, hipLaunchKernel(fn, dim3(nb), dim3(PB), kargs, 0, c->stream));
    c->pcg_last_plain = true;
  } else {
    HIP_TRY(c, hipLaunchCooperativeKernel(fn, dim3(nb), dim3(PB), kargs, 0, c->stream));
    c->pcg_last_plain = false;
  }
  return EFDC_OK;
}

// First exchange number of the next launch.  Launches are numbered
// 1 .. 4095, so within a cycle a slot never holds a number that is still to
// come; when the numbering starts a new cycle the slots are cleared.
static int next_tag0(efdc_ctx *c, unsigned &tag0) {
  const bool wrap = c->pcg_launch == PCG_LAUNCH_CYCLE;
  c->pcg_launch = c->pcg_launch % PCG_LAUNCH_CYCLE + 1u;
  if (wrap) {
    k_pcg_clear<<<512, 256, 0, c->stream>>>((u64 *)c->pcg_ps, 2 * PSLOTS * 2 * NVMAX,
                                            (u64 *)c->pcg_hx, 4 * (long)c->pcg_ncell);
    HIP_TRY(c, hipGetLastError());
  }
  tag0 = c->pcg_launch << PCG_TAG_BITS;
  return EFDC_OK;
}

static const void *p64_kernel(int cpt) {
  switch (cpt) {
    case 1: return (const void *)k_pcg64<1, false>;
    case 2: return (const void *)k_pcg64<2, false>;
    case 3: return (const void *)k_pcg64<3, false>;
    case 4: return (const void *)k_pcg64<4, false>;
    case 5: return (const void *)k_pcg64<5, false>;
    default: return (const void *)k_pcg64<6, false>;
  }
}
static const void *pseg_kernel(int cpt) {
  switch (cpt) {
    case 2: return (const void *)k_pcg64<2, true>;
    case 4: return (const void *)k_pcg64<4, true>;
    default: return (const void *)k_pcg64<6, true>;
  }
}

static int p64_args(efdc_ctx *c, int nb, const Bar &bar, P64Args &a) {
  a.ccc = c->dH[EFDC_CCC];
  a.ccs = c->dH[EFDC_CCS];
  a.ccw = c->dH[EFDC_CCW];
  a.ccn = c->dH[EFDC_CCN];
  a.cce = c->dH[EFDC_CCE];
  a.ccci = c->dH[EFDC_CCCI];
  a.fptmp = c->dH[EFDC_FPTMP];
  a.x = c->dH[EFDC_P];
  a.lw = c->dLW;
  a.le = c->dLE;
  a.ls = c->dLS;
  a.ln = c->dLN;
  a.nwet = c->n_wet();
  a.lc0 = c->LC - 1;
  a.rowmajor = c->rowmajor ? 1 : 0;
  a.mutual = c->mutual ? 1 : 0;
  a.xc = Xch{(u64 *)c->pcg_ps, (u64 *)c->pcg_hx, c->pcg_ncell, 0, nb};
  int s;
  if ((s = next_tag0(c, a.tag0))) return s;
  a.bar = bar;
  a.st = c->st;
  a.rsqm = c->prm.RSQM;
  a.rel_tol = c->prm.cg_rel_tol;
  a.iterm = c->prm.ITERM;
  a.wg = nullptr;
  a.wgseg = nullptr;
  a.segst = nullptr;
  a.xsave = nullptr;
  return EFDC_OK;
}

// Bounded waits: a plain launch may be given a small spin limit (to exercise
// the retry from the host); the cooperative one always has the full limit.
static Bar pcg_bar(efdc_ctx *c) {
  const bool plain = c->pcg_launch_mode == 0 && !c->pcg_force_coop;
  return Bar{c->pcg_ctr, c->pcg_abort,
             plain && c->pcg_spin_test > 0 ? c->pcg_spin_test : SPIN_MAX};
}

int pcg_solve(efdc_ctx *c, bool mixed, bool defer) {
  int s;
  if ((s = pcg_prepare(c))) return s;
  if (!c->pcg_reset_done) {
    k_pcg_reset<<<1, PCG_NCTR, 0, c->stream>>>(c->pcg_ctr, c->pcg_abort);
    HIP_TRY(c, hipGetLastError());
  }
  c->pcg_reset_done = false;  // this launch uses them
  int nb = 0;
  const Bar bar = pcg_bar(c);
  if (!mixed) {
    const int cpt = pcg_shape64(c, nb);
    if (!cpt) { c->err = "persistent CG: problem too large"; return EFDC_ERR_ARG; }
    P64Args a;
    if ((s = p64_args(c, nb, bar, a))) return s;
    const void *fn = nullptr;
    if (c->pcg64_pipe) {
      switch (cpt) {
        case 1: fn = (const void *)k_pcg64_pl<1>; break;
        case 2: fn = (const void *)k_pcg64_pl<2>; break;
        case 3: fn = (const void *)k_pcg64_pl<3>; break;
        case 4: fn = (const void *)k_pcg64_pl<4>; break;
        case 5: fn = (const void *)k_pcg64_pl<5>; break;
        default: fn = (const void *)k_pcg64_pl<6>; break;
      }
    } else {
      fn = p64_kernel(cpt);
    }
    TIMED(c, TK_PCG64, s = coop_launch(c, fn, nb, a));
    if (s) return s;
  } else {
    const int cpt = pcg_shape_mx(c, nb);
    if (!cpt) { c->err = "persistent CG: problem too large"; return EFDC_ERR_ARG; }
    if (!c->mx_coef_ok) {
      const int n = c->n_wet();
      k_mx_coef<<<(n + 255) / 256, 256, 0, c->stream>>>(
          c->dH[EFDC_CCC], c->dH[EFDC_CCS], c->dH[EFDC_CCW], c->dLS, n, c->LC - 1, c->dis,
          c->as32, c->aw32);
      HIP_TRY(c, hipGetLastError());
    }
    PMxArgs a;
    a.ccc = c->dH[EFDC_CCC];
    a.ccs = c->dH[EFDC_CCS];
    a.ccw = c->dH[EFDC_CCW];
    a.fptmp = c->dH[EFDC_FPTMP];
    a.dis = c->dis;
    a.as = c->as32;
    a.aw = c->aw32;
    a.x = c->dH[EFDC_P];
    a.ls = c->dLS;
    a.ln = c->dLN;
    a.nwet = c->n_wet();
    a.lc0 = c->LC - 1;
    a.xc = Xch{(u64 *)c->pcg_ps, (u64 *)c->pcg_hx, c->pcg_ncell, 0, nb};
    if ((s = next_tag0(c, a.tag0))) return s;
    a.bar = bar;
    a.st = c->st;
    a.rsqm = c->prm.RSQM;
    a.rel_tol = c->prm.cg_rel_tol;
    const double rtol = c->prm.mixed_inner_rtol > 0 ? c->prm.mixed_inner_rtol : 1e-5;
    a.rtol2 = rtol * rtol;
    a.iterm = c->prm.ITERM;
    a.max_outer = c->prm.mixed_max_outer;
    a.pdeg = c->prm.mixed_precond_degree > 0 ? c->prm.mixed_precond_degree
             : c->pcg_pdeg_tuned > 0         ? c->pcg_pdeg_tuned
                                             : PCG_PDEG_DEFAULT;
    const bool pl = cpt > PCGMX_CPT_SMALL || pcg_pipelined(c);
    const void *fn = nullptr;
    if (pl) {
      switch (cpt) {
        case 1: fn = (const void *)k_pcgmx_pl<1>; break;
        case 2: fn = (const void *)k_pcgmx_pl<2>; break;
        case 3: fn = (const void *)k_pcgmx_pl<3>; break;
        case 4: fn = (const void *)k_pcgmx_pl<4>; break;
        case 5: fn = (const void *)k_pcgmx_pl<5>; break;
        case 6: fn = (const void *)k_pcgmx_pl<6>; break;
        case 7: fn = (const void *)k_pcgmx_pl<7>; break;
        case 8: fn = (const void *)k_pcgmx_pl<8>; break;
        case 10: fn = (const void *)k_pcgmx_pl<10>; break;
        case 12: fn = (const void *)k_pcgmx_pl<12>; break;
        case 14: fn = (const void *)k_pcgmx_pl<14>; break;
        default: fn = (const void *)k_pcgmx_pl<16>; break;
      }
    } else {
      switch (cpt) {
        case 1: fn = (const void *)k_pcgmx<1>; break;
        case 2: fn = (const void *)k_pcgmx<2>; break;
        case 3: fn = (const void *)k_pcgmx<3>; break;
        case 4: fn = (const void *)k_pcgmx<4>; break;
        case 5: fn = (const void *)k_pcgmx<5>; break;
        case 6: fn = (const void *)k_pcgmx<6>; break;
        case 7: fn = (const void *)k_pcgmx<7>; break;
        default: fn = (const void *)k_pcgmx<8>; break;
      }
    }
    TIMED(c, TK_PCGMX, s = coop_launch(c, fn, nb, a));
    if (s) return s;
  }
  if (defer) {
    // the caller reads the state and the abort flag after the step
    c->pcg_deferred = true;
    return EFDC_OK;
  }
  HIP_TRY(c, hipMemcpyAsync(c->st_host, c->st, sizeof(CgState), hipMemcpyDeviceToHost,
                            c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  if (c->st_host->pabort) {
    if (c->pcg_last_plain) {
      // the plain launch was not co-resident: solve again, cooperatively,
      // from the P it reached (an iterate of the same system)
      ++c->pcg_retries;
      c->pcg_force_coop = true;
      s = pcg_solve(c, mixed, false);
      c->pcg_force_coop = false;
      return s;
    }
    c->err = "persistent CG: an exchange between workgroups timed out";
    return EFDC_ERR_HIP;
  }
  return EFDC_OK;
}

bool pcg_vec_applicable(efdc_ctx *c, int itmax) {
  int nb = 0;
  return c->prm.cg_kernel != EFDC_CG_KERNEL_MULTI && c->band <= WIN &&
         1L + 2L * itmax < PCG_TAGS_PER_LAUNCH && pcg_prepare(c) == EFDC_OK &&
         c->pcg_ncu > 0 && pcg_shape(c, c->pcg_occ64, PCG64_CPT_MAX, nb, PCG64_NB) > 0;
}

// A x = rhs with the matrix of the last step, from x; st and st_host receive
// the state (the adjoint's solve).
int pcg_vec_solve(efdc_ctx *c, double *x, const double *rhs, CgState *st, CgState *st_host,
                  double rel_tol, int itmax) {
  int s, nb = 0;
  const int cpt = pcg_shape(c, c->pcg_occ64, PCG64_CPT_MAX, nb, PCG64_NB);
  // the operator's symmetry flag comes from the forward solve
  HIP_TRY(c, hipMemcpyAsync(st, c->st, sizeof(CgState), hipMemcpyDeviceToDevice, c->stream));
  k_pcg_reset<<<1, PCG_NCTR, 0, c->stream>>>(c->pcg_ctr, &st->pabort);
  HIP_TRY(c, hipGetLastError());
  P64Args a;
  if ((s = p64_args(c, nb, pcg_bar(c), a))) return s;
  a.bar.abort = &st->pabort;
  a.x = x;
  a.fptmp = rhs;
  a.st = st;
  a.rsqm = 0.0;
  a.rel_tol = rel_tol;
  a.iterm = itmax;
  TIMED(c, TK_ADJ_CG, s = coop_launch(c, p64_kernel(cpt), nb, a));
  if (s) return s;
  HIP_TRY(c, hipMemcpyAsync(st_host, st, sizeof(CgState), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  if (!st_host->pabort) return EFDC_OK;
  if (!c->pcg_last_plain) {
    c->err = "persistent CG: an exchange between workgroups timed out";
    return EFDC_ERR_HIP;
  }
  // not co-resident: again, cooperatively, from the x it reached
  ++c->pcg_retries;
  c->pcg_force_coop = true;
  s = pcg_vec_solve(c, x, rhs, st, st_host, rel_tol, itmax);
  c->pcg_force_coop = false;
  return s;
}

// Cells per thread with which every basin's workgroups fit one co-resident
// grid together, and their number; 0 if they do not.
static int pcg_seg_shape(const efdc_ctx *c, int &nb) {
  for (int cpt = 2; cpt <= PCG64_CPT_MAX; cpt += 2) {
    const int cap = std::min(c->pcg_occseg[cpt] * c->pcg_ncu, PB);
    long need = 0;
    for (int q = 0; q < c->nseg; ++q)
      need += (c->seg_first[q + 1] - c->seg_first[q] + cpt * PB - 1) / (cpt * PB);
    if (need <= cap) {
      nb = (int)need;
      return cpt;
    }
  }
  return 0;
}

bool pcg_seg_applicable(efdc_ctx *c) {
  int nb = 0;
  return c->prm.cg_kernel != EFDC_CG_KERNEL_MULTI && c->band <= WIN &&
         1L + 2L * c->prm.ITERM < PCG_TAGS_PER_LAUNCH && pcg_prepare(c) == EFDC_OK &&
         c->pcg_ncu > 0 && pcg_seg_shape(c, nb) > 0;
}

// The FP64 solve of every basin in one persistent launch; the basins' states
// are in h_segst afterwards.
int pcg_seg_solve(efdc_ctx *c) {
  int s, nb = 0;
  const int cpt = pcg_seg_shape(c, nb);
  if (!c->pcg_segwg) {  // (dropped with the basins)
    std::vector<int4> wg;
    std::vector<int> seg;
    for (int q = 0; q < c->nseg; ++q) {
      const int w0 = (int)wg.size(), first = c->seg_first[q], end = c->seg_first[q + 1];
      for (int i = first; i < end; i += cpt * PB) {
        wg.push_back(make_int4(i, end, w0, (end - first + PB - 1) / PB));
        seg.push_back(q);
      }
    }
    void *tab = nullptr;  // the context's only once it is whole
    if ((s = dev_alloc(c, &tab, (sizeof(int4) + sizeof(int)) * wg.size()))) return s;
    hipError_t e = hipMemcpyAsync(tab, wg.data(), sizeof(int4) * wg.size(),
                                  hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync((int4 *)tab + wg.size(), seg.data(), sizeof(int) * seg.size(),
                         hipMemcpyHostToDevice, c->stream);
    const hipError_t es = hipStreamSynchronize(c->stream);
    if (e != hipSuccess || es != hipSuccess) {
      (void)hipFree(tab);
      HIP_TRY(c, e);
      HIP_TRY(c, es);
    }
    c->pcg_segwg = tab;
  }
  k_pcg_reset<<<1, PCG_NCTR, 0, c->stream>>>(c->pcg_ctr, c->pcg_abort);
  HIP_TRY(c, hipGetLastError());
  P64Args a;
  if ((s = p64_args(c, nb, pcg_bar(c), a))) return s;
  a.wg = (const int4 *)c->pcg_segwg;
  a.wgseg = (const int *)(a.wg + nb);
  a.segst = c->d_segst;
  a.xsave = c->r;  // (the launches' residual, which every solve of theirs writes first)
  TIMED(c, TK_PCG64, s = coop_launch(c, pseg_kernel(cpt), nb, a));
  if (s) return s;
  HIP_TRY(c, hipMemcpyAsync(c->h_segst, c->d_segst, sizeof(CgState) * c->nseg,
                            hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(c, hipMemcpyAsync(c->st_host, c->st, sizeof(CgState), hipMemcpyDeviceToHost,
                            c->stream));
  HIP_TRY(c, hipStreamSynchronize(c->stream));
  if (!c->st_host->pabort) return EFDC_OK;
  if (!c->pcg_last_plain) {
    c->err = "persistent CG: an exchange between workgroups timed out";
    return EFDC_ERR_HIP;
  }
  // not co-resident: again, cooperatively, from the P of the first launch
  // (some basins may have finished), so that every basin's bits stay its own
  HIP_TRY(c, hipMemcpyAsync(c->dH[EFDC_P] + 1, c->r + 1, sizeof(double) * c->n_wet(),
                            hipMemcpyDeviceToDevice, c->stream));
  ++c->pcg_retries;
  c->pcg_force_coop = true;
  s = pcg_seg_solve(c);
  c->pcg_force_coop = false;
  return s;
}

// Autotuner of the mixed persistent solve: the degree of the local
// preconditioner.  The solve is repeated from the same P for every
// candidate (timed with events), P is restored, and the fastest degree is
// kept for the following solves; the caller then solves once more.
int pcg_tune_degree(efdc_ctx *c) {
  int s;
  if (!c->tune_pbuf && (s = dev_alloc(c, (void **)&c->tune_pbuf, sizeof(double) * c->LCM)))
    return s;
  HIP_TRY(c, hipMemcpyAsync(c->tune_pbuf, c->dH[EFDC_P], sizeof(double) * c->LCM,
                            hipMemcpyDeviceToDevice, c->stream));
  hipEvent_t e0 = timer_event(c), e1 = timer_event(c);
  const int cand[5] = {1, 2, 3, 4, 6};
  float best_ms = 1e30f;
  int best = PCG_PDEG_DEFAULT, best_slot = -1;
  // the degrees are timed in the Chronopoulos-Gear form when the caller
  // leaves the form to the tuner
  // (past 8 cells per thread there is only the pipelined one)
  int tnb = 0;
  const bool forms = c->pcg_pipe_mode == 0 && pcg_shape_mx(c, tnb) <= PCGMX_CPT_SMALL;
  if (forms) c->pcg_pipe_tuned = false;
  for (int j = 0; j < 5; ++j) {
    c->pcg_pdeg_tuned = cand[j];
    float tot = 0.f;
    for (int r = 0; r < 3; ++r) {
      HIP_TRY(c, hipMemcpyAsync(c->dH[EFDC_P], c->tune_pbuf, sizeof(double) * c->LCM,
                                hipMemcpyDeviceToDevice, c->stream));
      HIP_TRY(c, hipEventRecord(e0, c->stream));
      if ((s = pcg_solve(c, true))) return s;
      HIP_TRY(c, hipEventRecord(e1, c->stream));
      HIP_TRY(c, hipEventSynchronize(e1));
      float ms = 0.f;
      HIP_TRY(c, hipEventElapsedTime(&ms, e0, e1));
      if (r > 0) tot += ms;  // the first solve is a warm-up
    }
    const float avg = tot / 2.f;
    if (c->tune_n < 8) {
      std::snprintf(c->tune_name[c->tune_n], 32, "pcg_mixed degree=%d", cand[j]);
      c->tune_ms[c->tune_n] = avg;
      ++c->tune_n;
    }
    if (avg < best_ms) {
      best_ms = avg;
      best = cand[j];
      best_slot = c->tune_n - 1;
    }
  }
  c->pcg_pdeg_tuned = best;
  // the pipelined form at that degree, when the caller leaves the choice
  if (forms) {
    c->pcg_pipe_tuned = true;
    float tot = 0.f;
    for (int r = 0; r < 3; ++r) {
      HIP_TRY(c, hipMemcpyAsync(c->dH[EFDC_P], c->tune_pbuf, sizeof(double) * c->LCM,
                                hipMemcpyDeviceToDevice, c->stream));
      HIP_TRY(c, hipEventRecord(e0, c->stream));
      if ((s = pcg_solve(c, true))) return s;
      HIP_TRY(c, hipEventRecord(e1, c->stream));
      HIP_TRY(c, hipEventSynchronize(e1));
      float ms = 0.f;
      HIP_TRY(c, hipEventElapsedTime(&ms, e0, e1));
      if (r > 0) tot += ms;
    }
    const float avg = tot / 2.f;
    c->pcg_pipe_tuned = avg < best_ms;
    if (c->tune_n < 8) {
      std::snprintf(c->tune_name[c->tune_n], 32, "pcg_mixed pipelined d=%d", best);
      c->tune_ms[c->tune_n] = avg;
      ++c->tune_n;
      if (c->pcg_pipe_tuned) best_slot = c->tune_n - 1;
    }
  }
  if (best_slot >= 0 && best_slot < 8) c->tune_chosen[best_slot] = 1;
  c->ev_pool.push_back(e0);
  c->ev_pool.push_back(e1);
  HIP_TRY(c, hipMemcpyAsync(c->dH[EFDC_P], c->tune_pbuf, sizeof(double) * c->LCM,
                            hipMemcpyDeviceToDevice, c->stream));
  return EFDC_OK;
}
