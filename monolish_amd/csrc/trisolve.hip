// trisolve.hip -- triangular sweeps: the SOR sweeps
// (src/equation/kernel/sor_kernel.hpp:5-73) and the IC / ILU triangular
// solves (csrsv2 in kernel/ic_kernel.hpp, ilu_kernel.hpp).
//
// Every such sweep has one form: out_i = fin(init_i - sum_d coef_d *
// out_{col_d}), the sum over the row's dependency entries in the row's
// storage order.  Each row does the serial loop's arithmetic in its order,
// so the result is bit-identical to the serial sweep.
//
// A sweep is one serial chain of rows as long as the matrix has levels
// (level of a row = 1 + the largest level of the rows it reads), so what
// bounds it is the time from one row's value to the row that reads it, not
// bandwidth: 2D Poisson 256^2 has 511 levels, 27-point 96^3 has 666.  The
// plan therefore keeps that step inside one wave or one workgroup wherever
// it can.  Rows are cut into chunks of consecutive rows in sweep order, one
// workgroup each, and a chunk into the ranges of its kChWaves waves:
//  - a wave runs its rows by level, the rows of a level side by side, with
//    no barrier: its own values come back through LDS in program order;
//  - a value of another wave of the chunk is read from LDS too, where a
//    marker (a signalling NaN) says that it is not there yet;
//  - a value of an earlier chunk is loaded from global memory ahead of its
//    first use and kept in a ring of the wave in LDS.
// Chunks are taken in sweep order and read only earlier ones, so they are
// done or running: the sweep cannot deadlock, however few workgroups run.
//
// A wave runs alone on its SIMD, so a level costs its instructions (about
// five clocks each) and one LDS round trip of 64 clocks, and the four waves
// share one vector memory unit (16 clocks a load).  The plan is therefore
// laid out in batches of up to 64 rows of several levels, one row per lane:
// a batch is loaded once, a few batches ahead, and each of its levels only
// reads its values from LDS, adds and writes.  Rows are filled up to D
// entries with coefficient 0 and a slot that holds 0 (x - 0 * 0 is x, bit
// for bit, but for a signalling NaN, which turns quiet: no row ever equals
// the marker); a row of more than D entries takes several batches.  A
// missing value shows as a NaN in the sum, so levels that miss nothing
// compare nothing else.
#include <algorithm>
#include <functional>
#include <future>
#include <vector>

#include "mgx_device.hpp"
#include "mgx_sweep.hpp"

namespace mgx {

namespace {

constexpr int kChWaves = 4;      // one per SIMD
constexpr int kRing = 1024;      // values of earlier chunks that a wave keeps
// Rows of a wave.  Narrow levels (2D grids): long ranges, so that the chain
// crosses few chunks.  Levels of kWideLevel rows on average or more (3D
// grids): short ranges, so that a level's rows spread over the chip.  Per
// SOR-PCG iteration, FP64, with 2048 / 1024 / 256 rows: 2D 5-point 256^2
// (128 rows a level) 0.37 / 0.40 / 0.42 ms, 1000^2 (500) 1.46 / 1.43 / 2.57
// ms; 3D 27-point 96^3 (1328) 2.06 / 1.87 / 1.68 ms, 128^3 (2356) 2.86 /
// 2.58 / 2.36 ms, 7-point 100^3 (3356) 0.95 / 0.82 / 0.77 ms.
constexpr int kWaveRows = 2048, kWaveRowsWide = 256, kWideLevel = 1000;
// Matrices whose rows read scattered rows gain less from chunks, or lose: the
// chain then crosses a chunk at almost every level, and a batch is cut short
// by the values of earlier chunks that it takes.  model_share runs the
// schedule of kModelRows rows from the middle, with what a batch, a level and
// a value's way measured, and sets it against kFlowLevelUs for each level of
// those rows, what one costs in the dependency-driven form: grids come to
// 0.09-0.2 of it, rows that read random rows of a band to 0.33-1.1, of the
// whole matrix to 1.4 and more.  From kScattered on a wave gets few rows, from
// kFlowBetter on the dependency-driven form runs where there are kFlowRows
// rows, kFlowMinWidth a level on average, and kFlowMinLevels levels (with
// fewer the entries take longer than the chain).  Per SOR-PCG iteration, FP64,
// in us, with 2048 / 256 / 64 rows a wave / dependency-driven:
//   band of 1000, 300000 rows (74 a level), share 0.33-0.43
//                                            11403 / 12522 / 24084 / 26392
//   band of 3000, 20000 rows (290), 0.75         567 / 516 / 500 / 565
//   band of 5000, 50000 rows (485), 1.0         1146 / 884 / 884 / 789
//   band of 5000, 200000 rows (350), 0.6-0.8   5464 / 4558 / 7150 / 4386
//   M-matrix, 20000 rows (400), 1.4             1371 / 700 / 560 / 559
//   M-matrix, 130000 rows (2321), 1.7          2987 / 1007 / 1254 / 696
//   M-matrix of 60 entries a row, 20000 rows (136), 3.9
//                                              4706 / 2651 / 1799 / 2078
//   5-point 700^2, rows permuted (13 levels), 1.0   501 / 352 / 482 / 426
constexpr int kWaveRowsScattered = 64;
constexpr int64_t kModelRows = 4096, kFlowRows = 32768, kFlowMinWidth = 256;
constexpr int kFlowMinLevels = 32;
constexpr double kScattered = 0.42, kFlowBetter = 0.6, kFlowLevelUs = 3.6;
// a batch, a level (and each of its entries' width), a value from an earlier
// chunk and from another wave of the chunk, in us
constexpr double kBatchUs = 0.73, kLevelUs = 0.11, kEntryUs = 0.023, kFarUs = 2.8, kNearUs = 0.09;
constexpr uint64_t kSpinTicks = 200000000;  // 2 s of the 100 MHz clock without progress
// 10 ms: a longer gap between two looks at the clock counts as this (nothing
// ran in it: the process was taken off the device)
constexpr uint64_t kSpinGap = 1000000;

// batch header: x, y = lanes whose row starts a level, z = rows | values of
// earlier chunks << 8 | kPart... (a batch with part of its rows' entries:
// one level, the sums go on in the next batch or come from the last)
constexpr uint32_t kPartFirst = 1u << 20, kPartMid = 1u << 21, kPartLast = 1u << 22;
// LDS slots: the chunk's crows values, the waves' rings, one slot that
// holds 0; then the ticket
constexpr uint32_t slot_zero(uint32_t crows) { return crows + kChWaves * kRing; }
static_assert(slot_zero(kChWaves * kWaveRows) < 65536, "slots are stored in 16 bits");

template <class T> struct SweepBits;
template <> struct SweepBits<double> {
  using U = uint64_t;
  static constexpr U kEmpty = 0x7ff0deadbeef0001ull, kNan = 0x7ff8000000000000ull;
};
template <> struct SweepBits<float> {
  using U = uint32_t;
  static constexpr U kEmpty = 0x7f80dea1u, kNan = 0x7fc00000u;
};

template <class T> struct TriArgs {
  int64_t n;
  int32_t crows, nchunk, rev;  // rows per chunk, chunks, sweep from the last row
  const int64_t *wave;
  const int4 *hdr;
  const int32_t *row, *ext;
  const uint16_t *slot;
  const T *coef, *isc;
  T *out;
  uint32_t *ticket;
};

// isc[2k] = the initial value of row[k] (out for the SOR backward sweep, in
// otherwise), then out of that row = kEmpty, a signalling NaN that no
// arithmetic produces; in may alias out
template <class T, int FIN>
__global__ __launch_bounds__(kBlock) void k_tri_init(int64_t n, const int32_t *__restrict__ row,
                                                     const T *in, T *out, T *isc,
                                                     uint32_t *ticket) {
  using U = typename SweepBits<T>::U;
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k == 0) *ticket = 0u;
  if (k < n) {
    const int32_t i = row[k];
    isc[2 * k] = FIN == 1 ? out[i] : in[i];
    reinterpret_cast<U *>(out)[i] = SweepBits<T>::kEmpty;
  }
}

// A wave waiting for values: true when nothing in the whole sweep has
// progressed for kSpinTicks (ticket[2] counts steps done, in groups); the
// wave then gives up (its rows become NaN) and ticket[1] makes the solver
// return MGX_ERR_TIMEOUT, so every wait ends.
struct SpinWatch {
  uint64_t last = 0, waited = 0;
  uint32_t seen = 0, spins = 0;
  __device__ __forceinline__ bool give_up(uint32_t *ticket) {
    if (__builtin_expect((++spins & 255u) != 0, 1)) return false;
    const uint32_t p = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)__hip_atomic_load(ticket + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    const uint64_t now = wall_clock64();
    const bool moved = spins == 256u || p != seen;
    waited = moved ? 0 : waited + min(now - last, kSpinGap);
    last = now;
    seen = p;
    if (moved) return false;
    if (waited <= kSpinTicks &&
        __hip_atomic_load(ticket + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
      return false;
    __hip_atomic_store(ticket + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  }
};

// plan data at a uniform address, by scalar loads: they don't queue behind
// the vector loads in flight
template <class V> __device__ __forceinline__ V scalar_get(const void *p, int64_t i) {
  typedef const __attribute__((address_space(4))) V CV;
  return ((CV *)p)[i];
}

// Entries per row and batch D (even): batches loaded ahead, registers of 64
// values of earlier chunks per batch, slots stored per lane and load
template <int D> struct Width {
  static constexpr int kAhead = D <= 4 ? 4 : 3, kFar = D <= 4 ? 1 : 3;
  static constexpr int kSlotLoad = D < 8 ? D : 8, kSlotLoads = (D + kSlotLoad - 1) / kSlotLoad;
  static constexpr int kSlots = kSlotLoad * kSlotLoads;
};

// one batch's data, in registers from kAhead batches before it runs
template <class T, int D> struct BatchRegs {
  T coef[D], init, sc;
  uint32_t slot[Width<D>::kSlots / 2];
  int32_t row, col[Width<D>::kFar];
  typename SweepBits<T>::U ext[Width<D>::kFar];
};

// FIN 0: out = acc * sc (SOR forward); 1: SOR backward, acc in double from
// 0, out = (T)((double)out - acc * (double)sc); 2: out = acc / sc; 3: out = acc
template <class T, int FIN, int D>
__global__ __launch_bounds__(64 * kChWaves) void k_tri_chunk(const TriArgs<T> a) {
  using U = typename SweepBits<T>::U;
  using Acc = typename std::conditional<FIN == 1, double, T>::type;
  using W = Width<D>;
  typedef int32_t I4 __attribute__((ext_vector_type(4)));
  typedef T V2 __attribute__((ext_vector_type(2)));
  typedef uint32_t SV __attribute__((ext_vector_type(W::kSlotLoad < 4 ? 2 : W::kSlotLoad / 2)));
  constexpr U kEmpty = SweepBits<T>::kEmpty;
  constexpr int P = W::kAhead, X = W::kFar, SL = W::kSlotLoad;
  extern __shared__ __align__(16) unsigned char tri_lds[];
  U *const s_val = reinterpret_cast<U *>(tri_lds);
  const uint32_t zero = slot_zero((uint32_t)a.crows);
  uint32_t *const s_ticket = reinterpret_cast<uint32_t *>(s_val + zero + 1);
  const uint32_t lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  U *const ob = reinterpret_cast<U *>(a.out);
  U *const ring = s_val + a.crows + w * kRing;
  auto lds_at = [&](uint32_t byte) -> U * { return reinterpret_cast<U *>(tri_lds + byte); };
  auto lds_get = [&](uint32_t byte) -> U {
    return __hip_atomic_load(lds_at(byte), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto far_get = [&](int32_t row) -> U {
    return __hip_atomic_load(ob + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (threadIdx.x == 0) s_val[zero] = (U)0;
  for (;;) {
    if (threadIdx.x == 0)
      *s_ticket =
          __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int i = (int)threadIdx.x; i < a.crows; i += 64 * kChWaves) s_val[i] = kEmpty;
    __syncthreads();
    const int32_t ch = __builtin_amdgcn_readfirstlane((int)*s_ticket);
    if (ch >= a.nchunk) break;
    // LDS slot of row i: its sweep position (i, or n - 1 - i) less the
    // chunk's first, as (i ^ flip) + off
    const uint32_t flip = a.rev ? ~0u : 0u;
    const uint32_t off = (a.rev ? (uint32_t)a.n : 0u) - (uint32_t)(ch * a.crows);
    const int64_t *const wv = a.wave + ((int64_t)ch * kChWaves + w) * 4;
    const int64_t s0 = scalar_get<int64_t>(wv, 0), s1 = scalar_get<int64_t>(wv, 4);
    int64_t le = scalar_get<int64_t>(wv, 1), lr = scalar_get<int64_t>(wv, 2),
            lx = scalar_get<int64_t>(wv, 3);
    uint32_t xpos = 0;  // values of earlier chunks taken so far
    BatchRegs<T, D> R[P];
    I4 h[P];
    auto load = [&](BatchRegs<T, D> &r, const I4 hd) {
      const uint32_t m = hd.z & 127u;
      // le counts rows: D coefficients (pairs of all rows, then the next
      // pairs) and kSlots slots each
      const V2 *cp = reinterpret_cast<const V2 *>(a.coef + le * D);
#pragma unroll
      for (int u = 0; u < D; u += 2, cp += m) {
        const V2 c2 = cp[lane];
        r.coef[u] = c2[0];
        r.coef[u + 1] = c2[1];
      }
      const uint32_t *sp = reinterpret_cast<const uint32_t *>(a.slot + le * W::kSlots);
#pragma unroll
      for (int g = 0; g < W::kSlotLoads; g++, sp += m * (SL / 2)) {
        if constexpr (SL == 2) {
          r.slot[g] = sp[lane];
        } else {
          const SV sv = reinterpret_cast<const SV *>(sp)[lane];
#pragma unroll
          for (int q = 0; q < SL / 2; q++) r.slot[g * (SL / 2) + q] = sv[q];
        }
      }
      const V2 is = reinterpret_cast<const V2 *>(a.isc + 2 * lr)[lane];
      r.init = is[0];
      r.sc = is[1];
      r.row = (a.row + lr)[lane];
#pragma unroll
      for (int q = 0; q < X; q++) r.col[q] = (a.ext + lx + 64 * q)[lane];
      le += m;
      lr += (hd.z & kPartLast) || !(hd.z & (kPartFirst | kPartLast | kPartMid)) ? m : 0u;
      lx += (hd.z >> 8) & 1023u;
    };
    auto far_load = [&](BatchRegs<T, D> &r, const I4 hd) {
      if ((hd.z >> 8) & 1023u) {
#pragma unroll
        for (int q = 0; q < X; q++) r.ext[q] = far_get(r.col[q]);
      }
    };
    if (s0 < s1) {
#pragma unroll
      for (int k = 0; k < P; k++) {
        h[k] = scalar_get<I4>(a.hdr, s0 + k);
        load(R[k], h[k]);
      }
      far_load(R[0], h[0]);
    }
    Acc carry = (Acc)0;
    for (int64_t s = s0; s < s1; s += P) {
#pragma unroll
      for (int k = 0; k < P; k++) {
        BatchRegs<T, D> &r = R[k];
        BatchRegs<T, D> &rn = R[(k + 1) % P];
        const I4 hd = h[k];
        const I4 hn = scalar_get<I4>(a.hdr, s + P + k);
        far_load(rn, h[(k + 1) % P]);
        const uint32_t m = hd.z & 127u, ne = (hd.z >> 8) & 1023u;
        // values that are not there yet go into the ring as the marker
        auto take = [&]() {
#pragma unroll
          for (int q = 0; q < X; q++)
            if (64 * q + lane < ne) ring[(xpos + 64 * q + lane) & (kRing - 1)] = r.ext[q];
          asm volatile("" ::: "memory");
        };
        if (ne) take();
        if (ne && m == 0) {
          // (no row of this batch will look again: wait here)
          SpinWatch sw;
          for (;;) {
            bool miss = false;
#pragma unroll
            for (int q = 0; q < X; q++) miss = miss || (64 * q + lane < ne && r.ext[q] == kEmpty);
            if (!__any(miss) || sw.give_up(a.ticket)) break;
#pragma unroll
            for (int q = 0; q < X; q++) r.ext[q] = far_get(r.col[q]);
          }
          take();
        }
        // the level of the lane's row in this batch, its values' and its own
        // place in LDS
        const uint64_t starts = (uint64_t)(uint32_t)hd.y << 32 | (uint32_t)hd.x;
        const int levels = __popcll(starts);
        int my = (int)__builtin_amdgcn_mbcnt_hi(
            (uint32_t)hd.y, __builtin_amdgcn_mbcnt_lo((uint32_t)hd.x, 0u));
        my += (int)((starts >> lane) & 1u) - 1;
        if (lane >= m) my = -1;
        uint32_t from[D];
#pragma unroll
        for (int u = 0; u < D; u++)
          from[u] = (u & 1 ? r.slot[u / 2] >> 16 : r.slot[u / 2] & 0xffffu) * (uint32_t)sizeof(U);
        U *const to = lds_at((((uint32_t)r.row ^ flip) + off) * (uint32_t)sizeof(U));
        U *const out = ob + r.row;
        const bool part = (hd.z & (kPartFirst | kPartMid | kPartLast)) != 0;
        Acc begin = FIN == 1 ? (Acc)0 : (Acc)r.init;
        if (part && !(hd.z & kPartFirst)) begin = carry;
        const bool last = !part || (hd.z & kPartLast);
        for (int j = 0; j < levels; j++) {
          Acc acc = begin;
          U z[D];
          auto sum = [&]() {
#pragma unroll
            for (int u = 0; u < D; u++) z[u] = lds_get(from[u]);
            acc = begin;
#pragma unroll
            for (int u = 0; u < D; u++) {
              const T p = r.coef[u] * __builtin_bit_cast(T, z[u]);
              if (FIN == 1)
                acc = acc + (double)p;
              else
                acc = acc - p;
            }
          };
          bool odd = false;
          if (my == j) {
            sum();
            odd = acc != acc;
          }
          if (__builtin_expect(__any(odd), 0)) {
            // a value that another wave of the chunk has not written yet, or
            // that an earlier chunk had not when it was asked for; or a NaN
            SpinWatch sw;
            for (;;) {
              if (ne) {
#pragma unroll
                for (int q = 0; q < X; q++) r.ext[q] = far_get(r.col[q]);
                take();
              }
              bool miss = false;
              if (my == j) {
                sum();
#pragma unroll
                for (int u = 0; u < D; u++) miss = miss || z[u] == kEmpty;
              }
              if (!__any(miss) || sw.give_up(a.ticket)) break;  // (the marker: a NaN row)
            }
          }
          if (my == j) {
            if (last) {
              T v;
              if (FIN == 0)
                v = acc * r.sc;
              else if (FIN == 1)
                v = (T)((double)r.init - acc * (double)r.sc);
              else if (FIN == 2)
                v = acc / r.sc;
              else
                v = acc;
              const U vb = __builtin_bit_cast(U, v);
              __hip_atomic_store(to, vb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              __hip_atomic_store(out, vb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
              carry = acc;
            }
          }
          asm volatile("" ::: "memory");  // the wave's next level reads these values
        }
        xpos += ne;
        h[k] = hn;
        load(r, hn);
      }
      if (lane == 0)
        __hip_atomic_fetch_add(a.ticket + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();  // the chunk's values are cleared next
  }
}

// The dependency-driven form, for matrices whose rows read scattered rows
// (kFlowBetter): hardly any dependency stays inside a chunk there, and what
// bounds the sweep is the number of values fetched. Persistent waves take 64
// consecutive level-order positions at a time from a ticket counter and each
// lane computes its row as soon as the rows it reads are written.  A lane
// loads its entries eight at a time (plain loads) and consumes them strictly
// in the row's order; at the first one still kEmpty it polls that one entry
// with a device-coherent atomic read (a plain load may keep seeing a cached
// copy) until it is written, then goes on, so the arithmetic is the serial
// sweep's. Rows only read rows of earlier levels, which sit at earlier
// positions, so their tickets were taken by waves that are already running:
// the sweep cannot deadlock.  A lane that has consumed none of its row's
// entries for kSpinTicks gives up: it publishes NaN and raises the plan's
// stall flag (ticket[1]), so the kernel always ends and the solver returns
// MGX_ERR_TIMEOUT. At most 1024 waves x 64 rows are in flight, so a valid
// plan's longest wait is 65536 dependency hops (measured 4-7 us each), far
// inside the 2 s limit.
constexpr int kFlowThreads = 256;
constexpr int kFlowBlocks = 256;
constexpr int kTriChunk = 8;

template <class T, int FIN>
__global__ __launch_bounds__(kFlowThreads) void k_tri_flow(
    int32_t n, const int4 *__restrict__ rec, const int32_t *__restrict__ dcol,
    const T *__restrict__ dcoef, const T *__restrict__ isc, T *out, uint32_t *ticket) {
  using U = typename SweepBits<T>::U;
  using Acc = typename std::conditional<FIN == 1, double, T>::type;
  U *ob = reinterpret_cast<U *>(out);
  const int lane = (int)(threadIdx.x & 63);
  const uint32_t nchunk = (uint32_t)((n + 63) / 64);
  for (;;) {
    uint32_t t = 0;
    if (lane == 0)
      t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t = (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
    if (t >= nchunk) break;
    const int32_t k = (int32_t)(t * 64u) + lane;
    const bool has = k < n;
    const int4 rc = has ? rec[k] : make_int4(0, 0, 0, 0);
    int32_t d = rc.y;
    const int32_t d1 = has ? rc.z : rc.y;
    const T init = has ? isc[2 * (int64_t)k] : (T)0;
    Acc acc = FIN == 1 ? (Acc)0 : (Acc)init;
    uint64_t last = wall_clock64(), waited = 0;  // since the lane's last progress
    int32_t wc = -1;  // >= 0: column of entry d, which was still kEmpty
    T wa = (T)0;
    // a lane publishes its row as soon as its last entry is consumed: a row
    // later in the same 64 may read it
    bool pending = has;
    while (__any(pending)) {
      if (pending && d < d1) {
        if (wc >= 0) {
          const U z = __hip_atomic_fetch_or(ob + wc, (U)0, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
          if (z != SweepBits<T>::kEmpty) {
            const T p = wa * __builtin_bit_cast(T, z);
            if (FIN == 1)
              acc = acc + (double)p;
            else
              acc = acc - p;
            d++;
            wc = -1;
            waited = 0;
          }
        } else {
          int32_t c[kTriChunk];
          T a[kTriChunk];
          U zb[kTriChunk];
#pragma unroll
          for (int u = 0; u < kTriChunk; u++) {
            const int32_t e = d + u < d1 ? d + u : d;
            c[u] = dcol[e];
            a[u] = dcoef[e];
          }
#pragma unroll
          // plain loads: out held kEmpty when this kernel started (k_tri_init,
          // an earlier kernel of the stream) and changes once, to the final
          // value, so a cached copy is either that value or a stale kEmpty,
          // which the device-coherent poll below resolves
          for (int u = 0; u < kTriChunk; u++) zb[u] = d + u < d1 ? ob[c[u]] : (U)0;
          bool stop = false;
          int32_t taken = 0;
#pragma unroll
          for (int u = 0; u < kTriChunk; u++) {
            if (!stop && d + u < d1) {
              if (zb[u] == SweepBits<T>::kEmpty) {
                stop = true;
                wc = c[u];
                wa = a[u];
              } else {
                const T p = a[u] * __builtin_bit_cast(T, zb[u]);
                if (FIN == 1)
                  acc = acc + (double)p;
                else
                  acc = acc - p;
                taken++;
              }
            }
          }
          d += taken;
          if (taken > 0) waited = 0;
        }
        const uint64_t now = wall_clock64();
        waited += min(now - last, kSpinGap);
        last = now;
        if (d < d1 && wc >= 0 && waited > kSpinTicks) {
          acc = (Acc)__builtin_bit_cast(T, SweepBits<T>::kNan);
          d = d1;
          __hip_atomic_store(ticket + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (pending && d >= d1) {
        const T s = isc[2 * (int64_t)k + 1];
        T v;
        if (FIN == 0)
          v = acc * s;
        else if (FIN == 1)
          v = (T)((double)init - acc * (double)s);
        else if (FIN == 2)
          v = acc / s;
        else
          v = acc;
        U vb = __builtin_bit_cast(U, v);
        if (vb == SweepBits<T>::kEmpty) vb = SweepBits<T>::kNan;
        __hip_atomic_exchange(ob + rc.x, vb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        pending = false;
      }
      if (__any(pending && wc >= 0)) __builtin_amdgcn_s_sleep(2);
    }
  }
}

// coef[d] = vals[dent[d]], 0 where the plan has no entry
template <class T>
__global__ __launch_bounds__(kBlock) void k_tri_pack(int64_t nd, const int32_t *__restrict__ dent,
                                                     const T *__restrict__ vals, T *coef) {
  const int64_t d = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (d < nd) coef[d] = dent[d] < 0 ? (T)0 : vals[dent[d]];
}

// isc[2k + 1] = vec[pos ? pos[row[k]] : row[k]]
template <class T>
__global__ __launch_bounds__(kBlock) void k_tri_scale(int64_t n, const int32_t *__restrict__ row,
                                                      const T *__restrict__ vec,
                                                      const int32_t *__restrict__ pos, T *isc) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k < n) {
    const int32_t i = row[k];
    isc[2 * k + 1] = vec[pos ? pos[i] : i];
  }
}

template <class T>
void tri_launch(Ctx *c, const TriPlan &P, void (*k)(TriArgs<T>), const TriArgs<T> &a) {
  const size_t lds = (slot_zero((uint32_t)P.crows) + 1) * sizeof(T) + 16;
  if (lds > 65536)
    MGX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  // small chunks: several workgroups share a compute unit
  const unsigned grid = (unsigned)std::min(P.nchunk, 4 * c->num_cus);
  k<<<grid, 64 * kChWaves, lds, c->stream>>>(a);
}

template <class T, int FIN>
void tri_run_t(Ctx *c, const TriOp &op, const T *in, T *out) {
  const TriPlan &P = *op.plan;
  if (P.n == 0) return;
  T *isc = static_cast<T *>(op.isc);
  k_tri_init<T, FIN><<<(unsigned)((P.n + kBlock - 1) / kBlock), kBlock, 0, c->stream>>>(
      P.n, P.d_row, in, out, isc, P.d_ticket);
  if (P.flow) {
    const int64_t want = (P.n + 63) / 64 / (kFlowThreads / 64) + 1;
    k_tri_flow<T, FIN><<<(unsigned)std::min<int64_t>(want, kFlowBlocks), kFlowThreads, 0,
                         c->stream>>>((int32_t)P.n, P.d_rec, P.d_dcol,
                                      static_cast<const T *>(op.coef), isc, out, P.d_ticket);
    MGX_HIP(hipGetLastError());
    return;
  }
  const TriArgs<T> a{P.n,     P.crows, P.nchunk, P.rev,
                     P.d_wave, P.d_hdr, P.d_row, P.d_ext, P.d_slot,
                     static_cast<const T *>(op.coef), isc, out,
                     P.d_ticket};
  if (P.width == 2)
    tri_launch(c, P, k_tri_chunk<T, FIN, 2>, a);
  else if (P.width == 4)
    tri_launch(c, P, k_tri_chunk<T, FIN, 4>, a);
  else if (P.width == 8)
    tri_launch(c, P, k_tri_chunk<T, FIN, 8>, a);
  else
    tri_launch(c, P, k_tri_chunk<T, FIN, 14>, a);
  MGX_HIP(hipGetLastError());
}

template <class T> void tri_run_fin(Ctx *c, const TriOp &op, const void *in, void *out) {
  const T *x = static_cast<const T *>(in);
  T *y = static_cast<T *>(out);
  switch (op.fin) {
    case kTriMul: tri_run_t<T, 0>(c, op, x, y); break;
    case kTriSorBack: tri_run_t<T, 1>(c, op, x, y); break;
    case kTriDiv: tri_run_t<T, 2>(c, op, x, y); break;
    default: tri_run_t<T, 3>(c, op, x, y); break;
  }
}

template <class V> V *upload(const std::vector<V> &h) {
  V *d = (V *)dev_alloc(std::max<size_t>(h.size(), 1) * sizeof(V));
  if (!h.empty()) MGX_HIP(hipMemcpy(d, h.data(), h.size() * sizeof(V), hipMemcpyHostToDevice));
  return d;
}

template <class P, class V> V *upload_parts(const std::vector<P> &parts, std::vector<V> P::*m) {
  size_t total = 0;
  for (const P &p : parts) total += (p.*m).size();
  V *d = (V *)dev_alloc(std::max<size_t>(total, 1) * sizeof(V));
  size_t o = 0;
  for (const P &p : parts) {
    const std::vector<V> &h = p.*m;
    if (!h.empty())
      MGX_HIP(hipMemcpy(d + o, h.data(), h.size() * sizeof(V), hipMemcpyHostToDevice));
    o += h.size();
  }
  return d;
}

struct WidthSizes {
  int ahead, far, slot_load, slots;
};
template <int D> WidthSizes width_sizes() {
  return {Width<D>::kAhead, Width<D>::kFar, Width<D>::kSlotLoad, Width<D>::kSlots};
}

// a batch without rows that takes the values of `rows`
void push_values(std::vector<int4> &hdr, std::vector<int32_t> &ext,
                 const std::vector<int32_t> &rows) {
  hdr.push_back(make_int4(0, 0, (int32_t)((uint32_t)rows.size() << 8 | kPartMid), 0));
  ext.insert(ext.end(), rows.begin(), rows.end());
}

bool dep_of(int filter, int64_t i, int32_t c) { return filter == 2 ? c > i : c < i; }

// the time of the sweep over positions [p0, p0 + pn) in chunks of kChWaves
// waves of srows rows (p0 a multiple of them), as a share of what the
// dependency-driven form takes for the levels of these rows.  for_reads(p, f)
// calls f with each position that position p reads (values from before p0
// are there); lev and cnt by position
template <class Lev, class Cnt, class Reads>
double model_share(int64_t n, int64_t p0, int64_t pn, int64_t srows, int D, int maxnew, Lev lev,
                   Cnt cnt, Reads for_reads) {
  std::vector<int32_t> depth(pn, 0), stamp(n, -1);
  int32_t levels = 1;
  for (int64_t p = p0; p < p0 + pn; p++) {
    int32_t d = 0;
    for_reads(p, [&](int64_t q) { if (q >= p0) d = std::max(d, depth[q - p0] + 1); });
    depth[p - p0] = d;
    levels = std::max(levels, d + 1);
  }
  std::vector<double> done(pn, 0.0);
  std::vector<int64_t> ord;
  double end = 0;
  int32_t v = 0;
  for (int64_t a = p0; a < p0 + pn; a += srows, v++) {
    const int64_t b = std::min(a + srows, p0 + pn), base = a - v % kChWaves * srows;
    ord.resize(b - a);
    for (int64_t p = a; p < b; p++) ord[p - a] = p;
    std::stable_sort(ord.begin(), ord.end(), [&](int64_t x, int64_t y) {
      return std::make_pair(lev(x), std::max(cnt(x), D)) < std::make_pair(lev(y), std::max(cnt(y), D));
    });
    double now = 0;
    for (size_t k = 0; k < ord.size();) {
      const bool lng = cnt(ord[k]) > D;
      size_t e = k;
      int fresh = 0, longest = 0;
      while (e < ord.size() && e - k < 64) {
        const int64_t p = ord[e];
        if ((cnt(p) > D) != lng || (lng && lev(p) != lev(ord[k]))) break;
        int news = 0;
        for_reads(p, [&](int64_t q) { news += q < base && stamp[q] != v; });
        if (e > k && fresh + news > maxnew) break;
        for_reads(p, [&](int64_t q) { if (q < base) stamp[q] = v; });
        fresh += news;
        longest = std::max(longest, cnt(p));
        e++;
      }
      const int parts = std::max(1, (longest + D - 1) / D);
      now += kBatchUs * parts;
      while (k < e) {
        const int32_t l = lev(ord[k]);
        const size_t k0 = k;
        double in = 0;
        for (; k < e && lev(ord[k]) == l; k++)
          for_reads(ord[k], [&](int64_t q) {
            if (q >= p0 && q < a) in = std::max(in, done[q - p0] + (q < base ? kFarUs : kNearUs));
          });
        now = std::max(now, in) + (kLevelUs + kEntryUs * D) * parts;
        for (size_t u = k0; u < k; u++) done[ord[u] - p0] = now;
      }
    }
    end = std::max(end, now);
  }
  return end / (kFlowLevelUs * levels);
}

}  // namespace

static void plan_free(TriPlan &P) {
  levels_free(P.lev);
  dev_free(P.d_hdr);
  dev_free(P.d_rec);
  dev_free(P.d_dcol);
  dev_free(P.d_slot);
  dev_free(P.d_dent);
  dev_free(P.d_ext);
  dev_free(P.d_row);
  dev_free(P.d_wave);
  dev_free(P.d_ticket);
  P = TriPlan();
}

void build_tri_plan(const std::vector<int32_t> &ptr, const std::vector<int32_t> &col,
                    const std::vector<int32_t> *ent, int64_t n, int filter, TriPlan &P) {
  plan_free(P);  // (what a build that ran out of memory left)
  // dependency entries of each row, in the row's order (filter 1 stops at
  // the first entry that is not left of the diagonal)
  std::vector<int32_t> cnt(n, 0), lev(n, 0);
  int32_t nlev = 0;
  auto for_deps = [&](int64_t i, auto &&f) {
    for (int32_t j = ptr[i]; j < ptr[i + 1]; j++) {
      if (dep_of(filter, i, col[j]))
        f(j);
      else if (filter == 1)
        break;
    }
  };
  if (filter == 2) {
    for (int64_t i = n - 1; i >= 0; i--) {
      int32_t l = 0;
      for_deps(i, [&](int32_t j) { l = std::max(l, lev[col[j]] + 1), cnt[i]++; });
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  } else {
    for (int64_t i = 0; i < n; i++) {
      int32_t l = 0;
      for_deps(i, [&](int32_t j) { l = std::max(l, lev[col[j]] + 1), cnt[i]++; });
      lev[i] = l;
      nlev = std::max(nlev, l + 1);
    }
  }
  SorLevels &L = P.lev;
  L.ptr.assign(nlev + 1, 0);
  for (int64_t i = 0; i < n; i++) L.ptr[lev[i] + 1]++;
  for (int32_t l = 0; l < nlev; l++) L.ptr[l + 1] += L.ptr[l];
  std::vector<int32_t> pos(L.ptr.begin(), L.ptr.end() - 1), rows(n);
  for (int64_t i = 0; i < n; i++) rows[pos[lev[i]]++] = (int32_t)i;
  L.nlev = nlev;
  L.max_width = 0;
  for (int32_t l = 0; l < nlev; l++) L.max_width = std::max(L.max_width, L.ptr[l + 1] - L.ptr[l]);
  P.n = n;
  P.rev = filter == 2;
  auto at = [&](int64_t i) { return P.rev ? n - 1 - i : i; };  // sweep position of row i
  // entries per row and batch: the smallest width that takes 98 % of the rows
  // in one batch (2, 3 and 13 entries on 5-, 7- and 27-point grids), a larger
  // one where the longest row is the longer chain, in batches, than the
  // levels: a wider level costs little then (diagonal, last row and last
  // column, 100000 rows: 25.3 / 13.3 / 10.3 / 7.7 ms an iteration of SOR-PCG
  // with 2 / 4 / 8 / 14)
  {
    const int widths[4] = {2, 4, 8, 14};
    int64_t over[4] = {0, 0, 0, 0};
    int32_t longest = 0;
    for (int64_t i = 0; i < n; i++) {
      for (int q = 0; q < 4; q++) over[q] += cnt[i] > widths[q];
      longest = std::max(longest, cnt[i]);
    }
    int q = 0;
    while (q < 3 && over[q] * 50 > n) q++;
    double least = 0;
    for (int u = q; u < 4; u++) {
      const double level = kLevelUs + kEntryUs * widths[u];
      const double us = nlev * level + (longest / widths[u]) * (kBatchUs + level);
      if (u == q || us < least) {
        least = us;
        P.width = widths[u];
      }
    }
  }
  const int D = P.width;
  const WidthSizes wd = D == 2   ? width_sizes<2>()
                        : D == 4 ? width_sizes<4>()
                        : D == 8 ? width_sizes<8>()
                                 : width_sizes<14>();
  const int maxnew = 64 * wd.far;
  double share = 0;  // (more than a chunk's rows, or nothing is handed over)
  if (n > kChWaves * kWaveRows) {
    const int64_t pn = std::min(n, kModelRows), span = kChWaves * kWaveRowsWide;
    share = model_share(
        n, (n - pn) / 2 / span * span, pn, kWaveRowsWide, D, maxnew,
        [&](int64_t p) { return lev[at(p)]; }, [&](int64_t p) { return cnt[at(p)]; },
        [&](int64_t p, auto &&f) { for_deps(at(p), [&](int32_t j) { f(at(col[j])); }); });
  }
  P.d_ticket = (uint32_t *)dev_alloc(256);  // [0] ticket, [1] stall flag, [2] batches done
  MGX_HIP(hipMemset(P.d_ticket, 0, 256));
  L.d_rows = upload(rows);
  L.d_ptr = upload(L.ptr);
  P.flow = n >= kFlowRows && share >= kFlowBetter && nlev >= kFlowMinLevels &&
           n >= kFlowMinWidth * (int64_t)nlev;
  if (P.flow) {
    int64_t nd = 0;
    for (int64_t i = 0; i < n; i++) nd += cnt[i];
    std::vector<int4> rec(n);
    std::vector<int32_t> dcol(std::max<int64_t>(nd, 1)), dent(std::max<int64_t>(nd, 1));
    int64_t d = 0;
    for (int64_t k = 0; k < n; k++) {
      const int32_t i = rows[k];
      rec[k] = make_int4(i, (int32_t)d, (int32_t)(d + cnt[i]), 0);
      for_deps(i, [&](int32_t j) {
        dcol[d] = col[j];
        dent[d++] = ent ? (*ent)[j] : j;
      });
    }
    P.ndeps = nd;
    P.nrow = n;
    P.d_rec = upload(rec);
    P.d_dcol = upload(dcol);
    P.d_dent = upload(dent);
    P.d_row = upload(rows);
    P.built = true;
    return;
  }
  // rows of each wave in level order
  const int64_t per = (n + kChWaves - 1) / kChWaves;
  const int64_t cap = share >= 1 && n < kFlowRows ? kWaveRowsScattered
                      : share >= kScattered || n >= kWideLevel * (int64_t)nlev ? kWaveRowsWide
                                                                             : kWaveRows;
  const int64_t srows = std::min<int64_t>(cap, std::max<int64_t>(64, (per + 63) / 64 * 64));
  P.crows = (int32_t)(kChWaves * srows);
  P.nchunk = (int32_t)((n + P.crows - 1) / P.crows);
  const int64_t nwave = (int64_t)P.nchunk * kChWaves;
  std::vector<int32_t> order(n);
  {
    std::vector<int32_t> next(nwave);
    for (int64_t v = 0; v < nwave; v++) next[v] = (int32_t)std::min<int64_t>(v * srows, n);
    for (int64_t k = 0; k < n; k++) order[next[at(rows[k]) / srows]++] = rows[k];
  }
  const uint16_t zero = (uint16_t)slot_zero((uint32_t)P.crows);
  std::vector<int64_t> wave((nwave + 1) * 4);
  // the waves' batches, by a few threads, each for a run of waves
  struct Part {
    std::vector<int4> hdr;
    std::vector<uint16_t> slot;
    std::vector<int32_t> dent, ext;
  };
  const int nthr = n < 65536 ? 1 : 4;
  std::vector<Part> part(nthr);
  // the rows of a level, in a wave, run in any order: those of one batch's
  // width first, longer ones by their length, so that a batch is not cut at
  // every change between them (2000-row M-matrix, half of its rows longer
  // than 14 entries: 0.89 -> 0.29 ms an iteration of SOR-PCG)
  auto sort_levels = [&](int64_t k0, int64_t k1) {
    for (int64_t k = k0; k < k1;) {
      int64_t e = k;
      bool lng = false;
      for (; e < k1 && lev[order[e]] == lev[order[k]]; e++) lng = lng || cnt[order[e]] > D;
      if (lng)
        std::stable_sort(order.begin() + k, order.begin() + e, [&](int32_t x, int32_t y) {
          return std::max(cnt[x], D) < std::max(cnt[y], D);
        });
      k = e;
    }
  };
  auto work = [&](int64_t v0, int64_t v1, Part &out) {
    std::vector<int4> &hdr = out.hdr;
    std::vector<uint16_t> &slot = out.slot;
    std::vector<int32_t> &dent = out.dent, &ext = out.ext;
    // per row: the wave that last took its value into its ring, and as which
    std::vector<int32_t> stamp(n, -1);
    std::vector<int64_t> taken(n);
    const int64_t mine = std::min<int64_t>(n, (v1 - v0) * srows) + 64;
    slot.reserve(mine * wd.slots);
    dent.reserve(mine * D);
    hdr.reserve(mine / 16);
    std::vector<int32_t> fresh, ent0(64);
    for (int64_t v = v0; v < v1; v++) {
      int64_t *const wv = &wave[v * 4];
      wv[0] = (int64_t)hdr.size();
      wv[1] = (int64_t)slot.size() / wd.slots;
      wv[2] = std::min<int64_t>(v * srows, n);
      wv[3] = (int64_t)ext.size();
      const int64_t k1 = std::min<int64_t>(wv[2] + srows, n);
      sort_levels(wv[2], k1);
      const int64_t base = v / kChWaves * P.crows;  // the chunk's first sweep position
      const uint32_t ring0 = (uint32_t)P.crows + (uint32_t)(v % kChWaves) * kRing;
      int64_t ntaken = 0;
      // a value of an earlier chunk: not in the ring, or no longer after the
      // new ones that may follow (counted from `since`) before it is read?
      int64_t since = 0;
      int most = maxnew;
      auto lacks = [&](int32_t q) {
        return stamp[q] != (int32_t)v || since + most - taken[q] > kRing;
      };
      for (int64_t k = wv[2]; k < k1;) {
        // the batch's rows: short ones of consecutive levels, or long ones of
        // one level
        const bool lng = cnt[order[k]] > D;
        int64_t ke = k;
        int longest = 0;
        uint64_t starts = 0;
        fresh.clear();
        since = ntaken;
        most = lng ? std::max(maxnew, 64 * D) : maxnew;
        auto take = [&](int32_t q) {
          stamp[q] = (int32_t)v;
          taken[q] = ntaken + (int64_t)fresh.size();
          fresh.push_back(q);
        };
        while (ke < k1 && ke - k < 64) {
          const int32_t i = order[ke];
          if ((cnt[i] > D) != lng) break;
          const bool level = ke == k || lev[order[ke - 1]] != lev[i];
          if (lng && ke > k && (level || longest > 2 * cnt[i] || cnt[i] > 2 * longest)) break;
          if (!lng) {
            int news = 0;
            for_deps(i, [&](int32_t j) { news += at(col[j]) < base && lacks(col[j]); });
            if (ke > k && (int)fresh.size() + news > maxnew) break;
            for_deps(i, [&](int32_t j) {
              if (at(col[j]) < base && lacks(col[j])) take(col[j]);
            });
          }
          if (level) starts |= 1ull << (ke - k);
          longest = std::max(longest, cnt[i]);
          ke++;
        }
        const int m = (int)(ke - k), parts = std::max(1, (longest + D - 1) / D);
        for (int l = 0; l < m; l++) ent0[l] = ptr[order[k + l]];
        for (int pt = 0; pt < parts; pt++) {
          const size_t s0 = slot.size(), c0 = dent.size();
          slot.resize(s0 + (size_t)m * wd.slots, zero);
          dent.resize(c0 + (size_t)m * D, -1);
          if (lng) {
            fresh.clear();
            since = ntaken;
          }
          for (int l = 0; l < m; l++) {
            const int32_t i = order[k + l], left = std::min(cnt[i] - pt * D, D);
            for (int u = 0; u < left; u++) {
              int32_t &j = ent0[l];
              while (!dep_of(filter, i, col[j])) j++;
              const int32_t q = col[j];
              dent[c0 + ((size_t)(u / 2) * m + l) * 2 + u % 2] = ent ? (*ent)[j] : j;
              j++;
              uint16_t sl;
              if (at(q) >= base) {
                sl = (uint16_t)(at(q) - base);
              } else {
                if (lng && lacks(q)) {
                  // (a full batch of new values: one that only takes them)
                  if ((int)fresh.size() == maxnew) {
                    push_values(hdr, ext, fresh);
                    ntaken += maxnew;
                    fresh.clear();
                  }
                  take(q);
                }
                sl = (uint16_t)(ring0 + (uint32_t)(taken[q] & (kRing - 1)));
              }
              slot[s0 + ((size_t)(u / wd.slot_load) * m + l) * wd.slot_load + u % wd.slot_load] = sl;
            }
          }
          const uint32_t flags = !lng              ? 0u
                                 : pt == 0         ? (parts == 1 ? kPartFirst | kPartLast : kPartFirst)
                                 : pt == parts - 1 ? kPartLast
                                                   : kPartMid;
          hdr.push_back(make_int4((int32_t)(uint32_t)starts, (int32_t)(uint32_t)(starts >> 32),
                                  (int32_t)((uint32_t)m | (uint32_t)fresh.size() << 8 | flags), 0));
          ext.insert(ext.end(), fresh.begin(), fresh.end());
          ntaken += (int64_t)fresh.size();
        }
        k = ke;
      }
      while ((int64_t)(hdr.size() - wv[0]) % wd.ahead) hdr.push_back(make_int4(0, 0, 0, 0));
    }
  };
  {
    std::vector<std::future<void>> run;
    for (int t = 1; t < nthr; t++)
      run.push_back(std::async(std::launch::async, work, nwave * t / nthr,
                               nwave * (t + 1) / nthr, std::ref(part[t])));
    work(0, nwave / nthr, part[0]);
    for (auto &r : run) r.get();
  }
  // behind each other; every array is loaded 64 lanes wide and up to `ahead`
  // batches past the end
  Part &last = part.back();
  wave[nwave * 4] = (int64_t)last.hdr.size();
  last.hdr.resize(last.hdr.size() + 2 * wd.ahead, make_int4(0, 0, 0, 0));
  last.slot.resize(last.slot.size() + 64 * wd.slots, zero);
  last.dent.resize(last.dent.size() + 64 * D, -1);
  last.ext.resize(last.ext.size() + 64 * (wd.far + 1), 0);
  int64_t at0[4] = {0, 0, 0, 0};
  for (int t = 0; t < nthr; t++) {
    const int64_t v1 = nwave * (t + 1) / nthr + (t + 1 == nthr);  // (and the end of the last)
    for (int64_t v = nwave * t / nthr; v < v1; v++)
      for (int q = 0; q < 4; q++) wave[v * 4 + q] += at0[q];
    at0[0] += (int64_t)part[t].hdr.size();
    at0[1] += (int64_t)part[t].slot.size() / wd.slots;
    at0[3] += (int64_t)part[t].ext.size();
  }
  std::vector<int32_t> prow(order);
  prow.resize(n + 128, 0);
  P.nrow = (int64_t)prow.size();
  P.ndeps = at0[1] * D;
  P.d_hdr = upload_parts(part, &Part::hdr);
  P.d_slot = upload_parts(part, &Part::slot);
  P.d_dent = upload_parts(part, &Part::dent);
  P.d_ext = upload_parts(part, &Part::ext);
  P.d_row = upload(prow);
  P.d_wave = upload(wave);
  P.built = true;
}

const TriPlan &tri_plan(Csr *A, int which) {
  TriPlan &P = A->tri[which];
  if (!P.built) {
    MGX_REQUIRE(which <= kTriUpper, "internal: the L^T plan is built by the IC set-up");
    const int64_t n = A->rows;
    std::vector<int32_t> rp(n + 1), ci;
    MGX_HIP(hipStreamSynchronize(A->ctx->stream));
    MGX_HIP(hipMemcpy(rp.data(), A->rp, (size_t)(n + 1) * 4, hipMemcpyDeviceToHost));
    ci.resize(std::max<int32_t>(rp[n], 0));
    if (!ci.empty())
      MGX_HIP(hipMemcpy(ci.data(), A->ci, ci.size() * 4, hipMemcpyDeviceToHost));
    build_tri_plan(rp, ci, nullptr, n, which, P);
  }
  return P;
}

TriOp tri_prepare(Csr *A, const TriPlan &P, mgx_dtype dt, int fin, const void *vals,
                  const void *scale, const int32_t *scale_pos) {
  Ctx *c = A->ctx;
  const size_t es = dt == MGX_F64 ? 8 : 4;
  TriOp op;
  op.plan = &P;
  op.fin = fin;
  op.coef = ws_get(c, (size_t)std::max<int64_t>(P.ndeps, 1) * es);
  op.isc = ws_get(c, (size_t)P.nrow * 2 * es);
  const unsigned gd = (unsigned)((P.ndeps + kBlock - 1) / kBlock);
  const int64_t n = P.n;
  const unsigned gn = (unsigned)((n + kBlock - 1) / kBlock);
  if (dt == MGX_F64) {
    if (P.ndeps > 0)
      k_tri_pack<double><<<gd, kBlock, 0, c->stream>>>(P.ndeps, P.d_dent, (const double *)vals,
                                                       (double *)op.coef);
    if (n > 0)
      k_tri_scale<double><<<gn, kBlock, 0, c->stream>>>(n, P.d_row, (const double *)scale,
                                                        scale_pos, (double *)op.isc);
  } else {
    if (P.ndeps > 0)
      k_tri_pack<float><<<gd, kBlock, 0, c->stream>>>(P.ndeps, P.d_dent, (const float *)vals,
                                                      (float *)op.coef);
    if (n > 0)
      k_tri_scale<float><<<gn, kBlock, 0, c->stream>>>(n, P.d_row, (const float *)scale,
                                                       scale_pos, (float *)op.isc);
  }
  MGX_HIP(hipGetLastError());
  return op;
}

void tri_run(Csr *A, const TriOp &op, mgx_dtype dt, const void *in, void *out) {
  if (dt == MGX_F64)
    tri_run_fin<double>(A->ctx, op, in, out);
  else
    tri_run_fin<float>(A->ctx, op, in, out);
}

void tri_check_stall(Csr *A) {
  for (TriPlan &P : A->tri) {
    if (!P.d_ticket) continue;
    uint32_t flag = 0;
    MGX_HIP(hipMemcpy(&flag, P.d_ticket + 1, 4, hipMemcpyDeviceToHost));
    if (flag) {
      MGX_HIP(hipMemset(P.d_ticket + 1, 0, 4));
      set_error("triangular sweep: no row was finished for more than 2 s; the sweep "
                "gave up (result NaN)");
      throw Error{MGX_ERR_TIMEOUT};
    }
  }
}

void levels_free(SorLevels &L) {
  dev_free(L.d_rows);
  dev_free(L.d_ptr);
  L = SorLevels();
}

void tri_free(Csr *A) {
  for (TriPlan &P : A->tri) plan_free(P);
}

}  // namespace mgx
