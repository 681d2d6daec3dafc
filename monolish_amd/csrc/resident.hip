// resident.hip -- a whole CG or BiCGSTAB solve of one small system in one
// cooperative launch, the system held in registers.
//
// An iteration of such a system moves little data (2D Poisson 256^2: 4 MB of
// matrix, 0.5 MB a vector), so one launch per stage is bound by the stages'
// boundaries: CG took 14.5 us an iteration in two launches, BiCGSTAB 61 us in
// five (250000 rows).  Here every thread keeps the rows 2t and 2t + 1 of its
// 512-row tiles -- their entries, and x, r, p, ... -- in registers for the
// whole solve.  The vector that an SpMV gathers (p = z + beta p; phat, shat)
// is also kept at the columns of the thread's entries and updated there, so
// only what its recurrence takes in crosses blocks: z in CG, r and v in
// BiCGSTAB, and the partial sums of the reductions, through device-coherent
// stores and loads (0.3-0.5 us from one compute unit to another).
//
// A reduction is one all-to-all step: each tile publishes its partial, and
// every block reads all of them and forms the canonical stage 2 itself (lane
// t adds the partials of tiles t, t + 256, ... in order, then the block
// tree), so no block waits for a combined result to come back.  A slot that
// has not been written holds a marker, a signalling NaN that no sum
// produces.  Three sets of slots take turns: a block has passed step k + 1
// only when every block has read step k, so it clears its slots of step k
// then, and they are clear before step k + 3 uses them (its own publication
// of step k + 2 comes after the clearing has completed).  The vector that the
// next SpMV gathers is stored before the partials are published, so the
// same step makes it visible.  Each partial is published once per XCD, so
// that an XCD's blocks poll lines of their own (one copy for all: 2.5 us more
// an iteration on 256^2).  Arithmetic and order are those of the
// launch-per-stage kernels (batch.hip), so the bits are the same.
//
// Per iteration, FP64, resident / launches (us): CG, 5-point 20^2 4.5 / 14.5,
// 256^2 4.9 / 13.4, 500^2 7.8 / 34.6, 700^2 11.8 / 49.3; 7-point 30^3 5.5 /
// 15.3, 60^3 8.5 / 36.1, 80^3 19.5 / 57.4 (two rounds of tiles, some
// registers spilled); BiCGSTAB, 5-point 100^2 8.1 / 28.3, 500^2 13.9 / 56.3;
// 7-point 60^3 17.1 / 53.5.  What is left of an iteration is latency: a store
// to memory, a poll, a gather, per step about 2 us.
#include <algorithm>

#include "mgx_batch.hpp"
#include "mgx_device.hpp"

namespace mgx {

namespace {

constexpr int kEnt = 7;           // most entries of a row (5: a form of its own)
constexpr int kResLanes = 4;      // partials per stage-2 lane: 1024 tiles
// copies of every partial, one for the blocks of each XCD
constexpr int kCopies = 8;
constexpr uint64_t kResTicks = 200000000;  // 2 s of the 100 MHz clock
constexpr uint64_t kResGap = 1000000;      // 10 ms, what 1024 reads never take

template <class T> struct Slot;
template <> struct Slot<double> {
  using U = uint64_t;
  static constexpr U kEmpty = 0x7ff0deadbeef0001ull;
};
template <> struct Slot<float> {
  using U = uint32_t;
  static constexpr U kEmpty = 0x7f80dea1u;
};

template <class V> __device__ __forceinline__ V rget(const V *p) {
  return __hip_atomic_load(const_cast<V *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class V> __device__ __forceinline__ void rput(V *p, V v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double rsqrt_of(double v) { return __builtin_sqrt(v); }
__device__ __forceinline__ float rsqrt_of(float v) { return __builtin_sqrtf(v); }

// before a launch; the first launch of a solve also keeps its x: when a wait
// of a launch gives up, some blocks may have stored their rows all the same
template <class T>
__global__ __launch_bounds__(kBlock) void k_res_clear(typename Slot<T>::U *slots, int64_t n,
                                                      uint32_t *err, const T *x, T *keep,
                                                      int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) slots[i] = Slot<T>::kEmpty;
  if (i == 0) *err = 0u;
  if (keep && i < rows) keep[i] = x[i];
}

// the descriptor's fields, read once by scalar loads into registers (read
// through a reference they were loaded anew, with a wait for everything in
// flight, at each use: 1.5 to 3.5 us more per iteration)
template <class T> struct ResDesc {
  const int32_t *rp, *ci;
  const T *val, *M;
  T *x, *r, *z, *pa, *pb, *r0, *va, *vb;
  double *rhist;
  int64_t rhist_len, n, ntiles;
  SolveState *st;
  __device__ __forceinline__ explicit ResDesc(const SysDesc<T> *sys) {
    typedef const __attribute__((address_space(4))) SysDesc<T> C;
    C *c = (C *)sys;
    rp = (decltype(rp))c->rp.p;
    ci = (decltype(ci))c->ci.p;
    val = (decltype(val))c->val.p;
    M = (decltype(M))c->M.p;
    x = (decltype(x))c->x.p;
    r = (decltype(r))c->r.p;
    z = (decltype(z))c->z.p;
    pa = (decltype(pa))c->pa.p;
    pb = (decltype(pb))c->pb.p;
    r0 = (decltype(r0))c->r0.p;
    va = (decltype(va))c->va.p;
    vb = (decltype(vb))c->vb.p;
    rhist = (decltype(rhist))c->rhist.p;
    st = (SolveState *)c->st.p;
    rhist_len = c->rhist_len, n = c->n, ntiles = c->ntiles;
  }
};

// TT tiles side by side in a block (256 threads each), TR rounds of them; KE:
// entries a row holds at most
template <class T, int TT, int TR, int KE> struct Resident {
  using U = typename Slot<T>::U;
  const ResDesc<T> &d;
  U *slots;       // 3 sets x kCopies x 2 sums x ntiles
  uint32_t *err;  // raised when a wait gave up
  T *sh;          // LDS: TT * TR * 8 wave sums, then 8, then 2 results
  int *bad;       // LDS
  int64_t tile[TR], row[TR];
  int nr[TR];  // rows held: 0..2
  T val[TR][2][KE];
  int32_t col[TR][2][KE];
  int len[TR][2];
  uint32_t step = 0;

  __device__ __forceinline__ Resident(const ResDesc<T> &desc, U *s, uint32_t *e, T *lds, int *b)
      : d(desc), slots(s), err(e), sh(lds), bad(b) {
    const int t = threadIdx.x & (kBlock - 1), g = threadIdx.x / kBlock;
#pragma unroll
    for (int q = 0; q < TR; q++) {
      tile[q] = ((int64_t)blockIdx.x * TR + q) * TT + g;
      row[q] = tile[q] * kTile + 2 * t;
      const int64_t left = d.n - row[q];
      nr[q] = left < 0 ? 0 : left > 2 ? 2 : (int)left;
#pragma unroll
      for (int e2 = 0; e2 < 2; e2++) {
        const int64_t i = row[q] + e2;
        const bool has = e2 < nr[q];
        const int32_t a = has ? d.rp[i] : 0;
        len[q][e2] = has ? d.rp[i + 1] - a : 0;
#pragma unroll
        for (int k = 0; k < KE; k++) {
          const bool in = k < len[q][e2];
          val[q][e2][k] = in ? d.val[a + k] : T(0);
          col[q][e2][k] = in ? d.ci[a + k] : 0;  // (row 0's value, not used)
        }
      }
    }
  }
  __device__ __forceinline__ T load(const T *v, int q, int e) const {
    return e < nr[q] ? v[row[q] + e] : T(0);
  }
  __device__ __forceinline__ void store(T *v, int q, int e, T x) const {
    if (e < nr[q]) rput(v + row[q] + e, x);
  }
  // x = the vector's values at the columns of the thread's entries
  __device__ __forceinline__ void gather(const T *v, T (&x)[TR][2][KE]) const {
#pragma unroll
    for (int q = 0; q < TR; q++)
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int k = 0; k < KE; k++) x[q][e][k] = rget(v + col[q][e][k]);
  }
  template <class F> __device__ __forceinline__ void each(F f) const {
#pragma unroll
    for (int q = 0; q < TR; q++)
#pragma unroll
      for (int e = 0; e < 2; e++)
#pragma unroll
        for (int k = 0; k < KE; k++) f(q, e, k);
  }
  // the rows' sums in storage order from 0
  __device__ __forceinline__ void spmv(T (&y)[TR][2], const T (&x)[TR][2][KE]) const {
#pragma unroll
    for (int q = 0; q < TR; q++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        T s = 0;
#pragma unroll
        for (int k = 0; k < KE; k++) {
          const T p = val[q][e][k] * x[q][e][k];
          if (k < len[q][e]) s = s + p;
        }
        y[q][e] = s;
      }
  }
  // One all-to-all step.  NV sums of a[v][q] (a lane's two rows of tile q
  // added); res[v] for every thread; false when a wait gave up
  template <int NV>
  __device__ __forceinline__ bool meet(const T (&a)[NV][TR], T (&res)[NV]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x / 64, g = threadIdx.x / kBlock;
    const int64_t nt = d.ntiles;
    U *const set = slots + (int64_t)(step % 3) * kCopies * 2 * nt;
    U *const prev = slots + (int64_t)((step + 2) % 3) * kCopies * 2 * nt;
    U *const mine = set + (int64_t)(blockIdx.x % kCopies) * 2 * nt;
    const int copy = threadIdx.x & (kBlock - 1);  // < kCopies: publishes that copy
    step++;
#pragma unroll
    for (int v = 0; v < NV; v++)
#pragma unroll
      for (int q = 0; q < TR; q++) {
        const T s = wave_tree(a[v][q]);
        if (lane == 0) sh[(v * TR + q) * 4 * TT + wv] = s;
      }
    __builtin_amdgcn_s_waitcnt(0);  // this thread's stores (and clearings) completed
    __syncthreads();
    if (copy < kCopies) {
#pragma unroll
      for (int q = 0; q < TR; q++)
        if (tile[q] < nt) {
#pragma unroll
          for (int v = 0; v < NV; v++) {
            const T *w = sh + (v * TR + q) * 4 * TT + 4 * g;
            const T lo = w[0] + w[1], hi = w[2] + w[3];
            const T r = lo + hi;
            rput(set + (int64_t)(2 * copy + v) * nt + tile[q], __builtin_bit_cast(U, r));
          }
        }
    }
    // the first 256 threads read all partials: lane t those of tiles t, t +
    // 256, ...
    int ok = 1;
    if (threadIdx.x < kBlock) {
      T lanev[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) lanev[v] = T(0);
      const int t = threadIdx.x;
      U got[NV][kResLanes];
#pragma unroll
      for (int j = 0; j < kResLanes; j++)
#pragma unroll
        for (int v = 0; v < NV; v++) got[v][j] = Slot<T>::kEmpty;
      uint64_t last = 0, waited = 0;
      bool late = false;  // out of time: one more read decides
      for (uint32_t spin = 0;; spin++) {
        // only what is missing is asked for again
        bool miss = false;
#pragma unroll
        for (int j = 0; j < kResLanes; j++)
          if (t + (int64_t)j * kBlock < nt) {
#pragma unroll
            for (int v = 0; v < NV; v++)
              if (got[v][j] == Slot<T>::kEmpty)
                got[v][j] = rget(mine + v * nt + t + (int64_t)j * kBlock);
          }
#pragma unroll
        for (int j = 0; j < kResLanes; j++)
          if (t + (int64_t)j * kBlock < nt) {
#pragma unroll
            for (int v = 0; v < NV; v++) miss = miss || got[v][j] == Slot<T>::kEmpty;
          }
        if (!__any(miss)) break;
        if (late) {
          rput(err, 1u);
          ok = 0;
          break;
        }
        if ((spin & 1023u) == 1023u) {
          // (a longer gap between two looks: all blocks stood still, the
          // process was taken off the device)
          const uint64_t now = wall_clock64();
          if (last) waited += min(now - last, kResGap);
          last = now;
          late = waited > kResTicks || rget(err) != 0u;
        }
      }
#pragma unroll
      for (int j = 0; j < kResLanes; j++)
        if (t + (int64_t)j * kBlock < nt) {
#pragma unroll
          for (int v = 0; v < NV; v++) lanev[v] = lanev[v] + __builtin_bit_cast(T, got[v][j]);
        }
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const T s = wave_tree(lanev[v]);
        if (lane == 0) sh[8 * TT * TR + 4 * v + wv] = s;
      }
      if (!ok && lane == 0) *bad = 1;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const T *w = sh + 8 * TT * TR + 4 * v;
      const T lo = w[0] + w[1], hi = w[2] + w[3];
      res[v] = lo + hi;
    }
    // every block has published this step, so all have read the one before
    if (copy < kCopies) {
#pragma unroll
      for (int q = 0; q < TR; q++)
        if (tile[q] < nt) {
#pragma unroll
          for (int v = 0; v < 2; v++)
            rput(prev + (int64_t)(2 * copy + v) * nt + tile[q], Slot<T>::kEmpty);
        }
    }
    return *bad == 0;
  }
};

// CG (cg.cpp:46-84) as k_cg_spmv / k_cg_update compute it; two all-to-all
// steps and one gather (z) an iteration
template <class T, int TT, int TR, int KE>
__global__ __launch_bounds__(kBlock *TT) void k_resident_cg(const SysDesc<T> *sys,
                                                            typename Slot<T>::U *slots,
                                                            uint32_t *err, int32_t *stopped,
                                                            int64_t max_iters) {
  __shared__ T sh[8 * TT * TR + 8];
  __shared__ int bad;
  const ResDesc<T> d(sys);
  SolveState *st = d.st;
  if (st->status != kStatRunning) return;
  if (threadIdx.x == 0) bad = 0;
  Resident<T, TT, TR, KE> R(d, slots, err, sh, &bad);
  T x[TR][2], r[TR][2], z[TR][2], p[TR][2], m[TR][2], q[TR][2];
  int64_t it = st->iter;
  bool first = st->first != 0;
  T beta = (T)st->beta, zr = (T)st->zr;
  const double tol = st->tol;
  const int64_t miniter = st->miniter, maxiter = st->maxiter;
  const int64_t stop_at = it + max_iters;
#pragma unroll
  for (int k = 0; k < TR; k++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      x[k][e] = R.load(d.x, k, e);
      r[k][e] = R.load(d.r, k, e);
      z[k][e] = R.load(d.z, k, e);
      p[k][e] = first ? T(0) : R.load((it & 1) ? d.pb : d.pa, k, e);
      m[k][e] = d.M ? R.load(d.M, k, e) : T(1);
    }
  int32_t s = kStatRunning;
  T resid = 0, rr = 0;
  T gp[TR][2][KE], gz[TR][2][KE];  // p and z at the entries' columns
  if (!first) R.gather((it & 1) ? d.pb : d.pa, gp);
  while (it < stop_at) {
    R.gather(d.z, gz);
    R.each([&](int k, int e, int j) {
      T pi = gz[k][e][j];
      if (!first) {
        const T bp = beta * gp[k][e][j];
        pi = gz[k][e][j] + bp;
      }
      gp[k][e][j] = pi;
    });
    R.spmv(q, gp);
    T a1[1][TR], pq[1];
#pragma unroll
    for (int k = 0; k < TR; k++) {
      T acc[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        T pi = z[k][e];
        if (!first) {
          const T bp = beta * p[k][e];
          pi = z[k][e] + bp;
        }
        p[k][e] = pi;
        acc[e] = e < R.nr[k] ? pi * q[k][e] : T(0);
      }
      a1[0][k] = acc[0] + acc[1];
    }
    if (!R.template meet<1>(a1, pq)) return;
    const T alpha = zr / pq[0], nalpha = -alpha;
    T a2[2][TR], red[2];
#pragma unroll
    for (int k = 0; k < TR; k++) {
      T zz[2], r2[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const T t1 = alpha * p[k][e];
        x[k][e] = t1 + x[k][e];
        const T t2 = nalpha * q[k][e];
        const T rv = t2 + r[k][e];
        r[k][e] = rv;
        const T zv = d.M ? m[k][e] * rv : rv;
        z[k][e] = zv;
        R.store(d.z, k, e, zv);
        zz[e] = e < R.nr[k] ? zv * rv : T(0);
        r2[e] = e < R.nr[k] ? rv * rv : T(0);
      }
      a2[0][k] = zz[0] + zz[1];
      a2[1][k] = r2[0] + r2[1];
    }
    if (!R.template meet<2>(a2, red)) return;
    const T zr_new = red[0];
    rr = red[1];
    beta = zr_new / zr;
    zr = zr_new;
    resid = rsqrt_of(rr);
    first = false;
    it++;
    if (blockIdx.x == 0 && threadIdx.x == 0 && d.rhist && it - 1 < d.rhist_len)
      d.rhist[it - 1] = (double)resid;
    if ((double)resid < tol && miniter <= it)
      s = MGX_OK;
    else if (resid != resid)
      s = MGX_SOLVER_RESIDUAL_NAN;
    else if (it >= maxiter)
      s = MGX_SOLVER_MAXITER;
    if (s != kStatRunning) break;
  }
#pragma unroll
  for (int k = 0; k < TR; k++)
#pragma unroll
    for (int e = 0; e < 2; e++)
      if (e < R.nr[k]) {
        const int64_t i = R.row[k] + e;
        d.x[i] = x[k][e];
        d.r[i] = r[k][e];
        ((it & 1) ? d.pb : d.pa)[i] = p[k][e];
      }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->beta = (double)beta;
    st->zr = (double)zr;
    st->rr = (double)rr;
    st->resid = (double)resid;
    st->iter = it;
    st->first = first;
    st->status = s;
    if (s != kStatRunning && stopped) atomicAdd(stopped, 1);
  }
}

// BiCGSTAB (bicgstab.cpp:53-129) as k_bcg_p ... k_bcg_update compute it; three
// all-to-all steps and two gathers (r, v) an iteration.  From one launch to
// the next p and v go through pa and vb, which are only written at a launch's
// end: va is written before the first step, when another block may not have
// taken the last launch's values yet
template <class T, int TT, int TR, int KE>
__global__ __launch_bounds__(kBlock *TT) void k_resident_bcg(const SysDesc<T> *sys,
                                                             typename Slot<T>::U *slots,
                                                             uint32_t *err, int32_t *stopped,
                                                             int64_t max_iters) {
  __shared__ T sh[8 * TT * TR + 8];
  __shared__ int bad;
  const ResDesc<T> d(sys);
  SolveState *st = d.st;
  if (st->status != kStatRunning) return;
  if (threadIdx.x == 0) bad = 0;
  Resident<T, TT, TR, KE> R(d, slots, err, sh, &bad);
  T x[TR][2], r[TR][2], r0[TR][2], p[TR][2], v[TR][2], m[TR][2], ph[TR][2], sv[TR][2], hv[TR][2],
      t[TR][2];
  int64_t it = st->iter;
  bool first = st->first != 0;
  T beta = (T)st->beta, rho = (T)st->rho, omega = (T)st->omega;
  double resid_out = st->resid;
  const double tol = st->tol;
  const int64_t miniter = st->miniter, maxiter = st->maxiter;
  const int64_t stop_at = it + max_iters;
#pragma unroll
  for (int k = 0; k < TR; k++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      x[k][e] = R.load(d.x, k, e);
      r[k][e] = R.load(d.r, k, e);
      r0[k][e] = R.load(d.r0, k, e);
      p[k][e] = first ? T(0) : R.load(d.pa, k, e);
      v[k][e] = first ? T(0) : R.load(d.vb, k, e);
      m[k][e] = d.M ? R.load(d.M, k, e) : T(1);
    }
  int32_t s = kStatRunning;
  // p, v, r, M at the entries' columns, and phat or shat there
  T gp[TR][2][KE], gv[TR][2][KE], gr[TR][2][KE], gm[TR][2][KE], gh[TR][2][KE];
  if (!first) {
    R.gather(d.pa, gp);
    R.gather(d.vb, gv);
  }
  if (d.M) R.gather(d.M, gm);
  while (it < stop_at) {
    const T nomega = -omega;
    auto next_p = [&](T rv, T vv, T pv) -> T {
      if (first) return rv;
      const T t1 = nomega * vv;
      const T p1 = t1 + pv;
      const T t2 = beta * p1;
      return rv + t2;
    };
    R.gather(d.r, gr);
#pragma unroll
    for (int k = 0; k < TR; k++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        p[k][e] = next_p(r[k][e], v[k][e], p[k][e]);
        ph[k][e] = d.M ? m[k][e] * p[k][e] : p[k][e];
      }
    R.each([&](int k, int e, int j) {
      gp[k][e][j] = next_p(gr[k][e][j], gv[k][e][j], gp[k][e][j]);
      gh[k][e][j] = d.M ? gm[k][e][j] * gp[k][e][j] : gp[k][e][j];
    });
    R.spmv(v, gh);
    T a1[1][TR], vr0[1];
#pragma unroll
    for (int k = 0; k < TR; k++) {
      const T b0 = 0 < R.nr[k] ? v[k][0] * r0[k][0] : T(0);
      const T b1 = 1 < R.nr[k] ? v[k][1] * r0[k][1] : T(0);
      a1[0][k] = b0 + b1;
      R.store(d.va, k, 0, v[k][0]);
      R.store(d.va, k, 1, v[k][1]);
    }
    if (!R.template meet<1>(a1, vr0)) return;
    const T alpha = rho / vr0[0], nalpha = -alpha;
    R.gather(d.va, gv);
    auto next_s = [&](T vv, T rv) -> T {
      const T t1 = nalpha * vv;
      return t1 + rv;
    };
#pragma unroll
    for (int k = 0; k < TR; k++)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        sv[k][e] = next_s(v[k][e], r[k][e]);
        hv[k][e] = d.M ? m[k][e] * sv[k][e] : sv[k][e];
      }
    R.each([&](int k, int e, int j) {
      const T si = next_s(gv[k][e][j], gr[k][e][j]);
      gh[k][e][j] = d.M ? gm[k][e][j] * si : si;
    });
    R.spmv(t, gh);
    T a2[2][TR], w[2];
#pragma unroll
    for (int k = 0; k < TR; k++) {
      T ts[2], tt[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        ts[e] = e < R.nr[k] ? t[k][e] * sv[k][e] : T(0);
        tt[e] = e < R.nr[k] ? t[k][e] * t[k][e] : T(0);
      }
      a2[0][k] = ts[0] + ts[1];
      a2[1][k] = tt[0] + tt[1];
    }
    if (!R.template meet<2>(a2, w)) return;
    omega = w[0] / w[1];
    if (omega == T(0)) {
      // breakdown: the residual reported is that of the current r
      it++;
      s = MGX_SOLVER_BREAKDOWN;
      break;
    }
    const T nom = -omega;
    T a3[2][TR], red[2];
#pragma unroll
    for (int k = 0; k < TR; k++) {
      T r2[2], rq[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const T b1 = alpha * ph[k][e];
        const T x1 = b1 + x[k][e];
        const T b2 = omega * hv[k][e];
        x[k][e] = b2 + x1;
        const T b3 = nom * t[k][e];
        const T rv = b3 + sv[k][e];
        r[k][e] = rv;
        R.store(d.r, k, e, rv);
        r2[e] = e < R.nr[k] ? rv * rv : T(0);
        rq[e] = e < R.nr[k] ? rv * r0[k][e] : T(0);
      }
      a3[0][k] = r2[0] + r2[1];
      a3[1][k] = rq[0] + rq[1];
    }
    if (!R.template meet<2>(a3, red)) return;
    const T resid = rsqrt_of(red[0]), rho_next = red[1];
    resid_out = (double)resid;
    if (blockIdx.x == 0 && threadIdx.x == 0 && d.rhist && it < d.rhist_len)
      d.rhist[it] = (double)resid;
    it++;
    if ((double)resid < tol && miniter <= it) {
      s = MGX_OK;
    } else if (resid != resid) {
      s = MGX_SOLVER_RESIDUAL_NAN;
    } else if (it >= maxiter) {
      s = MGX_SOLVER_MAXITER;
    } else if (rho_next == T(0)) {
      s = MGX_SOLVER_BREAKDOWN;  // at the top of the next iteration
      it++;
    } else {
      beta = (rho_next / rho) * (alpha / omega);
      rho = rho_next;
      first = false;
    }
    if (s != kStatRunning) break;
  }
#pragma unroll
  for (int k = 0; k < TR; k++)
#pragma unroll
    for (int e = 0; e < 2; e++)
      if (e < R.nr[k]) {
        const int64_t i = R.row[k] + e;
        d.x[i] = x[k][e];
        d.pa[i] = p[k][e];
        d.vb[i] = v[k][e];
      }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->beta = (double)beta;
    st->rho = (double)rho;
    st->omega = (double)omega;
    st->resid = resid_out;
    st->iter = it;
    st->first = first;
    st->status = s;
    if (s != kStatRunning && stopped) atomicAdd(stopped, 1);
  }
}

template <class T> using ResKernel = void (*)(const SysDesc<T> *, typename Slot<T>::U *,
                                              uint32_t *, int32_t *, int64_t);

template <class T, int KE> ResKernel<T> res_kernel(int method, int tt, int tr) {
  if (method == kMethodCG)
    return tt == 1   ? k_resident_cg<T, 1, 1, KE>
           : tr == 1 ? k_resident_cg<T, 2, 1, KE>
                     : k_resident_cg<T, 2, 2, KE>;
  return tt == 1 ? k_resident_bcg<T, 1, 1, KE> : k_resident_bcg<T, 2, 1, KE>;
}

// tiles side by side and rounds per block, so that every block has a compute
// unit of its own
struct ResShape {
  int tt, tr;
  int64_t grid;
};
ResShape res_shape(const Ctx *c, int64_t nt) {
  const int64_t cu = c->num_cus;
  const int tt = nt <= cu ? 1 : 2, tr = nt <= 2 * cu ? 1 : 2;
  return {tt, tr, (nt + tt * tr - 1) / (tt * tr)};
}

}  // namespace

// BiCGSTAB keeps five vectors at the entries' columns, too many registers
// for a second round of tiles
bool resident_fits(const Ctx *c, const Csr *A, int method) {
  const int64_t nt = ntiles_of(A->rows);
  const ResShape sp = res_shape(c, nt);
  return A->plan.max_row <= kEnt && nt <= (int64_t)kResLanes * kBlock && sp.grid <= c->num_cus &&
         (method == kMethodCG || sp.tr == 1);
}

// (the slots of FP64 sums; FP32 ones take half)
size_t resident_bytes(int64_t ntiles) { return 256 + (size_t)ntiles * 6 * kCopies * 8; }

template <class T>
bool resident_launch(Ctx *c, int method, const SysDesc<T> *sys, int64_t ntiles, int max_row,
                     void *scratch, int32_t *stopped, int64_t max_iters, const T *x, T *keep,
                     int64_t rows) {
  using U = typename Slot<T>::U;
  uint32_t *err = static_cast<uint32_t *>(scratch);
  U *slots = reinterpret_cast<U *>(static_cast<char *>(scratch) + 256);
  const int64_t n = 6 * kCopies * ntiles;
  const int64_t nc = keep ? std::max(n, rows) : n;
  k_res_clear<T><<<(unsigned)((nc + kBlock - 1) / kBlock), kBlock, 0, c->stream>>>(slots, n, err, x,
                                                                                   keep, rows);
  const ResShape sp = res_shape(c, ntiles);
  ResKernel<T> k = max_row <= 5 ? res_kernel<T, 5>(method, sp.tt, sp.tr)
                                : res_kernel<T, kEnt>(method, sp.tt, sp.tr);
  void *args[] = {(void *)&sys, (void *)&slots, (void *)&err, (void *)&stopped,
                  (void *)&max_iters};
  MGX_HIP(hipGetLastError());
  const hipError_t e =
      hipLaunchCooperativeKernel(reinterpret_cast<const void *>(k), dim3((unsigned)sp.grid),
                                 dim3((unsigned)(kBlock * sp.tt)), args, 0, c->stream);
  if (e == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}
template bool resident_launch<double>(Ctx *, int, const SysDesc<double> *, int64_t, int, void *,
                                      int32_t *, int64_t, const double *, double *, int64_t);
template bool resident_launch<float>(Ctx *, int, const SysDesc<float> *, int64_t, int, void *,
                                     int32_t *, int64_t, const float *, float *, int64_t);

}  // namespace mgx
