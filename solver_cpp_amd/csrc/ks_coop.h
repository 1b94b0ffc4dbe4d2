// ks_coop.h - Krylov iterations of a system that fits on chip, many to a launch.
//
// A CG step of a 256 x 256 grid moves 9 MB, a microsecond's worth, but as
// three dependent launches it takes 14 us: each launch costs 4 to 5 us
// whatever it does.  Here one launch runs up to kCoopIters steps.  The
// workgroups (one per CU at most, so all are resident together) own
// contiguous rows, up to four per thread (BiCG two), whose matrix entries and
// vector elements stay in the thread's registers between the steps, and of the
// most rows some in its scratch (FP64 CG with four 380 bytes, FP32 80; BiCG with
// two 390 and 200).  Two things cross workgroups:
//  * vectors that other rows' products gather: written with agent-scope
//    stores, which go through to memory, and gathered with agent-scope loads
//    (a workgroup's own part from LDS);
//  * reductions (Team::all_sum): every workgroup stores its sums, tagged with
//    the number of the reduction, and polls all the others'.  One store and
//    one load's latency, about 1.1 us for 64 workgroups, against 8 us and
//    more for a barrier with agent-scope fences (which write back and
//    invalidate the L2).  It is also the barrier between the steps: a
//    workgroup's vector stores are complete before its sums are stored.
// Sums form in a fixed order, the same in every workgroup, so solves are
// bit-identical run to run and control flow is uniform without a broadcast.
//
// Every wait is bounded (CoopArgs::spin polls).  A wait that runs out (the
// workgroups were not resident together, for instance beside another process)
// sets the fail word and ends the launch: its workgroups make no further wait,
// later launches return at once, the solve's and the host's stop flags keep the
// outer solver's steps from running on, and the host repeats the solve with one
// launch per operation (and does the context's next solves that way: ks_ctx).
#pragma once
#include "ks_kernels.h"

namespace ks {

// Threads of a workgroup and the most rows per thread: of one build, 512 threads
// were the fastest at most sizes (CG, 256 x 256 / 512 x 512 / 700 x 700: 6.4 / 8.6 /
// 13.2 us a step; 256 threads 6.7 / 9.8 / 41, 1024 threads 6.6 / 8.3 / 15.0): they
// leave 256 registers a thread.
constexpr int kCoopThreads = 512;
constexpr int kCoopRpt = 4;
constexpr int kCoopMaxWg = 256;
constexpr int kCoopRow = 8;       // entries of a row at most
constexpr int kCoopVals = 64;     // values of one reduction
constexpr int kCoopIters = 1024;  // steps per launch
constexpr int kCoopSpin = 1 << 21;
constexpr int64_t kCoopSlots = 2 * 2 * (int64_t)kCoopVals * kCoopMaxWg;

struct CoopArgs {
  unsigned long long* slots;  // kCoopSlots words: [parity][value][workgroup][2]
  unsigned* state;            // [0] tag of the last reduction, [1] fail
  int* stop;                  // a failure sets it: the stop flag of the solve around this one (nullable)
  int* host_stop;             // and the flag that the host looks at
  int spin;
};

template <class T>
__device__ __forceinline__ T shared_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void shared_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One workgroup's sum in a slot of 16 bytes: both halves carry the tag, so a
// reader that sees the tag in both has the whole value.
typedef unsigned slot_t __attribute__((ext_vector_type(4)));
constexpr int kSlotScope = 16;  // buffer instructions' sc1 bit: agent scope
struct Slots {
  __amdgpu_buffer_rsrc_t r;
  __device__ explicit Slots(unsigned long long* p)
      : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(kCoopSlots * 8), 0x00027000)) {}
  __device__ void put(int slot, unsigned tag, double v) const {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const slot_t q = {(unsigned)b, tag, (unsigned)(b >> 32), tag};
    __builtin_amdgcn_raw_buffer_store_b128(q, r, slot * 16, 0, kSlotScope);
  }
  __device__ slot_t get(int slot) const {
    return __builtin_amdgcn_raw_buffer_load_b128(r, slot * 16, 0, kSlotScope);
  }
};

// The workgroups, of NT threads, of one launch.  Every thread of every workgroup calls each
// member together.
template <int NT>
struct Team {
  static constexpr int kWaves = NT / 64;
  CoopArgs a;
  unsigned round;  // tag of the last reduction
  bool good;       // no wait has run out

  int* out;        // LDS: a wait of this workgroup ran out

  __device__ Team(const CoopArgs& args, int* out_) : a(args), out(out_) {
    round = a.state[0];
    good = shared_load(a.state + 1) == 0;
    if (threadIdx.x == 0) *out = 0;  // ordered by the first reduction's barrier
  }
  // v[i] summed over all threads of all workgroups, i < NV, in every thread;
  // nothing once a wait has run out.
  template <int NV>
  __device__ void all_sum(double (&v)[NV]) {
    static_assert(NV <= kCoopVals, "slots");
    if (!good) return;
    __shared__ double red[NV][kWaves];
    __shared__ double tot[NV];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, W = gridDim.x;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const double s = wave_sum(v[i]);
      if (lane == 0) red[i][w] = s;
    }
    // this thread's vector stores are complete
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ++round;
    const Slots slots(a.slots);
    const int base = (round & 1) * kCoopVals * kCoopMaxWg;
    if ((int)threadIdx.x < NV) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < kWaves; ++k) s += red[threadIdx.x][k];
      slots.put(base + (int)threadIdx.x * kCoopMaxWg + blockIdx.x, round, s);
    }
    // value i is collected by wavefront i % kWaves: lane u polls workgroups u,
    // u + 64, .. together
    for (int i = w; i < NV; i += kWaves) {
      constexpr int kQ = kCoopMaxWg / 64;
      const int q = base + i * kCoopMaxWg + lane;
      slot_t t[kQ];
      for (int k = 0;; ++k) {
        bool all = true;
#pragma unroll
        for (int u = 0; u < kQ; ++u)
          if (64 * u < W) t[u] = slots.get(q + (lane + 64 * u < W ? 64 * u : 0));
#pragma unroll
        for (int u = 0; u < kQ; ++u)
          if (64 * u < W) all &= lane + 64 * u >= W || (t[u][1] == round && t[u][3] == round);
        if (all) break;
        if (k >= a.spin) { *out = 1; break; }
        asm volatile("" ::: "memory");  // load again
      }
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < kQ; ++u)
        if (lane + 64 * u < W) s += __builtin_bit_cast(double, ((uint64_t)t[u][2] << 32) | t[u][0]);
      s = wave_sum(s);
      if (lane == 0) tot[i] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = tot[i];
    if (*out) good = false;
  }
  // at the end of the launch: the next launch's first tag, or the failure
  __device__ void close() {
    if (threadIdx.x != 0) return;
    if (!good) {
      shared_store(a.state + 1, 1u);
      if (a.stop) shared_store(a.stop, 1);
      *(volatile int*)a.host_stop = 1;
    } else if (blockIdx.x == 0) a.state[0] = round;
  }
};

// The rows of one thread: their entries in registers, and the products with a
// vector whose own part lies in LDS.  Row j of the thread is row0 + NT j +
// threadIdx.x; workgroup b owns rows [b * per, (b + 1) * per).
template <class T, int NT, int RPT>
struct CoopRows {
  T a[RPT][kCoopRow];
  int32_t c[RPT][kCoopRow];
  int len[RPT];
  int32_t row0, own;  // the workgroup's first row and number of rows
  __device__ void load(int64_t n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ col,
                       const T* __restrict__ val) {
    const int64_t per = (int64_t)RPT * NT, r0 = (int64_t)blockIdx.x * per;
    row0 = (int32_t)r0;
    own = (int32_t)(n - r0 < per ? n - r0 : per);
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      const int i = at(j);
      const int32_t s = i < own ? ptr[row0 + i] : 0, e = i < own ? ptr[row0 + i + 1] : 0;
      len[j] = e - s;
#pragma unroll
      for (int k = 0; k < kCoopRow; ++k) {
        a[j][k] = k < len[j] ? val[s + k] : T(0);
        c[j][k] = k < len[j] ? col[s + k] : 0;
      }
    }
  }
  __device__ static int at(int j) { return j * NT + (int)threadIdx.x; }
  __device__ bool has(int j) const { return at(j) < own; }
  __device__ bool local(int32_t i) const { return (unsigned)(i - row0) < (unsigned)own; }
  // Row sums in CSR order, products rounded before the add, as the SpMV
  // kernels form them.  far(c) loads what x of another workgroup's row c is
  // formed from, near(that, beta) forms it: the loads of two rows go out
  // together before the first is used (waited for one by one they cost 0.7 us
  // each).
  template <class Far, class Near>
  __device__ __forceinline__ void mul(const T* xl, double beta, Far far, Near near, T (&y)[RPT]) const {
    constexpr int J = RPT < 2 ? RPT : 2;
#pragma unroll
    for (int j0 = 0; j0 < RPT; j0 += J) {
      decltype(far(0)) f[J][kCoopRow];
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int k = 0; k < kCoopRow; ++k)
          if (k < len[j0 + j] && !local(c[j0 + j][k])) f[j][k] = far(c[j0 + j][k]);
      // near()'s beta comes after the loads: the compiler otherwise moves its
      // one fma up to each load and waits for them one by one (256 x 256: 6.3
      // against 5.9 us a step)
      asm volatile("" : "+v"(beta));
#pragma unroll
      for (int j = 0; j < J; ++j) {
        T s = T(0);
#pragma unroll
        for (int k = 0; k < kCoopRow; ++k)
          if (k < len[j0 + j]) {
            const int32_t i = c[j0 + j][k];
            s = mul_add_rn(s, a[j0 + j][k], local(i) ? xl[i - row0] : near(f[j][k], beta));
          }
        y[j0 + j] = s;
      }
    }
  }
};

// beta p + r, a row's new direction.  Its owner forms it and so does every
// workgroup that gathers it, and the two must agree bit for bit: one rounding,
// not what the compiler makes of a product and a sum at each place.
template <class T>
__device__ __forceinline__ T direction(double beta, T p, T r) {
  return (T)fma(beta, (double)p, (double)r);
}

// Whether a CG-family solve ends at count with (r, r) = rr; -1 goes on, else
// its status (cg_check's rule).
__device__ inline int cg_stop(long long count, long long maxloop, double rr, double bnorm, double eps) {
  if (count > maxloop) return 2;
  const double num = sqrt(rr), err = (bnorm == 0.0 && num == 0.0) ? 0.0 : num / bnorm;
  return err <= eps ? 0 : !finite(err) ? 3 : -1;
}

// The residual history as one thread writes it, its length in a register
// (cg_check's entries).
struct CoopHist {
  double* h;
  long long n, cap;
  __device__ void add(long long count, long long maxloop, double rr, double bnorm) {
    if (count > maxloop) return;
    const double num = sqrt(rr);
    if (h && n < cap) {
      h[2 * n] = (double)count;
      h[2 * n + 1] = (bnorm == 0.0 && num == 0.0) ? 0.0 : num / bnorm;
    }
    ++n;
  }
};

// CG (cg.cpp:148-272), up to `iters` steps.  mode 0 goes on from the last
// launch (x in xs, r and p in vec, the scalars in c), 1 starts from
// r = (T)src and x = 0, 2 from the r (in vec), x and scalars that other kernels
// left.  A step:
//   p = beta p + r, q = A p
//   alpha = rr / (p, q)              first reduction
//   x += alpha p, r -= alpha q
//   beta = rr' / rr, stop test       second reduction
// A gathered p_j of another workgroup is formed from its r_j and the step
// before's p_j, as that workgroup forms it, so no third reduction has to wait
// for the new p.  vec holds r (written between the reductions, read after the
// second) and two p, by parity of the step: a workgroup that is a step ahead
// of another does not write what that one still reads.
// last: no launch follows; xout (FP32 solves) receives x when the solve ends.
// Measured (5-point grids, FP64, per step against three launches): see
// coop_fits.
template <class T, int NT, int RPT>
__global__ __launch_bounds__(NT) void k_cg_coop(int64_t n, const int32_t* __restrict__ ptr,
                                                const int32_t* __restrict__ col, const T* __restrict__ val,
                                                const double* __restrict__ src, T* xs, T* vec, int64_t ld,
                                                double* xout, Ctl* c, CoopArgs ca, int mode, int last, int iters,
                                                Gate g, StatArgs st) {
  if (g.off()) return;
  __shared__ int s_out;
  Team<NT> team(ca, &s_out);
  if (!team.good) return;
  __shared__ T pl[RPT * NT];
  CoopRows<T, NT, RPT> A;
  A.load(n, ptr, col, val);
  T x[RPT], r[RPT], p[RPT], q[RPT];
  const double eps = c->eps;
  const long long maxloop = c->maxloop;
  long long count = mode ? 1 : c->count;
  double bnorm = c->bnorm, rr = c->rr, alpha = 0.0, beta = mode ? 0.0 : c->beta;
  CoopHist hist{c->hist, mode == 1 ? 0 : c->nhist, c->hist_cap};
  int stop = -1;
  const bool boss = blockIdx.x == 0 && threadIdx.x == 0;
  bool fresh = mode != 0;  // p is r
  T* now = vec + (count & 1 ? 2 * ld : ld);  // this step's p
  T* old = vec + (count & 1 ? ld : 2 * ld);  // the last one's
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    x[j] = r[j] = p[j] = T(0);
    if (A.has(j)) {
      const int32_t i = A.row0 + A.at(j);
      if (mode == 1) r[j] = (T)src[i];
      else { x[j] = xs[i]; r[j] = vec[i]; }
      if (mode == 0) p[j] = old[i];
    }
  }
  if (mode == 1) {
    double s[1] = {0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (A.has(j)) shared_store(vec + A.row0 + A.at(j), r[j]);
      s[0] += (double)r[j] * (double)r[j];
    }
    team.all_sum(s);
    rr = s[0];
    bnorm = sqrt(rr);
    stop = team.good ? cg_stop(count, maxloop, rr, bnorm, eps) : 3;
    if (boss) hist.add(count, maxloop, rr, bnorm);
  }
  int done = 0;
  while (stop < 0 && done < iters) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      p[j] = fresh ? r[j] : direction(beta, p[j], r[j]);
      pl[A.at(j)] = p[j];
      if (A.has(j)) shared_store(now + A.row0 + A.at(j), p[j]);
    }
    __syncthreads();
    struct Raw {
      T r, p;
    };
    if (fresh)
      A.mul(pl, beta, [&](int32_t i) { return shared_load(vec + i); }, [](T ri, double) { return ri; }, q);
    else
      A.mul(pl, beta, [&](int32_t i) { return Raw{shared_load(vec + i), shared_load(old + i)}; },
            [](Raw f, double b) { return direction(b, f.p, f.r); }, q);
    double s[1] = {0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) s[0] = fma((double)p[j], (double)q[j], s[0]);
    team.all_sum(s);
    alpha = rr / s[0];
    s[0] = 0.0;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      x[j] = (T)(alpha * (double)p[j] + (double)x[j]);
      r[j] = (T)((-alpha) * (double)q[j] + (double)r[j]);
      if (A.has(j)) shared_store(vec + A.row0 + A.at(j), r[j]);
      s[0] = fma((double)r[j], (double)r[j], s[0]);
    }
    team.all_sum(s);
    if (!team.good) break;
    beta = s[0] / rr;
    rr = s[0];
    ++count;
    ++done;
    fresh = false;
    T* t = now;
    now = old;
    old = t;
    stop = cg_stop(count, maxloop, rr, bnorm, eps);
    if (boss) hist.add(count, maxloop, rr, bnorm);
  }
  if (team.good) {
#pragma unroll
    for (int j = 0; j < RPT; ++j)
      if (A.has(j)) {
        const int32_t i = A.row0 + A.at(j);
        xs[i] = x[j];
        if (xout && (stop >= 0 || last)) xout[i] = (double)x[j];
      }
    if (boss) {
      if (mode == 1) { c->done = 0; c->ksz = 0; c->steps = 0; c->bnorm = bnorm; }
      c->count = count;
      c->nhist = hist.n;
      const double num = sqrt(rr);
      c->err = (bnorm == 0.0 && num == 0.0) ? 0.0 : num / bnorm;
      c->rr = rr;
      c->alpha = alpha;
      c->beta = beta;
      c->steps += done;
      c->tsteps += done;
      c->stop = 0;
      c->status = 2;
      if (stop >= 0) ctl_stop(c, stop);
      st.count_many(done, (unsigned long long)done * 2 * sizeof(T) * n);  // p and r of each step
    }
  }
  team.close();
}

// BiCG (bicg.cpp:162-310), as k_cg_coop: a step is both products (A p and
// A^T p*), the reduction of
// (p*, A p), the updates, and the reduction of (r*, r) and (r, r).  vec holds
// r, r*, then p and p* of even and of odd steps.  Both matrices' entries are
// kept, so a thread takes at most two rows (at two, 390 bytes of them in scratch
// in FP64 and 200 in FP32; BicgLevel::kRpt).
// Measured (7-point grids, us a step, on chip against five launches): FP64 16^3
// 6.1 / 23.2, 32^3 8.0 / 23.6, 50^3 11.5 / 27.2, 64^3 20.7 / 28.4; FP32 inside
// VPGMRES 16^3 7.8 / 24.9, 50^3 13.4 / 25.5, 64^3 18.1 / 25.5.
template <class T, int NT, int RPT>
__global__ __launch_bounds__(NT) void k_bicg_coop(int64_t n, const int32_t* __restrict__ ptr,
                                                  const int32_t* __restrict__ col, const T* __restrict__ val,
                                                  const int32_t* __restrict__ tptr, const int32_t* __restrict__ tcol,
                                                  const T* __restrict__ tval, const double* __restrict__ src, T* xs,
                                                  T* vec, int64_t ld, double* xout, Ctl* c, CoopArgs ca, int mode,
                                                  int last, int iters, Gate g, StatArgs st) {
  if (g.off()) return;
  __shared__ int s_out;
  Team<NT> team(ca, &s_out);
  if (!team.good) return;
  __shared__ T pl[RPT * NT], psl[RPT * NT];
  CoopRows<T, NT, RPT> A, B;
  A.load(n, ptr, col, val);
  B.load(n, tptr, tcol, tval);
  T x[RPT], r[RPT], rs[RPT], p[RPT], ps[RPT], q[RPT], qs[RPT];
  const double eps = c->eps;
  const long long maxloop = c->maxloop;
  long long count = mode ? 1 : c->count;
  // rz = (r*, r); rr = (r, r), which the test looks at
  double bnorm = c->bnorm, rz = c->rr, rr = c->gamma, alpha = 0.0, beta = mode ? 0.0 : c->beta;
  CoopHist hist{c->hist, mode == 1 ? 0 : c->nhist, c->hist_cap};
  int stop = -1;
  const bool boss = blockIdx.x == 0 && threadIdx.x == 0;
  bool fresh = mode != 0;  // p is r, p* is r*
  T* const rv = vec;
  T* const rsv = vec + ld;
  T* now = vec + (count & 1 ? 4 * ld : 2 * ld);  // this step's p, then p*
  T* old = vec + (count & 1 ? 2 * ld : 4 * ld);
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    x[j] = r[j] = rs[j] = p[j] = ps[j] = T(0);
    if (A.has(j)) {
      const int32_t i = A.row0 + A.at(j);
      if (mode == 1) r[j] = rs[j] = (T)src[i];
      else { x[j] = xs[i]; r[j] = rv[i]; rs[j] = rsv[i]; }
      if (mode == 0) { p[j] = old[i]; ps[j] = old[ld + i]; }
    }
  }
  if (mode == 1) {
    double s[1] = {0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      if (A.has(j)) {
        shared_store(rv + A.row0 + A.at(j), r[j]);
        shared_store(rsv + A.row0 + A.at(j), rs[j]);
      }
      s[0] += (double)r[j] * (double)r[j];
    }
    team.all_sum(s);
    rz = rr = s[0];
    bnorm = sqrt(rr);
    stop = team.good ? cg_stop(count, maxloop, rr, bnorm, eps) : 3;
    if (boss) hist.add(count, maxloop, rr, bnorm);
  }
  int done = 0;
  while (stop < 0 && done < iters) {
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      p[j] = fresh ? r[j] : direction(beta, p[j], r[j]);
      ps[j] = fresh ? rs[j] : direction(beta, ps[j], rs[j]);
      pl[A.at(j)] = p[j];
      psl[A.at(j)] = ps[j];
      if (A.has(j)) {
        shared_store(now + A.row0 + A.at(j), p[j]);
        shared_store(now + ld + A.row0 + A.at(j), ps[j]);
      }
    }
    __syncthreads();
    struct Raw {
      T r, p;
    };
    if (fresh) {
      const auto same = [](T v, double) { return v; };
      A.mul(pl, beta, [&](int32_t i) { return shared_load(rv + i); }, same, q);
      B.mul(psl, beta, [&](int32_t i) { return shared_load(rsv + i); }, same, qs);
    } else {
      const auto near = [](Raw f, double b) { return direction(b, f.p, f.r); };
      A.mul(pl, beta, [&](int32_t i) { return Raw{shared_load(rv + i), shared_load(old + i)}; }, near, q);
      B.mul(psl, beta, [&](int32_t i) { return Raw{shared_load(rsv + i), shared_load(old + ld + i)}; }, near, qs);
    }
    double s1[1] = {0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) s1[0] = fma((double)ps[j], (double)q[j], s1[0]);
    team.all_sum(s1);
    alpha = rz / s1[0];
    double s[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      x[j] = (T)(alpha * (double)p[j] + (double)x[j]);
      r[j] = (T)((-alpha) * (double)q[j] + (double)r[j]);
      rs[j] = (T)((-alpha) * (double)qs[j] + (double)rs[j]);
      if (A.has(j)) {
        shared_store(rv + A.row0 + A.at(j), r[j]);
        shared_store(rsv + A.row0 + A.at(j), rs[j]);
      }
      s[0] = fma((double)rs[j], (double)r[j], s[0]);
      s[1] = fma((double)r[j], (double)r[j], s[1]);
    }
    team.all_sum(s);
    if (!team.good) break;
    beta = s[0] / rz;
    rz = s[0];
    rr = s[1];
    ++count;
    ++done;
    fresh = false;
    T* t = now;
    now = old;
    old = t;
    stop = cg_stop(count, maxloop, rr, bnorm, eps);
    if (boss) hist.add(count, maxloop, rr, bnorm);
  }
  if (team.good) {
#pragma unroll
    for (int j = 0; j < RPT; ++j)
      if (A.has(j)) {
        const int32_t i = A.row0 + A.at(j);
        xs[i] = x[j];
        if (xout && (stop >= 0 || last)) xout[i] = (double)x[j];
      }
    if (boss) {
      if (mode == 1) { c->done = 0; c->ksz = 0; c->steps = 0; c->bnorm = bnorm; }
      c->count = count;
      c->nhist = hist.n;
      const double num = sqrt(rr);
      c->err = (bnorm == 0.0 && num == 0.0) ? 0.0 : num / bnorm;
      c->rr = rz;
      c->gamma = rr;
      c->alpha = alpha;
      c->beta = beta;
      c->steps += done;
      c->tsteps += done;
      c->stop = 0;
      c->status = 2;
      if (stop >= 0) ctl_stop(c, stop);
      st.count_many(2 * done, (unsigned long long)done * 4 * sizeof(T) * n);
    }
  }
  team.close();
}

}  // namespace ks
