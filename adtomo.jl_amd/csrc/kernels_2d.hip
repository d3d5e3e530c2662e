// 2D forward and adjoint of one event by one workgroup, each wave a band of
// rows, working values in LDS or registers.
//
// Forward (Eikonal.h:22-93).  a is the shorter axis, b the longer.  Lane p of a
// wave owns row p of its band of H <= 64 rows; step v updates the nodes
// (p, b = v - p), counted along the sweep: the reference's lexicographic pass in
// hyperplane order, so the values are its bits.  (a, b -+ 1) are the lane's own
// registers, (a -+ 1, b) the neighbouring lane's (one DPP shift), at a band's
// edges its neighbours' rows.  A wave runs as far as its neighbours' step counts
// allow; within an iteration nothing else synchronises the waves.  Two sets of
// waves take the even and the odd sweeps, so that a sweep follows the one before
// it by one axis length: 2 M_a + 3 N_b steps an iteration, not 4 (M_a + N_b).  Travel times
// sit in LDS with a border of +inf (a missing neighbour: the minimum ignores it),
// or, where they do not fit, in memory.
//
// What bounds it: the latency of a step (one local solve is a chain of some 20
// dependent FP64 operations), one wave a SIMD.  Measured against
// fwd2_event_kernel (one barrier a hyperplane, all values in memory), whole
// calls, FP64: 101 x 101 2.07 -> 0.47 ms (3 iterations, 0.26 us a step), 151 x
// 301 3.31 -> 0.90 ms, 400 x 400 (values in memory) 7.2 -> 2.9 ms, 1024 x 1500
// 68 -> 40 ms.
#include "buffer_ops.hpp"
#include "eikonal_device.hpp"
#include "kernels.hpp"

namespace adt {

namespace {

__device__ __forceinline__ int uni2(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ void fence2() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ int ld_lds(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st_lds(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int CTRL>
__device__ __forceinline__ double shift2(double edge, double x) {
  const uint64_t e = (uint64_t)__double_as_longlong(edge), b = (uint64_t)__double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)e, (int)b, CTRL, 0xf, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), CTRL,
                                                            0xf, 0xf, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ float shift2(float edge, float x) {
  return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(
      (int)__float_as_uint(edge), (int)__float_as_uint(x), CTRL, 0xf, 0xf, false));
}

// Slowness with which the fast solve gives the reference's bits: finite and far
// from overflow, f h zero or f and f h with squares above the subnormals (the
// root's argument is at least (f h)^2 where it is used).
template <typename T>
__device__ __forceinline__ bool tame2(T f, T h) {
  const T lo = sizeof(T) == 8 ? T(0x1p-380) : T(0x1p-60f), hi = sizeof(T) == 8 ? T(0x1p240) : T(0x1p20f);
  const T a = Real<T>::fabs_(f), b = Real<T>::fabs_(f * h);
  return a < hi && b < hi && (b == T(0) || (b >= lo && a >= lo));
}

// Eikonal.h:14-20 for tame operands, both branches evaluated.
template <typename T>
__device__ __forceinline__ T fast2(T a, T b, T f, T h) {
  const T fh = f * h, c = a - b, d = Real<T>::fabs_(c);
  const T one = Real<T>::min1_(a, b) + fh;
  const T two = (a + b + Real<T>::refine_(T(2.0) * f * f * h * h - c * c)) / T(2.0);
  return d >= fh ? one : two;
}

}  // namespace

// MEM: the travel times stay in memory.  Reports fault = 2 (nothing done) if
// the slowness is not tame, 1 if a wait ran out; u is then to be solved anew.
template <typename T, bool MEM>
__global__ void __launch_bounds__(1024) fwd2_band_kernel(Event2Desc ev, int max_iter) {
  __shared__ __attribute__((aligned(16))) char store[MEM ? 16 : kFwd2Lds];
  __shared__ int prog[4][16];  // steps done by each band in each sweep
  __shared__ T red[2][16];
  __shared__ int flag[3];
  T* const ul = (T*)store;
  const int m1 = ev.m + 1, n1 = ev.n + 1;
  const bool a_is_j = n1 <= m1;
  const int Ma = a_is_j ? n1 : m1, Nb = a_is_j ? m1 : n1;
  const int sA = a_is_j ? m1 : 1, sB = a_is_j ? 1 : m1;  // u[j * (m + 1) + i]
  const int N = Ma * Nb;
  const int as = a_is_j ? ev.jx : ev.ix, bs = a_is_j ? ev.ix : ev.jx;
  const int P = (Nb + 3) & ~1;  // LDS pitch, even: diagonals spread over the banks
  const int nt = (int)blockDim.x, waves = nt >> 6;
  const int NW = (Ma + 63) >> 6, sets = waves / NW;  // bands; sets of waves (1 or 2)
  const int wave = uni2(threadIdx.x >> 6), p = threadIdx.x & 63;
  const int w = wave % NW, set = wave / NW;
  const int H = (Ma + NW - 1) / NW;
  const T h = (T)ev.h, inf = (T)__builtin_inf();
  T* const u = (T*)ev.u;
  T* const uold = (T*)ev.uold;
  const T* const f = (const T*)ev.f;
  if (threadIdx.x < 2) flag[threadIdx.x] = 0;
  if (threadIdx.x == 0) *ev.info = adt_info{};
  __syncthreads();
  bool ok = Real<T>::fabs_(h) < T(0x1p20f);
  for (int q = threadIdx.x; q < N; q += nt) {
    ok = (int)ok & (int)tame2(f[q], h);
    const T v = q == ev.jx * m1 + ev.ix ? T(0) : T(100000.0);
    u[q] = v;
    uold[q] = v;
  }
  if constexpr (!MEM) {
    for (int q = threadIdx.x; q < (Ma + 2) * P; q += nt) {
      const int a = q / P - 1, b = q % P - 1;
      const bool in = a >= 0 && a < Ma && b >= 0 && b < Nb;
      ul[q] = !in ? inf : (a == as && b == bs) ? T(0) : T(100000.0);
    }
  }
  if (!ok) flag[0] = 1;
  __syncthreads();
  if (flag[0]) {
    if (threadIdx.x == 0) ev.info->fault = 2;
    return;
  }
  const rsrc_t ru = make_rsrc(u, (uint64_t)N * sizeof(T));
  const rsrc_t rf = make_rsrc(f, (uint64_t)N * sizeof(T));
  auto rows = [&](int band) {
    const int r = Ma - band * H;
    return r < H ? r : H;
  };
  const int nrow = rows(w);
  int it;
  bool conv = false;
  T err = T(0);
  for (it = 0; it < max_iter; ++it) {
    if (threadIdx.x < 64) prog[threadIdx.x >> 4][threadIdx.x & 15] = 0;
    __syncthreads();
    for (int sw = set; sw < 4; sw += sets) {
      const int dir = kDir2[sw];
      const bool fa = a_is_j ? (dir & 2) : (dir & 1), fb = a_is_j ? (dir & 1) : (dir & 2);
      const int prev = sw > 0 ? kDir2[sw > 0 ? sw - 1 : 0] ^ dir : 0;
      const bool Fa = a_is_j ? (prev & 2) : (prev & 1), Fb = a_is_j ? (prev & 1) : (prev & 2);
      // the bands before and after this one along the sweep
      const int wu = fa ? w + 1 : w - 1, wd = fa ? w - 1 : w + 1;
      const bool has_u = wu >= 0 && wu < NW, has_d = wd >= 0 && wd < NW;
      const int V = nrow + Nb - 1;
      const int hu = has_u ? rows(wu) : 0, hd = has_d ? rows(wd) : 0;
      const int capu = hu + Nb - 1, capd = hd + Nb - 1;
      // see allowed()
      const int kd = (Fa ? hd - 1 : 0) + (Fb ? Nb : 1);
      const int ko = 4 + (Fa ? nrow - 1 : 0) + (Fb ? Nb - 1 : 0);
      int* const pu = &prog[sw][has_u ? wu : w];
      int* const pd = &prog[sw > 0 ? sw - 1 : 0][has_d ? wd : w];
      int* const po = &prog[sw > 0 ? sw - 1 : 0][w];
      const bool row = p < nrow;
      const int ra = w * H + (fa ? nrow - 1 - p : p);  // the lane's row
      const int tA = fa ? -1 : 1, tB = fb ? -1 : 1;
      const int rbs = fb ? Nb - 1 - bs : bs;           // the source's canonical b
      const bool srow = row && ra == as;
      const bool first = p == 0, last = p == nrow - 1;
      // byte offset of (row, canonical b) in memory, and with MEM off its LDS
      // address; both advance by one column a step
      const int gB = (fb ? -sB : sB) * (int)sizeof(T), gA = tA * sA * (int)sizeof(T);
      const int lB = tB, lA = tA * P;
      int gq = (ra * sA + (fb ? (Nb - 1) * sB : 0)) * (int)sizeof(T) - p * gB;  // b = -p
      int lq = ((row ? ra : 0) + 1) * P + 1 + (fb ? Nb - 1 : 0) - p * lB;
      struct Fl {
        T old, f, up, dn;
      };
      auto in = [&](int b) { return (unsigned)b < (unsigned)Nb; };
      auto goff = [&](bool on, int q) -> uint32_t { return on ? (uint32_t)q : kOOB; };
      // what the step of column b (`k` columns from the current one) reads:
      // old(b + 1), f(b), the rows beyond the band; LDS cell 0 is +inf
      auto issue = [&](Fl& F, int b, int k) {
        const bool i0 = in(b), i1 = in(b + 1);
        F.f = bload(rf, goff(row && i0, gq + k * gB), T(0));
        if constexpr (MEM) {
          F.up = bload(ru, goff(first && has_u && i0, gq + k * gB - gA), T(0));
          F.dn = bload(ru, goff(last && has_d && i0, gq + k * gB + gA), T(0));
          F.old = bload(ru, goff(row && i1, gq + (k + 1) * gB), T(0));
        } else {
          const int c = lq + k * lB;
          F.old = ul[i1 ? c + lB : 0];
          F.up = ul[i0 ? c - lA : 0];
          F.dn = ul[i0 ? c + lA : 0];
        }
      };
      // The last step whose loads (those of step v + 2) the counts allow: in this
      // sweep the band before has finished the column of its last row next to our
      // first; in the sweep before, the band after has finished the column next
      // to our last, and our own band diagonal v + 3 (a flipped axis adds its
      // length).
      const int inf_v = 1 << 30;
      auto allowed = [&]() -> int {
        int r = inf_v;
        if (has_u) {
          const int c = uni2(ld_lds(pu));
          r = c >= capu ? r : c - 2 - hu;
        }
        if (sw > 0) {
          const int o = uni2(ld_lds(po));
          const int ro = o >= V ? inf_v : o - ko;
          r = ro < r ? ro : r;
          if (has_d) {
            const int c = uni2(ld_lds(pd));
            int rd = c >= capd ? inf_v : Fb ? (c >= kd ? inf_v : nrow - 4) : c - kd - 3 + nrow;
            rd = rd < nrow - 4 ? nrow - 4 : rd;  // its column 0 is not needed before
            r = rd < r ? rd : r;
          }
        }
        return r;
      };
      // Every count is reached, as a wave waits only for earlier steps in the order
      // (sweep, band); how long it takes grows with the grid (a sweep that flips the
      // long axis waits for all of the one before it).  So the bound is on the time
      // in which no count of the workgroup moves; past it a fault is reported.
      int safe = -2;
      auto wait = [&](int v) {
        int seen = -1;
        uint64_t t0 = 0;
        for (int spin = 0; (safe = allowed()) < v; ++spin) {
          if (uni2(ld_lds(&flag[1]))) {
            safe = inf_v;
            break;
          }
          if ((spin & 1023) == 1023) {
            const int c = ld_lds(&prog[p >> 4][p & 15]);
            const bool moved = __builtin_amdgcn_ballot_w64(c != seen) != 0;
            const uint64_t now = wall_clock64();
            seen = c;
            t0 = moved ? now : t0;
            if (now - t0 > kTeamPatience) st_lds(&flag[1], 1);
          }
          __builtin_amdgcn_s_sleep(1);
        }
        fence2();
      };
      int b = -p;
      Fl A, B;
      wait(-1);
      T OLDN, OWN, NEWP = inf;  // old(v+1), old(v) -> new(v), new(v-1)
      {
        T x;
        if constexpr (MEM) {
          x = bload(ru, goff(row && in(b), gq), T(0));
          x = row && in(b) ? x : inf;
        } else {
          x = ul[in(b) ? lq : 0];
        }
        OLDN = x;
      }
      // (each followed by stores like a step's, to nowhere: the loop is entered
      // with the operations in flight that its end leaves)
      auto no_store = [&]() {
        if constexpr (MEM) {
          bstore(ru, kOOB, inf);
        } else {
          if (p == 0) {
            ul[0] = inf;
            st_lds(&flag[2], 0);
          }
        }
        fence2();
      };
      issue(A, b, 0);
      no_store();
      issue(B, b + 1, 1);
      no_store();
      auto step = [&](int v, Fl& F) {
        OWN = OLDN;
        if constexpr (MEM)
          OLDN = row && in(b + 1) ? F.old : inf;
        else
          OLDN = F.old;
        T eu = F.up, ed = F.dn;
        if constexpr (MEM) {
          eu = has_u ? eu : inf;
          ed = has_d ? ed : inf;
        }
        const T ff = F.f;
        const T ua = shift2<0x138>(eu, NEWP);
        T da = shift2<0x130>(ed, OLDN);
        da = last ? ed : da;
        const T ma = Real<T>::min1_(ua, da);
        const T mb = Real<T>::min1_(NEWP, OLDN);
        asm volatile("" ::"v"(OLDN), "v"(ff) : "memory");
        if (__builtin_expect(v > safe, 0)) wait(v);
        fence2();
        issue(F, b + 2, 2);
        const bool val = row && in(b);
        // the reference's a is the x axis, b the y axis
        const T ax = a_is_j ? mb : ma, ay = a_is_j ? ma : mb;
        const T cand = fast2(ax, ay, ff, h);
        const bool upd = val && !(srow && b == rbs);
        const T nw = Real<T>::min1_(OWN, cand);
        OWN = upd ? nw : OWN;
        if constexpr (MEM) {
          bstore(ru, goff(val, gq), OWN);
          fence2();
          // loads that this step consumed were issued after step v-3's store
          if (p == 0) st_lds(&prog[sw][w], v > 2 ? v - 2 : 0);
        } else {
          ul[val ? lq : 1] = val ? OWN : inf;  // cell 1: border as well
          fence2();
          if (p == 0) st_lds(&prog[sw][w], v + 1);
        }
        NEWP = OWN;
        ++b;
        gq += gB;
        lq += lB;
      };
      int v = 0;
      for (; v + 1 < V; v += 2) {
        step(v, A);
        step(v + 1, B);
      }
      if (v < V) step(v, A);
      if constexpr (MEM) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      fence2();
      if (p == 0) st_lds(&prog[sw][w], V);
    }
    __syncthreads();
    // a wait ran out: over (nothing is written to the flag until the next sweeps)
    if (uni2(ld_lds(&flag[1]))) break;
    if constexpr (!MEM) {
      for (int q = threadIdx.x; q < N; q += nt) {
        const int j = q / m1, i = q - j * m1;
        const int a = a_is_j ? j : i, b = a_is_j ? i : j;
        u[q] = ul[(a + 1) * P + b + 1];
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    // ||u - u_old|| / ||u_old||, summed in the order of 1024 threads (node q on
    // thread q mod 1024), whatever the number of waves
    for (int vw = wave; vw < 16; vw += waves) {
      T sd = T(0), so = T(0);
      for (int q = vw * 64 + p; q < N; q += 1024) {
        const T x = u[q], y = uold[q];
        const T d = x - y;
        sd = sd + d * d;
        so = so + y * y;
        uold[q] = x;
      }
      for (int o = 32; o > 0; o >>= 1) {
        sd = sd + __shfl_xor(sd, o);
        so = so + __shfl_xor(so, o);
      }
      if (p == 0) {
        red[0][vw] = sd;
        red[1][vw] = so;
      }
    }
    __syncthreads();
    T sd = T(0), so = T(0);
    for (int q = 0; q < 16; ++q) {
      sd = sd + red[0][q];
      so = so + red[1][q];
    }
    err = Real<T>::sqrt_(sd) / Real<T>::sqrt_(so);
    if (threadIdx.x == 0 && it < kMaxLoggedIters) ev.info->err_log[it] = (double)err;
    if (err < T(1e-8)) {
      conv = true;
      break;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (flag[1]) ev.info->fault = ADT_FAULT;
    ev.info->iterations = conv ? it + 1 : it;
    ev.info->converged = conv ? 1 : 0;
    ev.info->err = (double)err;
    const double e = (double)err, thr = (double)T(1e-8);
    ev.info->ambiguous = (e > thr * (1 - 1e-12) && e < thr * (1 + 1e-12)) ? 1 : 0;
  }
}

template __global__ void fwd2_band_kernel<double, false>(Event2Desc, int);
template __global__ void fwd2_band_kernel<double, true>(Event2Desc, int);
template __global__ void fwd2_band_kernel<float, false>(Event2Desc, int);
template __global__ void fwd2_band_kernel<float, true>(Event2Desc, int);

// -------------------------------------------------------------- adjoint ---
//
// The triangular solve of Eikonal.h:95-199 level by level (a node resolves once
// every node that takes it as an upwind neighbour has), as adj2_kahn_kernel
// does it, with what a level touches in LDS: one byte per node (bits 0-1 the
// upwind side along x, 2-3 along y, 4-6 feeders not yet resolved, 7 the
// source; a singular node has no side and 7 feeders), the multipliers (LAM;
// else in memory) and the queues of this and the next level (entries past
// kAdj2Q in memory).  What bounds it: a level costs one barrier and one chain of
// LDS reads, a division and LDS atomics, about 1 us.  Measured, whole calls,
// FP64: 101 x 101 (LAM) 0.47 -> 0.20 ms, 151 x 301 (multipliers in memory) 1.14
// -> 0.50 ms, 330 x 340 2.26 -> 1.00 ms.  512 threads: 128 are slower from 300
// nodes a level on (151 x 301 0.83 ms), 256 at 0.58.

template <typename T, bool LAM>
__global__ void __launch_bounds__(512) adj2_lds_kernel(Event2Desc ev) {
  __shared__ __attribute__((aligned(16))) char store[kAdj2Lds];
  __shared__ int queue[2][kAdj2Q];
  __shared__ int cnt[3];
  __shared__ int nact, nsing;
  const int W = ev.m + 1, N = W * (ev.n + 1);
  const int nt = (int)blockDim.x;
  // one row of nothing before and after the grid: neighbours are read without
  // bounds (a row's end never takes the next row's start as its upwind side)
  uint8_t* const cd = (uint8_t*)store + ((W + 3) & ~3);
  T* const laml = (T*)(store + adj2_codes(W, N)) + W;
  gptr<T> const lamg = (gptr<T>)ev.lam;
  const rsrc_t ru = make_rsrc(ev.u, (uint64_t)N * sizeof(T));
  const rsrc_t rl = make_rsrc(ev.lam, (uint64_t)N * sizeof(T));
  // (an index before the array's start would wrap in the range check: such a
  // neighbour, which nothing uses, reads node 0)
  auto at = [](int q) { return (uint32_t)(q > 0 ? q : 0) * (uint32_t)sizeof(T); };
  auto get_u = [&](int q) { return bload(ru, at(q), T(0)); };
  auto put_lam = [&](int q, T x) {
    if constexpr (LAM)
      laml[q] = x;
    else
      lamg[q] = x;
  };
  auto get_lam = [&](int q) -> T {
    if constexpr (LAM)
      return laml[q];
    else
      return bload(rl, at(q), T(0));
  };
  for (int q = threadIdx.x; q < adj2_codes(W, N) / 4; q += nt) ((int*)store)[q] = 0;
  if (threadIdx.x == 0) {
    *ev.info = adt_info{};
    cnt[0] = cnt[1] = cnt[2] = 0;
    nact = nsing = 0;
  }
  if constexpr (LAM) {
    for (int q = threadIdx.x; q < W; q += nt) laml[q - W] = laml[N + q] = T(0);
  }
  __syncthreads();
  // --- sides (Eikonal.h:107-185); a multiplier starts as its source
  gptr<const T> const g = (gptr<const T>)ev.grad_u;
  for (int q = threadIdx.x; q < N; q += nt) {
    const int j = q / W, i = q - j * W;
    uint8_t c = 0;
    if (i == ev.ix && j == ev.jx) {
      c = 0x80;
    } else {
      const T up = get_u(q);
      const T xp = get_u(q + 1), xm = get_u(q - 1), yp = get_u(q + W), ym = get_u(q - W);
      const bool left = i > 0 && (i == ev.m || xp > xm);
      const bool down = j > 0 && (j == ev.n || yp > ym);
      if (up > (left ? xm : xp)) c |= left ? 1 : 2;
      if (up > (down ? ym : yp)) c |= down ? 4 : 8;
      if (!c) {
        c = 0x70;
        atomicAdd(&nsing, 1);
      }
    }
    put_lam(q, c == 0x70 ? T(0) : g[q]);
    cd[q] = c;
  }
  __syncthreads();
  // Appends one or two nodes of a lane to the queue of the level that `which`
  // counts.
  auto push = [&](bool on0, int node0, bool on1, int node1, int which, int par) {
    const uint64_t b0 = __ballot(on0), b1 = __ballot(on1);
    if (!(b0 | b1)) return;
    const int n0 = __builtin_popcountll(b0);
    int base = 0;
    if ((threadIdx.x & 63) == 0) base = atomicAdd(&cnt[which], n0 + __builtin_popcountll(b1));
    base = __builtin_amdgcn_readfirstlane(base);
    auto put = [&](bool on, uint64_t bal, int at, int node) {
      const int pos = at + (int)__builtin_amdgcn_mbcnt_hi(
                               (uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
      if (on) {
        if (pos < kAdj2Q)
          queue[par][pos] = node;
        else
          ev.queue[(int64_t)par * N + pos] = node;
      }
    };
    put(on0, b0, base, node0);
    put(on1, b1, base + n0, node1);
  };
  // --- feeders
  for (int q0 = 0; q0 < N; q0 += nt) {
    const int q = q0 + threadIdx.x;
    int c = 0x70, k = 0;
    if (q < N) {
      c = cd[q];
      k = ((cd[q - 1] & 3) == 2 ? 1 : 0) + ((cd[q + 1] & 3) == 1 ? 1 : 0) +
          ((cd[q - W] & 12) == 8 ? 1 : 0) + ((cd[q + W] & 12) == 4 ? 1 : 0);
      if (c != 0x70) cd[q] = (uint8_t)(c | (k << 4));
    }
    const bool act = c != 0x70;
    const uint64_t bal = __ballot(act);
    if ((threadIdx.x & 63) == 0 && bal) atomicAdd(&nact, __builtin_popcountll(bal));
    push(act && k == 0, q, false, 0, 0, 0);
  }
  __syncthreads();
  // --- levels
  int lev = 0, done = 0;
  for (;; ++lev) {
    const int cur = lev % 3, nxt = (lev + 1) % 3, par = lev & 1;
    const int n = cnt[cur];
    if (n == 0) break;
    if (threadIdx.x == 0) cnt[(lev + 2) % 3] = 0;
    done += n;
    for (int e0 = (threadIdx.x & ~63); e0 < n; e0 += nt) {
      const int e = e0 + (threadIdx.x & 63);
      const bool on = e < n;
      const int r = !on ? 0 : e < kAdj2Q ? queue[par][e] : ev.queue[(int64_t)par * N + e];
      const int q[4] = {r - 1, r + 1, r - W, r + W};
      T un[4], ln[4];
      int cn[4];
      const T ur = get_u(r);
#pragma unroll
      for (int k = 0; k < 4; ++k) un[k] = get_u(q[k]);
      const int c = cd[r];
      T num = get_lam(r);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        cn[k] = cd[q[k]];
        ln[k] = get_lam(q[k]);
      }
      T D = T(0);
      bool have = false;
#pragma unroll
      for (int d = 0; d < 2; ++d) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int k = 2 * d + s;
          const bool feeds = ((cn[k] >> (2 * d)) & 3) == (s ? 1 : 2);
          const T x = num + (T(2.0) * (un[k] - ur)) * ln[k];
          num = feeds ? x : num;
        }
        const int sd = (c >> (2 * d)) & 3;
        const T t = T(2.0) * (ur - (sd == 1 ? un[2 * d] : un[2 * d + 1]));
        D = sd ? (have ? D + t : t) : D;
        have = have || sd;
      }
      if (c & 0x80) D = T(1.0);
      if (on) put_lam(r, num / D);
      bool ready[2];
      int t[2];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int sd = (c >> (2 * d)) & 3;
        t[d] = sd == 1 ? q[2 * d] : q[2 * d + 1];
        const int ct = sd == 1 ? cn[2 * d] : cn[2 * d + 1];
        ready[d] = false;
        // a singular neighbour (no side, not the source) is never released
        if (on && sd && (ct & 0x8f)) {
          const int sh = (t[d] & 3) * 8 + 4;
          const unsigned old = atomicSub((unsigned*)(cd + (t[d] & ~3)), 1u << sh);
          ready[d] = ((old >> sh) & 7u) == 1u;
        }
      }
      push(ready[0], t[0], ready[1], t[1], nxt, par ^ 1);
    }
    if constexpr (!LAM) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  const T h = (T)ev.h;
  gptr<const T> const f = (gptr<const T>)ev.f;
  gptr<T> const gf = (gptr<T>)ev.grad_f;
  const int src = ev.jx * W + ev.ix;
  for (int q = threadIdx.x; q < N; q += nt) {
    T dFdf = T(-2.0) * f[q] * h * h;
    if (q == src) dFdf = T(0.0);
    gf[q] = -get_lam(q) * dFdf;
  }
  if (threadIdx.x == 0) {
    ev.info->n_singular = nsing;
    ev.info->adj_sweeps = lev;
    ev.info->adj_converged = done == nact ? 1 : 0;
  }
}

template __global__ void adj2_lds_kernel<double, true>(Event2Desc);
template __global__ void adj2_lds_kernel<double, false>(Event2Desc);
template __global__ void adj2_lds_kernel<float, true>(Event2Desc);
template __global__ void adj2_lds_kernel<float, false>(Event2Desc);

}  // namespace adt
