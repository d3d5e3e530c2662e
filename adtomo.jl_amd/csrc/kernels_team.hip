// 3D forward of events that leave compute units idle: several workgroups
// per event ("team"), all on one XCD.
//
// Work items.  The (a, b, k) grid of an event (a the shorter horizontal axis,
// b the longer, k contiguous) is cut into regions: bands of H <= 64 rows of a
// times slabs of kTW * LW nodes of k (LW = 16 bytes of nodes), each with all
// of b.  One item is one region of one sweep, done by one workgroup of kTW
// waves: wave w owns LW nodes of k, lane p row p of the band, and step v
// processes the anti-diagonal b = v - p of the region in every lane
// (hyperplane order, as in kernels_diag.hip, so the values are the reference's bit for
// bit).  Neighbours come from
//   (a, b -+ 1)  the lane's own registers (new values of diagonal v-1, old
//                values of v+1),
//   (a -+ 1, b)  the neighbouring lane's registers (one DPP shift); at the
//                ends of the band from memory,
//   (a, b, c-1)  the wave before through an LDS ring, at the slab's first wave
//                from memory; (a, b, c+1) from memory, one step ahead.
// Neighbours outside the grid are +inf, which the minimum ignores.
//
// Order between items.  Each region counts the diagonals of the current sweep
// whose new values are in memory.  An item runs as far as the counts it
// needs allow: in its own sweep those of the regions upwind along a and k, in
// the sweep before its own region's and those of the regions downwind.  The
// counts follow from the two sweeps' directions, so a sweep that flips a (b,
// k) runs one M_a (N_b, a few slabs) of steps behind the sweep before it: an
// iteration takes about 4 (M_a + N_b) + 30 slabs + 80 steps instead of the
// 8 (M_a + N_b + l) of sweeps run one after the other.
// (Several sweeps run on one region at a time, so a region has a count for each
// of four consecutive sweeps: any three flips in a row include one of a and one
// of b, so a sweep is complete before the third after it begins.)
//
// Items are numbered in an order in which each depends on lower numbers only,
// and workgroups draw the numbers of an event in order, so every wait is for
// an item that a running workgroup holds, whatever part of the grid is
// resident.
//
// One XCD per event.  A workgroup reads the XCD it runs on and joins an event
// that XCD has taken, so all of an event's values pass through that XCD's L2:
// stores reach it (the vector L1 writes through) and loads of travel times
// bypass the L1 (device scope), which is all the coherence the exchange needs.
// Store order: a wave's memory operations complete in the order issued, so a
// value loaded after a store proves the store complete.
//
// What bounds it.  One event: the latency of a step, about 2000 cycles of one
// wave per SIMD (two dependent local solves 870, the neighbours' minima 300, the
// next loads 270, progress checks and hand-over 580); 2700 where u and f exceed
// the XCD's 4 MB L2.  Two FP64 nodes per lane, because four would make a step 1.55
// times as long for 6% fewer of them.  Many events: the L2's rate of 16-byte
// accesses from 64 different columns (about 0.44 us per wave step and CU).
//
// Many events are taken by the wide form: eight nodes of k per lane (a slab is
// then 32 nodes), whose memory accesses cover whole 64-byte columns and change
// hands between lanes in LDS, one step ahead.  Its steps are 2.3 times as long, so
// an event alone takes twice the time, but the accesses cost a fifth, and what
// bounds it is the local solves (0.6 us per wave step and CU, two waves a SIMD: the
// 223 registers of FP64 allow no third, and one with spills is slower; the 152 of
// FP32 and 167 with FP64 solves would, which was not tried).
//
// Measured, forward alone, one workgroup per event -> 16 bytes -> eight nodes, ms of
// 20 iterations: 128x128x64 FP64 185, 37, 63; 64x64x32 94, 12, 30; 64 events of
// 128x128x64 with FP32 storage 180, 112, 78; 200 of 200x200x80 FP64 1237, 2196, 878;
// 256 of 128x128x64 FP64 250, 897, 297.  16 events of 400x400x160 with FP32 storage,
// up to their stop rule, 1476, 196, 106.
//
// Values the fast local solve does not cover (NaN, -0, infinities, values of
// 2^240 and more, discriminants below 2^-767) set the event's abort word; the
// diagonal kernel launched behind this one then solves the event from u0.  Such an
// event costs more than with that kernel alone: its first sweep here (256 uneven
// events with u0 infinite 52.0 -> 53.1 ms), and, where it is the only one of many, a
// solve behind the others' (46.8 -> 67.4 ms).
#include <type_traits>

#include "buffer_ops.hpp"
#include "eikonal_device.hpp"
#include "kernels.hpp"
#include "team_device.hpp"
#include "team_gate.hpp"

namespace adt {

namespace {

template <typename T>
using lptr = __attribute__((address_space(3))) T*;
using u32x4 = __attribute__((ext_vector_type(4))) unsigned int;

constexpr int kAuxDev = 16;  // sc1: device scope, past the vector L1
constexpr int kRing = 8;     // diagonals of the k exchange in LDS

template <typename T>
constexpr int kTL = 16 / (int)sizeof(T);  // nodes of k per lane

__device__ __forceinline__ int ld_wg(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st_wg(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The event is finished or aborted: nobody waits for its items any more.
__device__ __forceinline__ bool gone(gptr<const int> words) {
  return ld_dev(&words[kTeamState]) >= kTeamOver || ld_dev(&words[kTeamAbort]) != 0;
}
// Bounded polling: call with every unsuccessful poll.  True when the wait is
// to be given up; one that ran out of time aborts the event (which the
// diagonal kernel then solves).
struct TPatience {
  int spin = 0;
  uint64_t t0 = 0;
  __device__ __forceinline__ bool over(words_t words) {
    if (++spin > 2) __builtin_amdgcn_s_sleep(1);
    if ((spin & 63) != 0) return false;
    if (uni(gone(words) ? 1 : 0)) return true;
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (now - t0 <= kTeamPatience) return false;
    st_xcd(&words[kTeamAbort], 2);
    return true;
  }
};
__device__ __forceinline__ double ld_old(rsrc_t r, uint32_t off, double) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kAuxDev));
}
__device__ __forceinline__ float ld_old(rsrc_t r, uint32_t off, float) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kAuxDev));
}

// The lane's LW nodes in canonical order (FC: the sweep runs k downwards);
// a segment of cnt < LW nodes (FULL off) keeps the rest of the array unused.
template <typename T, bool FULL, bool FC, int AUX>
__device__ __forceinline__ void ld_seg(T (&x)[kTL<T>], rsrc_t r, uint32_t off, int cnt) {
  constexpr int LW = kTL<T>;
  if constexpr (FULL) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
    const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = FC ? LW - 1 - e : e;
      if constexpr (sizeof(T) == 8)
        x[e] = __longlong_as_double((long long)(((uint64_t)w[2 * m + 1] << 32) | w[2 * m]));
      else
        x[e] = __uint_as_float(w[m]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = FC ? cnt - 1 - e : e;
      const uint32_t o = (off != kOOB && e < cnt) ? off + (uint32_t)(m * (int)sizeof(T)) : kOOB;
      if constexpr (sizeof(T) == 8)
        x[e] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, AUX));
      else
        x[e] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, AUX));
    }
  }
}

template <typename T, bool FULL, bool FC>
__device__ __forceinline__ void st_seg(const T (&x)[kTL<T>], rsrc_t r, uint32_t off, int cnt) {
  constexpr int LW = kTL<T>;
  if constexpr (FULL) {
    unsigned w[4];
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = FC ? LW - 1 - e : e;
      if constexpr (sizeof(T) == 8) {
        const uint64_t b = (uint64_t)__double_as_longlong(x[e]);
        w[2 * m] = (unsigned)b;
        w[2 * m + 1] = (unsigned)(b >> 32);
      } else {
        w[m] = __float_as_uint(x[e]);
      }
    }
    u32x4 v;
    v.x = w[0];
    v.y = w[1];
    v.z = w[2];
    v.w = w[3];
    __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 0);
  } else {
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = FC ? cnt - 1 - e : e;
      const uint32_t o = (off != kOOB && e < cnt) ? off + (uint32_t)(m * (int)sizeof(T)) : kOOB;
      bstore(r, o, x[e]);
    }
  }
}

// The value of the lane before (after); the first (last) lane keeps `edge`.
template <int CTRL>
__device__ __forceinline__ double dpp_shift(double edge, double x) {
  const uint64_t e = (uint64_t)__double_as_longlong(edge), b = (uint64_t)__double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)e, (int)b, CTRL, 0xf, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(e >> 32), (int)(b >> 32), CTRL,
                                                            0xf, 0xf, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ float dpp_shift(float edge, float x) {
  return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(
      (int)__float_as_uint(edge), (int)__float_as_uint(x), CTRL, 0xf, 0xf, false));
}
constexpr int kDppUp = 0x138;  // wave_shr:1: lane p reads lane p - 1
constexpr int kDppDn = 0x130;  // wave_shl:1: lane p reads lane p + 1

// Uniform description of one item (one region of one sweep).
template <typename T>
struct TItem {
  int Hr, Nb, V;      // rows of the band, nodes of b, diagonals Hr + Nb - 1
  int l, k0, cnt;     // k extent; this wave's lowest node and its node count
  int nw;             // active waves (segments) of the slab
  int off0;           // byte offset of (row 0, b = 0, node k0), canonical
  int dA, dB;         // byte steps of one canonical row / column
  bool up, dn;        // the band has a neighbour before / after it
  bool first;         // the event's first sweep: old values are u0
  int seqbase;        // count base of this sweep
  T h;
  double hd;
  rsrc_t u, src, f;
};

// What lane i < 5 of the first wave watches (a region's count), and what the
// loads issued in step v (those of step v + 2) need of it.
struct TWatch {
  gptr<const int> ptr;
  int base, xo, sg, K, cap;
  int have;
  __device__ __forceinline__ int need(int v) const {
    const int x = v + xo;
    const int n = sg * x + K;
    return x < 0 ? base : base + (n < cap ? n : cap);
  }
};

// Waits until every watched count is high enough; false if the event is gone.
__device__ __forceinline__ bool watch_wait(TWatch& W, int v, int lane, words_t words) {
  TPatience wait;
  for (;;) {
    const bool ok = lane >= 5 || W.have >= W.need(v);
    if (__builtin_amdgcn_ballot_w64(!ok) == 0) return true;
    W.have = ld_dev(W.ptr);
    // here, not after the loop, where every step would wait for it
    asm volatile("" ::"v"(W.have));
    if (wait.over(words)) return false;
  }
}

// A wave's progress for the wave after it: steps finished and, below, the
// diagonals whose stores it and the waves before it have completed.
__device__ __forceinline__ void put_prog(uint64_t* p, int steps, int done) {
  __hip_atomic_store(p, ((uint64_t)(unsigned)steps << 32) | (unsigned)done, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int get_prog(const uint64_t* p, int& done) {
  const uint64_t x = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  done = uni((int)(unsigned)x);
  return uni((int)(x >> 32));
}

// A copy in registers of its own (the compiler would otherwise keep the value
// where it is and move the load that takes its place, waiting for it).
__device__ __forceinline__ float own_copy(float x) {
  float r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}
__device__ __forceinline__ double own_copy(double x) {
  double r;
  asm volatile("v_mov_b64 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// What a step reads, two steps ahead.
template <typename T>
struct TFlight {
  T old[kTL<T>];  // old(v+1)
  T f[kTL<T>];    // slowness of v
  T xd;           // old value past the segment's end
  T up[kTL<T>];   // first lane: new values of the row before the band
  T dn[kTL<T>];   // last lane of a 64-row band: old values of the row after it
  T xc;           // first wave: new value before the segment
  int have;       // first wave: the watched counts
};

// Steps of one wave of an item; false if the event is gone.  Two sets of
// registers take the loads of even and odd steps, issued two steps ahead, so
// no load in flight is copied (a copy would wait for it, and for the stores
// behind it).
template <typename T, bool MIX, bool FULL, bool FC>
__device__ __forceinline__ bool team_sweep(const TItem<T>& S, TWatch W, int w, words_t count,
                                           words_t words, lptr<T> ring, uint64_t* prog,
                                           int* stop) {
  constexpr int LW = kTL<T>;
  constexpr int SZ = (int)sizeof(T);
  const int p = threadIdx.x & 63;
  const int cnt = FULL ? LW : S.cnt;
  const T inf = (T)__builtin_inf();
  const bool lastw = w == S.nw - 1;
  // canonical c-1 of the segment's first node and c+1 of its last
  const int klo = S.k0 - 1, khi = S.k0 + cnt;
  const bool has_cm = FC ? khi < S.l : klo >= 0;
  const bool has_cp = FC ? klo >= 0 : khi < S.l;
  const int dcm = FC ? cnt * SZ : -SZ, dcp = FC ? -SZ : cnt * SZ;
  const bool mem_cm = w == 0 && has_cm;
  const bool row = p < S.Hr;
  // lane Hr (where there is one) only loads: the row after the band
  const bool loads = row || (p == S.Hr && S.dn);
  const bool edge64 = S.Hr == 64 && S.dn;
  const bool top = p == 0, bot = p == 63;
  // byte offset of the lane's column at diagonal v, and its b
  int off = S.off0 + p * (S.dA - S.dB);  // v = 0
  int b = -p;
  auto sel = [](bool ok, int o) -> uint32_t { return ok ? (uint32_t)o : kOOB; };
  bool unsafe = false;
  auto wild = [&](const T (&x)[LW]) {
    bool r = false;
#pragma unroll
    for (int e = 0; e < LW; ++e)
      if (FULL || e < cnt) r = (int)r | (int)Real<T>::wild_(x[e]) | (int)Real<T>::odd_(x[e]);
    return r;
  };
  // What the step of column (o, bb) reads: first what only some items read (a
  // load that may be left out sits before those that are always there, so the
  // waits for these stay exact), then old(v+1), the slowness and the old value
  // past the segment's end.
  auto issue = [&](TFlight<T>& F, int o, int bb) {
    const bool in = (unsigned)bb < (unsigned)S.Nb;
    if (S.up) ld_seg<T, FULL, FC, kAuxDev>(F.up, S.u, sel(in && top, o - S.dA), cnt);
    if (edge64) ld_seg<T, FULL, FC, kAuxDev>(F.dn, S.src, sel(in && bot, o + S.dA), cnt);
    if (mem_cm) F.xc = ld_old(S.u, sel(in && row, o + dcm), T(0));
    if (w == 0) F.have = ld_dev(W.ptr);
    code_fence();
    ld_seg<T, FULL, FC, kAuxDev>(
        F.old, S.src, sel(loads && (unsigned)(bb + 1) < (unsigned)S.Nb, o + S.dB), cnt);
    code_fence();
    ld_seg<T, FULL, FC, 0>(F.f, S.f, sel(in && row, o), cnt);
    code_fence();
    F.xd = ld_old(S.src, sel(in && row && has_cp, o + dcp), T(0));
  };

  // prologue: old(0), and what step 0 reads
  bool ok = true;
  if (w == 0) {
    ok = watch_wait(W, -1, p, words);
    if (!ok) st_wg(stop, 1);
  } else {
    int d;
    while (get_prog(&prog[w - 1], d) < 0) {
      if (uni(ld_wg(stop))) {
        ok = false;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (!ok) return false;
  code_fence();
  TFlight<T> A, B;
  A.xc = B.xc = inf;
#pragma unroll
  for (int e = 0; e < LW; ++e) A.up[e] = A.dn[e] = B.up[e] = B.dn[e] = inf;
  T NEWP[LW], OWN[LW], OLDN[LW];  // new(v-1), old(v) -> new(v), old(v+1)
  ld_seg<T, FULL, FC, kAuxDev>(OWN, S.src, sel(loads && (unsigned)b < (unsigned)S.Nb, off), cnt);
  code_fence();
  // (each followed by a store like a step's, which the range check drops: the
  // loop is entered with the operations in flight that its end leaves)
  issue(A, off, b);
  code_fence();
  st_seg<T, FULL, FC>(OWN, S.u, kOOB, cnt);
  code_fence();
  issue(B, off + S.dB, b + 1);
  code_fence();
  st_seg<T, FULL, FC>(OWN, S.u, kOOB, cnt);
  code_fence();
  if (p == 0) put_prog(&prog[w], 0, 0);
  {
    const bool in = loads && (unsigned)b < (unsigned)S.Nb;
    if (S.first) unsafe = (int)unsafe | (int)wild(OWN);
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      NEWP[e] = inf;
      OLDN[e] = in ? OWN[e] : inf;  // becomes OWN in the first step
    }
  }
  // One step: F holds what it reads and then takes the loads of the step after
  // the next.  Once the event is gone (ok is off) the remaining steps run
  // without waiting: its travel times are then written anew by the diagonal
  // kernel, and no path leaves a step early (the waits for loads would lose
  // count).
  int dn_seen = 0;  // steps the wave after has finished, as last read
  auto step = [&](int v, TFlight<T>& F) {
    // the wave before: progress, then the value it hands over (the LDS reads
    // of a wave run in order: the value is there if the progress says so)
    uint64_t pr = 0;
    T xr = inf;
    if (w > 0) {
      pr = __hip_atomic_load(&prog[w - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      code_fence();
      xr = ring[((w - 1) * kRing + (v & (kRing - 1))) * 64 + p];
    }
    const bool in1 = loads && (unsigned)(b + 1) < (unsigned)S.Nb;
    const bool val = row && (unsigned)b < (unsigned)S.Nb;
    T ma[LW], mb[LW], f[LW];
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      OWN[e] = OLDN[e];
      OLDN[e] = in1 ? F.old[e] : inf;
      f[e] = own_copy(F.f[e]);
      // minima along a and b (the neighbouring lanes; at the band's ends from memory)
      const T ua = dpp_shift<kDppUp>(F.up[e], NEWP[e]);
      const T da = dpp_shift<kDppDn>(F.dn[e], OLDN[e]);
      ma[e] = Real<T>::min1_(ua, da);
      mb[e] = Real<T>::min1_(NEWP[e], OLDN[e]);
    }
    const T xd = has_cp ? own_copy(F.xd) : inf;
    T xc = own_copy(F.xc);
    if (S.first) {
      unsafe = (int)unsafe | (int)wild(F.old);
      bool r = false;
#pragma unroll
      for (int e = 0; e < LW; ++e)
        if (FULL || e < cnt) r = (int)r | (int)Real<T>::wild_(f[e]);
      unsafe = (int)unsafe | (int)r;
    }
    // these loads were issued after step v-3's stores, which are complete then
    asm volatile("" ::"v"(OLDN[0]), "v"(f[0]), "v"(xd) : "memory");
    int done = v - 2 > 0 ? v - 2 : 0;
    if (w > 0) {
      if (__builtin_expect(uni((int)(pr >> 32)) < v + 1, 0)) {
        int d;
        while (get_prog(&prog[w - 1], d) < v + 1 && ok) {
          if (uni(ld_wg(stop))) ok = false;
        }
        pr = (unsigned)d;
        code_fence();
        xr = ring[((w - 1) * kRing + (v & (kRing - 1))) * 64 + p];
      }
      const int up_done = uni((int)(unsigned)pr);
      done = done < up_done ? done : up_done;
      xc = xr;
    } else {
      W.have = F.have;
      const bool low = p < 5 && W.have < W.need(v);
      if (__builtin_amdgcn_ballot_w64(low) != 0 && ok && !watch_wait(W, v, p, words)) {
        st_wg(stop, 1);
        ok = false;
      }
    }
    code_fence();
    // ---- loads of the step after the next
    issue(F, off + 2 * S.dB, b + 2);
    // ---- the lane's nodes
    if (val) {
#pragma unroll
      for (int e = 0; e < LW; ++e) {
        if (FULL || e < cnt) {
          const T cm = e == 0 ? xc : OWN[e == 0 ? 0 : e - 1];
          const T cp = (FULL ? e + 1 < LW : e + 1 < cnt) ? OWN[e + 1 < LW ? e + 1 : e] : xd;
          const T mc = Real<T>::min1_(cm, cp);
          T cand;
          if constexpr (MIX)
            cand = (T)solution3d<double, true>(ma[e], mb[e], mc, f[e], S.hd, unsafe);
          else
            cand = solution3d<T, true>(ma[e], mb[e], mc, f[e], S.h, unsafe);
          unsafe = (int)unsafe | (int)Real<T>::odd_(cand);
          OWN[e] = Real<T>::min1_(cand, OWN[e]);
        }
      }
    }
    // ---- hand over: the last node to the wave after, the values to memory
    // (a wave's LDS operations run in order: the value before the progress)
    if (!lastw) {
      T xo = OWN[LW - 1];
      if constexpr (!FULL) {
#pragma unroll
        for (int e = 0; e < LW; ++e)
          if (e == cnt - 1) xo = OWN[e];
      }
      // slot v & 7 was read by the wave after at its step v - 8
      while (dn_seen < v - kRing + 1 && ok) {
        int d;
        dn_seen = get_prog(&prog[w + 1], d);
        if (dn_seen < v - kRing + 1 && uni(ld_wg(stop))) ok = false;
      }
      ring[(w * kRing + (v & (kRing - 1))) * 64 + p] = xo;
      code_fence();
    }
    if (p == 0) {
      put_prog(&prog[w], v + 1, done);
      if (lastw) st_xcd(count, S.seqbase + done);
    }
    st_seg<T, FULL, FC>(OWN, S.u, sel(val, off), cnt);
    code_fence();
#pragma unroll
    for (int e = 0; e < LW; ++e) NEWP[e] = OWN[e];
    off += S.dB;
    ++b;
  };
  int v = 0;
  for (; v + 1 < S.V; v += 2) {
    step(v, A);
    step(v + 1, B);
  }
  if (v < S.V) step(v, A);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (__builtin_amdgcn_ballot_w64(unsafe) != 0 && p == 0) st_xcd(&words[kTeamAbort], 1);
  return ok;
}

// ---- the wide form: eight nodes of k per lane
//
// Memory is read and written in 16-byte pieces, the NP pieces of a column by
// neighbouring lanes (64 / NP columns an instruction), and the pieces change hands
// in LDS.  Staging of a wave: 64 columns of NP pieces, those of FP64 rotated by
// their column's number so that neither side has bank conflicts, and behind them
// the rows beyond the band.
constexpr int kTWide = 8;  // nodes of k per lane
template <typename T>
constexpr int kNP = kTWide * (int)sizeof(T) / 16;  // pieces of a column
template <typename T>
constexpr int kStage = 66 * kNP<T>;                // pieces of a staging area
template <typename T>
__device__ __forceinline__ int stage_rot(int col) {
  return kNP<T> == 4 ? (col >> 2) & 3 : 0;
}

// What a step of the wide form reads, one step ahead.
template <typename T>
struct TWideFlight {
  // piece lane % NP of columns j 64 / NP + lane / NP
  u32x4 old[kNP<T>], f[kNP<T>];
  u32x4 up, dn;  // the first NP lanes: pieces of the rows beyond the band
  T xd, xc;
  int have;
};

// Nodes of one column out of the staging area (`at`: its first piece; rot: its
// rotation), canonical order; entries from cnt on are not used.
template <typename T, bool FULL, bool FC>
__device__ __forceinline__ void from_stage(T (&x)[kTWide], lptr<u32x4> st, int at, int rot, int cnt) {
  constexpr int LW = kTWide, PER = 16 / (int)sizeof(T), NP = kNP<T>;
  if constexpr (FULL) {
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      const u32x4 v = st[at + ((c + rot) & (NP - 1))];
      const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int m = c * PER + i, e = FC ? LW - 1 - m : m;
        if constexpr (sizeof(T) == 8)
          x[e] = __longlong_as_double((long long)(((uint64_t)w[2 * i + 1] << 32) | w[2 * i]));
        else
          x[e] = __uint_as_float(w[i]);
      }
    }
  } else {
    const lptr<T> q = (lptr<T>)st;
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = e < cnt ? (FC ? cnt - 1 - e : e) : 0;
      x[e] = q[(at + ((m / PER + rot) & (NP - 1))) * PER + m % PER];
    }
  }
}
template <typename T, bool FULL, bool FC>
__device__ __forceinline__ void to_stage(const T (&x)[kTWide], lptr<u32x4> st, int at, int rot, int cnt) {
  constexpr int LW = kTWide, PER = 16 / (int)sizeof(T), NP = kNP<T>;
  if constexpr (FULL) {
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      unsigned w[4];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int m = c * PER + i, e = FC ? LW - 1 - m : m;
        if constexpr (sizeof(T) == 8) {
          const uint64_t b = (uint64_t)__double_as_longlong(x[e]);
          w[2 * i] = (unsigned)b;
          w[2 * i + 1] = (unsigned)(b >> 32);
        } else {
          w[i] = __float_as_uint(x[e]);
        }
      }
      u32x4 v;
      v.x = w[0];
      v.y = w[1];
      v.z = w[2];
      v.w = w[3];
      st[at + ((c + rot) & (NP - 1))] = v;
    }
  } else {
    const lptr<T> q = (lptr<T>)st;
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      const int m = FC ? cnt - 1 - e : e;
      if (e < cnt) q[(at + ((m / PER + rot) & (NP - 1))) * PER + m % PER] = x[e];
    }
  }
}

// As team_sweep, with loads one step ahead: what a step consumes was issued
// after the stores of the step two before it.
template <typename T, bool MIX, bool FULL, bool FC>
__device__ __forceinline__ bool team_sweep_wide(const TItem<T>& S, TWatch W, int w, words_t count,
                                                words_t words, lptr<T> ring, lptr<u32x4> st,
                                                uint64_t* prog, int* stop) {
  constexpr int LW = kTWide;
  constexpr int SZ = (int)sizeof(T), PER = 16 / SZ, NP = kNP<T>, CP = 64 / NP;
  const int p = threadIdx.x & 63;
  const int cnt = FULL ? LW : S.cnt;
  const T inf = (T)__builtin_inf();
  const bool lastw = w == S.nw - 1;
  const int klo = S.k0 - 1, khi = S.k0 + cnt;
  const bool has_cm = FC ? khi < S.l : klo >= 0;
  const bool has_cp = FC ? klo >= 0 : khi < S.l;
  const int dcm = FC ? cnt * SZ : -SZ, dcp = FC ? -SZ : cnt * SZ;
  const bool mem_cm = w == 0 && has_cm;
  const bool row = p < S.Hr;
  const bool loads = row || (p == S.Hr && S.dn);
  const bool edge64 = S.Hr == 64 && S.dn;
  const int dC = S.dA - S.dB;  // bytes from a column to the next of its diagonal
  int off = S.off0 + p * dC, b = -p;                    // the lane's column
  int qoff = S.off0 + (p / NP) * dC + (p % NP) * 16;     // the lane's piece, first of four
  int qb = -(p / NP);
  const bool piece = FULL || (p % NP) * PER < cnt;       // (pieces past the segment: not read)
  // (the rotation of column CP j + p / NP does not depend on j)
  const int qat = (p / NP) * NP + ((p % NP + stage_rot<T>(p / NP)) & (NP - 1));  // its place in the staging area
  const int at = p * NP, rot = stage_rot<T>(p);             // the lane's column there
  auto sel = [](bool ok, int o) -> uint32_t { return ok ? (uint32_t)o : kOOB; };
  bool unsafe = false;
  auto wild = [&](const T (&x)[LW]) {
    bool r = false;
#pragma unroll
    for (int e = 0; e < LW; ++e)
      if (FULL || e < cnt) r = (int)r | (int)Real<T>::wild_(x[e]) | (int)Real<T>::odd_(x[e]);
    return r;
  };
  auto in = [&](int bb) { return (unsigned)bb < (unsigned)S.Nb; };
  auto ld_old4 = [&](u32x4 (&x)[NP], int o, int bb) {  // old values of the columns at (o, bb)
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int col = CP * j + (p / NP);
      const bool ok = piece && (col < S.Hr || (col == S.Hr && S.dn)) && in(bb - CP * j);
      x[j] = __builtin_amdgcn_raw_buffer_load_b128(S.src, sel(ok, o + CP * j * dC), 0, kAuxDev);
    }
  };
  auto put4 = [&](const u32x4 (&x)[NP]) {
#pragma unroll
    for (int j = 0; j < NP; ++j) st[qat + 64 * j] = x[j];
  };
  // what step v reads (v = the diagonal of off, b, qoff, qb plus k columns)
  auto issue = [&](TWideFlight<T>& F, int v, int k) {
    const bool ends = p < NP && piece;
    if (S.up)
      F.up = __builtin_amdgcn_raw_buffer_load_b128(
          S.u, sel(ends && in(v), S.off0 + v * S.dB - S.dA + p * 16), 0, kAuxDev);
    if (edge64)
      F.dn = __builtin_amdgcn_raw_buffer_load_b128(
          S.src, sel(ends && in(v - 63), S.off0 + v * S.dB + 63 * dC + S.dA + p * 16), 0, kAuxDev);
    if (mem_cm) F.xc = ld_old(S.u, sel(in(b + k) && row, off + k * S.dB + dcm), T(0));
    if (w == 0) F.have = ld_dev(W.ptr);
    code_fence();
    ld_old4(F.old, qoff + (k + 1) * S.dB, qb + k + 1);
    code_fence();
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const bool ok = piece && CP * j + (p / NP) < S.Hr && in(qb + k - CP * j);
      F.f[j] = __builtin_amdgcn_raw_buffer_load_b128(S.f, sel(ok, qoff + k * S.dB + CP * j * dC), 0, 0);
    }
    code_fence();
    F.xd = ld_old(S.src, sel(in(b + k) && row && has_cp, off + k * S.dB + dcp), T(0));
  };
  // the diagonal's values out of the staging area into memory
  auto st4 = [&](int o, int bb, bool on) {
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const bool ok = on && piece && CP * j + (p / NP) < S.Hr && in(bb - CP * j);
      const u32x4 x = st[qat + 64 * j];
      const uint32_t a = sel(ok, o + CP * j * dC);
      if constexpr (FULL) {
        __builtin_amdgcn_raw_buffer_store_b128(x, S.u, a, 0, 0);
      } else {
        const unsigned y[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          const uint32_t ai = ok && (p % NP) * PER + i < cnt ? a + (uint32_t)(i * SZ) : kOOB;
          if constexpr (sizeof(T) == 8)
            bstore(S.u, ai, __longlong_as_double((long long)(((uint64_t)y[2 * i + 1] << 32) | y[2 * i])));
          else
            bstore(S.u, ai, __uint_as_float(y[i]));
        }
      }
    }
  };

  bool ok = true;
  if (w == 0) {
    ok = watch_wait(W, -1, p, words);
    if (!ok) st_wg(stop, 1);
  } else {
    int d;
    while (get_prog(&prog[w - 1], d) < 0) {
      if (uni(ld_wg(stop))) {
        ok = false;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (!ok) return false;
  code_fence();
  TWideFlight<T> F;
  F.xc = inf;
  T NEWP[LW], OWN[LW], OLDN[LW];  // new(v-1), old(v) -> new(v), old(v+1)
  ld_old4(F.old, qoff, qb);
  put4(F.old);
  code_fence();
  from_stage<T, FULL, FC>(OWN, st, at, rot, cnt);
  code_fence();
  issue(F, 0, 0);
  code_fence();
  st4(qoff, qb, false);
  code_fence();
  if (p == 0) put_prog(&prog[w], 0, 0);
  {
    const bool i0 = loads && in(b);
    if (S.first) unsafe = (int)unsafe | (int)wild(OWN);
#pragma unroll
    for (int e = 0; e < LW; ++e) {
      NEWP[e] = inf;
      OLDN[e] = i0 ? OWN[e] : inf;
    }
  }
  int dn_seen = 0;
  for (int v = 0; v < S.V; ++v) {
    uint64_t pr = 0;
    T xr = inf;
    if (w > 0) {
      pr = __hip_atomic_load(&prog[w - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      code_fence();
      xr = ring[((w - 1) * kRing + (v & (kRing - 1))) * 64 + p];
    }
    const bool in1 = loads && in(b + 1);
    const bool val = row && in(b);
    T ma[LW], f[LW];
    {
      T x[LW];
      code_fence();
      put4(F.old);
      code_fence();
      from_stage<T, FULL, FC>(x, st, at, rot, cnt);
      code_fence();
      put4(F.f);
      code_fence();
      from_stage<T, FULL, FC>(f, st, at, rot, cnt);
      if (S.first) {
        unsafe = (int)unsafe | (int)wild(x);
        bool r = false;
#pragma unroll
        for (int e = 0; e < LW; ++e)
          if (FULL || e < cnt) r = (int)r | (int)Real<T>::wild_(f[e]);
        unsafe = (int)unsafe | (int)r;
      }
#pragma unroll
      for (int e = 0; e < LW; ++e) {
        OWN[e] = OLDN[e];
        OLDN[e] = in1 ? x[e] : inf;
      }
      T eu[LW], ed[LW];
#pragma unroll
      for (int e = 0; e < LW; ++e) eu[e] = ed[e] = inf;
      if (S.up) {
        if (p < NP) st[64 * NP + p] = F.up;
        code_fence();
        from_stage<T, FULL, FC>(eu, st, 64 * NP, 0, cnt);
      }
      if (edge64) {
        if (p < NP) st[65 * NP + p] = F.dn;
        code_fence();
        from_stage<T, FULL, FC>(ed, st, 65 * NP, 0, cnt);
      }
      code_fence();
#pragma unroll
      for (int e = 0; e < LW; ++e)
        ma[e] = Real<T>::min1_(dpp_shift<kDppUp>(eu[e], NEWP[e]), dpp_shift<kDppDn>(ed[e], OLDN[e]));
    }
    const T xd = has_cp ? own_copy(F.xd) : inf;
    T xc = own_copy(F.xc);
    // these loads were issued after step v-2's stores, which are complete then
    asm volatile("" ::"v"(OLDN[0]), "v"(f[0]), "v"(xd) : "memory");
    int done = v - 1 > 0 ? v - 1 : 0;
    if (w > 0) {
      if (__builtin_expect(uni((int)(pr >> 32)) < v + 1, 0)) {
        int d;
        while (get_prog(&prog[w - 1], d) < v + 1 && ok) {
          if (uni(ld_wg(stop))) ok = false;
          __builtin_amdgcn_s_sleep(1);
        }
        pr = (unsigned)d;
        code_fence();
        xr = ring[((w - 1) * kRing + (v & (kRing - 1))) * 64 + p];
      }
      const int up_done = uni((int)(unsigned)pr);
      done = done < up_done ? done : up_done;
      xc = xr;
    } else {
      W.have = F.have;
      const bool low = p < 5 && W.have < W.need(v - 1);
      if (__builtin_amdgcn_ballot_w64(low) != 0 && ok && !watch_wait(W, v - 1, p, words)) {
        st_wg(stop, 1);
        ok = false;
      }
    }
    code_fence();
    issue(F, v + 1, 1);
    // (ahead of the other wave of the SIMD until the step's values are on their
    // way: 64 events of 128x128x64 with FP32 storage 13.8 -> 12.2 ms)
    __builtin_amdgcn_s_setprio(3);
    // ---- the lane's nodes
    if (val) {
#pragma unroll
      for (int e = 0; e < LW; ++e) {
        if (FULL || e < cnt) {
          const T cm = e == 0 ? xc : OWN[e == 0 ? 0 : e - 1];
          const T cp = (FULL ? e + 1 < LW : e + 1 < cnt) ? OWN[e + 1 < LW ? e + 1 : e] : xd;
          const T mc = Real<T>::min1_(cm, cp);
          const T mb = Real<T>::min1_(NEWP[e], OLDN[e]);
          T cand;
          if constexpr (MIX)
            cand = (T)solution3d<double, true>(ma[e], mb, mc, f[e], S.hd, unsafe);
          else
            cand = solution3d<T, true>(ma[e], mb, mc, f[e], S.h, unsafe);
          unsafe = (int)unsafe | (int)Real<T>::odd_(cand);
          OWN[e] = Real<T>::min1_(cand, OWN[e]);
        }
      }
    }
    if (!lastw) {
      T xo = OWN[LW - 1];
      if constexpr (!FULL) {
#pragma unroll
        for (int e = 0; e < LW; ++e)
          if (e == cnt - 1) xo = OWN[e];
      }
      while (dn_seen < v - kRing + 1 && ok) {
        int d;
        dn_seen = get_prog(&prog[w + 1], d);
        if (dn_seen < v - kRing + 1 && uni(ld_wg(stop))) ok = false;
      }
      ring[(w * kRing + (v & (kRing - 1))) * 64 + p] = xo;
      code_fence();
    }
    if (p == 0) {
      put_prog(&prog[w], v + 1, done);
      if (lastw) st_xcd(count, S.seqbase + done);
    }
    code_fence();
    to_stage<T, FULL, FC>(OWN, st, at, rot, cnt);
    code_fence();
    st4(qoff, qb, true);
    code_fence();
#pragma unroll
    for (int e = 0; e < LW; ++e) NEWP[e] = OWN[e];
    __builtin_amdgcn_s_setprio(0);
    off += S.dB;
    ++b;
    qoff += S.dB;
    ++qb;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (__builtin_amdgcn_ballot_w64(unsafe) != 0 && p == 0) st_xcd(&words[kTeamAbort], 1);
  return ok;
}

// max |u - snapshot| over nodes [lo, hi) and the next snapshot = u.
template <typename T>
__device__ __forceinline__ uint64_t err_chunk(const T* u, const T* snap, T* dst, int64_t lo,
                                              int64_t hi) {
  uint64_t key = 0;
  constexpr int U = 4;
  for (int64_t j = lo + threadIdx.x; j < hi; j += (int64_t)blockDim.x * U) {
    T a[U], s[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t x = j + (int64_t)q * blockDim.x;
      if (x < hi) {
        a[q] = __hip_atomic_load(u + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s[q] = __hip_atomic_load(snap + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
#pragma unroll
    for (int q = 0; q < U; ++q) {
      const int64_t x = j + (int64_t)q * blockDim.x;
      if (x < hi) {
        const uint64_t k = maxkey(Real<T>::fabs_(a[q] - s[q]));
        key = k > key ? k : key;
        dst[x] = a[q];
      }
    }
  }
  return key;
}

}  // namespace

template <typename T, bool MIX, bool WIDE>
__global__ void __launch_bounds__(kTW * 64, WIDE ? 2 : 4)
    fwd3_team_kernel(const EventDesc* __restrict__ evs, const TeamDesc* __restrict__ teams,
                     TeamShared* sh, int nteam, int per_group, int max_iter) {
  constexpr int LW = WIDE ? kTWide : kTL<T>;
  __shared__ T ring_s[kTW * kRing * 64];
  __shared__ u32x4 stage_s[WIDE ? kTW * kStage<T> : 1];
  __shared__ uint64_t prog[kTW];
  __shared__ int stop;
  __shared__ uint64_t red[kTW];
  __shared__ TDraw draw;
  __shared__ int rank_s;
  const unsigned xcc = xcd_id();
  const int p = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) rank_s = add_dev((words_t)&sh->arrived[xcc * 16], 1);
  __syncthreads();
  const int rank = uni(rank_s);
  TeamClaim claim(sh, xcc, rank, per_group);
  int team = -1;
  for (;;) {
    // ---- an event to work on
    if (threadIdx.x == 0) {
      if (team < 0)
        team = claim_event(sh, nteam, claim, [](int) { return true; },
                           [&](int e) { return gone((words_t)teams[e].words); });
      draw.team = team;
      if (team >= 0) {
        draw.ticket = add_dev((words_t)&teams[team].words[kTeamTicket], 1);
        draw.quit = gone((words_t)teams[team].words) ? 1 : 0;
      }
      stop = 0;
    }
    if (threadIdx.x < kTW) put_prog(&prog[threadIdx.x], -1, 0);
    __syncthreads();
    const int tm = uni(draw.team);
    if (tm < 0) return;
    const TeamDesc& td = teams[tm];
    const EventDesc& ev = evs[td.ev];
    const words_t words = (words_t)td.words;
    const int per_it = 8 * td.R + td.E;
    const int ticket = uni(draw.ticket);
    const int it = ticket / per_it, rem = ticket - it * per_it;
    const bool sweep = rem < 8 * td.R;
    const int sw = rem / td.R;
    // the iteration before is over (first sweep), the sweeps are done (error pass)
    const bool dropped = team_gate(
        draw, it >= max_iter, sweep ? sw == 0 && it > 0 : true, threadIdx.x == 0,
        [](int x) { return uni(x); },
        [&]() {
          const words_t word = &words[sweep ? kTeamState : kTeamSwept];
          const int need = sweep ? it : td.R * (it + 1);
          TPatience wait;
          while (ld_dev(word) < need)
            if (wait.over(words)) break;
          return gone(words);
        },
        []() { __syncthreads(); });
    if (dropped) {
      team = -1;
      __syncthreads();
      continue;
    }
    const int64_t N = (int64_t)ev.m * ev.n * ev.l;
    const uint64_t bytes = (uint64_t)N * sizeof(T);
    if (sweep) {
      const int idx = rem - sw * td.R;
      const int cb = idx / td.ns, cs = idx - cb * td.ns;  // canonical band and slab
      const int dir = kDir3[sw];
      const bool a_is_i = ev.m <= ev.n;
      const int Ma = a_is_i ? ev.m : ev.n, Nb = a_is_i ? ev.n : ev.m;
      const int sA = a_is_i ? ev.n * ev.l : ev.l, sB = a_is_i ? ev.l : ev.n * ev.l;
      const bool fi = dir & 1, fj = dir & 2, fk = dir & 4;
      const bool fa = a_is_i ? fi : fj, fb = a_is_i ? fj : fi;
      const int rb = fa ? td.bands - 1 - cb : cb;  // real band, real slab
      const int rs = fk ? td.ns - 1 - cs : cs;
      auto rows = [&](int band) {
        const int r = Ma - band * td.H;
        return r < td.H ? r : td.H;
      };
      TItem<T> S;
      S.Hr = rows(rb);
      S.Nb = Nb;
      S.V = S.Hr + Nb - 1;
      S.l = ev.l;
      const int nseg = (ev.l + LW - 1) / LW;
      const int seg0 = rs * kTW;
      S.nw = nseg - seg0 < kTW ? nseg - seg0 : kTW;
      S.up = cb > 0;
      S.dn = cb + 1 < td.bands;
      S.first = it == 0 && sw == 0;
      const int seq = it * 8 + sw;
      S.seqbase = seq << kTeamSeqShift;
      S.dA = (fa ? -sA : sA) * (int)sizeof(T);
      S.dB = (fb ? -sB : sB) * (int)sizeof(T);
      S.h = (T)ev.h;
      S.hd = ev.h;
      S.u = make_rsrc(ev.u, bytes);
      S.src = make_rsrc(S.first ? ev.u0 : ev.u, bytes);
      S.f = make_rsrc(ev.f, bytes);
      if (w < S.nw) {
        const int seg = seg0 + (fk ? S.nw - 1 - w : w);
        S.k0 = seg * LW;
        S.cnt = ev.l - S.k0 < LW ? ev.l - S.k0 : LW;
        const int row0 = rb * td.H + (fa ? S.Hr - 1 : 0);
        S.off0 = (int)((uint32_t)(row0 * (int64_t)sA + (fb ? (int64_t)(Nb - 1) * sB : 0) + S.k0) *
                       (uint32_t)sizeof(T));
        // the counts lane i of the first wave watches
        TWatch W;
        W.ptr = &words[kTeamAbort];
        W.base = 0;
        W.xo = 0;
        W.sg = 0;
        W.K = 0;
        W.cap = 0;
        W.have = 0;
        if (w == 0 && p < 5) {
          const int prev = sw > 0 ? kDir3[sw > 0 ? sw - 1 : 0] ^ dir : 0;
          const bool Fa = a_is_i ? prev & 1 : prev & 2, Fb = a_is_i ? prev & 2 : prev & 1;
          const int nrb = fa ? rb - 1 : rb + 1, prb = fa ? rb + 1 : rb - 1;
          const int nrs = fk ? rs - 1 : rs + 1, prs = fk ? rs + 1 : rs - 1;
          int b2 = -1, s2 = rs;
          if (p == 0 && sw > 0) {  // own region, sweep before
            b2 = rb;
            W.xo = 3;
            W.sg = 1;
            W.K = 1 + (Fa ? S.Hr - 1 : 0) + (Fb ? Nb - 1 : 0);
          } else if (p == 1 && sw > 0 && S.dn) {  // next band, sweep before
            b2 = nrb;
            W.xo = 3 - S.Hr;
            W.sg = Fb ? 0 : 1;
            W.K = 1 + (Fa ? rows(nrb) - 1 : 0) + (Fb ? Nb - 1 : 0);
          } else if (p == 2 && sw > 0 && cs + 1 < td.ns) {  // next slab, sweep before
            b2 = rb;
            s2 = nrs;
            W.xo = 2;
            W.sg = 1;
            W.K = 1 + (Fa ? S.Hr - 1 : 0) + (Fb ? Nb - 1 : 0);
          } else if (p == 3 && cb > 0) {  // band before, this sweep
            b2 = prb;
            W.xo = 2;
            W.sg = 1;
            W.K = rows(prb);
          } else if (p == 4 && cs > 0) {  // slab before, this sweep
            b2 = rb;
            s2 = prs;
            W.xo = 2;
            W.sg = 1;
            W.K = 1;
          }
          if (b2 >= 0) {
            const int of = p < 3 ? seq - 1 : seq;
            W.ptr = &words[kTeamCounts + 16 * (b2 * td.ns + s2) + (of & 3)];
            W.base = of << kTeamSeqShift;
            W.cap = rows(b2) + Nb - 1;
          }
        }
        const words_t count = &words[kTeamCounts + 16 * (rb * td.ns + rs) + (seq & 3)];
        const lptr<T> ring = (lptr<T>)ring_s;
        auto sweep = [&](auto full, auto down) {
          constexpr bool FULL = decltype(full)::value, FC = decltype(down)::value;
          if constexpr (WIDE)
            team_sweep_wide<T, MIX, FULL, FC>(S, W, w, count, words, ring,
                                              (lptr<u32x4>)stage_s + w * kStage<T>, prog, &stop);
          else
            team_sweep<T, MIX, FULL, FC>(S, W, w, count, words, ring, prog, &stop);
        };
        const std::true_type yes;
        const std::false_type no;
        if (S.cnt == LW) {
          if (fk)
            sweep(yes, yes);
          else
            sweep(yes, no);
        } else {
          if (fk)
            sweep(no, yes);
          else
            sweep(no, no);
        }
      }
      __syncthreads();  // every wave's stores are complete
      if (threadIdx.x == 0) {
        if (stop) {
          draw.quit = 1;
        } else {
          st_xcd(&words[kTeamCounts + 16 * (rb * td.ns + rs) + (seq & 3)], S.seqbase + S.V);
          if (sw == 7) add_dev(&words[kTeamSwept], 1);
        }
      }
    } else {
      // ---- error pass: err = max |u - u_old| (Eikonal3D.cpp:79-81), u_old = u
      const int c = rem - 8 * td.R;
      const int64_t lo = N * c / td.E, hi = N * (c + 1) / td.E;
      const T* snap = (const T*)(it == 0 ? ev.u0 : ev.uold);
      uint64_t key = err_chunk<T>((const T*)ev.u, snap, (T*)ev.uold, lo, hi);
      for (int o = 32; o > 0; o >>= 1) {
        const uint64_t k = __shfl_xor(key, o);
        key = k > key ? k : key;
      }
      if (p == 0) red[w] = key;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0) {
        for (int q = 1; q < kTW; ++q) key = red[q] > key ? red[q] : key;
        unsigned long long* const kw = (unsigned long long*)&td.words[kTeamKey + 2 * (it & 1)];
        __hip_atomic_fetch_max(kw, (unsigned long long)key, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (add_dev(&words[kTeamErred], 1) == td.E * (it + 1) - 1) {
          // the iteration's last chunk: the stop rule
          const uint64_t k =
              __hip_atomic_load(kw, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const T err = key_to_real(k, T(0));
          const bool conv = err < (T)ev.tol, over = conv || it + 1 >= max_iter;
          if (it < kMaxLoggedIters) ev.info->err_log[it] = (double)err;
          if (over) {
            ev.info->iterations = it + 1;
            ev.info->converged = conv ? 1 : 0;
            ev.info->err = (double)err;
          }
          // the other key word serves the next iteration
          __hip_atomic_store((unsigned long long*)&td.words[kTeamKey + 2 * ((it + 1) & 1)], 0ull,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          st_dev(&words[kTeamState], over ? kTeamOver : it + 1);
        }
      }
    }
    if (threadIdx.x == 0 && draw.quit) team = -1;
    __syncthreads();
  }
}

#define ADT_TEAM(T, MIX, WIDE)                                                                  \
  template __global__ void fwd3_team_kernel<T, MIX, WIDE>(const EventDesc*, const TeamDesc*,    \
                                                          TeamShared*, int, int, int);
ADT_TEAM(double, false, false)
ADT_TEAM(float, false, false)
ADT_TEAM(float, true, false)
ADT_TEAM(double, false, true)
ADT_TEAM(float, false, true)
ADT_TEAM(float, true, true)
#undef ADT_TEAM

}  // namespace adt
