// 3D adjoint as a tile-ordered topological solve, with any number of
// workgroups per event.
//
// The system is the one of Eikonal3D.cpp:96-198: the reference assembles the
// upwind Jacobian and solves A^T lambda = g with a sparse LU.  Every edge of
// the upwind graph (node c "feeds" node r when r is c's argmin neighbour
// along one of c's active dimensions) goes from a larger to a smaller travel
// time, so A is triangular in decreasing u and each node resolves once all
// its feeders have:
//     lambda_r = (g_r + sum_c 2 (u_c - u_r) lambda_c) / D_r,
//     D_r = sum over r's active dimensions (x, y, z order) of 2 (u_r - u_up),
// the feeders pulled in the fixed order (i-1, i+1, j-1, j+1, k-1, k+1).
// The result does not depend on the order in which nodes are resolved.
//
// The event is cut into 8x8x8 tiles.  A wave works on one tile at a time: it
// loads travel times and sources with a one-node halo into LDS, resolves every
// node that the multipliers final outside the tile allow, stores the results,
// and tells the neighbouring tiles that it has resolved a feeder of theirs.  Codes
// and multipliers are kept tile by tile (512 entries each, i j k order), so a
// tile is one contiguous piece; a multiplier that is not final holds a NaN of
// its own (Raw::open), so the value is its own flag.  The k faces of a tile, whose
// nodes each lie in another 64-byte sector, are kept a second time, travel times
// and multipliers, so that a neighbour reads 64 nodes in 8 sectors.
//
// Inside a tile lane (i, j) owns the row k = 0..7.  What is resolved, what
// feeds what and along which sides are 8-bit masks in registers; the lanes
// exchange their masks (two DPP shifts, a rotation, one permute), which gives
// the row's ready nodes, and each lane resolves one of them a round: about 22
// rounds where the rays cross the tile along all three axes.
//
// Scheduling.  Each tile counts the deliveries it has not yet taken account
// of; the delivery that finds the count at zero puts the tile in the event's
// queue, so a tile is in the queue or with a wave, never twice.  (A tile
// with feeders still to come may be put back while others wait, see kWindow.)  A wave that
// takes it reads the count, then the halo, and afterwards takes the count it
// read away: if anything was delivered meanwhile it goes on with the tile, the
// halo's multipliers read anew.  The queue starts with the tiles that hold a
// node without feeders.  A wave without work draws a place of the queue and
// waits for it to be filled.  The tile graph may have cycles; the node graph
// has none: an unresolved node whose feeders are all final lies in a tile with
// a delivery not yet taken account of, or in one of the first queue.
//
// All waves of an event run on one XCD (see kernels_team.hip): its values pass
// through that XCD's L2, which the stores reach and the halo's loads (device
// scope) read.  A delivery is made after the wave's stores have completed.
//
// What bounds it.  One event: the chain of tiles along the rays, for each a load
// (5000 cycles), some 25 rounds of 900 cycles (LDS reads, six products in order,
// a division) and the hand-over (4000).  Many events: memory (the tiles of 256
// events of 128x128x64 read and write 34.7 GB in 7.6 ms, all three kernels 50.7 in
// 10.8), with two waves a SIMD to hide its latency (LDS holds no more).  Measured,
// prepare and solve, against one workgroup per event with its scheduling in LDS:
// 128x128x64 FP64 12.7 -> 1.8 ms, 200x200x80 43 -> 4 ms, 400x400x160 460 -> 21 ms;
// 64 events of 128x128x64 FP32 14.6 -> 4.5 ms; 256 of them FP64, 30 to 120 sources
// each, 17.1 -> 12.7 ms (the benchmark's, 60 each, 10.8).
#include "adjoint3.hpp"
#include "buffer_ops.hpp"
#include "eikonal_device.hpp"
#include "kernels.hpp"
#include "team_device.hpp"

namespace adt {

namespace {

constexpr int kT = 8;                   // tile edge (nodes)
constexpr int kTN = kT * kT * kT;       // nodes per tile
constexpr int kFaces = 2 * kT * kT;     // nodes of its k faces
static_assert(kTileNodes == kTN && kTileFaces == kFaces, "tile workspace");
constexpr int kBJ = kT + 2, kBI = kBJ * kBJ, kBox = kBI * kBJ;  // box with halo: strides, size
constexpr uint64_t kAllZ = 0x4040404040404040ull;  // a row of Z codes (or of no nodes)
// Word of a tile: deliveries not yet taken account of (16 bits); edges into it
// from unresolved nodes of other tiles (10 bits); it has been worked on before.
constexpr int kCountMask = 0xffff, kEdge = 1 << 16, kEdgeMask = 0x3ff, kSeen = 1 << 30;
// Queue entry: tile + 1 (24 bits), kSeen.
constexpr int kTileMask = 0xffffff;
// While the queue holds kLong tiles (`pick`) a wave takes kWindow of them at once, works on
// the one with the fewest edges still to come and puts the others back; a tile
// that it made ready itself it keeps only with at most kFew.  On 256 events of
// 128x128x64 that makes 2.1 passes a tile instead of 4, on 200 of 200x200x80 2.3
// instead of 4.6 (windows of 4, 8, 32, 64: 18.3, 16.8, 16.6, 17.4 ms whole calls
// for the first against 16.6).
constexpr int kWindow = 16, kLong = 20, kFew = 48;
__device__ __forceinline__ int edges_of(int w) { return (w >> 16) & kEdgeMask; }
constexpr int kWaves = kAdjWaves;

template <typename T>
struct Raw;
template <>
struct Raw<double> {
  using U = uint64_t;
  static constexpr U open = 0x7ff4a5a55a5a5a5aull;
};
template <>
struct Raw<float> {
  using U = uint32_t;
  static constexpr U open = 0x7fa5a5a5u;
};

// A node of the box: travel time and multiplier (the source g until resolved).
template <typename T>
struct alignas(2 * sizeof(T)) Node {
  T u, l;
};

// Per-event constants.
template <typename T>
struct Ev {
  int m, n, l;
  int nti, ntj, ntk, ntiles;
  T h;
  gptr<const T> u, u0, g, f;
  gptr<T> gu0, gf, lam, uface, lface;  // faces: per tile k = 0, k = 7, 64 nodes each
  gptr<uint8_t> code;
  words_t hdr, word, ring;
  int cap;
  __device__ explicit Ev(const EventDesc& ev) {
    m = ev.m;
    n = ev.n;
    l = ev.l;
    nti = (m + kT - 1) / kT;
    ntj = (n + kT - 1) / kT;
    ntk = (l + kT - 1) / kT;
    ntiles = nti * ntj * ntk;
    h = (T)ev.h;
    u = (gptr<const T>)ev.u;
    u0 = (gptr<const T>)ev.u0;
    g = (gptr<const T>)ev.grad_u;
    f = (gptr<const T>)ev.f;
    gu0 = (gptr<T>)ev.grad_u0;
    gf = (gptr<T>)ev.grad_f;
    lam = (gptr<T>)ev.lam;
    uface = lam + (int64_t)ntiles * kTN;
    lface = uface + (int64_t)ntiles * kFaces;
    code = (gptr<uint8_t>)ev.code;
    hdr = (words_t)ev.queue;
    word = hdr + kAdjHdr;
    ring = word + ntiles;
    cap = adj_ring(ntiles);
  }
};

struct Tile {
  int t, i, j, k;  // number, coordinates in tiles
};
template <typename T>
__device__ __forceinline__ Tile tile_of(const Ev<T>& E, int t) {
  Tile x;
  x.t = t;
  x.k = t % E.ntk;
  const int ij = t / E.ntk;
  x.j = ij % E.ntj;
  x.i = ij / E.ntj;
  return x;
}
// The neighbouring tile in direction q (i-1, i+1, j-1, j+1, k-1, k+1), or -1.
template <typename T>
__device__ __forceinline__ int tile_nb(const Ev<T>& E, const Tile& X, int q) {
  const int d = q >> 1, s = (q & 1) ? 1 : -1;
  const int c = (d == 0 ? X.i : d == 1 ? X.j : X.k) + s;
  const int ext = d == 0 ? E.nti : d == 1 ? E.ntj : E.ntk;
  const int st = d == 0 ? E.ntj * E.ntk : d == 1 ? E.ntk : 1;
  return c >= 0 && c < ext ? X.t + s * st : -1;
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// Wave-level ordering of LDS accesses by different lanes (the wave's LDS
// instructions execute in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Bit `b` of the eight bytes of x as an 8-bit mask.
__device__ __forceinline__ unsigned bits_of(uint64_t x, int b) {
  const unsigned lo = ((unsigned)x >> b) & 0x01010101u, hi = ((unsigned)(x >> 32) >> b) & 0x01010101u;
  return __builtin_amdgcn_udot4(hi, 0x80402010u, __builtin_amdgcn_udot4(lo, 0x08040201u, 0u, false),
                                false);
}
// A lane's number (< 32) summed over the wave.
__device__ __forceinline__ int wave_count(unsigned x) {
  int n = 0;
#pragma unroll
  for (int b = 0; b < 5; ++b) n += __builtin_popcountll(__ballot((x >> b) & 1u)) << b;
  return n;
}

// What a lane knows of its row: masks over k (bit k = node k of the row).
struct Row {
  unsigned nz;     // not Z
  unsigned F[6];   // has a feeder in direction q
  unsigned S[6];   // has its upwind neighbour in direction q
  unsigned out[6]; // that one lies in the neighbouring tile and is not Z
};

// From the codes of the row and its neighbours (a neighbour at -1 feeds if its
// upwind is at +1, and the reverse; a Z code has no sides).
template <typename T, bool SIDES>
__device__ __forceinline__ Row row_masks(const Ev<T>& E, const Tile& X) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  gptr<const uint64_t> const c8 = (gptr<const uint64_t>)E.code;
  const int64_t at = (int64_t)X.t * 64 + lane;
  const int64_t sI = (int64_t)E.ntj * E.ntk * 64, sJ = (int64_t)E.ntk * 64;
  const bool pi = X.i > 0 || i > 0, ni = X.i + 1 < E.nti || i < 7;
  const bool pj = X.j > 0 || j > 0, nj = X.j + 1 < E.ntj || j < 7;
  const bool pk = X.k > 0, nk = X.k + 1 < E.ntk;
  const uint64_t c = c8[at];
  uint64_t im = c8[!pi ? at : i > 0 ? at - 8 : at - sI + 56];
  uint64_t ip = c8[!ni ? at : i < 7 ? at + 8 : at + sI - 56];
  uint64_t jm = c8[!pj ? at : j > 0 ? at - 1 : at - sJ + 7];
  uint64_t jp = c8[!nj ? at : j < 7 ? at + 1 : at + sJ - 7];
  uint64_t km = c8[!pk ? at : at - 64];
  uint64_t kp = c8[!nk ? at : at + 64];
  im = pi ? im : kAllZ;
  ip = ni ? ip : kAllZ;
  jm = pj ? jm : kAllZ;
  jp = nj ? jp : kAllZ;
  km = pk ? km : kAllZ;
  kp = nk ? kp : kAllZ;
  const uint64_t kmw = (c << 8) | (km >> 56), kpw = (c >> 8) | (kp << 56);
  Row R;
  R.nz = bits_of(~c, 6);
  R.F[0] = bits_of(im, 1);
  R.F[1] = bits_of(ip, 0);
  R.F[2] = bits_of(jm, 3);
  R.F[3] = bits_of(jp, 2);
  R.F[4] = bits_of(kmw, 5);
  R.F[5] = bits_of(kpw, 4);
  if constexpr (SIDES) {
#pragma unroll
    for (int q = 0; q < 6; ++q) R.S[q] = bits_of(c, q);
    R.out[0] = i == 0 ? R.S[0] & bits_of(~im, 6) : 0;
    R.out[1] = i == 7 ? R.S[1] & bits_of(~ip, 6) : 0;
    R.out[2] = j == 0 ? R.S[2] & bits_of(~jm, 6) : 0;
    R.out[3] = j == 7 ? R.S[3] & bits_of(~jp, 6) : 0;
    R.out[4] = R.S[4] & (unsigned)(~km >> 62) & 1u;
    R.out[5] = (R.S[5] & 0x80u) & ((unsigned)(~kp >> 6) << 7);
  }
  return R;
}

// Multiplier words as the event's XCD has them now.
template <typename T>
__device__ __forceinline__ typename Raw<T>::U ld_lam(gptr<const T> p) {
  using U = typename Raw<T>::U;
  return __hip_atomic_load((gptr<const U>)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bounded wait (30 s): call with every unsuccessful poll; true when the time
// is over.
struct Patience {
  int spin = 0;
  uint64_t t0 = 0;
  __device__ __forceinline__ bool over() {
    if (++spin > 2) __builtin_amdgcn_s_sleep(1);
    if ((spin & 255) != 0) return false;
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    return now - t0 > kTeamPatience;
  }
};

__device__ __forceinline__ void give_up(const EventDesc& ev, words_t hdr) {
  ev.info->fault = ADT_FAULT;
  st_dev(&hdr[kAdjOver], 2);
}

// Puts an entry into place `at` of the queue, drawn before.
template <typename T>
__device__ __forceinline__ void put_entry(const Ev<T>& E, const EventDesc& ev, int at, int entry) {
  const words_t slot = &E.ring[(unsigned)at % (unsigned)E.cap];
  if ((unsigned)at >= (unsigned)E.cap) {
    Patience wait;  // the wave that drew this place one round ago empties it
    while (ld_dev(slot) != 0) {
      if (wait.over()) {
        give_up(ev, E.hdr);
        break;
      }
    }
  }
  st_xcd(slot, entry);
}

// The entry of this lane's place, once it is there (0: the event is over), out
// of the queue.
template <typename T>
__device__ __forceinline__ int get_entry(const Ev<T>& E, const EventDesc& ev, int at) {
  const words_t slot = &E.ring[(unsigned)at % (unsigned)E.cap];
  Patience wait;
  int entry;
  for (;;) {
    entry = ld_dev(slot);
    const int over = ld_dev(&E.hdr[kAdjOver]);
    if (over) return 0;
    if (entry) break;
    if (wait.over()) give_up(ev, E.hdr);
  }
  st_xcd(slot, 0);
  return entry;
}

// The wave's work on the tile of `entry`, with `taken` deliveries to it, until
// nothing more is delivered.  Returns the queue entry of a tile that it has
// made ready and takes next, with that tile's word, or 0.  `busy`: the queue is
// long.
template <typename T>
__device__ int work_tile(const Ev<T>& E, const EventDesc& ev, Node<T>* const box, int entry, int taken,
                         bool busy, int& keep_word) {
  using U = typename Raw<T>::U;
  const int lane = lane_id(), la = lane >> 3, lb = lane & 7;
  const Tile X = tile_of(E, (entry & kTileMask) - 1);
  const bool seen = entry & kSeen;
  const int64_t base = (int64_t)X.t * kTN;
  const int nbt[6] = {tile_nb(E, X, 0), tile_nb(E, X, 1), tile_nb(E, X, 2),
                      tile_nb(E, X, 3), tile_nb(E, X, 4), tile_nb(E, X, 5)};
  U hw[6];
  auto load_halo = [&]() {
    const int hx[4] = {7 * 64 + lane, lane, la * 64 + 56 + lb, la * 64 + lb};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      hw[q] = ld_lam<T>(E.lam + (nbt[q] >= 0 ? (int64_t)nbt[q] * kTN + hx[q] : base));
    hw[4] = ld_lam<T>(E.lface + (nbt[4] >= 0 ? (int64_t)nbt[4] * kFaces + 64 + lane : 0));
    hw[5] = ld_lam<T>(E.lface + (nbt[5] >= 0 ? (int64_t)nbt[5] * kFaces + lane : 0));
  };
  // ---- travel times of the box; sources and slowness of the tile
  int bx[14];
  T fr[8];
  int64_t gx[8];
  bool in[8];
  {
    T uv[14], gv[8];
    const int i0 = X.i * kT, j0 = X.j * kT, k0 = X.k * kT;
    const int64_t sI = (int64_t)E.n * E.l;
    const rsrc_t ru = make_rsrc((const void*)E.u, (uint64_t)E.m * sI * sizeof(T));
    const rsrc_t rg = make_rsrc((const void*)E.g, (uint64_t)E.m * sI * sizeof(T));
    const rsrc_t rf = make_rsrc((const void*)E.f, (uint64_t)E.m * sI * sizeof(T));
#pragma unroll
    for (int s = 0; s < 14; ++s) {
      // slots 0-7: slabs i = s; 8, 9: the i faces, 10, 11 the j faces, 12, 13 the k faces
      const int ii = s < 8 ? s : s == 8 ? -1 : s == 9 ? kT : la;
      const int jj = s < 10 ? la : s == 10 ? -1 : s == 11 ? kT : lb;
      const int kk = s < 12 ? lb : s == 12 ? -1 : kT;
      bx[s] = (ii + 1) * kBI + (jj + 1) * kBJ + kk + 1;
      const int gi = i0 + ii, gj = j0 + jj, gk = k0 + kk;
      const bool on = gi >= 0 && gi < E.m && gj >= 0 && gj < E.n && gk >= 0 && gk < E.l;
      const int64_t x = (int64_t)gi * sI + (int64_t)gj * E.l + gk;
      const uint32_t off = boff<T>(on, x);
      if (s < 12)
        uv[s] = bload(ru, off, T(0));
      else if (s == 12)
        uv[s] = E.uface[nbt[4] >= 0 ? (int64_t)nbt[4] * kFaces + 64 + lane : 0];
      else
        uv[s] = E.uface[nbt[5] >= 0 ? (int64_t)nbt[5] * kFaces + lane : 0];
      if (s < 8) {
        in[s] = on;
        gx[s] = x;
        gv[s] = bload(rg, off, T(0));
        fr[s] = bload(rf, off, T(0));
      }
    }
    load_halo();
#pragma unroll
    for (int s = 0; s < 14; ++s) box[bx[s]].u = uv[s];
#pragma unroll
    for (int s = 0; s < 8; ++s) box[bx[s]].l = gv[s];
  }
  // ---- masks
  const Row R = row_masks<T, true>(E, X);
  unsigned done = 0;
  if (seen) {  // nodes resolved before, by any wave
    U w[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) w[s] = ld_lam<T>(E.lam + base + s * 64 + lane);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const uint64_t b = __ballot(w[s] != Raw<T>::open);
      done = la == s ? (unsigned)(b >> (8 * lb)) & 0xffu : done;
      if (w[s] != Raw<T>::open) box[bx[s]].l = __builtin_bit_cast(T, w[s]);
    }
  }
  // feeders inside the tile, by where the exchange brings their lane's mask
  // from: lane ^ 8 of the 16 (A), the lane 8 away on the other side (B), ...
  const bool odd = lane & 8;
  const unsigned f0 = la > 0 ? R.F[0] : 0, f1 = la < 7 ? R.F[1] : 0;
  const unsigned fA = odd ? f0 : f1, fB = odd ? f1 : f0;
  const int peer = (odd ? lane + 8 : lane - 8) << 2;
  const unsigned fC = lb > 0 ? R.F[2] : 0, fD = lb < 7 ? R.F[3] : 0;
  const unsigned fE = R.F[4] & 0xfeu, fG = R.F[5] & 0x7fu;
  const unsigned p0 = R.F[0] | R.F[1] << 8 | R.F[2] << 16 | R.F[3] << 24;
  const unsigned p1 = R.F[4] | R.F[5] << 8 | R.S[0] << 16 | R.S[1] << 24;
  const unsigned p2 = R.S[2] | R.S[3] << 8 | R.S[4] << 16 | R.S[5] << 24;
  const int row = (la + 1) * kBI + (lb + 1) * kBJ + 1;
  bool first = !seen;
  for (;;) {
    // ---- the halo's multipliers, and which of its nodes are final
    unsigned blocked = 0;
    {
      uint64_t fin[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        box[bx[8 + q]].l = __builtin_bit_cast(T, hw[q]);
        fin[q] = __ballot(hw[q] != Raw<T>::open);
      }
      blocked |= la == 0 ? R.F[0] & ~(unsigned)(fin[0] >> (8 * lb)) : 0;
      blocked |= la == 7 ? R.F[1] & ~(unsigned)(fin[1] >> (8 * lb)) : 0;
      blocked |= lb == 0 ? R.F[2] & ~(unsigned)(fin[2] >> (8 * la)) : 0;
      blocked |= lb == 7 ? R.F[3] & ~(unsigned)(fin[3] >> (8 * la)) : 0;
      blocked |= R.F[4] & (hw[4] == Raw<T>::open ? 1u : 0u);
      blocked |= R.F[5] & (hw[5] == Raw<T>::open ? 0x80u : 0u);
    }
    const unsigned cand = R.nz & ~blocked;
    const unsigned before = done;
    unsigned nd = ~done;
    wave_sync();
    // ---- rounds
    for (;;) {
      const unsigned ra = __builtin_amdgcn_update_dpp(0, (int)nd, 0x128, 0xf, 0xf, true);
      const unsigned rb = __builtin_amdgcn_ds_bpermute(peer, (int)nd);
      const unsigned rc = __builtin_amdgcn_update_dpp(0, (int)nd, 0x111, 0xf, 0xf, true);
      const unsigned rd = __builtin_amdgcn_update_dpp(0, (int)nd, 0x101, 0xf, 0xf, true);
      const unsigned wait = (fA & ra) | (fB & rb) | (fC & rc) | (fD & rd) | (fE & (nd << 1)) |
                            (fG & (nd >> 1));
      const unsigned ready = cand & nd & ~wait;
      if (__ballot(ready != 0) == 0) break;
      const int k = ready ? __builtin_ctz(ready) : 0;
      Node<T>* const x = box + row + k;
      const Node<T> own = *x;
      const Node<T> nb[6] = {x[-kBI], x[kBI], x[-kBJ], x[kBJ], x[-1], x[1]};
      const unsigned s0 = p0 >> k, s1 = p1 >> k, s2 = p2 >> k;
      T w[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) w[q] = T(2.0) * (nb[q].u - own.u);
      T num = own.l;
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        const T c = num + w[q] * nb[q].l;
        num = ((q < 4 ? s0 >> (8 * q) : s1 >> (8 * (q - 4))) & 1u) ? c : num;
      }
      // 2 (u_r - u_up) is -w of the upwind side, exactly
      T D = T(0);
      D = D - (((s1 >> 16) & 1u) ? w[0] : ((s1 >> 24) & 1u) ? w[1] : T(0));
      D = D - ((s2 & 1u) ? w[2] : ((s2 >> 8) & 1u) ? w[3] : T(0));
      D = D - (((s2 >> 16) & 1u) ? w[4] : ((s2 >> 24) & 1u) ? w[5] : T(0));
      const T lr = num / D;
      wave_sync();
      if (ready) x->l = lr;
      nd &= ~(ready & (0u - ready));
      wave_sync();
    }
    done = ~nd & 0xffu;
    const unsigned now = done & ~before;
    // ---- results, then the deliveries
    const bool any = __ballot(now != 0) != 0;
    if (any) {
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const unsigned r = (unsigned)__builtin_amdgcn_ds_bpermute((s * 8 + la) << 2, (int)now);
        if ((r >> lb) & 1u) {
          const T lr = box[bx[s]].l;
          E.lam[base + s * 64 + lane] = lr == lr ? lr : T(__builtin_nan(""));
          const T rhs = T(-2.0) * fr[s] * E.h * E.h;  // Eikonal3D.cpp:113-116, 194-196
          E.gf[gx[s]] = -lr * rhs;
        }
      }
      // the k faces: this lane's row ends
      const T l0 = box[row].l, l7 = box[row + 7].l;
      if (now & 1u) E.lface[(int64_t)X.t * kFaces + lane] = l0 == l0 ? l0 : T(__builtin_nan(""));
      if (now & 0x80u) E.lface[(int64_t)X.t * kFaces + 64 + lane] = l7 == l7 ? l7 : T(__builtin_nan(""));
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const bool left = __ballot((R.nz & ~done) != 0) != 0;
    const int nres = wave_count(__builtin_popcount(now));
    // edges released on each face; lane q < 6 has those in direction q
    int nt = -1, rel = 0;
    {
      const int xi = __builtin_popcount(now & (la == 0 ? R.out[0] : R.out[1]));
      const int xj = __builtin_popcount(now & (lb == 0 ? R.out[2] : R.out[3]));
      int n[6] = {0, 0, 0, 0, __builtin_popcountll(__ballot((now & R.out[4]) != 0)),
                  __builtin_popcountll(__ballot((now & R.out[5]) != 0))};
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint64_t bi = __ballot((xi >> b) & 1), bj = __ballot((xj >> b) & 1);
        n[0] += __builtin_popcountll(bi & 0xffull) << b;
        n[1] += __builtin_popcountll(bi >> 56) << b;
        n[2] += __builtin_popcountll(bj & 0x0101010101010101ull) << b;
        n[3] += __builtin_popcountll(bj & 0x8080808080808080ull) << b;
      }
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        rel = lane == q ? n[q] : rel;
        nt = lane == q && n[q] ? nbt[q] : nt;
      }
    }
    // lane 6: nodes left; 7: this tile; 8: passes
    words_t word = E.hdr;
    int add = 0;
    if (nt >= 0) {
      word = &E.word[nt];
      add = 1 - rel * kEdge;
    } else if (lane == 6) {
      word = &E.hdr[kAdjLeft];
      add = -nres;
    } else if (lane == 7 && left) {
      word = &E.word[X.t];
      add = (first ? kSeen : 0) - taken;
    } else if (lane == 8) {
      word = &E.hdr[kAdjPasses];
      add = 1;
    }
    const int old = add ? add_xcd(word, add) : 0;
    const int nodes = __builtin_amdgcn_readlane(old, 6);
    const int mine = __builtin_amdgcn_readlane(old, 7) & kCountMask;
    first = false;
    if (nres > 0 && nodes == nres) {  // the event's last node
      if (lane == 0) {
        ev.info->adj_sweeps = ld_dev(&E.hdr[kAdjPasses]);
        ev.info->adj_converged = 1;
        st_dev(&E.hdr[kAdjOver], 1);
      }
      return 0;
    }
    // neighbours that were idle: into the queue, but for one that this wave
    // takes itself if its own tile has nothing more to do
    const bool again = left && mine != taken;
    if (again) {
      taken = mine - taken;
      load_halo();
    }
    const bool idle = nt >= 0 && (old & kCountMask) == 0;
    const uint64_t m = __ballot(idle);
    int keep = 0;
    if (m) {
      const int ent = (nt + 1) | (old & kSeen);
      const uint64_t m0 = __ballot(idle && edges_of(old) - rel <= kFew);
      const int sel = again ? -1 : m0 ? __builtin_ctzll(m0) : busy ? -1 : __builtin_ctzll(m);
      if (sel >= 0) {
        keep = __builtin_amdgcn_readlane(ent, sel);
        keep_word = __builtin_amdgcn_readlane(old + add, sel);
      }
      if (idle && lane != sel) put_entry(E, ev, add_xcd(&E.hdr[kAdjTail], 1), ent);
    }
    if (!again) return keep;
  }
}

}  // namespace

// Codes of every tile (the reference's Z rule, Eikonal3D.cpp:105-171), grad_u0
// = g where u == u0 (:105-110; g is read only there) and 0 elsewhere, dL/df =
// -0 * (-2 f h h) on Z (the value the reference's final loop gives those
// nodes, :194-196), no multiplier final, counts and queues empty, and the
// words of `sh` zero.  A wave takes a tile, a lane (j, k) its column of i.
template <typename T>
__global__ void __launch_bounds__(256)
    adj3_codes_kernel(const EventDesc* __restrict__ evs, int chunks, int* sh, int64_t sh_words) {
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < sh_words; q += (int64_t)gridDim.x * 256)
    sh[q] = 0;
  const EventDesc& ev = evs[blockIdx.x / chunks];
  if (ev.adj_algo != 0) return;
  const Ev<T> E(ev);
  const int c = blockIdx.x % chunks;
  const int words = (int)adj_words(E.ntiles);
  for (int q = c * 256 + threadIdx.x; q < words; q += chunks * 256) E.hdr[q] = 0;
  const int lane = lane_id(), la = lane >> 3, lb = lane & 7;
  const int64_t sI = (int64_t)E.n * E.l;
  const int ex[3] = {E.m, E.n, E.l};
  for (int t = c * kWaves + uni(threadIdx.x >> 6); t < E.ntiles; t += chunks * kWaves) {
    const Tile X = tile_of(E, t);
    const int i0 = X.i * kT, j = X.j * kT + la, k = X.k * kT + lb;
    const bool on = j < E.n && k < E.l;
    const int cj = j < E.n ? j : E.n - 1, ck = k < E.l ? k : E.l - 1;
    const int64_t col = (int64_t)cj * E.l + ck;
    // (a neighbour outside the grid is never looked at)
    const int64_t jm = col - (cj > 0 ? E.l : 0), jp = col + (cj + 1 < E.n ? E.l : 0);
    const int64_t km = col - (ck > 0 ? 1 : 0), kp = col + (ck + 1 < E.l ? 1 : 0);
    T own[kT + 2];
    T v0[kT], nj[kT][4];
#pragma unroll
    for (int s = 0; s < kT + 2; ++s) {
      const int i = i0 + s - 1;
      const int64_t x = (int64_t)(i < 0 ? 0 : i < E.m ? i : E.m - 1) * sI;
      own[s] = E.u[x + col];
      if (s >= 1 && s <= kT) {
        v0[s - 1] = E.u0[x + col];
        nj[s - 1][0] = E.u[x + jm];
        nj[s - 1][1] = E.u[x + jp];
        nj[s - 1][2] = E.u[x + km];
        nj[s - 1][3] = E.u[x + kp];
      }
    }
    const int64_t base = (int64_t)t * kTN + lane, fb = (int64_t)t * kFaces + (lb ? 64 : 0) + la;
    if (lb == 0 || lb == 7) {
#pragma unroll
      for (int s = 0; s < kT; ++s) {
        E.uface[fb + s * 8] = own[s + 1];
        *((gptr<typename Raw<T>::U>)E.lface + fb + s * 8) = Raw<T>::open;
      }
    }
#pragma unroll
    for (int s = 0; s < kT; ++s) {
      const int i = i0 + s;
      const bool in = on && i < E.m;
      const int64_t x = (int64_t)(i < E.m ? i : E.m - 1) * sI + col;
      const T nb[6] = {own[s], own[s + 2], nj[s][0], nj[s][1], nj[s][2], nj[s][3]};
      const int co[3] = {i, j, k};
      const uint32_t code = in ? code3<T>(own[s + 1], v0[s], nb, co, ex) : kZ;
      E.code[base + s * 64] = (uint8_t)code;
      *((gptr<typename Raw<T>::U>)E.lam + base + s * 64) = Raw<T>::open;
      if (in) {
        if (E.gu0) E.gu0[x] = own[s + 1] == v0[s] ? E.g[x] : T(0);
        if (code & kZ) {
          const T rhs = T(-2.0) * E.f[x] * E.h * E.h;
          E.gf[x] = -T(0) * rhs;
        }
      }
    }
  }
}

// The number of nodes to resolve and the first queue: tiles that hold a node
// without feeders.
template <typename T>
__global__ void __launch_bounds__(256)
    adj3_seeds_kernel(const EventDesc* __restrict__ evs, int chunks) {
  const EventDesc& ev = evs[blockIdx.x / chunks];
  if (ev.adj_algo != 0) return;
  const Ev<T> E(ev);
  const int c = blockIdx.x % chunks;
  for (int t = c * kWaves + uni(threadIdx.x >> 6); t < E.ntiles; t += chunks * kWaves) {
    const Row R = row_masks<T, false>(E, tile_of(E, t));
    const unsigned fed = R.F[0] | R.F[1] | R.F[2] | R.F[3] | R.F[4] | R.F[5];
    const bool seed = __ballot((R.nz & ~fed) != 0) != 0;
    const int n = wave_count(__builtin_popcount(R.nz));
    const int lane = lane_id(), i = lane >> 3, j = lane & 7;
    unsigned e = __builtin_popcount(R.nz & R.F[4] & 1u) + __builtin_popcount(R.nz & R.F[5] & 0x80u);
    e += i == 0 ? __builtin_popcount(R.nz & R.F[0]) : 0;
    e += i == 7 ? __builtin_popcount(R.nz & R.F[1]) : 0;
    e += j == 0 ? __builtin_popcount(R.nz & R.F[2]) : 0;
    e += j == 7 ? __builtin_popcount(R.nz & R.F[3]) : 0;
    const int edges = wave_count(e);
    if (lane == 0 && n > 0) {
      add_dev(&E.hdr[kAdjLeft], n);
      st_dev(&E.word[t], edges * kEdge + (seed ? 1 : 0));
      if (seed) st_dev(&E.ring[add_dev(&E.hdr[kAdjTail], 1)], t + 1);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(kWaves * 64, 2)
    adj3_tile_kernel(const EventDesc* __restrict__ evs, TeamShared* sh, int nev, int per_group,
                     bool pick) {
  __shared__ Node<T> box[kWaves][kBox];
  __shared__ int event_s, rank_s;
  const unsigned xcd = xcd_id();
  const int w = uni(threadIdx.x >> 6);
  if (threadIdx.x == 0) rank_s = add_dev((words_t)&sh->arrived[xcd * 16], 1);
  __syncthreads();
  TeamClaim claim(sh, xcd, uni(rank_s), per_group);
  for (;;) {
    if (threadIdx.x == 0)
      event_s = claim_event(
          sh, nev, claim, [&](int e) { return evs[e].adj_algo == 0; },
          [&](int e) { return ld_dev((words_t)evs[e].queue + kAdjOver) != 0; });
    __syncthreads();
    const int e = uni(event_s);
    if (e < 0) return;
    const EventDesc& ev = evs[e];
    const Ev<T> E(ev);
    // no node to resolve at all (the words left and over: 0 and 0)
    if (threadIdx.x == 0 && ld_dev(&E.hdr[kAdjLeft]) == 0 && ld_dev(&E.hdr[kAdjOver]) == 0) {
      ev.info->adj_converged = 1;
      st_dev(&E.hdr[kAdjOver], 1);
    }
    int entry = 0, word = 0;
    bool busy = false;
    for (;;) {
      if (!entry) {
        const int lane = lane_id();
        int at = -1;
        if (busy) {  // a window of places that are filled, or being filled
          if (lane == 0) {
            int h = ld_dev(&E.hdr[kAdjHead]);
            const int tail = ld_dev(&E.hdr[kAdjTail]);
            if (tail - h >= kLong &&
                __hip_atomic_compare_exchange_strong(&E.hdr[kAdjHead], &h, h + kWindow, __ATOMIC_RELAXED,
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
              at = h;
          }
          at = uni(at);
        }
        if (at >= 0) {
          int mine = 0, mw = 0;
          unsigned key = ~0u;
          if (lane < kWindow) {
            mine = get_entry(E, ev, at + lane);
            if (mine) mw = ld_dev(&E.word[(mine & kTileMask) - 1]);
            key = mine ? (unsigned)edges_of(mw) << 8 | lane : ~0u;
          }
#pragma unroll
          for (int o = 1; o < kWindow; o <<= 1) {
            const unsigned k = __shfl_xor(key, o);
            key = k < key ? k : key;
          }
          key = uni(key);
          if (key == ~0u) break;  // over
          const int sel = key & 0xff;
          const bool back = lane < kWindow && lane != sel && mine != 0;
          const uint64_t bm = __ballot(back);
          int to = 0;
          if (lane == 0) to = add_xcd(&E.hdr[kAdjTail], __builtin_popcountll(bm));
          to = uni(to);
          if (back) put_entry(E, ev, to + __builtin_popcountll(bm & ((1ull << lane) - 1)), mine);
          entry = __builtin_amdgcn_readlane(mine, sel);
          word = __builtin_amdgcn_readlane(mw, sel);
        } else {
          int head = 0;
          if (lane == 0) head = add_xcd(&E.hdr[kAdjHead], 1);
          head = uni(head);
          entry = uni(get_entry(E, ev, head));
          if (!entry) break;
          word = uni(ld_dev(&E.word[(entry & kTileMask) - 1]));
          busy = pick && uni(ld_dev(&E.hdr[kAdjTail])) - head >= kLong;
        }
      }
      code_fence();
      entry = work_tile(E, ev, box[w], entry, word & kCountMask, busy, word);
    }
    __syncthreads();
  }
}

#define ADT_ADJ3_TILE(T)                                                             \
  template __global__ void adj3_codes_kernel<T>(const EventDesc*, int, int*, int64_t); \
  template __global__ void adj3_seeds_kernel<T>(const EventDesc*, int);              \
  template __global__ void adj3_tile_kernel<T>(const EventDesc*, TeamShared*, int, int, bool);
ADT_ADJ3_TILE(double)
ADT_ADJ3_TILE(float)
#undef ADT_ADJ3_TILE

}  // namespace adt
