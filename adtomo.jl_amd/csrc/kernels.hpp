// Internal kernel descriptors and launch declarations.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/adtomo_hip.h"

namespace adt {

constexpr int kMaxLoggedIters = ADT_MAX_LOGGED_ITERS;

struct MisfitNodes;

// One 3D event as seen by the persistent kernels (device resident).
struct EventDesc {
  int m, n, l;
  // launch setting of this event (its box class's, or the global one):
  // forward on the diagonal-streaming kernel (else k-streaming), c segments
  // of that kernel (1..8), adjoint traversal (0 tiles, 1 node by node)
  int8_t fwd_diag, fwd_segs, adj_algo, pad;
  double h, tol;
  const void* u0;
  const void* f;
  const void* grad_u;
  void* u;
  void* uold;      // workspace: iteration snapshot [N]
  void* lam;       // workspace: adjoint multipliers [N]
  uint8_t* code;   // workspace: upwind codes [N]
  uint8_t* indeg;  // workspace: unresolved incoming count per node [N] (word-aligned)
  int32_t* queue;  // workspace: topological order of the adjoint [N]
  void* grad_u0;
  void* grad_f;
  adt_info* info;  // device
  // Optional (device, NULL if absent): the receiver misfit whose gradient
  // becomes grad_u between the forward and the adjoint (fused kernel), and
  // the receiver coordinates it reads.
  const adt_misfit3d* mis;
  const MisfitNodes* mnodes;
  const double* rx;
  const double* ry;
  const double* rz;
  int64_t nrec;
  // An event that fwd3_team_kernel solves: its words (device); the diagonal
  // kernel then takes it only if the abort word is set.  NULL otherwise.
  const int* team_words;
};

// An event of fwd3_team_kernel: bands of at most H rows of the shorter
// horizontal axis, ns slabs of kTW segments along k, R = bands * ns regions,
// E chunks of the error pass; words: its counters, zeroed before the launch.
struct TeamDesc {
  int ev;  // index of its EventDesc
  int bands, H, ns, R, E;
  int* words;
};
constexpr int kTW = 4;             // waves per workgroup
constexpr int kTeamXcds = 16;      // XCD ids are below this
constexpr int kTeamGroups = 256;   // groups of workgroups per XCD
constexpr int kTeamOver = 1 << 20;  // state of a finished event
constexpr int kTeamSeqShift = 22;  // a count is (sweep << 22) + diagonals
constexpr uint64_t kTeamPatience = 3000000000ull;  // 30 s of the 100 MHz clock
// Word indices (16 words = 64 bytes apart: each is polled by itself).
enum {
  kTeamTicket = 0,   // items drawn
  kTeamState = 16,   // iterations finished, or kTeamOver
  kTeamAbort = 32,   // 1: values beyond the fast solve, 2: a wait ran out
  kTeamSwept = 48,   // regions that have finished an iteration's last sweep
  kTeamErred = 64,   // chunks of the error passes done
  kTeamKey = 80,     // error keys of even / odd iterations (two 64-bit words)
  kTeamCounts = 96   // per region: diagonals in memory
};
constexpr size_t team_words(int R) { return (size_t)kTeamCounts + 16 * (size_t)R; }
// State of one launch, zeroed before it; `list` holds kTeamXcds * nteam ints.
struct TeamShared {
  unsigned long long group[kTeamXcds][kTeamGroups];
  int arrived[kTeamXcds * 16];
  int owned[kTeamXcds * 16];
  int next;
  int pad[15];
  int list[1];
};

// One 2D event.
struct Event2Desc {
  int m, n, ix, jx;
  double h;
  const void* f;
  const void* grad_u;
  void* u;
  void* uold;
  void* lam;
  uint8_t* code;
  uint8_t* indeg;
  int32_t* queue;
  void* grad_f;
  adt_info* info;
};

// Objective kernels use the public descriptors directly (plain C layout).
using SourceDesc = adt_source3d;
using MisfitDesc = adt_misfit3d;

// A solve's receivers grouped by interpolation node (built on the host for
// each box of a receiver set): node[u] (flat index, increasing, u < nuniq)
// takes the entries ent[off[u] .. off[u+1]), each (receiver j) * 8 +
// corner (bit 2: the x1 / x2 side, bit 1: y, bit 0: z), in increasing j.
// gj: the solve's scratch of nrec adjoint seeds d loss / d t_j.
struct MisfitNodes {
  const int64_t* node;
  const int64_t* off;
  const int64_t* ent;
  int64_t nuniq;
  void* gj;
};

// Tables passed as kernel arguments (kernel arguments are at most 4 KB).
struct SourceTable {
  SourceDesc s[64];
};
struct ArrayTable {
  const void* a[256];
};
static_assert(sizeof(SourceTable) <= 3584 && sizeof(ArrayTable) <= 3584, "kernel arguments");

template <typename T>
__global__ void source_u0_kernel(SourceTable tab, const T* vel0, int m, int n, int l, T h, int parts);
template <typename T>
__global__ void misfit_kernel(const MisfitDesc* d, const MisfitNodes* nodes, const double* rx,
                              const double* ry, const double* rz, int nrec, int parts);
template <typename T>
__global__ void misfit_nodes_kernel(const MisfitDesc* d, const MisfitNodes* nodes, const double* rx,
                                    const double* ry, const double* rz, int parts);
template <typename T>
__global__ void model_kernel(const T* x, const T* vel0, int64_t N, T* fvar, T* f);
template <typename T, bool MORE>
__global__ void sum_arrays_kernel(ArrayTable tab, const void* const* more, int nin, int64_t N,
                                  T* out);
template <typename T, int R>
__global__ void smooth_pass1_kernel(const T* fvar, int m, int n, int l, int rh, int rv, T wgt,
                                    T* sgn, T* partial);
template <typename T, int R>
__global__ void smooth_pass2_kernel(const T* sgn, int m, int n, int l, int rh, int rv, T wgt,
                                    T lambda, T* grad, const T* partial, int npart, T* value);
template <typename T>
__global__ void slowness_kernel(const T* fvar, int64_t N, T scale, T* f_s);
template <typename T>
__global__ void slowness_grad_kernel(const T* fvar, int64_t N, T scale, const T* grad_fs,
                                     T* grad_fvar, T* partial);
template <typename T>
__global__ void sum_partials_kernel(const T* partial, int npart, T* out);
template <typename T>
__global__ void model_grad_kernel(const T* x, const T* fvar, const T* grad_f, const T* grad_fvar,
                                  int64_t N, T* grad_x);

template <typename T>
__global__ void fwd3_plane_kernel(T* u, const T* f, T h, int m, int n, int l, int dir, int s,
                                  int a_lo, int a_cnt);
// MIX (T = float only): FP32 storage with every local solve in FP64,
// rounded once to FP32.
template <typename T, bool MIX>
__global__ void fwd3_stream_kernel(const EventDesc* evs, int max_iter);
// Bytes of one node's record in the 3D adjoint workspace (lambda and three
// coefficients).
template <typename T>
constexpr size_t kAdjRecBytes = 4 * sizeof(T);
// Launch setting diag_max_l meaning "every k extent on fwd3_diag_kernel"
// (it sweeps the k axis in chunks of 64 nodes).
constexpr int kDiagAll = 1 << 30;
template <typename T, bool MIX>
__global__ void fwd3_diag_kernel(const EventDesc* evs, int max_iter);
// Several workgroups per event, all on one XCD (kernels_team.hip).
template <typename T, bool MIX, bool WIDE>
__global__ void fwd3_team_kernel(const EventDesc* evs, const TeamDesc* teams, TeamShared* sh,
                                 int nteam, int per_group, int max_iter);
// Forward then adjoint of each event in one workgroup (every event on the
// diagonal forward).
template <typename T, bool MIX>
__global__ void fwd_adj3_diag_kernel(const EventDesc* evs, int max_iter);
__global__ void info_clear_kernel(adt_info* info, int n, int* words, int64_t nwords);
template <typename T>
__global__ void strided_copy_kernel(const T* src, T* dst, int64_t N, int64_t d1, int64_t d2,
                                    int64_t s0, int64_t s1, int64_t s2, int to_rowmajor);
template <typename T>
__global__ void copy_kernel(T* dst, const T* src, int64_t N);
template <typename T>
__global__ void maxdiff_kernel(const T* a, const T* b, int64_t N, const unsigned long long* from,
                               unsigned long long* out);
template <typename T>
__global__ void lastnan_kernel(const T* a, const T* b, int64_t N, unsigned long long* last);
template <typename T>
__global__ void adj3_prep_kernel(const T* u, const T* u0, const T* g, int m, int n, int l,
                                 uint8_t* code, T* lam, T* grad_u0);
template <typename T>
__global__ void adj3_plane_kernel(const T* u, const T* g, const uint8_t* code, T* lam, int m,
                                  int n, int l, int dir, int s, int a_lo, int a_cnt, int* changed);
template <typename T>
__global__ void adj3_finish_kernel(const T* lam, const T* f, T h, int64_t N, T* grad_f);
template <typename T>
__global__ void fwd2_event_kernel(const Event2Desc* evs, int max_iter);
// 2D forward by bands of rows, one wave each (at most 1024 rows): travel times
// in LDS (kFwd2Lds bytes with their border), or in memory (MEM).
template <typename T, bool MEM>
__global__ void fwd2_band_kernel(Event2Desc ev, int max_iter);
constexpr int kFwd2Lds = 150 * 1024;
// 2D adjoint with its working values in LDS: a byte per node (adj2_codes bytes
// with a row before and after), and with LAM the multipliers, in kAdj2Lds;
// queue: 2 N ints.
template <typename T, bool LAM>
__global__ void adj2_lds_kernel(Event2Desc ev);
constexpr int kAdj2Lds = 112 * 1024, kAdj2Q = 4096;
__host__ __device__ constexpr int64_t adj2_codes(int64_t W, int64_t N) {
  return (N + 2 * (W + 4) + 15) & ~int64_t(15);
}
template <typename T>
__global__ void adj3_kahn_kernel(const EventDesc* evs);
// Tile-ordered 3D adjoint (kernels_adjoint_tile.hip), for events of at most
// kTileMax tiles of 8^3 nodes: codes, first queue, traversal; `chunks`
// workgroups per event prepare, groups of per_group resolve.  Workspace per
// event, tile by tile: lam = multipliers (T), code = upwind codes (bytes), 512
// each per tile, and behind the multipliers travel times and multipliers of the k
// faces, 128 each; queue = adj_words(): header, a count per tile, the queue.
template <typename T>
__global__ void adj3_codes_kernel(const EventDesc* evs, int chunks, int* sh, int64_t sh_words);
template <typename T>
__global__ void adj3_seeds_kernel(const EventDesc* evs, int chunks);
template <typename T>
__global__ void adj3_tile_kernel(const EventDesc* evs, TeamShared* sh, int nev, int per_group,
                                 bool pick);
constexpr int kTileEdge = 8, kTileNodes = 512, kTileFaces = 128;
constexpr int kTileMax = 65536;
constexpr int kAdjWaves = 4;  // per workgroup
// Header words (64 bytes apart): places of the queue drawn and filled, nodes
// left, 1 when the event is over (2: a wait ran out), passes over tiles.
enum { kAdjHead = 0, kAdjTail = 16, kAdjLeft = 32, kAdjOver = 48, kAdjPasses = 64, kAdjHdr = 80 };
// Places of the queue: every tile once and one for each wave that may wait; with
// more, a place is seldom used twice (which costs the check that it is empty).
constexpr int kAdjWaiters = 4096;
__host__ __device__ constexpr int adj_ring(int ntiles) { return 8 * ntiles + kAdjWaiters; }
constexpr size_t adj_words(int64_t ntiles) {
  return (size_t)kAdjHdr + (size_t)ntiles + (size_t)adj_ring((int)ntiles);
}
template <typename T>
__global__ void adj2_kahn_kernel(const Event2Desc* evs);
template <typename T>
__global__ void arith_kernel(int op, const T* a, const T* b, T* out, int64_t N);

}  // namespace adt
