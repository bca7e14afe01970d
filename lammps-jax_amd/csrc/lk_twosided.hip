// Two-sided accumulation schemes on the packed edges: LK_ACCUM_PLAIN and LK_ACCUM_HALF.
//
// PLAIN is the sparse-edge atom-force bundle (wrap_energy_fn, python/lammps_jax/export.py:153-209
// over make_setfl_energy(half_edges=False), eam.py:265-333, or the LJ energy of
// examples/export_model.py:16-50): density and pair energy sit on the sender; the energy sums
// the owned rows, or every row when an edge starts on a ghost row (export.py:183-194), or the
// owned rows only for n_hops > 1 / communicating bundles; forces are -dE/dx, so the sender takes
// +g and the receiver -g and ghost rows carry force rows for the reverse comm.
// HALF is the communicating half-edge bundle (eam.py:303-317): density to both ends, the sender
// carries the whole pair energy, ghost density partials fold into their owners (reverse comm),
// ghost F' is the owner's, and both ends take the pair force.
// In both, the engine's f gains scale * F over nall rows with newton on (AddForcesFunctor,
// cpp/pair_jax_kokkos.cpp:175-192, 959-987) and the virial is f.r over the nall rows of the
// total f (VirialFDotRFunctor, cpp:227-245), reported only with newton on (cpp:733-736).
//
// Every per-atom sum is a segmented reduction over the atom's incident edges in ascending edge
// order, so results are bitwise reproducible without float atomics:
//   count    incident-edge count per atom (integer atomics; exact)
//   scan     exclusive offsets (two-level: 4096-element chunks, then the chunk totals)
//   fill     (edge << 1 | side) into each atom's segment (atomicSub: the counts return to zero,
//            ready for the next step)
//   sort     one wave per atom ranks its segment by edge id and stores the other atom of each
//            edge with the side in the top bit (side 1: this atom is the receiver)
//   sweeps   16 lanes per atom walk the sorted segment; a fixed butterfly sums the lanes.

#include <algorithm>
#include <climits>
#include <cmath>
#include <limits>

#include "lk_eam_common.h"

namespace lk {

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanChunk = kScanThreads * kScanItems;
constexpr int kRowBlock = 1024;                // threads per row-sweep block
constexpr int kRowAtoms = 64;                  // atoms per partial tile (energy, virial slots)
// Lanes per atom in the row sweeps: a block holds kRowBlock / G atoms, kRowBlock / G / kRowAtoms
// partial tiles. Sixteen lanes for float64, eight for float32, whose lists of 50 to 100 entries
// leave fewer lanes idle that way (C4 force sweep 498 -> 404 us, density 239 -> 216 us, C5 LJ
// sweep 146 -> 122 us); the float64 steps of the small systems lost with eight (C2 0.097 ->
// 0.104 ms/step).
template <typename S>
constexpr int kLanesPerAtom = sizeof(S) == 4 ? 8 : 16;
constexpr int kIncLds = 7680;                  // 120 KB table window
constexpr int kIncDensLds = 4096;              // 64 KB density-table window (two blocks per CU)
// Force sweep two blocks per CU with the density-sized window: fp32 (fp64 would spill).
template <typename S>
constexpr bool kForceTwoBlocks = sizeof(S) == 4;

struct IncArgs {
  const int *senders;
  const int *receivers;
  const unsigned char *mask;
  const StepResult *result;
  int max_edges;
  int nrows;  // atoms that may appear on an edge (max_atoms)
  int *deg;   // [nrows + 1], zero between steps
  int *loc;   // [nrows + 1] offsets within each scan chunk
  int *part;  // [chunks] exclusive chunk offsets
  uint32_t *tmp;
  int *inc;
  int2 *span;  // [nrows] first entry and entries of each atom's list
};

__device__ __forceinline__ long live_edges(const StepResult *r, int max_edges)
{
  const long c = r->edge_count;
  return c < max_edges ? c : max_edges;
}

__global__ __launch_bounds__(256) void k_clear_int(int *p, long n)
{
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__device__ __forceinline__ int inc_off(const int *loc, const int *part, int a)
{
  return loc[a] + part[a / kScanChunk];
}

__device__ __forceinline__ bool edge_ends(const IncArgs &a, long e, int &s, int &r)
{
  if (!a.mask[e]) return false;
  s = a.senders[e];
  r = a.receivers[e];
  return s >= 0 && s < a.nrows && r >= 0 && r < a.nrows;
}

__global__ __launch_bounds__(256) void k_inc_count(IncArgs a)
{
  const long n = live_edges(a.result, a.max_edges);
  for (long e = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < n;
       e += static_cast<long>(gridDim.x) * blockDim.x) {
    int s, r;
    if (!edge_ends(a, e, s, r)) continue;
    atomicAdd(&a.deg[s], 1);
    atomicAdd(&a.deg[r], 1);
  }
}

// Exclusive scan of in[0, n) within 4096-element chunks; chunk totals to part[].
__global__ __launch_bounds__(kScanThreads) void k_scan_chunks(const int *__restrict__ in, int n,
                                                              int *__restrict__ out,
                                                              int *__restrict__ part)
{
  __shared__ int wsum[kScanThreads / kWave];
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const long base = static_cast<long>(blockIdx.x) * kScanChunk + static_cast<long>(t) * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    v[q] = base + q < n ? in[base + q] : 0;
    s += v[q];
  }
  int incl = s;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int y = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += y;
  }
  if (lane == kWave - 1) wsum[wave] = incl;
  __syncthreads();
  if (wave == 0) {
    const int w = lane < kScanThreads / kWave ? wsum[lane] : 0;
    int wi = w;
#pragma unroll
    for (int off = 1; off < kScanThreads / kWave; off <<= 1) {
      const int y = __shfl_up(wi, off, kWave);
      if (lane >= off) wi += y;
    }
    if (lane < kScanThreads / kWave) wsum[lane] = wi - w;
  }
  __syncthreads();
  int run = wsum[wave] + incl - s;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    if (base + q < n) out[base + q] = run;
    run += v[q];
  }
  if (t == kScanThreads - 1) part[blockIdx.x] = run;
}

// Exclusive scan of the chunk totals in place (one block).
__global__ __launch_bounds__(kScanThreads) void k_scan_parts(int *__restrict__ part, int nparts)
{
  __shared__ int wsum[kScanThreads / kWave];
  __shared__ int carry;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int b0 = 0; b0 < nparts; b0 += kScanThreads) {
    const int i = b0 + t;
    const int v = i < nparts ? part[i] : 0;
    int incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) wsum[wave] = incl;
    __syncthreads();
    if (wave == 0) {
      const int w = lane < kScanThreads / kWave ? wsum[lane] : 0;
      int wi = w;
#pragma unroll
      for (int off = 1; off < kScanThreads / kWave; off <<= 1) {
        const int y = __shfl_up(wi, off, kWave);
        if (lane >= off) wi += y;
      }
      if (lane < kScanThreads / kWave) wsum[lane] = wi - w;
    }
    __syncthreads();
    const int c = carry;
    if (i < nparts) part[i] = c + wsum[wave] + incl - v;
    __syncthreads();
    if (t == kScanThreads - 1) carry = c + wsum[wave] + incl;
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void k_inc_fill(IncArgs a)
{
  const long n = live_edges(a.result, a.max_edges);
  for (long e = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < n;
       e += static_cast<long>(gridDim.x) * blockDim.x) {
    int s, r;
    if (!edge_ends(a, e, s, r)) continue;
    const uint32_t key = static_cast<uint32_t>(e) << 1;
    const int ps = inc_off(a.loc, a.part, s) + atomicSub(&a.deg[s], 1) - 1;
    a.tmp[ps] = key;
    const int pr = inc_off(a.loc, a.part, r) + atomicSub(&a.deg[r], 1) - 1;
    a.tmp[pr] = key | 1u;
  }
}

// One wave per atom: the rank of each entry is the number of smaller keys in the segment
// (keys are distinct), so the store order is ascending edge id whatever order fill left.
__global__ __launch_bounds__(256) void k_inc_sort(IncArgs a, int nsort)
{
  const int atom = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (atom >= nsort) return;  // whole wave
  const int b = inc_off(a.loc, a.part, atom);
  const int L = inc_off(a.loc, a.part, atom + 1) - b;
  if (lane == 0) a.span[atom] = make_int2(b, L);
  for (int c0 = 0; c0 < L; c0 += kWave) {
    const bool mine = c0 + lane < L;
    const uint32_t v = mine ? a.tmp[b + c0 + lane] : 0xFFFFFFFFu;
    int rank = 0;
    for (int c1 = 0; c1 < L; c1 += kWave) {
      const uint32_t w = c1 + lane < L ? a.tmp[b + c1 + lane] : 0xFFFFFFFFu;
#pragma unroll 16
      for (int m = 0; m < kWave; ++m) {
        // lane m's key broadcast through a scalar register (v_readlane), not the LDS crossbar
        const uint32_t wm =
            static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w), m));
        rank += wm < v ? 1 : 0;
      }
    }
    if (mine) {
      const long e = v >> 1;
      const uint32_t side = v & 1u;
      const int other = side ? a.senders[e] : a.receivers[e];
      a.inc[b + rank] = static_cast<int>(static_cast<uint32_t>(other) | (side << 31));
    }
  }
}

// Incidence lists from the neighbour-list slots (once per list). Slot (ii, jj) passes the
// list's static filters of PackNeighborFunctor (cpp:84-94: rows past max_atoms, jj >= numneigh,
// j >= max_atoms, the half filter j < i); its distance filter is applied each step. Atom a's
// list is its out-entries (the kept slots of its own row, in slot order: other = j) followed by
// its in-entries (slots of other rows naming a: other = i, side bit set) in ascending i.

// How the bins of the build are laid out (k_inc_lists).
struct BinLayout {
  int bin_log;   // atoms per bin: 1 << bin_log
  int per_atom;  // in-entries kept in LDS per atom; 0: none, the bins sort theirs
  int pitch;     // slots per staged row
};
struct ListArgs {
  const int *ilist;
  const int *numneigh;
  const int *neighbors;
  long stride;
  int rows;
  int maxneighs;
  int max_atoms;
  int half_filter;
  int *out_n;   // list slots of each atom's row (0: the atom is no row)
  int *row_of;  // list row of each atom that is one; null without inc_bit
  int2 *span;   // first entry and entries of each atom
  int *inc;
  uint32_t *inc_bit;  // each entry's place among the validity bits, rows of words `bit_pitch` apart;
                      // null: not wanted
  int bit_pitch;
  uint32_t *claim;  // the sorted path's marks where LDS does not hold them, a word per in-entry
  int fold;         // the plain scheme's fold
  int slots;        // the entries carry their slots
  BinLayout layout;
  int *longest;  // lists with room for longer rows than 32-atom bins take: the longest row, which
                 // the layout then goes by; else null
};

// The row atom of list row ii and its slot count, or -1 when the row packs nothing.
__device__ __forceinline__ int list_row(const ListArgs &L, int ii, int &nn)
{
  const int i = L.ilist[ii];
  nn = 0;
  if (i < 0 || i >= L.max_atoms) return -1;
  nn = min(L.numneigh[i], L.maxneighs);
  return i;
}

__device__ __forceinline__ bool list_neighbor(const ListArgs &L, int i, int jj, int &j)
{
  j = L.neighbors[static_cast<long>(jj) * L.stride + i] & kNeighMask;
  if (j >= L.max_atoms) return false;
  return !(L.half_filter && j < i);
}

// The place of slot jj of list row ii among the validity bits: word (jj >> 5) * pitch + ii, bit jj & 31.
__device__ __forceinline__ uint32_t slot_bit(const ListArgs &L, int ii, int jj)
{
  return ((static_cast<uint32_t>(jj >> 5) * static_cast<uint32_t>(L.bit_pitch) +
           static_cast<uint32_t>(ii)) << 5) | static_cast<uint32_t>(jj & 31);
}

// An in-entry (row i names atom a) whose reverse slot is one of a's out-entries (a's row names
// i) gives a the same pair force in the plain scheme: the two slots pass the pack's distance
// filter together (r^2 is the same sum of the negated differences), and a's plain-scheme share of
// edge i -> a, -g = coef (x_i - x_a), equals that of a -> i (coef depends on r only). Such an
// in-entry is dropped and the out-entry marked (kIncPaired), and the sweeps weigh the out-entry
// by the ends whose rows count. Each owned pair is then evaluated once per end instead of twice.
constexpr uint32_t kIncPaired = 1u << 30;
constexpr uint32_t kIncAtom = 0x3FFFFFFFu;
constexpr uint32_t kIncNone = 0xFFFFFFFFu;

// ---------------------------------------------------------------------------------------------
// The list-built incidence lists through bins of atoms (once per list)
// ---------------------------------------------------------------------------------------------
// The kept slots keyed by the atom they name are brought together in bins of 64 atoms (fewer for
// rows too long for LDS): a count per bin, an exclusive scan, a scatter into the bins' ranges,
// then one block per bin puts its atoms' lists together in LDS. The scatter's order inside a bin
// follows atomic claims; the last pass orders each atom's in-entries by row atom, so the lists are
// the same from run to run. The list is read four times, the entries written twice and read twice;
// a radix sort of (atom, slot) pairs, the placing of out- and in-entries and the fold went over
// the entries nine times: build of 256,000 atoms' half list (12.6 M entries) 566 -> 261 us,
// of a 131,072-atom list with ghost rows (14 M entries, nearly all folded) 890 -> 295 us.
constexpr int kBinLog = 6;
constexpr int kBinAtoms = 1 << kBinLog;  // at most
constexpr int kBinMeasureLog = 5;        // room for smaller bins than this: the rows are measured
constexpr int kBinPool = 62 * 1024;      // LDS of a bin's lists (two blocks or more share a CU)
constexpr int kBinWaves = 16;            // waves of a counting block: kBinWaves / W 64-row tiles
constexpr int kBinTable = 2048;          // bins a block counts in LDS; others go to memory at once
constexpr int kBinProbes = 8;

// An entry on its way: the atom's place in its bin above the row atom, in 32 bits where atoms stay
// below 2^26 - 1; in 64 past that, and where the lists keep their slots' validity bit addresses: the
// slot is then below the row atom.
template <typename E>
struct Entry;
template <>
struct Entry<uint32_t> {
  static constexpr bool kSlot = false;
  static __device__ __forceinline__ uint32_t make(int place, int row_atom, int)
  {
    return (static_cast<uint32_t>(place) << 26) | static_cast<uint32_t>(row_atom);
  }
  static __device__ __forceinline__ uint32_t who(uint32_t v) { return v; }  // without the slot
  static __device__ __forceinline__ int place(uint32_t v) { return static_cast<int>(v >> 26); }
  static __device__ __forceinline__ uint32_t row_atom(uint32_t v) { return v & ((1u << 26) - 1); }
  static __device__ __forceinline__ int slot(uint32_t) { return 0; }
};
template <>
struct Entry<uint64_t> {
  static constexpr bool kSlot = true;
  static __device__ __forceinline__ uint64_t make(int place, int row_atom, int slot)
  {
    return (static_cast<uint64_t>(place) << 56) | (static_cast<uint64_t>(row_atom) << 26) |
           static_cast<uint64_t>(slot);
  }
  static __device__ __forceinline__ uint64_t who(uint64_t v) { return v >> 26; }
  static __device__ __forceinline__ int place(uint64_t v) { return static_cast<int>(v >> 56); }
  static __device__ __forceinline__ uint32_t row_atom(uint64_t v)
  {
    return static_cast<uint32_t>(v >> 26) & ((1u << 30) - 1);
  }
  static __device__ __forceinline__ int slot(uint64_t v)
  {
    return static_cast<int>(v & ((1u << 26) - 1));
  }
};

// Atoms per bin: 64, or fewer where the out-entries of that many rows and their in-entries (with
// a fold, hash tables four fifths full at the longest row's length) would take more than kBinPool.
// Rows past 1,760 slots (1,980 without a fold) keep bins of four atoms and sort. Entries with slots
// take 16 bits more each (rows past 1,376 and 1,584).
__host__ __device__ inline BinLayout bin_layout(long longest, bool fold, bool slots)
{
  const long per = fold ? (longest * 5 / 4 + 7) / 4 * 4 : (longest + 7) / 4 * 4;
  const long pitch = longest | 1, atom = 4 * (per + pitch) + (slots ? 2 * per : 0);
  BinLayout y{kBinLog, 0, 0};
  while (y.bin_log > kBinMinLog && atom << y.bin_log > kBinPool) --y.bin_log;
  if (atom << y.bin_log <= kBinPool) {
    y.per_atom = static_cast<int>(per);
    y.pitch = static_cast<int>(pitch);
  }
  return y;
}

// An engine's list may have room for far more slots than its rows have, so where the room alone
// would make the bins smaller than 32 atoms the rows are measured on the device first. By the room,
// the step on a new list of 32,000 LJ atoms with 80 slots a row (plain) took 245 us at room for 240
// slots, 998 at 700 and 6,390 at 1,700; by the rows it takes 164 at each (153 at room for 80). The
// measuring takes 10 to 14 us: rows that do fill room for 108 to 218 slots would lose that for
// nothing.
__device__ __forceinline__ BinLayout bin_layout_of(const ListArgs &L)
{
  return L.longest ? bin_layout(*L.longest, L.fold != 0, L.slots != 0) : L.layout;
}

__device__ __forceinline__ int bin_count(const ListArgs &L, const BinLayout &y)
{
  return (L.max_atoms + (1 << y.bin_log) - 1) >> y.bin_log;
}

__global__ __launch_bounds__(256) void k_inc_longest(ListArgs L)
{
  const int ii = blockIdx.x * blockDim.x + threadIdx.x;
  int nn = 0;
  if (ii < L.rows) list_row(L, ii, nn);
  const int most = wave_max_int(nn);
  if ((threadIdx.x & (kWave - 1)) == 0 && most > 0) atomicMax(L.longest, most);
}

// The bins' counters and offsets, [cap] each (offsets [cap + 1]).
struct Bins {
  int cap;    // bins there is room for
  int *next;  // in-entries, then the scatter's next free place
  int *out;   // out-entries (list slots)
  int *off;   // first in-entry in the scatter's output
  int *loff;  // first entry in the lists
};

__global__ __launch_bounds__(256) void k_inc_clear(ListArgs L, Bins B)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < L.max_atoms) L.out_n[i] = 0;
  if (i < B.cap) {
    B.next[i] = 0;
    B.out[i] = 0;
  }
}

// Count (SCATTER false: the in- and out-entries of each bin; also out_n) and scatter.
// One lane per row, the W waves of a tile sharing its slots; entries of adjacent lanes in the same
// bin (adjacent rows' k-th neighbours mostly are) count as one run, so a wave does one LDS update
// per run.
template <bool SCATTER, typename E, int W>
__global__ __launch_bounds__(kBinWaves *kWave) LK_EIGHT_WAVES
void k_inc_bins(ListArgs L, Bins B, E *__restrict__ tmp)
{
  __shared__ int tag[kBinTable], cnt[kBinTable];
  __shared__ int aux[kBinTable];  // count: out-entries; scatter: the block's first place
  constexpr int kThreads = kBinWaves * kWave, kTiles = kBinWaves / W;
  const int wave = wave_in_block(), lane = threadIdx.x & (kWave - 1);
  const int wq = wave % W;
  const int ii = (blockIdx.x * kTiles + wave / W) * kWave + lane;
  for (int k = threadIdx.x; k < kBinTable; k += kThreads) {
    tag[k] = -1;
    cnt[k] = 0;
    aux[k] = 0;
  }
  int nn = 0, i = -1;
  if (ii < L.rows) i = list_row(L, ii, nn);
  const int nmax = wave_max_int(nn);
  const int bin_log = bin_layout_of(L).bin_log;
  __syncthreads();
  // the LDS slot of bin b, or -1 when the probed slots hold other bins (they keep them: the same
  // answer in both walks of the scatter)
  auto slot_of = [&](int b) -> int {
    uint32_t h = (static_cast<uint32_t>(b) * 2654435761u) >> 21;  // kBinTable = 2^11
    for (int probe = 0; probe < kBinProbes; ++probe) {
      int old = __hip_atomic_load(&tag[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (old == -1) old = atomicCAS(&tag[h], -1, b);
      if (old == -1 || old == b) return static_cast<int>(h);
      h = (h + 1) & (kBinTable - 1);
    }
    return -1;
  };
  if (!SCATTER && wq == 0 && i >= 0) {
    L.out_n[i] = nn;
    if (L.row_of) L.row_of[i] = ii;
    const int q = slot_of(i >> bin_log);
    atomicAdd(q >= 0 ? &aux[q] : &B.out[i >> bin_log], nn);
  }
  auto walk = [&](auto &&use) {
    constexpr int kBatch = 8;
    for (int j0 = wq; j0 < nmax; j0 += W * kBatch) {
      int raw[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int jj = j0 + W * u;
        raw[u] = jj < nn ? L.neighbors[static_cast<long>(jj) * L.stride + i] : 0;
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (j0 + W * u >= nmax) break;  // wave-uniform
        const int j = raw[u] & kNeighMask;
        // list_neighbor's filter on the loaded entry
        const bool ok = j0 + W * u < nn && j < L.max_atoms && !(L.half_filter && j < i);
        const int b = ok ? j >> bin_log : -1;
        const int before = __shfl_up(b, 1, kWave);
        const bool head = lane == 0 || before != b;
        const uint64_t heads = wave_ballot(head);
        const uint64_t upto = (2ull << lane) - 1ull;  // lanes up to this one
        const uint64_t next = heads & ~upto;
        const int n = (next ? __builtin_ctzll(next) : kWave) - lane;  // a head's run
        use(j, j0 + W * u, b, head, n, 63 - __builtin_clzll(heads & upto));
      }
    }
  };
  walk([&](int, int, int b, bool head, int n, int) {
    if (!head || b < 0) return;
    const int q = slot_of(b);
    if (q >= 0)
      atomicAdd(&cnt[q], n);
    else if (!SCATTER)
      atomicAdd(&B.next[b], n);
  });
  __syncthreads();
  for (int k = threadIdx.x; k < kBinTable; k += kThreads) {
    if (tag[k] < 0) continue;
    if constexpr (SCATTER) {
      if (cnt[k] == 0) continue;
      aux[k] = atomicAdd(&B.next[tag[k]], cnt[k]);
      cnt[k] = 0;
    } else {
      if (cnt[k]) atomicAdd(&B.next[tag[k]], cnt[k]);
      if (aux[k]) atomicAdd(&B.out[tag[k]], aux[k]);
    }
  }
  if constexpr (SCATTER) {
    __syncthreads();
    walk([&](int j, int jj, int b, bool head, int n, int first) {
      int at = 0;
      if (head && b >= 0) {
        const int q = slot_of(b);
        at = q >= 0 ? aux[q] + atomicAdd(&cnt[q], n) : atomicAdd(&B.next[b], n);
      }
      at = __shfl(at, first, kWave) + lane - first;
      if (b >= 0)
        tmp[at] = Entry<E>::make(j & ((1 << bin_log) - 1), i, jj);
    });
  }
}

// Exclusive scans of the bins' in-entries (off, and next in place) and of all their entries (loff),
// one block.
__global__ __launch_bounds__(kScanThreads) void k_inc_bin_scan(ListArgs L, Bins B)
{
  const int nbins = bin_count(L, bin_layout_of(L));
  __shared__ int wsum[2][kScanThreads / kWave];
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  int carry = 0, carry_l = 0;
  for (int b0 = 0; b0 < nbins; b0 += kScanChunk) {
    int v[kScanItems], w[kScanItems], s = 0, sl = 0;
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
      const int k = b0 + t * kScanItems + q;
      v[q] = k < nbins ? B.next[k] : 0;
      w[q] = k < nbins ? v[q] + B.out[k] : 0;
      s += v[q];
      sl += w[q];
    }
    int incl = s, incl_l = sl;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int y = __shfl_up(incl, o, kWave), yl = __shfl_up(incl_l, o, kWave);
      if (lane >= o) {
        incl += y;
        incl_l += yl;
      }
    }
    if (lane == kWave - 1) {
      wsum[0][wave] = incl;
      wsum[1][wave] = incl_l;
    }
    __syncthreads();
    int run = carry + incl - s, run_l = carry_l + incl_l - sl;
    for (int q = 0; q < kScanThreads / kWave; ++q) {
      run += q < wave ? wsum[0][q] : 0;
      run_l += q < wave ? wsum[1][q] : 0;
      carry += wsum[0][q];
      carry_l += wsum[1][q];
    }
#pragma unroll
    for (int q = 0; q < kScanItems; ++q) {
      const int k = b0 + t * kScanItems + q;
      if (k < nbins) {
        B.next[k] = run;
        B.off[k] = run;
        B.loff[k] = run_l;
      }
      run += v[q];
      run_l += w[q];
    }
    __syncthreads();
  }
  if (t == 0) B.off[nbins] = carry;
}

__device__ __forceinline__ uint32_t bin_hash(uint32_t atom, uint32_t slots)
{
  return static_cast<uint32_t>((static_cast<uint64_t>(atom * 2654435761u) * slots) >> 32);
}

// Values below v among the `n4` groups of four at `v4`. TIES: values equal to v before index `at`
// count too, so that equal values (a list that names an atom twice) take places of their own.
template <bool TIES>
__device__ __forceinline__ int rank_of(const uint4 *v4, int n4, uint32_t v, int at)
{
  int rank = 0;
  for (int m = 0; m < n4; ++m) {
    const uint4 q = v4[m];
    rank += (q.x < v ? 1 : 0) + (q.y < v ? 1 : 0) + (q.z < v ? 1 : 0) + (q.w < v ? 1 : 0);
    if (TIES)
      rank += (q.x == v && 4 * m + 0 < at ? 1 : 0) + (q.y == v && 4 * m + 1 < at ? 1 : 0) +
              (q.z == v && 4 * m + 2 < at ? 1 : 0) + (q.w == v && 4 * m + 3 < at ? 1 : 0);
  }
  return rank;
}

// One wave gives use(rank, value, index) the `c` values of slots[0, n) below 2^31 (`n` a multiple of
// four) with their places in ascending order. Distinct values have the ranks 0 .. c - 1, which sum to
// c (c - 1) / 2; any other sum means equal ones, and the ranks are taken again with ties broken.
template <class Use>
__device__ __forceinline__ void store_ranked(const uint32_t *slots, int n, int c, Use &&use)
{
  const uint4 *v4 = reinterpret_cast<const uint4 *>(slots);
  const int lane = threadIdx.x & (kWave - 1);
  int sum = 0;
  for (int q = lane; q < n; q += kWave) {
    const uint32_t v = slots[q];
    if (v >> 31) continue;
    const int r = rank_of<false>(v4, n / 4, v, q);
    use(r, v, q);
    sum += r;
  }
  if (wave_sum(sum) == c * (c - 1) / 2) return;
  for (int q = lane; q < n; q += kWave) {
    const uint32_t v = slots[q];
    if (v >> 31) continue;
    use(rank_of<true>(v4, n / 4, v, q), v, q);
  }
}

// One block per bin: the lists of its atoms. Their out-entries are staged in LDS, `pitch` slots per
// atom (odd: no bank conflicts), and their in-entries meet in `per_atom` slots per atom: for
// the half scheme as segments, for the plain one as hash tables of row atoms, in which the
// out-entries look up their reverse (one that finds it is marked, and the in-entry leaves). The
// out-entries are written without their gaps, what is left of the in-entries ranked by row atom.
// A bin whose in-entries do not fit, one with a row that names an atom twice and whose reverse is
// there, and every bin when `per_atom` is 0, sorts its in-entries instead (in LDS where they fit its
// `pool_words`, else where they are) and finds them by bisection. By either path the m-th slot of a
// row naming an atom pairs with the m-th slot of that atom's row naming it back.
// A search of the bin's rows and entries for each entry stood in place of the sort: with rows of
// 2,117 slots (4,000 LJ atoms, 8.4 M entries, plain) 45.5 ms; the sort takes 0.46 ms.
constexpr int kListThreads = 1024;
constexpr int kSortHead = 256;  // words of the sorted path's offsets at the start of the pool

// Ascending sort of T[0, n) by a whole block: bitonic merges whose every comparison leaves the
// smaller value at the lower place, so places past n, taken as largest, need not exist.
template <typename E>
__device__ __forceinline__ void sort_entries(E *T, int n)
{
  auto order = [&](int lo, int hi) {
    if (hi >= n) return;
    const E u = T[lo], v = T[hi];
    if (v < u) {
      T[lo] = v;
      T[hi] = u;
    }
  };
  for (int half = 1, log = 0; half < n; half <<= 1, ++log) {
    // blocks of 2 half places, each half sorted: the first half against the second reversed
    for (int q = threadIdx.x; (q >> log) * 2 * half < n; q += kListThreads) {
      const int at = (q >> log) * 2 * half, k = q & (half - 1);
      order(at + k, at + 2 * half - 1 - k);
    }
    __syncthreads();
    for (int j = half >> 1, jl = log - 1; j > 0; j >>= 1, --jl) {
      for (int q = threadIdx.x; (q >> jl) * 2 * j < n; q += kListThreads) {
        const int at = (q >> jl) * 2 * j + (q & (j - 1));
        order(at, at + j);
      }
      __syncthreads();
    }
  }
}

// First place of ascending T[0, n) that is not below v.
template <typename E>
__device__ __forceinline__ int lower_bound(const E *T, int n, E v)
{
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if (T[mid] < v)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

template <typename E, bool FOLD>
__global__ __launch_bounds__(kListThreads) LK_EIGHT_WAVES
void k_inc_lists(ListArgs L, Bins B, E *__restrict__ tmp, int pool_words)
{
  extern __shared__ __align__(16) uint32_t pool[];  // [atoms][per_atom], [atoms][pitch], slots
  __shared__ int nin[kBinAtoms], nout[kBinAtoms], rown[kBinAtoms];
  __shared__ int start[kBinAtoms], seg[kBinAtoms], next[kBinAtoms];
  __shared__ int spill;
  constexpr int kWaves = kListThreads / kWave;
  const int tid = threadIdx.x, wave = wave_in_block(), lane = tid & (kWave - 1);
  const BinLayout y = bin_layout_of(L);
  if (static_cast<int>(blockIdx.x) >= bin_count(L, y)) return;  // whole block
  const int per_atom = y.per_atom, pitch = y.pitch;
  const int na = 1 << y.bin_log, a0 = blockIdx.x << y.bin_log;
  const int e0 = B.off[blockIdx.x], n = B.off[blockIdx.x + 1] - e0;
  const int slots = na * per_atom;
  uint32_t *outs = pool + slots;
  // the in-entries' slots, which 16 bits hold: longer rows than these sort
  uint16_t *in_slot = reinterpret_cast<uint16_t *>(outs + na * pitch);
  auto atom_of = [](E v) { return Entry<E>::place(v); };
  auto row_atom = [](E v) { return Entry<E>::row_atom(v); };
  if (tid < kBinAtoms) {
    nin[tid] = 0;
    nout[tid] = 0;
    next[tid] = 0;
    rown[tid] = tid < na && a0 + tid < L.max_atoms ? L.out_n[a0 + tid] : 0;
  }
  if (tid == 0) spill = per_atom == 0;
  for (int k = tid; k < slots; k += kListThreads) pool[k] = kIncNone;
  __syncthreads();
  // the places of the atoms' lists from their counts, by the first wave
  auto place = [&]() {
    if (wave == 0) {
      const int c4 = (nin[lane] + 3) & ~3, c = nin[lane] + nout[lane];
      int incl = c, incl4 = c4;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int y = __shfl_up(incl, o, kWave), y4 = __shfl_up(incl4, o, kWave);
        if (lane >= o) {
          incl += y;
          incl4 += y4;
        }
      }
      start[lane] = B.loff[blockIdx.x] + incl - c;
      seg[lane] = incl4 - c4;
      if (!FOLD && incl4 > slots) spill = 1;  // the half scheme's segments
      if (lane < na && a0 + lane < L.max_atoms) {
        L.span[a0 + lane] = make_int2(start[lane], c);
      }
    }
    __syncthreads();
  };
  // thread t stages the slots t / na, + threads / na, ... of atom t % na
  const int d_own = tid & (na - 1), q0 = tid >> y.bin_log, qstep = kListThreads >> y.bin_log;
  // The expectations keep the sorted path out of the way of the others (142.5 -> 139.9 us of the lists
  // of 256,000 atoms' half list, what they take without it).
  if (__builtin_expect(per_atom > 0, 1)) {
    if constexpr (FOLD) {
      for (int e = tid; e < n; e += kListThreads) {
        const E v = tmp[e0 + e];
        uint32_t *keys = pool + atom_of(v) * per_atom;
        uint32_t h = bin_hash(row_atom(v), per_atom);
        bool in = false;
        for (int probe = 0; probe < per_atom && !in; ++probe) {
          in = atomicCAS(&keys[h], kIncNone, row_atom(v)) == kIncNone;
          if constexpr (Entry<E>::kSlot)
            if (in) in_slot[atom_of(v) * per_atom + h] = static_cast<uint16_t>(Entry<E>::slot(v));
          if (++h == static_cast<uint32_t>(per_atom)) h = 0;
        }
        if (!in) spill = 1;
      }
      __syncthreads();
    } else {
      for (int e = tid; e < n; e += kListThreads) atomicAdd(&nin[atom_of(tmp[e0 + e])], 1);
    }
    uint32_t *keys = pool + d_own * per_atom;
    for (int b0 = q0; b0 < rown[d_own]; b0 += 4 * qstep) {
      int raw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int jj = b0 + u * qstep;
        raw[u] = jj < rown[d_own]
                     ? L.neighbors[static_cast<long>(jj) * L.stride + a0 + d_own] & kNeighMask
                     : INT_MAX;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int jj = b0 + u * qstep, j = raw[u];
        if (jj >= rown[d_own]) break;
        uint32_t v = static_cast<uint32_t>(j);
        if (j >= L.max_atoms || (L.half_filter && j < a0 + d_own)) {
          v = kIncNone;  // list_neighbor's filter
        } else if constexpr (FOLD) {
          // the claim is made once, past the search: inside it each step waits for the atomic
          // (131,072 LJ atoms with ghost rows, 14 M entries: lists 239 -> 166 us)
          uint32_t h = bin_hash(v, per_atom), k = kIncNone;
          for (int probe = 0; probe < per_atom; ++probe) {
            k = keys[h];
            if (k == kIncNone || (k & ~(1u << 31)) == static_cast<uint32_t>(j)) break;
            k = kIncNone;
            if (++h == static_cast<uint32_t>(per_atom)) h = 0;
          }
          if (k != kIncNone) {
            if (!(k >> 31) && !(atomicOr(&keys[h], 1u << 31) >> 31))
              v |= kIncPaired;
            else
              spill = 1;  // the row names j again: the sorted path tells its slots apart
          }
        }
        outs[d_own * pitch + jj] = v;
      }
    }
    __syncthreads();
    for (int d = wave; d < na; d += kWaves) {
      int c = 0, ci = 0;
      for (int k = 0; k < rown[d]; k += kWave)
        c += __popcll(wave_ballot(k + lane < rown[d] && outs[d * pitch + k + lane] != kIncNone));
      if (FOLD)
        for (int k = 0; k < per_atom; k += kWave)
          ci += __popcll(wave_ballot(k + lane < per_atom && !(pool[d * per_atom + k + lane] >> 31)));
      if (lane == 0) {
        nout[d] = c;
        if (FOLD) nin[d] = ci;
      }
    }
    __syncthreads();
    const bool fits = !FOLD || !spill;
    if (fits) place();
    if (__builtin_expect(fits && !spill, 1)) {
      if constexpr (!FOLD) {
        for (int e = tid; e < n; e += kListThreads) {
          const E v = tmp[e0 + e];
          const int d = atom_of(v), at = seg[d] + atomicAdd(&next[d], 1);
          pool[at] = row_atom(v);
          if constexpr (Entry<E>::kSlot) in_slot[at] = static_cast<uint16_t>(Entry<E>::slot(v));
        }
        __syncthreads();
      }
      for (int d = wave; d < na; d += kWaves) {
        int to = start[d];
        int ii = 0;
        if constexpr (Entry<E>::kSlot)
          if (L.inc_bit && rown[d] > 0) ii = L.row_of[a0 + d];
        for (int k = 0; k < rown[d]; k += kWave) {
          const uint32_t v = k + lane < rown[d] ? outs[d * pitch + k + lane] : kIncNone;
          const uint64_t M = wave_ballot(v != kIncNone);
          if (v != kIncNone) {
            L.inc[to + lanes_below(M)] = static_cast<int>(v);
            if constexpr (Entry<E>::kSlot)
              if (L.inc_bit) L.inc_bit[to + lanes_below(M)] = slot_bit(L, ii, k + lane);
          }
          to += __popcll(M);
        }
        const int in0 = FOLD ? d * per_atom : seg[d];
        if (nin[d] > 0)
          store_ranked(pool + in0, FOLD ? per_atom : (nin[d] + 3) & ~3, nin[d],
                       [&](int r, uint32_t v, int q) {
                         L.inc[to + r] = static_cast<int>(v | (1u << 31));
                         if constexpr (Entry<E>::kSlot)
                           if (L.inc_bit)
                             L.inc_bit[to + r] = slot_bit(L, L.row_of[v], in_slot[in0 + q]);
                       });
      }
      return;
    }
    __syncthreads();  // every wave has left the pool
  }
  // The sorted path. first: each atom's first in-entry; the waves share the atoms' slots and
  // in-entries out in strips, each first counted, then written from the place the counts leave it.
  int *first = reinterpret_cast<int *>(pool);  // [na + 1]
  int *strip_out = first + 2 * kBinAtoms, *strip_in = strip_out + kBinAtoms;
  static_assert(4 * kBinAtoms <= kSortHead && kWaves <= kBinAtoms, "the offsets fit");
  const int strips = na < kWaves ? kWaves / na : 1;  // of an atom
  auto sorted_lists = [&](const E *T, uint32_t *claims, bool in_lds) {
    for (int d = tid; d <= na; d += kListThreads)
      first[d] = d < na ? lower_bound(T, n, Entry<E>::make(d, 0, 0)) : n;
    auto same = [](E u, E v) { return Entry<E>::who(u) == Entry<E>::who(v); };
    // The place of the in-entry from row j to atom d, the first of equal ones, or -1.
    auto find = [&](int d, int j) -> int {
      const E key = Entry<E>::make(d, j, 0);
      const int at = lower_bound(T, n, key);
      return at < n && same(T[at], key) ? at : -1;
    };
    // A run's first entry: its row atom is named by a slot of the atom's own row, and by another.
    const int marks = (n + 31) >> 5;
    uint32_t *named = claims, *again = claims + marks;
    auto marked = [](const uint32_t *set, int at) -> bool {
      return (__hip_atomic_load(&set[at >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >>
              (at & 31)) & 1u;
    };
    if constexpr (FOLD) {
      for (int k = tid; k < 2 * marks; k += kListThreads)
        __hip_atomic_store(&named[k], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // writes L2 back, most of the time of a small bin (4.56 ms for the 0.46 ms above)
      if (!in_lds) __threadfence();
      __syncthreads();
      for (int jj = q0; jj < rown[d_own]; jj += qstep) {
        int j;
        if (!list_neighbor(L, a0 + d_own, jj, j)) continue;
        const int at = find(d_own, j);
        if (at < 0) continue;
        const uint32_t bit = 1u << (at & 31);
        if (atomicOr(&named[at >> 5], bit) & bit) atomicOr(&again[at >> 5], bit);
      }
      if (!in_lds) __threadfence();
    }
    __syncthreads();
    // slots of atom d's row below `end` that name j
    auto naming = [&](int d, int end, int j) -> int {
      int c = 0;
      for (int k = 0; k < end; ++k) {
        int jk;
        c += list_neighbor(L, a0 + d, k, jk) && jk == j ? 1 : 0;
      }
      return c;
    };
    auto paired = [&](int d, int jj, int j) -> bool {
      const int at = find(d, j);
      if (at < 0 || !marked(again, at)) return at >= 0;
      const int mth = at + naming(d, jj, j);
      return mth < n && same(T[mth], T[at]);
    };
    auto folded = [&](int d, int e) -> bool {
      int at = e;
      while (at > 0 && same(T[at - 1], T[e])) --at;
      if (at == e || !marked(again, at)) return at == e && marked(named, at);
      return e - at < naming(d, rown[d], static_cast<int>(row_atom(T[e])));
    };
    // out(u, d, jj, j, rank) for the kept slots of strip u of atom d, in(u, d, e, rank) for its
    // unfolded in-entries, end(u, slots, in-entries)
    auto walk = [&](auto &&out, auto &&in, auto &&end) {
      for (int u = wave; u < na * strips; u += kWaves) {
        const int d = u / strips, part = u % strips;
        auto range = [&](int len, int &lo, int &hi) {
          const int per = (len + strips - 1) / strips;
          lo = min(part * per, len);
          hi = min(lo + per, len);
        };
        int lo, hi, c = 0, ci = 0;
        range(rown[d], lo, hi);
        for (int k = lo; k < hi; k += kWave) {
          int j = 0;
          const bool kept = k + lane < hi && list_neighbor(L, a0 + d, k + lane, j);
          const uint64_t M = wave_ballot(kept);
          if (kept) out(u, d, k + lane, j, c + lanes_below(M));
          c += __popcll(M);
        }
        range(first[d + 1] - first[d], lo, hi);
        for (int k = lo; k < hi; k += kWave) {
          const int e = first[d] + k + lane;
          const bool kept = k + lane < hi && !(FOLD && folded(d, e));
          const uint64_t M = wave_ballot(kept);
          if (kept) in(u, d, e, ci + lanes_below(M));
          ci += __popcll(M);
        }
        end(u, c, ci);
      }
    };
    walk([](int, int, int, int, int) {}, [](int, int, int, int) {},
         [&](int u, int c, int ci) {
           if (lane == 0) {
             strip_out[u] = c;
             strip_in[u] = ci;
           }
         });
    __syncthreads();
    if (tid < kBinAtoms) {
      int c = 0, ci = 0;
      for (int u = tid * strips; tid < na && u < (tid + 1) * strips; ++u) {
        const int k = strip_out[u], ki = strip_in[u];
        strip_out[u] = c;
        strip_in[u] = ci;
        c += k;
        ci += ki;
      }
      nout[tid] = c;
      nin[tid] = ci;
    }
    __syncthreads();
    place();
    walk(
        [&](int u, int d, int jj, int j, int rank) {
          const int at = start[d] + strip_out[u] + rank;
          L.inc[at] = static_cast<int>(static_cast<uint32_t>(j) |
                                       (FOLD && paired(d, jj, j) ? kIncPaired : 0u));
          if constexpr (Entry<E>::kSlot)
            if (L.inc_bit) L.inc_bit[at] = slot_bit(L, L.row_of[a0 + d], jj);
        },
        [&](int u, int d, int e, int rank) {
          const int at = start[d] + nout[d] + strip_in[u] + rank;
          L.inc[at] = static_cast<int>(row_atom(T[e]) | (1u << 31));
          if constexpr (Entry<E>::kSlot)
            if (L.inc_bit)
              L.inc_bit[at] = slot_bit(L, L.row_of[row_atom(T[e])], Entry<E>::slot(T[e]));
        },
        [](int, int, int) {});
  };
  // with a fold, two marks per entry behind the entries, or in LDS alone, or in memory
  const int room = pool_words - kSortHead, words = static_cast<int>(sizeof(E) / 4);
  const int marks = FOLD ? 2 * ((n + 31) >> 5) : 0;
  uint32_t *head = pool + kSortHead;
  if (n <= room / words && n * words + marks <= room) {
    E *T = reinterpret_cast<E *>(head);
    for (int e = tid; e < n; e += kListThreads) T[e] = tmp[e0 + e];
    __syncthreads();
    sort_entries(T, n);
    sorted_lists(T, head + n * words, true);
  } else {
    sort_entries(tmp + e0, n);
    if (marks <= room)
      sorted_lists(tmp + e0, head, true);
    else
      sorted_lists(tmp + e0, L.claim + e0, false);
  }
}

template <int G, typename T>
__device__ __forceinline__ T group_sum(T v)
{
#pragma unroll
  for (int m = G / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

// Arguments of the two-sided sweeps besides the model block.
struct TwoSided {
  const int2 *span;  // first entry and entries of each atom
  const int *inc;
  int nall;
  int nlocal;
  int nadd;             // rows that take the force add: nall with newton on, else nlocal
  int owned_rows_only;  // export.py:190-192 (n_hops > 1 or a communicating bundle)
  int fdotr;            // newton on: the f.r virial is reported
  const double *x;      // engine positions for the virial
  const int *ghost_off;
  const int *ghost_list;
  int nblk;             // 64-atom partial tiles over nall
  const uint32_t *bits;     // kFromBits: the pack's validity bits
  const uint32_t *inc_bit;  // kFromBits: each entry's place in them
  double cutsq_pack;        // the pack's filter: rsq <= cutsq in float64 (cpp:91)
  float cutsq_lo, cutsq_hi; // cutsq_pack rounded down and up to float
  const int *ghost_flag;    // 1 when a packed edge starts on a ghost row (the pack's flag)
  FusedPack pack;           // a fused pack of this step: tail reset and counts (else unused)
};

// Whether the pack kept an entry's list slot this step, decided from the entry's own geometry
// wherever that decides it, so the sweeps gather no validity word. The pack keeps rsq <= cutsq,
// rsq formed in float64 from the engine's positions without contraction (cpp:84-91); for a
// list-built entry that is the whole per-step filter (the list's other filters are applied when
// the lists are built). Float64 records hold those positions, and r2 is the same sum of the same
// squared differences (negated or not): the same value, so the same decision.
// Float32 records hold them rounded to float. With u = 2^-24, l1 = |dx| + |dy| + |dz| and
// s = l1 + (the 1-norms of both positions), each difference is within
// b_c = u (|d_c| + |x_a,c| + |x_o,c|) / (1 - u) of the float64 one, so
// |sum d^2 - sum D^2| <= sum b_c (2|d_c| + b_c) <= u s (2 l1 + u s) / (1 - u)^2, and r2 is within
// 3u r2 / (1 - 3u) of sum d^2 (float64 rounding adds far less). band = 2u (s (2 l1 + u s) + 4 r2),
// computed in float, exceeds twice that bound and at least 8u r2, which covers the rounding of
// r2 +- band against cutsq rounded down (up) to float. Only an r2 inside the band looks further:
// where the pack ran in this call it forms rsq from the engine's positions as the pack did (the
// sign of the differences does not matter), else it reads the validity bit of the entry's slot. Per
// row, BandRow bounds the band of every entry the model's cutoff lets through (l1 <= sqrt(3)
// rc_model, and the neighbour's 1-norm <= the row's + l1), so most entries are decided by one
// comparison with a row threshold. Lists built from packed edges hold kept slots only (no
// filter).
template <typename S>
struct BandRow {
  S sa;       // the row atom's 1-norm
  S fast_lo;  // r2 <= fast_lo: kept
  S fast_hi;  // r2 > fast_hi: dropped
};

template <typename S>
__device__ __forceinline__ BandRow<S> band_row(const TwoSided &t, const Atom4<S> &xa, S cutsq_model)
{
  BandRow<S> br{};
  if constexpr (sizeof(S) == 4) {
    constexpr float u = 5.9604645e-8f;  // 2^-24
    br.sa = fabsf(xa.x) + fabsf(xa.y) + fabsf(xa.z);
    const float l1m = 1.7320509f * sqrtf(cutsq_model) * 1.0001f;
    const float sm = 2.0f * (br.sa + l1m);
    const float band = 2.0f * u * (sm * (2.0f * l1m + u * sm) + 4.0f * t.cutsq_hi) * 1.0001f;
    br.fast_lo = t.cutsq_lo - 1.25f * band;
    br.fast_hi = t.cutsq_hi + 1.25f * band;
  }
  return br;
}

// How a sweep tells the kept entries, a template parameter of the sweeps: inside the band from
// the positions of this call's pack, or from the validity bits of an earlier one. (Both in one
// kernel held 94 SGPRs in the float32 density sweep: one block per CU, 59 -> 71 us at 256,000 atoms.)
enum Filter { kAllKept = 0, kFromX = 1, kFromBits = 2 };

// The decision inside the band: entry q of atom a's list, with atom o.
template <int FILTER>
__device__ __forceinline__ bool kept_by_pack(const TwoSided &t, int a, int o, int q)
{
  if constexpr (FILTER == kFromX) {
#pragma clang fp contract(off)
    double rsq = 0.0;
#pragma unroll 1  // rare: few registers before few instructions
    for (int c = 0; c < 3; ++c) {
      const double d = t.x[3L * a + c] - t.x[3L * o + c];
      rsq = rsq + d * d;
    }
    return !(rsq > t.cutsq_pack);
  } else {
    const uint32_t at = t.inc_bit[q];
    return ((t.bits[at >> 5] >> (at & 31u)) & 1u) != 0;
  }
}

template <int FILTER, typename S>
__device__ __forceinline__ bool slot_kept(const TwoSided &t, int a, uint32_t v, int q, S r2, S dx,
                                          S dy, S dz, const BandRow<S> &br, const Atom4<S> &xo)
{
  if constexpr (FILTER == kAllKept) return true;
  if constexpr (sizeof(S) == 8) {
    (void)a;
    (void)v;
    (void)q;
    (void)dx;
    (void)dy;
    (void)dz;
    (void)br;
    (void)xo;
    return !(r2 > t.cutsq_pack);
  } else {
    if (r2 <= br.fast_lo) return true;
    if (r2 > br.fast_hi) return false;
    constexpr float u = 5.9604645e-8f;  // 2^-24
    const float l1 = fabsf(dx) + fabsf(dy) + fabsf(dz);
    const float s = l1 + br.sa + (fabsf(xo.x) + fabsf(xo.y) + fabsf(xo.z));
    const float band = 2.0f * u * (s * (2.0f * l1 + u * s) + 4.0f * r2);
    if (r2 + band <= t.cutsq_lo) return true;
    if (r2 - band > t.cutsq_hi) return false;
    return kept_by_pack<FILTER>(t, a, static_cast<int>(v & kIncAtom), q);
  }
}

// The fp64 force sweep's walk over its atom's incident entries k = gl, gl + 16, ... with the
// next entry in flight while the current one is computed. Per entry the sweep issues, in this
// order: the neighbour's record and F', then advance(): the next entry's load goes out after
// this entry's gathers, so waiting for the gathers never waits for it. A skipped entry gathers
// its own row's record instead (cached), so no branch surrounds a load. (The density and LJ
// sweeps measured slower with it, also at eight waves per SIMD: C4 density 404 -> 464 us, C5 LJ
// 181 -> 183 us; they take two entries at a time instead.)
template <int G>
struct IncCursor {
  uint32_t v = 0;
  int b, last;
  __device__ __forceinline__ IncCursor(const TwoSided &t, int b_, int L, int gl) : b(b_), last(b_ + L - 1)
  {
    if (gl < L) load(t, b + gl);
  }
  __device__ __forceinline__ void load(const TwoSided &t, int q_)
  {
    v = static_cast<uint32_t>(t.inc[q_]);
  }
  __device__ __forceinline__ void advance(const TwoSided &t, int k)
  {
    asm volatile("" ::: "memory");  // keep these loads behind the current entry's gathers
    load(t, min(b + k + G, last));
  }
};

// Rows whose energy counts (export.py:183-194).
__device__ __forceinline__ int energy_rows(const TwoSided &t, bool half)
{
  if (half || t.owned_rows_only) return t.nlocal;
  return *t.ghost_flag ? t.nall : t.nlocal;
}

template <typename S>
__device__ __forceinline__ S geometry(const Atom4<S> &xa, const Atom4<S> &xo, S &dx, S &dy, S &dz)
{
#pragma clang fp contract(off)
  dx = xo.x - xa.x;
  dy = xo.y - xa.y;
  dz = xo.z - xa.z;
  return dx * dx + dy * dy + dz * dz;
}

// Density per row (eam.py:298-314); PAIR: also the row's pair energy (the edge-force path, whose
// edge sweep keeps no per-row energy). Without it the window holds the density tables only, so
// two blocks fit on a CU; the force sweep then sums the pair energy.
template <typename S, bool HALF, bool PAIR, int FILTER, int G>
__global__ __launch_bounds__(kRowBlock) LK_EIGHT_WAVES
void k_eam_density_inc(EamArgs<S> m, TwoSided t, S *__restrict__ rho_part, S *__restrict__ epair)
{
  constexpr int kLds = PAIR ? kIncLds : kIncDensLds;
  constexpr int APB = kRowBlock / G;  // atoms per block
  __shared__ LdsEntry<S> lds[kLds];
  // the tail reset's bounds load before the window's loads and its stores go out after them
  const TailBounds tb = tail_bounds(t.pack);
  const Window<S> win = fill_window_issue<S>(lds, kLds, m, PAIR ? m.n_rtab : m.n_el, kRowBlock);
  fused_tail_reset(t.pack, tb, kRowBlock);
  window_ready();
  const int g = threadIdx.x / G, gl = threadIdx.x % G;
  const int nsb = (t.nall + APB - 1) / APB;
  for (int blk = blockIdx.x; blk < nsb; blk += gridDim.x) {
    const int a = blk * APB + g;
    S rho = S(0), ep = S(0);
    if (a < t.nall) {
      const Atom4<S> xa = m.atoms[a];
      const BandRow<S> br = band_row(t, xa, m.cutsq);
      const int za = clamp_species(static_cast<int>(xa.w), m.n_el);
      const int2 span = t.span[a];
      const int b = span.x, L = span.y;
      // Two entries per lane at a time (k and k + G): both entries load together, then both
      // records, so a pair of entries costs two memory round trips; a skipped or missing entry
      // gathers the row's own record.
      auto dens = [&](uint32_t v, int q, const Atom4<S> &xo) {
        const bool in = (v >> 31) != 0;
        if (!HALF && in) return;  // plain: density and pair energy stay on the sender
        S dx, dy, dz;
        const S r2 = geometry(xa, xo, dx, dy, dz);
        if (!(r2 < m.cutsq)) return;
        if (!slot_kept<FILTER>(t, a, v, q, r2, dx, dy, dz, br, xo)) return;
        const S rinv = rsqrt_nr(r2);
        const S rr = r2 * rinv;
        const Locator<S> L2 = locate_mul(rr, m.inv_dr, m.nr);
        const int zo = clamp_species(static_cast<int>(xo.w), m.n_el);
        // the window alone when every active lane's node lies in it (a wave-uniform branch; the
        // density window usually holds the whole table), so the lookup waits on LDS only
        const Coef<S> c = wave_ballot(L2.node < win.lo) == 0 ? rcoef_lds(win, L2.node, zo)
                                                             : rcoef_split(win, m, L2.node, zo);
        rho += cvalue(c, L2.t);
        if (PAIR && !in) {
          const S phi = cvalue(rcoef(win, m, L2.node, m.n_el + pair_row(za, zo)), L2.t) * rinv;
          ep += HALF ? phi : S(0.5) * phi;  // half: the sender carries both halves
        }
      };
      for (int k = gl; k < L; k += 2 * G) {
        const bool two = k + G < L;
        const int q1 = b + k, q2 = b + (two ? k + G : k);
        uint32_t v1 = static_cast<uint32_t>(t.inc[q1]);
        uint32_t v2 = static_cast<uint32_t>(t.inc[q2]);
        // both entries in flight before either is used: without this the compiler moves the
        // first entry's use (and so the wait for it) above the second entry's load (C4 density
        // 271 -> 250 us; the same in the LJ sweep measured slower at C5, 146 -> 150 us)
        asm volatile("" : "+v"(v1), "+v"(v2));
        const bool s1 = !HALF && (v1 >> 31) != 0, s2 = !two || (!HALF && (v2 >> 31) != 0);
        const Atom4<S> x1 = m.atoms[s1 ? a : static_cast<int>(v1 & kIncAtom)];
        const Atom4<S> x2 = m.atoms[s2 ? a : static_cast<int>(v2 & kIncAtom)];
        dens(v1, q1, x1);
        if (two) dens(v2, q2, x2);
      }
    }
    rho = group_sum<G>(rho);
    if (PAIR) ep = group_sum<G>(ep);
    if (gl == 0 && a < t.nall) {
      rho_part[a] = rho;
      if (PAIR) epair[a] = ep;
    }
  }
}

// Embedding: F and F' per row (eam.py:319-321); half folds ghost densities into their owners
// first and hands the owner's F' to its ghost images. Energy partial of the tile into slot 0:
// F, plus the row's pair energy when the density sweep kept it (epair not null).
template <typename S, bool HALF>
__global__ __launch_bounds__(kWave) void k_eam_embed_inc(EamArgs<S> m, TwoSided t,
                                                         const S *__restrict__ rho_part,
                                                         const S *__restrict__ epair)
{
  const int tile = blockIdx.x;
  const int a = tile * kWave + threadIdx.x;
  const int erows = energy_rows(t, HALF);
  double e_row = 0.0;
  if (HALF) {
    if (a < t.nlocal) {
      S rho = rho_part[a];
      if (t.ghost_off)
        for (int q = t.ghost_off[a]; q < t.ghost_off[a + 1]; ++q) rho += rho_part[t.ghost_list[q]];
      S F, Fp;
      embed(m, clamp_species(static_cast<int>(m.atoms[a].w), m.n_el), rho, F, Fp);
      m.fp[a] = Fp;
      m.rho[a] = rho;
      if (t.ghost_off)
        for (int q = t.ghost_off[a]; q < t.ghost_off[a + 1]; ++q) {
          m.fp[t.ghost_list[q]] = Fp;
          m.rho[t.ghost_list[q]] = S(0);
        }
      e_row = static_cast<double>(epair ? epair[a] + F : F);
    }
  } else if (a < t.nall) {
    const S rho = rho_part[a];
    S F, Fp;
    embed(m, clamp_species(static_cast<int>(m.atoms[a].w), m.n_el), rho, F, Fp);
    m.fp[a] = Fp;
    m.rho[a] = rho;
    if (a < erows) e_row = static_cast<double>(epair ? epair[a] + F : F);
  }
  const double esum = wave_sum(e_row);
  if (threadIdx.x == 0 && tile < t.nblk) put_partial(m.partials + 8L * tile, esum);
}

// Per-row f.r virial of the total f after the add, summed over the 64 rows of each partial tile
// in a fixed order by the first wave, which stores the partials. vt is [6][APB], one column per
// atom of the block.
template <bool VIRIAL, int APB>
__device__ __forceinline__ void add_row_force(double *f, const double *x, int a, int nadd,
                                              int nall, int fdotr, double scale, double fx,
                                              double fy, double fz, double (*vt)[APB], int g)
{
  double w[6] = {0, 0, 0, 0, 0, 0};
  if (a < nall) {
    double *fa = f + 3L * a;
    double tx = fa[0], ty = fa[1], tz = fa[2];
    if (a < nadd) {
      tx += scale * fx;
      ty += scale * fy;
      tz += scale * fz;
      fa[0] = tx;
      fa[1] = ty;
      fa[2] = tz;
    }
    if (VIRIAL && fdotr) {
      const double *xa = x + 3L * a;
      w[0] = tx * xa[0];
      w[1] = ty * xa[1];
      w[2] = tz * xa[2];
      w[3] = ty * xa[0];
      w[4] = tz * xa[0];
      w[5] = tz * xa[1];
    }
  }
  if (VIRIAL)
    for (int c = 0; c < 6; ++c) vt[c][g] = w[c];
}

// The partials of the block's tiles, from columns [64 q, 64 q + 64) of vt and et for its tile
// q (the atoms blk * APB + 64 q ...): called by the first wave only, after a barrier. The pair
// energy goes to slot 7; write_energy: et holds the rows' whole energy, into slot 0.
template <bool VIRIAL, int APB>
__device__ __forceinline__ void store_block_partials(double *partials, int blk, int nall,
                                                     double (*vt)[APB], const double *et,
                                                     bool write_energy)
{
  const int lane = threadIdx.x;
#pragma unroll
  for (int q = 0; q < APB / kRowAtoms; ++q) {
    const int tile = blk * (APB / kRowAtoms) + q;
    if (tile * kRowAtoms >= nall) break;  // uniform over the wave
    if (VIRIAL) {
      for (int c = 0; c < 6; ++c) {
        const double v = wave_sum(vt[c][q * kRowAtoms + lane]);
        if (lane == 0) put_partial(partials + 8L * tile + 1 + c, v);
      }
    }
    const double e = wave_sum(et[q * kRowAtoms + lane]);
    if (lane == 0) {
      put_partial(partials + 8L * tile + 7, write_energy ? 0.0 : e);
      if (write_energy) put_partial(partials + 8L * tile, e);
    }
  }
}

// Force sweep (eam.py:336-409 closed form; export.py:197-204 autodiff convention), and the pair
// energy of the counted rows (eam.py:300-307) from the phi it evaluates anyway: on the sender,
// both halves in the half scheme, half per directed edge in the plain one.
template <typename S, bool HALF, bool VIRIAL, int FILTER, int G>
__device__ __forceinline__ void eam_force_inc_rows(const EamArgs<S> &m, const TwoSided &t,
                                                   LdsEntry<S> *lds, int lds_entries)
{
  constexpr int APB = kRowBlock / G;  // atoms per block
  __shared__ double vt[6][APB];
  __shared__ double et[APB];
  // float32: the window holds Hermite rows (more nodes per byte); float64: (f, d) entries
  Window<S> win{};
  HWindow hw{};
  if constexpr (sizeof(S) == 4)
    hw = fill_hwindow(reinterpret_cast<float *>(lds), lds_entries * 4, m.htab, m.htab_w, m.nr,
                      kRowBlock);
  else
    win = fill_window<S>(lds, lds_entries, m, m.n_rtab, kRowBlock);
  const int g = threadIdx.x / G, gl = threadIdx.x % G;
  const int erows = energy_rows(t, HALF);
  const int nsb = (t.nall + APB - 1) / APB;
  for (int blk = blockIdx.x; blk < nsb; blk += gridDim.x) {
    const int a = blk * APB + g;
    S fx = S(0), fy = S(0), fz = S(0), ep = S(0);
    if (a < t.nall) {
      const Atom4<S> xa = m.atoms[a];
      const BandRow<S> br = band_row(t, xa, m.cutsq);
      const int za = clamp_species(static_cast<int>(xa.w), m.n_el);
      const S fpa = m.fp[a];
      const int2 span = t.span[a];
      const int b = span.x, L = span.y;
      // The gathers of an entry: its neighbour's record and F' (the row's own when the entry
      // is skipped, so no branch surrounds a load).
      struct Gathered {
        uint32_t v;
        int q;  // the entry's index
        bool skip;
        Atom4<S> xo;
        S fpo;
      };
      auto gather = [&](uint32_t v, int q, bool present) -> Gathered {
        Gathered e;
        e.v = v;
        e.q = q;
        const bool in = (v >> 31) != 0;
        const int o = static_cast<int>(v & kIncAtom);
        // plain: an uncounted sender gives no gradient; a folded pair counts each counted end
        const bool paired = !HALF && (v & kIncPaired) != 0;
        const bool ca = a < erows, co = o < erows;
        e.skip = !present || (!HALF && (paired ? !(ca || co) : !(in ? co : ca)));
        e.xo = m.atoms[e.skip ? a : o];
        e.fpo = m.fp[(HALF || in || paired) && !e.skip ? o : a];
        return e;
      };
      auto edge = [&](const Gathered &e) {
        if (e.skip) return;
        const uint32_t v = e.v;
        const Atom4<S> &xo = e.xo;
        const S fpo = e.fpo;
        const bool in = (v >> 31) != 0;
        const int o = static_cast<int>(v & kIncAtom);
        const bool paired = !HALF && (v & kIncPaired) != 0;
        const bool ca = a < erows, co = o < erows;
        S dx, dy, dz;
        const S r2 = geometry(xa, xo, dx, dy, dz);
        if (!(r2 < m.cutsq)) return;
        if (!slot_kept<FILTER>(t, a, v, e.q, r2, dx, dy, dz, br, xo)) return;
        const S rinv = rsqrt_nr(r2);
        const S rr = r2 * rinv;
        const Locator<S> L2 = locate_mul(rr, m.inv_dr, m.nr);
        const int zo = clamp_species(static_cast<int>(xo.w), m.n_el);
        // Past the table the non-extrapolated lookups saturate: slope 0 (eam.py:150).
        const bool inside = !(L2.t_raw > S(1));
        const int zs = in ? zo : za, zr = in ? za : zo;
        const S fps = in ? fpo : fpa;
        // Slopes in t of the density tables zr and t3, and the pair table's value and slope:
        // from the LDS window alone when every active lane's node lies in it (a wave-uniform
        // branch), else from the tables in memory (or the window, lane by lane), whose loads'
        // waits also wait for the entries already in flight for the next round.
        const int tp = m.n_el + pair_row(za, zo);
        const int t3 = HALF ? zs : za;
        const bool three = HALF || paired;
        S sr, z2, z2s, s3 = S(0);
        if constexpr (sizeof(S) == 4) {
          if (wave_ballot(L2.node < hw.lo) == 0) {
            const HermBasisF hb = herm_basis_f(L2.t);
            sr = hslope_density(hw, L2.node, zr, hb);
            hpair(hw, L2.node, 2 * m.n_el + 3 * (tp - m.n_el), hb, z2, z2s);
            if (three) s3 = hslope_density(hw, L2.node, t3, hb);
          } else {
            const Coef<S> cp = rcoef_global(m, L2.node, tp);
            sr = cslope_t(rcoef_global(m, L2.node, zr), L2.t);
            z2 = cvalue(cp, L2.t);
            z2s = cslope_t(cp, L2.t);
            if (three) s3 = cslope_t(rcoef_global(m, L2.node, t3), L2.t);
          }
        } else {
          Coef<S> cr, cp, c3;
          if (wave_ballot(L2.node < win.lo) == 0) {
            cr = rcoef_lds(win, L2.node, zr);
            cp = rcoef_lds(win, L2.node, tp);
            if (three) c3 = rcoef_lds(win, L2.node, t3);
          } else {
            cr = rcoef_split(win, m, L2.node, zr);
            cp = rcoef_split(win, m, L2.node, tp);
            if (three) c3 = rcoef_split(win, m, L2.node, t3);
          }
          sr = cslope_t(cr, L2.t);
          z2 = cvalue(cp, L2.t);
          z2s = cslope_t(cp, L2.t);
          if (three) s3 = cslope_t(c3, L2.t);
        }
        const S rho_r_p = inside ? sr * m.inv_dr : S(0);
        const S phi = z2 * rinv;
        if (!in) ep += HALF ? phi : S(0.5) * phi;
        const S z2p = inside ? z2s * m.inv_dr : S(0);
        const S phip = (z2p - phi) * rinv;
        S coef;
        if (HALF) {
          const S fpr = in ? fpa : fpo;
          const S rho_s_p = inside ? s3 * m.inv_dr : S(0);
          coef = (fps * rho_r_p + fpr * rho_s_p + phip) * rinv;
        } else if (paired) {
          // both directed edges: a -> o on a's counted row, o -> a on o's
          const S rho_a_p = inside ? s3 * m.inv_dr : S(0);
          const S ga = ca ? fpa * rho_r_p + S(0.5) * phip : S(0);
          const S go = co ? fpo * rho_a_p + S(0.5) * phip : S(0);
          coef = (ga + go) * rinv;
        } else {
          coef = (fps * rho_r_p + S(0.5) * phip) * rinv;
        }
        // sender += coef d, receiver -= coef d with d = x_r - x_s: either way coef (x_o - x_a)
        fx += coef * dx;
        fy += coef * dy;
        fz += coef * dz;
      };
      // float32: entries k and k + G of this lane at a time: both gathers go out together,
      // then the next pair's entries (clamped to the list's last entry, so every load is
      // unconditional and waiting for the gathers never waits for them), then both edges are
      // computed (C4 force sweep 750 -> 739 us). float64 takes one entry at a time with the next
      // in flight (two at a time measured 2% slower there, at 97 VGPRs and four waves per SIMD).
      if constexpr (sizeof(S) == 8) {
        IncCursor<G> cur(t, b, L, gl);
        for (int k = gl; k < L; k += G) {
          const Gathered e = gather(cur.v, 0, true);  // float64 needs no index
          cur.advance(t, k);
          edge(e);
        }
      } else if (gl < L) {
        const int last = b + L - 1;
        int q1 = b + gl, q2 = min(b + gl + G, last);
        uint32_t v1 = static_cast<uint32_t>(t.inc[q1]);
        uint32_t v2 = static_cast<uint32_t>(t.inc[q2]);
        for (int k = gl; k < L; k += 2 * G) {
          const Gathered e1 = gather(v1, q1, true);
          const Gathered e2 = gather(v2, q2, k + G < L);
          asm volatile("" ::: "memory");  // keep the next entries' loads behind the gathers
          q1 = min(b + k + 2 * G, last);
          q2 = min(b + k + 3 * G, last);
          v1 = static_cast<uint32_t>(t.inc[q1]);
          v2 = static_cast<uint32_t>(t.inc[q2]);
          edge(e1);
          edge(e2);
        }
      }
    }
    fx = group_sum<G>(fx);
    fy = group_sum<G>(fy);
    fz = group_sum<G>(fz);
    ep = group_sum<G>(ep);
    if (gl == 0) {
      add_row_force<VIRIAL, APB>(m.f, t.x, a, t.nadd, t.nall, t.fdotr, m.scale,
                                 static_cast<double>(fx), static_cast<double>(fy),
                                 static_cast<double>(fz), vt, g);
      et[g] = a < erows ? static_cast<double>(ep) : 0.0;
    }
    __syncthreads();
    if (threadIdx.x < kWave)
      store_block_partials<VIRIAL, APB>(m.partials, blk, t.nall, vt, et, false);
    __syncthreads();
  }
  finalize_last_block(m.partials, t.nblk, m.scale, 1.0, m.flags, m.result, m.done,
                      reinterpret_cast<double *>(lds), t.pack, m.mirror);
}

// One block per CU: the 120 KB table window (all of a 2000-node r-grid of two elements).
template <typename S, bool HALF, bool VIRIAL, int FILTER, int G>
__global__ __launch_bounds__(kRowBlock) void k_eam_force_inc(EamArgs<S> m, TwoSided t)
{
  __shared__ LdsEntry<S> lds[kIncLds];
  eam_force_inc_rows<S, HALF, VIRIAL, FILTER, G>(m, t, lds, kIncLds);
}

// Two blocks per CU (eight waves per SIMD) with the 64 KB window: twice the gathers in flight for
// more lookups below the window (L2-resident). The fp32 sweep fits 64 VGPRs without spills
// (C4 force sweep 814 -> 748 us); the fp64 one would spill.
template <typename S, bool HALF, bool VIRIAL, int FILTER, int G>
__global__ __launch_bounds__(kRowBlock) __attribute__((amdgpu_waves_per_eu(8))) LK_EIGHT_WAVES
void k_eam_force_inc_2b(EamArgs<S> m, TwoSided t)
{
  __shared__ LdsEntry<S> lds[kIncDensLds];
  eam_force_inc_rows<S, HALF, VIRIAL, FILTER, G>(m, t, lds, kIncDensLds);
}

template <typename S>
struct LjModel {
  const Atom4<S> *atoms;
  S cutsq, sigsq, four_eps, edge_scale;
  double scale;
  double *f;
  double *partials;
  StepResult *result;
  int *done;
  int flags;
  StepResult *mirror;
};

// LJ 12-6 plain (examples/export_model.py:16-50): e per edge on the sender row, g = 2 de/d(r^2) d
// (times edge_energy_scale) to the sender and minus it to the receiver.
template <typename S, bool VIRIAL, int FILTER, int G>
__global__ __launch_bounds__(kRowBlock) __attribute__((amdgpu_waves_per_eu(8))) LK_EIGHT_WAVES
void k_lj_inc(LjModel<S> m, TwoSided t)
{
  constexpr int APB = kRowBlock / G;  // atoms per block
  __shared__ double vt[6][APB];
  __shared__ double et[APB];
  __shared__ double scratch[7 * kRowBlock];
  fused_tail_reset(t.pack, tail_bounds(t.pack), kRowBlock);
  const int g = threadIdx.x / G, gl = threadIdx.x % G;
  const int erows = energy_rows(t, false);
  const S tiny = static_cast<S>(1.0e-12);
  const int nsb = (t.nall + APB - 1) / APB;
  for (int blk = blockIdx.x; blk < nsb; blk += gridDim.x) {
    const int a = blk * APB + g;
    S en = S(0), fx = S(0), fy = S(0), fz = S(0);
    if (a < t.nall) {
      const Atom4<S> xa = m.atoms[a];
      const BandRow<S> br = band_row(t, xa, m.cutsq);
      const int2 span = t.span[a];
      const int b = span.x, L = span.y;
      // counted ends of an entry: its sender's row, or both rows of a folded pair (the pair
      // force on a is the same from either directed edge)
      auto ends = [&](uint32_t v) -> int {
        const bool in = (v >> 31) != 0;
        const int co = static_cast<int>(v & kIncAtom) < erows ? 1 : 0;
        return (in ? 0 : (a < erows ? 1 : 0)) + ((in || (v & kIncPaired)) ? co : 0);
      };
      auto pair = [&](uint32_t v, int q, int w, const Atom4<S> &xo) {
        if (w == 0) return;
        S dx, dy, dz;
        const S r2 = geometry(xa, xo, dx, dy, dz);
        if (!(r2 > tiny && r2 < m.cutsq)) return;  // export_model.py:22
        if (!slot_kept<FILTER>(t, a, v, q, r2, dx, dy, dz, br, xo)) return;
        const S inv_r2 = m.sigsq / r2;
        const S inv_r6 = inv_r2 * inv_r2 * inv_r2;
        if (!(v >> 31)) en += m.edge_scale * (m.four_eps * (inv_r6 * inv_r6 - inv_r6));
        const S dedr2 = -m.four_eps * (S(6) * inv_r6 * inv_r6 - S(3) * inv_r6) / r2;
        const S coef = static_cast<S>(w) * (m.edge_scale * S(2) * dedr2);
        fx += coef * dx;
        fy += coef * dy;
        fz += coef * dz;
      };
      // Two entries per lane at a time (k and k + G), as in the density sweep: both entries,
      // then both records (an uncounted or missing entry gathers the row's own record).
      for (int k = gl; k < L; k += 2 * G) {
        const bool two = k + G < L;
        const int q1 = b + k, q2 = b + (two ? k + G : k);
        const uint32_t v1 = static_cast<uint32_t>(t.inc[q1]);
        const uint32_t v2 = static_cast<uint32_t>(t.inc[q2]);
        const int w1 = ends(v1), w2 = two ? ends(v2) : 0;
        const Atom4<S> x1 = m.atoms[w1 ? static_cast<int>(v1 & kIncAtom) : a];
        const Atom4<S> x2 = m.atoms[w2 ? static_cast<int>(v2 & kIncAtom) : a];
        pair(v1, q1, w1, x1);
        pair(v2, q2, w2, x2);
      }
    }
    en = group_sum<G>(en);
    fx = group_sum<G>(fx);
    fy = group_sum<G>(fy);
    fz = group_sum<G>(fz);
    if (gl == 0) {
      et[g] = a < erows ? static_cast<double>(en) : 0.0;
      add_row_force<VIRIAL, APB>(m.f, t.x, a, t.nadd, t.nall, t.fdotr, m.scale,
                                 static_cast<double>(fx), static_cast<double>(fy),
                                 static_cast<double>(fz), vt, g);
    }
    __syncthreads();
    if (threadIdx.x < kWave)
      store_block_partials<VIRIAL, APB>(m.partials, blk, t.nall, vt, et, true);
    __syncthreads();
  }
  finalize_last_block(m.partials, t.nblk, m.scale, 1.0, m.flags, m.result, m.done, scratch,
                      t.pack, m.mirror);
}

static int grid_for(const Handle &h, long work, int per_block, int blocks_per_cu)
{
  long want = (work + per_block - 1) / per_block;
  const long cap = static_cast<long>(blocks_per_cu) * (h.num_cus > 0 ? h.num_cus : 256);
  if (want > cap) want = cap;
  if (want < 1) want = 1;
  return static_cast<int>(want);
}

static hipError_t build_incidence(Handle &h, hipStream_t s, int nall)
{
  IncArgs ia;
  ia.senders = h.d_senders;
  ia.receivers = h.d_receivers;
  ia.mask = h.d_mask;
  ia.result = h.d_result;
  ia.max_edges = h.contract.max_edges;
  ia.nrows = h.contract.max_atoms;
  ia.deg = h.d_deg;
  ia.loc = h.d_inc_loc;
  ia.part = h.d_inc_part;
  ia.tmp = h.d_inc_tmp;
  ia.inc = h.d_inc;
  ia.span = h.d_inc_span;
  const int egrid = grid_for(h, h.contract.max_edges, 256, 16);
  {
    StageTimer timer(h, s, "inc_count");
    // the counts start from zero whatever the previous build left (a list-built one keeps the
    // rows' slot counts there)
    const long n = static_cast<long>(h.contract.max_atoms) + 1;
    hipLaunchKernelGGL(k_clear_int, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s,
                       h.d_deg, n);
    hipLaunchKernelGGL(k_inc_count, dim3(egrid), dim3(256), 0, s, ia);
  }
  {
    StageTimer timer(h, s, "inc_scan");
    const int n = h.contract.max_atoms + 1;
    const int chunks = (n + kScanChunk - 1) / kScanChunk;
    hipLaunchKernelGGL(k_scan_chunks, dim3(chunks), dim3(kScanThreads), 0, s, h.d_deg, n,
                       h.d_inc_loc, h.d_inc_part);
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(kScanThreads), 0, s, h.d_inc_part, chunks);
  }
  {
    StageTimer timer(h, s, "inc_fill");
    hipLaunchKernelGGL(k_inc_fill, dim3(egrid), dim3(256), 0, s, ia);
  }
  if (nall > 0) {
    StageTimer timer(h, s, "inc_sort");
    hipLaunchKernelGGL(k_inc_sort, dim3((nall + 3) / 4), dim3(256), 0, s, ia, nall);
  }
  return hipGetLastError();
}

static hipError_t build_incidence_from_list(Handle &h, hipStream_t s, bool fold, bool bits)
{
  ListArgs L{};
  L.ilist = h.list_ilist;
  L.numneigh = h.list_numneigh;
  L.neighbors = h.list_neighbors;
  L.stride = h.list_stride;
  L.rows = h.list_rows;
  L.maxneighs = h.list_maxneighs;
  L.max_atoms = h.contract.max_atoms;
  L.half_filter = h.list_half_filter;
  L.out_n = h.d_deg;
  L.span = h.d_inc_span;
  L.inc = h.d_inc;
  L.fold = fold ? 1 : 0;
  const int atoms = L.max_atoms;
  L.slots = bits || atoms > kBinAtoms32 ? 1 : 0;
  L.layout = bin_layout(L.maxneighs, fold, L.slots != 0);
  L.inc_bit = bits ? h.d_inc_bit : nullptr;
  L.row_of = bits ? h.d_row_of : nullptr;
  L.bit_pitch = h.contract.max_atoms;
  Bins B;
  B.cap = (atoms + (1 << L.layout.bin_log) - 1) >> L.layout.bin_log;
  B.next = h.d_bins;
  B.out = B.next + B.cap;
  B.off = B.out + B.cap;
  B.loff = B.off + B.cap + 1;
  const bool measure = L.layout.bin_log < kBinMeasureLog;
  L.longest = measure ? B.loff + B.cap : nullptr;
  const size_t lds = measure ? kBinPool
                             : static_cast<size_t>(4 * (L.layout.per_atom + L.layout.pitch) +
                                                   (L.slots ? 2 * L.layout.per_atom : 0))
                                   << L.layout.bin_log;
  // Waves per 64-row tile of the counting blocks: many where the tiles are few, so that the blocks
  // reach the CUs; two past eight tiles per CU, where a block's eight tiles share the bins they
  // name and so its LDS counts (fewer claims in memory). Count and scatter together in us by waves
  // 2, 4, 8, 16, chosen starred; two at every size before:
  //   16 tiles (1,024 rows, plain)  65, 38, 26, 20*    1,024 tiles (65,536, plain) 81, 57*, 62, 88
  //   500 tiles (32,000, plain)     76, 51, 45*, 53    2,048 tiles (131,072, half) 74, 56*, 75, 98
  //                                                    4,000 tiles (256,000, half) 105*, 117, 134, 163
  // The line between sixteen and eight waves lies where they meet: both stages by events, 8 and 16,
  //   64 tiles (4,096, plain)  42.6, 41.7*    192 tiles (12,288, half)  41.6*, 40.9
  //   96 tiles (6,144, plain)  45.7*, 45.7    256 tiles (16,384, plain) 50.7*, 53.8
  //   128 tiles (8,192, half)  40.2*, 38.8    400 tiles (25,600, half)  45.8*, 47.6
  const int cus = h.num_cus > 0 ? h.num_cus : 256, tiles = (L.rows + kWave - 1) / kWave;
  auto bins = [&](auto scatter, auto *tmp) {
    using E = std::remove_pointer_t<decltype(tmp)>;
    auto launch = [&](auto waves) {
      constexpr int W = decltype(waves)::value, kTiles = kBinWaves / W;
      hipLaunchKernelGGL((k_inc_bins<decltype(scatter)::value, E, W>),
                         dim3((tiles + kTiles - 1) / kTiles), dim3(kBinWaves * kWave), 0, s, L, B,
                         tmp);
    };
    if (4 * tiles <= cus)
      launch(std::integral_constant<int, 16>{});
    else if (tiles <= 2 * cus)
      launch(std::integral_constant<int, 8>{});
    else if (tiles <= 8 * cus)
      launch(std::integral_constant<int, 4>{});
    else
      launch(std::integral_constant<int, 2>{});
  };
  {
    StageTimer timer(h, s, "inc_count");
    if (measure) {
      hipLaunchKernelGGL(k_clear_int, dim3(1), dim3(256), 0, s, L.longest, 1L);
      if (L.rows > 0)
        hipLaunchKernelGGL(k_inc_longest, dim3((L.rows + 255) / 256), dim3(256), 0, s, L);
    }
    hipLaunchKernelGGL(k_inc_clear, dim3((atoms + 255) / 256), dim3(256), 0, s, L, B);
    if (L.rows > 0)
      bins(std::false_type{}, static_cast<uint32_t *>(nullptr));
    hipLaunchKernelGGL(k_inc_bin_scan, dim3(1), dim3(kScanThreads), 0, s, L, B);
  }
  auto finish = [&](auto *tmp) {
    using E = std::remove_pointer_t<decltype(tmp)>;
    if (L.rows > 0) {
      StageTimer timer(h, s, "inc_fill");
      bins(std::true_type{}, tmp);
    }
    StageTimer timer(h, s, "inc_place");
    if (fold)
      hipLaunchKernelGGL((k_inc_lists<E, true>), dim3(B.cap), dim3(kListThreads), lds, s, L, B,
                         tmp, static_cast<int>(lds / 4));
    else
      hipLaunchKernelGGL((k_inc_lists<E, false>), dim3(B.cap), dim3(kListThreads), lds, s, L, B,
                         tmp, static_cast<int>(lds / 4));
  };
  // d_inc_tmp holds an entry and a word of marks per list slot (ensure_incidence)
  L.claim = h.d_inc_tmp + static_cast<long>(L.rows) * L.maxneighs * (L.slots ? 2 : 1);
  if (!L.slots)
    finish(h.d_inc_tmp);
  else
    finish(reinterpret_cast<uint64_t *>(h.d_inc_tmp));
  return hipGetLastError();
}

static Handle::IncKey list_key(const Handle &h, bool fold)
{
  Handle::IncKey key;
  key.epoch = h.list_epoch;
  key.ilist = h.list_ilist;
  key.neighbors = h.list_neighbors;
  key.stride = h.list_stride;
  key.rows = h.list_rows;
  key.maxneighs = h.list_maxneighs;
  key.half_filter = h.list_half_filter;
  key.fold = fold ? 1 : 0;
  return key;
}

// The incidence lists of the neighbour list, built once per list: by the engine's epoch (or every
// step when it gives none) and the list's shape; `bits`: with the entries' validity bit addresses,
// for sweeps that read them. A build that failed leaves no lists to reuse.
static hipError_t lists_of_list(Handle &h, hipStream_t s, bool fold, bool bits)
{
  const Handle::IncKey key = list_key(h, fold);
  if (h.list_epoch >= 0 && key == h.inc_key && (!bits || h.inc_bits)) return hipSuccess;
  h.inc_key = Handle::IncKey{};
  const hipError_t e = build_incidence_from_list(h, s, fold, bits);
  if (e == hipSuccess) {
    h.inc_key = key;
    h.inc_bits = bits;
  }
  return e;
}

// A pack called on its own over the list that incidence lists without bit addresses stand for (a fused
// step built them): its sweeps will want the addresses, and the list is there to read now.
hipError_t launch_list_bits(Handle &h, hipStream_t s)
{
  const bool fold = h.inc_key.fold != 0;
  if (h.list_epoch < 0 || h.inc_bits || !h.d_inc_bit || !(list_key(h, fold) == h.inc_key))
    return hipSuccess;
  return lists_of_list(h, s, fold, true);
}

// The incidence lists of the packed edges, built every step.
static hipError_t lists_of_edges(Handle &h, hipStream_t s, int nall)
{
  h.inc_key = Handle::IncKey{};  // no list's any more
  return build_incidence(h, s, nall);
}

// The sweeps' filter: none for lists built from packed edges or from a matrix, whose slots the
// model masks itself.
static int sweep_filter(const Handle &h, bool from_list, const FusedPack &pack)
{
  if (!from_list || !h.list_bits_filter) return kAllKept;
  return pack.state ? kFromX : kFromBits;
}

// Whether sweeps over the list's entries after this pack read validity bits (float64 ones decide every
// entry from its own r2).
static bool reads_bits(const Handle &h, const FusedPack &pack)
{
  return h.d_inc_bit && sweep_filter(h, true, pack) == kFromBits;
}

// Calls f with `filter` as a constant. Float64 sweeps decide every entry from its own r2, so one
// filtering form serves both.
template <typename S, class F>
static void with_filter(int filter, F &&f)
{
  if (filter == kAllKept)
    f(std::integral_constant<int, kAllKept>{});
  else if (sizeof(S) == 8 || filter == kFromX)
    f(std::integral_constant<int, kFromX>{});
  else if constexpr (sizeof(S) == 4)
    f(std::integral_constant<int, kFromBits>{});
}

static TwoSided two_sided_args(Handle &h, int nlocal, int nghost, const double *x)
{
  TwoSided t;
  t.span = h.d_inc_span;
  t.inc = h.d_inc;
  t.nall = nlocal + nghost;
  t.nlocal = nlocal;
  t.nadd = h.contract.newton_pair ? t.nall : nlocal;
  t.owned_rows_only = (h.contract.n_hops > 1 || h.contract.comm) ? 1 : 0;
  t.fdotr = h.contract.newton_pair ? 1 : 0;
  t.x = x;
  t.ghost_off = nghost > 0 ? h.d_ghost_off : nullptr;
  t.ghost_list = h.d_ghost_list;
  t.nblk = (t.nall + kRowAtoms - 1) / kRowAtoms;
  t.bits = h.d_bits;
  t.inc_bit = h.d_inc_bit;
  t.cutsq_pack = h.contract.cutoff * h.contract.cutoff;
  t.cutsq_lo = static_cast<float>(t.cutsq_pack);
  t.cutsq_hi = t.cutsq_lo;
  if (static_cast<double>(t.cutsq_lo) > t.cutsq_pack)
    t.cutsq_lo = std::nextafter(t.cutsq_lo, -std::numeric_limits<float>::infinity());
  if (static_cast<double>(t.cutsq_hi) < t.cutsq_pack)
    t.cutsq_hi = std::nextafter(t.cutsq_hi, std::numeric_limits<float>::infinity());
  t.ghost_flag = &h.d_result->ghost_sender;
  t.pack = FusedPack{};
  return t;
}

// A fused pack (`pack.state` set) leaves the demand count and the ghost-sender flag in its
// state words and the previous pack's tail to reset; the sweeps take both from there.
static void use_pack(TwoSided &t, const FusedPack &pack)
{
  if (!pack.state) return;
  t.pack = pack;
  t.ghost_flag = pack.state + kGhostFlag;
}

template <typename S, bool HALF>
static hipError_t eam_two_sided(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                                double scale, double *f, const double *x, bool from_list,
                                const FusedPack &pack, int phase)
{
  EamArgs<S> m = eam_args<S>(h, nlocal, scale, f);
  TwoSided t = two_sided_args(h, nlocal, nghost, x);
  use_pack(t, pack);
  const int filter = sweep_filter(h, from_list, pack);
  m.flags = flags;
  // Split passes exchange the handle's rho rows: the density sweep writes its partials there and
  // the embedding reads them back completed (every row, ghosts included, holding its atom's
  // whole density), so no ghost map folds or copies; only owned rows count their energy.
  const bool split = phase != kPhaseAll;
  S *rho_part = static_cast<S *>(split ? h.d_rho : h.d_rho_part);
  if (split) {
    t.ghost_off = nullptr;
    t.owned_rows_only = 1;
  }
  constexpr int G = kLanesPerAtom<S>;
  const int nsb = t.nall > 0 ? (t.nall + kRowBlock / G - 1) / (kRowBlock / G) : 1;
  const int grid = grid_for(h, nsb, 1, 1);
  if (t.nblk > 0 && phase != kPhaseForce) {
    StageTimer timer(h, s, "eam_density");
    with_filter<S>(filter, [&](auto F) {
      hipLaunchKernelGGL((k_eam_density_inc<S, HALF, false, F.value, G>),
                         dim3(grid_for(h, nsb, 1, 2)), dim3(kRowBlock), 0, s, m, t, rho_part,
                         static_cast<S *>(nullptr));
    });
  }
  if (phase == kPhaseDensity) return hipGetLastError();
  if (t.nblk > 0) {
    StageTimer timer(h, s, "eam_embed");
    if (split)  // every row from its completed density
      hipLaunchKernelGGL((k_eam_embed_inc<S, false>), dim3(t.nblk), dim3(kWave), 0, s, m, t,
                         static_cast<const S *>(rho_part), static_cast<const S *>(nullptr));
    else
      hipLaunchKernelGGL((k_eam_embed_inc<S, HALF>), dim3(t.nblk), dim3(kWave), 0, s, m, t,
                         static_cast<const S *>(rho_part), static_cast<const S *>(nullptr));
  }
  // one launch even with no rows: its last block writes the step result
  StageTimer timer(h, s, "eam_force");
  with_filter<S>(filter, [&](auto F) {
    auto launch = [&](auto virial) {
      if constexpr (kForceTwoBlocks<S>)
        hipLaunchKernelGGL((k_eam_force_inc_2b<S, HALF, virial.value, F.value, G>),
                           dim3(grid_for(h, nsb, 1, 2)), dim3(kRowBlock), 0, s, m, t);
      else
        hipLaunchKernelGGL((k_eam_force_inc<S, HALF, virial.value, F.value, G>), dim3(grid),
                           dim3(kRowBlock), 0, s, m, t);
    };
    if (flags & LK_VIRIAL)
      launch(std::true_type{});
    else
      launch(std::false_type{});
  });
  return hipGetLastError();
}

template <typename S>
static hipError_t lj_two_sided(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                               double scale, double *f, const double *x, bool from_list,
                               const FusedPack &pack)
{
  LjModel<S> m;
  m.atoms = static_cast<const Atom4<S> *>(h.d_atoms);
  m.cutsq = static_cast<S>(h.lj.cutoff * h.lj.cutoff);
  m.sigsq = static_cast<S>(h.lj.sigma * h.lj.sigma);
  m.four_eps = static_cast<S>(4.0 * h.lj.epsilon);
  m.edge_scale = static_cast<S>(h.lj.edge_energy_scale);
  m.scale = scale;
  m.f = f;
  m.partials = h.d_partials;
  m.result = h.d_result;
  m.done = h.d_done;
  m.flags = flags;
  m.mirror = h.d_host_result;
  TwoSided t = two_sided_args(h, nlocal, nghost, x);
  use_pack(t, pack);
  const int filter = sweep_filter(h, from_list, pack);
  constexpr int G = kLanesPerAtom<S>;
  const int nsb = t.nall > 0 ? (t.nall + kRowBlock / G - 1) / (kRowBlock / G) : 1;
  const int grid = grid_for(h, nsb, 1, 2);
  StageTimer timer(h, s, "lj_rows");
  with_filter<S>(filter, [&](auto F) {
    if (flags & LK_VIRIAL)
      hipLaunchKernelGGL((k_lj_inc<S, true, F.value, G>), dim3(grid), dim3(kRowBlock), 0, s, m, t);
    else
      hipLaunchKernelGGL((k_lj_inc<S, false, F.value, G>), dim3(grid), dim3(kRowBlock), 0, s, m, t);
  });
  return hipGetLastError();
}

// ----------------------------------------------------------------------------------------------
// Edge-force output (force_output = edge-force). The model's output is the force on each packed
// edge's sender, [max_edges][3] at the contract precision: make_setfl_edge_force for the
// communicating half-edge EAM export (eam.py:336-409: the half scheme's density and F' above,
// then psip / r * r_ij per edge) and make_lj_edge_force (examples/export_model.py:52-74:
// dU/d(r_ij)). The pair style then adds them into f (AddEdgeForcesFunctor,
// cpp/pair_jax_kokkos.cpp:194-225, 959-970): f(s) += scale * F_e over [0, count), and with newton
// pair f(r) -= scale * F_e, with atomic adds as the reference's functor does. The virial is f.r
// of the total f over nall rows after the add (cpp:1092-1100). Slots from the count up to the
// previous step's count are cleared, so the buffer past the live edges holds zeros.
// ----------------------------------------------------------------------------------------------
template <typename S>
struct EdgeOut {
  const int *senders;
  const int *receivers;
  const unsigned char *mask;
  const StepResult *count;  // the pack's demand count of this step
  int max_edges;
  const int *state;         // pack state: kEdgeForceLive slots hold the previous compute's forces
  S *edge_f;
  double *f;
  double scale;
  double *partials;
  int ntiles;               // partial tiles the finalize reduces
  int slot0_from;           // first tile whose slot 0 (row energy) this launch clears
  int block_energy;         // each block stores its edge energy in its own slot 7
  int nlocal;
  int nall;
};

template <typename S>
__device__ __forceinline__ long live_edges(const EdgeOut<S> &o)
{
  const long c = o.count->edge_count;
  return c < o.max_edges ? c : o.max_edges;
}

template <typename S, bool NEWTON>
__device__ __forceinline__ void store_edge_force(const EdgeOut<S> &o, long e, int snd, int rcv,
                                                 S gx, S gy, S gz, bool live)
{
  S *q = o.edge_f + 3 * e;
  q[0] = gx;
  q[1] = gy;
  q[2] = gz;
  if (!live) return;
  const double vx = o.scale * static_cast<double>(gx);
  const double vy = o.scale * static_cast<double>(gy);
  const double vz = o.scale * static_cast<double>(gz);
  atomicAdd(o.f + 3L * snd + 0, vx);
  atomicAdd(o.f + 3L * snd + 1, vy);
  atomicAdd(o.f + 3L * snd + 2, vz);
  if (NEWTON) {
    atomicAdd(o.f + 3L * rcv + 0, -vx);
    atomicAdd(o.f + 3L * rcv + 1, -vy);
    atomicAdd(o.f + 3L * rcv + 2, -vz);
  }
}

// Clears the slots of the previous step past this step's count and the partial slots this
// launch owns (7 everywhere, 0 from slot0_from on).
template <typename S>
__device__ __forceinline__ void edge_tail_and_slots(const EdgeOut<S> &o, long ne)
{
  const long stride = static_cast<long>(gridDim.x) * blockDim.x;
  const long tid = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  const long reset_end = o.state[kEdgeForceLive];
  for (long e = ne + tid; e < reset_end; e += stride) {
    S *q = o.edge_f + 3 * e;
    q[0] = S(0);
    q[1] = S(0);
    q[2] = S(0);
  }
  for (long t = tid; t < o.ntiles; t += stride) {
    if (!o.block_energy || t >= gridDim.x) put_partial(o.partials + 8L * t + 7, 0.0);
    if (t >= o.slot0_from) put_partial(o.partials + 8L * t, 0.0);
  }
}

template <typename S, bool NEWTON>
__global__ __launch_bounds__(kRowBlock) void k_eam_edge_force(EamArgs<S> m, EdgeOut<S> o)
{
  __shared__ LdsEntry<S> lds[kIncLds];
  const Window<S> win = fill_window<S>(lds, kIncLds, m, m.n_rtab, kRowBlock);
  const long ne = live_edges(o);
  const long stride = static_cast<long>(gridDim.x) * blockDim.x;
  for (long e = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < ne; e += stride) {
    const int snd = o.senders[e], rcv = o.receivers[e];
    S gx = S(0), gy = S(0), gz = S(0);
    bool live = false;
    if (o.mask[e] && snd < o.nall && rcv < o.nall) {
      const Atom4<S> xs = m.atoms[snd], xr = m.atoms[rcv];
      S dx, dy, dz;
      const S r2 = geometry(xs, xr, dx, dy, dz);  // d = x_r - x_s
      if (r2 < m.cutsq) {
        const S rinv = rsqrt_nr(r2);
        const S rr = r2 * rinv;
        const Locator<S> L = locate_mul(rr, m.inv_dr, m.nr);
        const int zs = clamp_species(static_cast<int>(xs.w), m.n_el);
        const int zr = clamp_species(static_cast<int>(xr.w), m.n_el);
        // Past the table the non-extrapolated lookups saturate: slope 0 (eam.py:150).
        const bool inside = !(L.t_raw > S(1));
        const S rhojp = inside ? cslope_t(rcoef(win, m, L.node, zr), L.t) * m.inv_dr : S(0);
        const S rhoip = inside ? cslope_t(rcoef(win, m, L.node, zs), L.t) * m.inv_dr : S(0);
        const Coef<S> cp = rcoef(win, m, L.node, m.n_el + pair_row(zs, zr));
        const S phi = cvalue(cp, L.t) * rinv;
        const S z2p = inside ? cslope_t(cp, L.t) * m.inv_dr : S(0);
        const S phip = (z2p - phi) * rinv;
        const S coef = (m.fp[snd] * rhojp + m.fp[rcv] * rhoip + phip) * rinv;
        gx = coef * dx;
        gy = coef * dy;
        gz = coef * dz;
        live = true;
      }
    }
    store_edge_force<S, NEWTON>(o, e, snd, rcv, gx, gy, gz, live);
  }
  edge_tail_and_slots(o, ne);
}

// LJ: the per-edge energy (scale edge_energy_scale) of senders below the energy rows goes to the
// block's partial slot 7, summed in a fixed order.
template <typename S, bool NEWTON>
__global__ __launch_bounds__(256) void k_lj_edge_force(LjModel<S> m, EdgeOut<S> o)
{
  __shared__ double red[256];
  const long ne = live_edges(o);
  const int erows = o.count->ghost_sender ? o.nall : o.nlocal;  // export.py:183-194
  const S tiny = static_cast<S>(1.0e-12);
  const long stride = static_cast<long>(gridDim.x) * blockDim.x;
  double en = 0.0;
  for (long e = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < ne; e += stride) {
    const int snd = o.senders[e], rcv = o.receivers[e];
    S gx = S(0), gy = S(0), gz = S(0);
    bool live = false;
    if (o.mask[e] && snd < o.nall && rcv < o.nall) {
      const Atom4<S> xs = m.atoms[snd], xr = m.atoms[rcv];
      S dx, dy, dz;
      const S r2 = geometry(xs, xr, dx, dy, dz);
      if (r2 > tiny && r2 < m.cutsq) {  // export_model.py:22
        const S u = m.sigsq / r2;
        const S u3 = u * u * u;
        if (snd < erows) en += static_cast<double>(m.edge_scale * (m.four_eps * (u3 * u3 - u3)));
        const S dedr2 = -m.four_eps * (S(6) * u3 * u3 - S(3) * u3) / r2;
        const S coef = S(2) * dedr2;
        gx = coef * dx;
        gy = coef * dy;
        gz = coef * dz;
        live = true;
      }
    }
    store_edge_force<S, NEWTON>(o, e, snd, rcv, gx, gy, gz, live);
  }
  red[threadIdx.x] = en;
  __syncthreads();
  for (int off = blockDim.x / 2; off >= 1; off >>= 1) {
    if (static_cast<int>(threadIdx.x) < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0 && static_cast<int>(blockIdx.x) < o.ntiles)
    put_partial(o.partials + 8L * blockIdx.x + 7, red[0]);
  edge_tail_and_slots(o, ne);
}

// f.r of the total f over the nall rows (cpp:227-245) into slots 1..6 of each 64-row tile, then
// the last block reduces every slot into the step result. The edge-force launch before it has
// finished: its live slot count becomes the next compute's reset bound.
template <bool VIRIAL>
__global__ __launch_bounds__(256) void k_fdotr_rows(const double *__restrict__ f,
                                                    const double *__restrict__ x, int nall,
                                                    int fdotr, double *partials, int ntiles,
                                                    double escale, int flags, StepResult *result,
                                                    int *done, StepResult *mirror, int *state,
                                                    int max_edges)
{
  constexpr int kWaves = 256 / kWave;
  __shared__ double scratch[7 * 256];
  __shared__ double tp[kWaves][6];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = wave_in_block();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int c = result->edge_count;
    state[kEdgeForceLive] = c < max_edges ? c : max_edges;
  }
  // Each wave sums one tile; the first wave stores the block's tiles. The loop bounds are the
  // block's, for the barriers.
  for (int t0 = blockIdx.x * kWaves; t0 < ntiles; t0 += static_cast<int>(gridDim.x) * kWaves) {
    const int t = t0 + wave;
    const int a = t * kWave + lane;
    double w[6] = {0, 0, 0, 0, 0, 0};
    if (VIRIAL && fdotr && t < ntiles && a < nall) {
      const double *fa = f + 3L * a;
      const double *xa = x + 3L * a;
      w[0] = fa[0] * xa[0];
      w[1] = fa[1] * xa[1];
      w[2] = fa[2] * xa[2];
      w[3] = fa[1] * xa[0];
      w[4] = fa[2] * xa[0];
      w[5] = fa[2] * xa[1];
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const double v = wave_sum(w[c]);
      if (lane == 0) tp[wave][c] = v;
    }
    __syncthreads();
    if (threadIdx.x < kWaves * 6) {
      const int q = threadIdx.x / 6, c = threadIdx.x % 6;
      if (t0 + q < ntiles) put_partial(partials + 8L * (t0 + q) + 1 + c, tp[q][c]);
    }
    __syncthreads();
  }
  finalize_last_block(partials, ntiles, escale, 1.0, flags, result, done, scratch, FusedPack{},
                      mirror);
}

template <typename S>
static EdgeOut<S> edge_out(Handle &h, int nlocal, int nghost, double scale, double *f, int ntiles,
                           int slot0_from, int block_energy)
{
  EdgeOut<S> o;
  o.senders = h.d_senders;
  o.receivers = h.d_receivers;
  o.mask = h.d_mask;
  o.count = h.d_result;
  o.max_edges = h.contract.max_edges;
  o.state = h.d_pack_state;
  o.edge_f = static_cast<S *>(h.d_edge_f);
  o.f = f;
  o.scale = scale;
  o.partials = h.d_partials;
  o.ntiles = ntiles;
  o.slot0_from = slot0_from;
  o.block_energy = block_energy;
  o.nlocal = nlocal;
  o.nall = nlocal + nghost;
  return o;
}

static hipError_t launch_fdotr(Handle &h, hipStream_t s, double *f, const double *x, int nall,
                               int ntiles, double scale, int flags)
{
  const int fdotr = h.contract.newton_pair ? 1 : 0;
  const int grid = grid_for(h, ntiles, 4, 2);
  StageTimer timer(h, s, "virial_fdotr");
  if ((flags & LK_VIRIAL) && fdotr)
    hipLaunchKernelGGL((k_fdotr_rows<true>), dim3(grid), dim3(256), 0, s, f, x, nall, fdotr,
                       h.d_partials, ntiles, scale, flags, h.d_result, h.d_done, h.d_host_result,
                       h.d_pack_state, h.contract.max_edges);
  else
    hipLaunchKernelGGL((k_fdotr_rows<false>), dim3(grid), dim3(256), 0, s, f, x, nall, fdotr,
                       h.d_partials, ntiles, scale, flags, h.d_result, h.d_done, h.d_host_result,
                       h.d_pack_state, h.contract.max_edges);
  return hipGetLastError();
}

template <typename S>
static hipError_t eam_edge_force(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                                 double scale, double *f, const double *x, bool from_list)
{
  EamArgs<S> m = eam_args<S>(h, nlocal, scale, f);
  TwoSided t = two_sided_args(h, nlocal, nghost, x);
  m.flags = flags;
  S *rho_part = static_cast<S *>(h.d_rho_part);
  S *epair = static_cast<S *>(h.d_epair);
  if (t.nblk > 0) {
    StageTimer timer(h, s, "eam_density");
    with_filter<S>(sweep_filter(h, from_list, FusedPack{}), [&](auto F) {
      hipLaunchKernelGGL((k_eam_density_inc<S, true, true, F.value, 16>),
                         dim3(grid_for(h, (t.nall + kRowBlock / 16 - 1) / (kRowBlock / 16), 1, 1)),
                         dim3(kRowBlock), 0, s, m, t, rho_part, epair);
    });
  }
  if (t.nblk > 0) {
    StageTimer timer(h, s, "eam_embed");
    hipLaunchKernelGGL((k_eam_embed_inc<S, true>), dim3(t.nblk), dim3(kWave), 0, s, m, t,
                       static_cast<const S *>(rho_part), static_cast<const S *>(epair));
  }
  int egrid = grid_for(h, h.contract.max_edges, kRowBlock, 1);
  if (egrid > h.partial_slots) egrid = h.partial_slots;
  const int ntiles = t.nblk > egrid ? t.nblk : egrid;
  const EdgeOut<S> o = edge_out<S>(h, nlocal, nghost, scale, f, ntiles, t.nblk, 0);
  {
    StageTimer timer(h, s, "edge_force");
    if (h.contract.newton_pair)
      hipLaunchKernelGGL((k_eam_edge_force<S, true>), dim3(egrid), dim3(kRowBlock), 0, s, m, o);
    else
      hipLaunchKernelGGL((k_eam_edge_force<S, false>), dim3(egrid), dim3(kRowBlock), 0, s, m, o);
  }
  return launch_fdotr(h, s, f, x, nlocal + nghost, ntiles, scale, flags);
}

template <typename S>
static hipError_t lj_edge_force(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                                double scale, double *f, const double *x)
{
  LjModel<S> m{};
  m.atoms = static_cast<const Atom4<S> *>(h.d_atoms);
  m.cutsq = static_cast<S>(h.lj.cutoff * h.lj.cutoff);
  m.sigsq = static_cast<S>(h.lj.sigma * h.lj.sigma);
  m.four_eps = static_cast<S>(4.0 * h.lj.epsilon);
  m.edge_scale = static_cast<S>(h.lj.edge_energy_scale);
  const int nall = nlocal + nghost;
  const int nblk = (nall + kWave - 1) / kWave;
  int egrid = grid_for(h, h.contract.max_edges, 256, 4);
  if (egrid > h.partial_slots) egrid = h.partial_slots;
  const int ntiles = nblk > egrid ? nblk : egrid;
  const EdgeOut<S> o = edge_out<S>(h, nlocal, nghost, scale, f, ntiles, 0, 1);
  {
    StageTimer timer(h, s, "edge_force");
    if (h.contract.newton_pair)
      hipLaunchKernelGGL((k_lj_edge_force<S, true>), dim3(egrid), dim3(256), 0, s, m, o);
    else
      hipLaunchKernelGGL((k_lj_edge_force<S, false>), dim3(egrid), dim3(256), 0, s, m, o);
  }
  return launch_fdotr(h, s, f, x, nall, ntiles, scale, flags);
}

hipError_t launch_edge_force(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                             double scale, double *f, const double *x, bool from_list)
{
  const bool f64 = h.contract.precision == LK_FLOAT64;
  if (h.model == 2)
    return f64 ? lj_edge_force<double>(h, s, nlocal, nghost, flags, scale, f, x)
               : lj_edge_force<float>(h, s, nlocal, nghost, flags, scale, f, x);
  hipError_t e = hipSuccess;
  if (from_list) {
    e = lists_of_list(h, s, false, reads_bits(h, FusedPack{}));  // whole lists
  } else {
    e = lists_of_edges(h, s, nlocal + nghost);
  }
  if (e != hipSuccess) return e;
  return f64 ? eam_edge_force<double>(h, s, nlocal, nghost, flags, scale, f, x, from_list)
             : eam_edge_force<float>(h, s, nlocal, nghost, flags, scale, f, x, from_list);
}

hipError_t launch_two_sided(Handle &h, hipStream_t s, int nlocal, int nghost, int flags,
                            double scale, double *f, const double *x, bool from_list,
                            const FusedPack &pack, int phase)
{
  hipError_t e = hipSuccess;
  if (phase == kPhaseForce) {
    // the incidence lists are the ones this step's density pass used
  } else if (from_list) {
    e = lists_of_list(h, s, h.accum == LK_ACCUM_PLAIN, reads_bits(h, pack));
  } else {
    e = lists_of_edges(h, s, nlocal + nghost);
  }
  if (e != hipSuccess) return e;
  const bool f64 = h.contract.precision == LK_FLOAT64;
  const bool half = h.accum == LK_ACCUM_HALF;
  if (h.model == 1) {
    if (f64)
      return half ? eam_two_sided<double, true>(h, s, nlocal, nghost, flags, scale, f, x,
                                                from_list, pack, phase)
                  : eam_two_sided<double, false>(h, s, nlocal, nghost, flags, scale, f, x,
                                                 from_list, pack, phase);
    return half ? eam_two_sided<float, true>(h, s, nlocal, nghost, flags, scale, f, x, from_list,
                                             pack, phase)
                : eam_two_sided<float, false>(h, s, nlocal, nghost, flags, scale, f, x, from_list,
                                              pack, phase);
  }
  if (f64) return lj_two_sided<double>(h, s, nlocal, nghost, flags, scale, f, x, from_list, pack);
  return lj_two_sided<float>(h, s, nlocal, nghost, flags, scale, f, x, from_list, pack);
}

}  // namespace lk
