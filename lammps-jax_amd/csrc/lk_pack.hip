// Neighbour-list packing on gfx950: cutoff filter + stream compaction of the LAMMPS Kokkos list
// into the bundle's sender/receiver/mask arrays (reference: cpp/pair_jax_kokkos.cpp:54-118,
// 157-173, 811-874), and the atom staging copy (cpp:35-52, 794-809).
//
// Layout of the packed edges ("row tiles"). The list is LayoutLeft (atom-fastest), so a wave
// reads it coalesced only with one lane per row. A wave therefore owns a tile of 64 consecutive
// list rows. Within a tile the edges are ordered by their ordinal k among the row's kept
// entries, then by row: at step k every row with more than k kept entries writes one edge, and
// the wave's writes land contiguously (ballot + mbcnt compaction). Tiles follow each other in
// row order, so the packed range [0, count) has no holes. The order is deterministic; the
// reference's atomic counter gives an arbitrary order, and the two agree after canonical sort.
//
// Three launches: count (filter, per-row counts, validity bits), a scan of the tile totals, and
// the compacted write; then the tail reset of slots the previous step used.

#include <mutex>

#include "lk_device.h"
#include "lk_internal.h"
#include "lk_tile.h"
#include "lk_pack.h"

namespace lk {

// PackAtomsFunctor (cpp/pair_jax_kokkos.cpp:35-52): positions narrowed to the contract precision,
// species = type - 1. The record keeps the species beside the position for one-gather lookups.
// `state` (optional, the pack state words) starts the fused pack that follows: the demand counter
// and the ghost-sender flag are zeroed and the live slot count of the previous pack is kept as
// the bound of this pack's tail reset.
template <typename S>
__global__ __launch_bounds__(256) void k_pack_atoms(const double *__restrict__ x,
                                                     const int *__restrict__ type, int span,
                                                     Atom4<S> *__restrict__ atoms,
                                                     int *__restrict__ species,
                                                     int *__restrict__ state)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (state && i == 0) {
    state[kPrevLive] = state[kLive];
    state[kDemand] = 0;
    state[kGhostFlag] = 0;
  }
  if (i >= span) return;
  const int sp = type[i] - 1;
  Atom4<S> a;
  a.x = static_cast<S>(x[3L * i + 0]);
  a.y = static_cast<S>(x[3L * i + 1]);
  a.z = static_cast<S>(x[3L * i + 2]);
  a.w = static_cast<S>(sp);
  atoms[i] = a;
  species[i] = sp;
}

constexpr int kCountWords = 8;  // validity words of a row held in LDS

constexpr int kPackWaves = 8;  // waves per 64-row tile

// Pass 1: one lane per list row, eight waves per 64-row tile. Wave w takes the slots w, w + 8, ... of
// every row: it reads them (coalesced across the rows) and applies the filter; the bits meet in LDS
// and go out as validity words (LayoutLeft). Each slot costs two dependent round trips (its entry,
// then the neighbour's position), so two slots of a row go at a time: both positions gather while
// the next two entries load; every load is unconditional, so waiting for the gathers never waits
// for the next entries. 108,000 atoms, 96 slots a row: 42 -> 34 us (four waves of one 32-slot word each,
// the fourth nearly empty, before; four slots at a time 34, sixteen waves 37, four 37).
__global__ __launch_bounds__(kPackWaves * kWave) void k_pack_count(PackArgs a)
{
  constexpr int W = kPackWaves, U = 2;
  static_assert(32 % (W * U) == 0, "a round's slots lie in one validity word");
  __shared__ int part[W][kWave];
  __shared__ uint32_t sbits[kCountWords][kWave];
  const int tile = tile_of_block();
  if (tile * kWave >= a.num_rows) return;
  const int wave = wave_in_block();
  const int lane = threadIdx.x & (kWave - 1);
  const int ii = tile * kWave + lane;
  const bool row = ii < a.num_rows;
  int i = -1;
  int nn = 0;
  if (row) {
    i = a.ilist[ii];
    if (i < a.max_atoms) {
      nn = min(a.numneigh[i], a.maxneighs);
    } else {
      i = -1;  // cpp:84: rows past max_atoms pack nothing
    }
  }
  double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0;
  if (i >= 0) {
    xi0 = a.x[3L * i + 0];
    xi1 = a.x[3L * i + 1];
    xi2 = a.x[3L * i + 2];
  }
  const int nn_max = wave_max_int(nn);  // the same in every wave
  int cnt = 0;
  // The row of a lane whose slots reach nn_max: every slot below it exists there, so a lane past its
  // own row reads that one (unused) and the loads need no branch.
  const int longest = __shfl(i, __builtin_ctzll(wave_ballot(nn == nn_max)), kWave);
  auto slot_entry = [&](int jj) -> int {
    const int at = min(jj, nn_max - 1);  // uniform
    const int *col = a.neighbors + static_cast<long>(at) * a.stride;
    return col[static_cast<unsigned>(at < nn ? i : longest)] & kNeighMask;
  };
  // 256 slots of every row at a time: their validity words fill LDS.
  for (int c0 = 0; c0 < nn_max; c0 += 32 * kCountWords) {
    const int c1 = min(c0 + 32 * kCountWords, nn_max);
    const int nwords = (c1 - c0 + 31) >> 5;
    for (int w = wave; w < nwords; w += W) sbits[w][lane] = 0u;
    __syncthreads();
    if (c0 + wave < c1) {
      int e[U];
#pragma unroll
      for (int q = 0; q < U; ++q) e[q] = slot_entry(c0 + wave + q * W);
      for (int jj = c0 + wave; jj < c1; jj += U * W) {
        double x[U][3];
        int ne[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {
          const long at = (jj + q * W < nn && e[q] < a.max_atoms) ? e[q] : 0;
          for (int c = 0; c < 3; ++c) x[q][c] = a.x[3 * at + c];
        }
#pragma unroll
        for (int q = 0; q < U; ++q) ne[q] = slot_entry(jj + (U + q) * W);
        uint32_t word = 0;
#pragma unroll
        for (int q = 0; q < U; ++q) {
          const int slot = jj + q * W;
          const bool keep = slot < nn && e[q] < a.max_atoms &&
                            keep_entry(a, i, xi0, xi1, xi2, e[q], x[q][0], x[q][1], x[q][2]);
          word |= keep ? 1u << (slot & 31) : 0u;
          e[q] = ne[q];
        }
        if (word) atomicOr(&sbits[(jj - c0) >> 5][lane], word);
      }
    }
    __syncthreads();
    for (int w = wave; w < nwords; w += W) {
      const uint32_t word = sbits[w][lane];
      cnt += __popc(word);
      if (row) a.bits[static_cast<long>((c0 >> 5) + w) * a.pitch + ii] = word;
    }
  }
  part[wave][lane] = cnt;
  __syncthreads();
  if (wave != 0) return;
  cnt = part[0][lane];
#pragma unroll
  for (int w = 1; w < W; ++w) cnt += part[w][lane];
  if (row) {
    a.row_count[ii] = cnt;
    a.row_atom[ii] = i;
  }
  const int edges = cnt * (a.duplicate ? 2 : 1);
  const int total = wave_sum(edges);
  const bool ghost_row = i >= a.nlocal && cnt > 0;
  const uint64_t gmask = wave_ballot(ghost_row);
  if (lane == 0) {
    a.tile_count[tile] = total;
    a.tile_flags[tile] = gmask != 0 ? 1 : 0;
  }
}

// Pass 2: exclusive scan of the tile totals in one block, in a fixed order. Writes the tile
// offsets, the demand count and overflow flag (cpp:103-108 semantics: overflow when the count
// exceeds max_edges), and whether any kept edge starts on a ghost row. prev_live: the previous
// pack's live slots, the bound of the tail reset (negative: the count the state holds).
__global__ __launch_bounds__(1024) void k_tile_scan(const int *__restrict__ tile_count,
                                                     const int *__restrict__ tile_flags,
                                                     int ntiles, int max_edges,
                                                     int *__restrict__ tile_off,
                                                     StepResult *__restrict__ result,
                                                     int *__restrict__ state, int prev_live)
{
  __shared__ long part[1024 / kWave];
  __shared__ int flag_any;
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  if (t == 0) flag_any = 0;
  const int per = (ntiles + blockDim.x - 1) / blockDim.x;
  const int lo = min(t * per, ntiles);
  const int hi = min(lo + per, ntiles);
  long sum = 0;
  int flags = 0;
  for (int k = lo; k < hi; ++k) {
    sum += tile_count[k];
    flags |= tile_flags[k];
  }
  long incl = sum;  // inclusive over the wave
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const long v = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += v;
  }
  if (lane == kWave - 1) part[wave] = incl;
  __syncthreads();
  if (flags) atomicOr(&flag_any, 1);
  long run = incl - sum;  // exclusive prefix of this thread's range
  for (int w = 0; w < wave; ++w) run += part[w];
  for (int k = lo; k < hi; ++k) {
    tile_off[k] = static_cast<int>(run);
    run += tile_count[k];
  }
  if (t == static_cast<int>(blockDim.x) - 1) {
    const long total = run;
    tile_off[ntiles] = static_cast<int>(total);
    result->edge_count = static_cast<int>(total);
    result->edge_overflow = total > max_edges ? 1 : 0;
    // the write pass resets [count, previous live count) after the new edges
    state[kPrevLive] = prev_live >= 0 ? prev_live : state[kLive];
    state[kLive] = static_cast<int>(total < max_edges ? total : max_edges);
  }
  __syncthreads();
  if (t == 0) result->ghost_sender = flag_any;
}

// Pass 3: compacted write, eight waves per tile. The rows with more than k kept entries form the
// ballot M of ordinal k and write M's popcount consecutive edges. Wave w writes one contiguous range
// of ordinals: its first slot is the sum over the rows of min(count, first ordinal), and each lane
// skips its row's entries before that once. The validity words come from LDS (from memory past 256
// slots). 108,000 atoms, 7.0 M edges: 33.5 -> 29 us, 3.6 TB/s of list and packed edges (every wave
// popped every ordinal before; four waves 32.6, sixteen 32, eight ordinals at a time 30).
__device__ __forceinline__ void pack_write_tile(const PackArgs &a, int tile,
                                                const int *__restrict__ tile_off,
                                                int *__restrict__ senders,
                                                int *__restrict__ receivers,
                                                unsigned char *__restrict__ mask,
                                                uint32_t (*sbits)[kWave])
{
  constexpr int W = kPackWaves, B = 4;  // B: ordinals whose list re-reads go out together
  const int wave = wave_in_block();
  const int lane = threadIdx.x & (kWave - 1);
  const int ii = tile * kWave + lane;
  const bool row = ii < a.num_rows;
  const int cnt = row ? a.row_count[ii] : 0;
  const int i = row ? a.row_atom[ii] : -1;
  const int mult = a.duplicate ? 2 : 1;
  const long base = tile_off[tile];
  const int nn_max = wave_max_int(i >= 0 ? min(a.numneigh[i], a.maxneighs) : 0);
  const int nwords = min((nn_max + 31) >> 5, kCountWords);
  for (int w = wave; w < nwords; w += W)
    sbits[w][lane] = row ? a.bits[static_cast<long>(w) * a.pitch + ii] : 0u;
  __syncthreads();
  auto read = [&](int w) -> uint32_t {
    return w < kCountWords ? sbits[w][lane] : a.bits[static_cast<long>(w) * a.pitch + ii];
  };
  const int kmax = wave_max_int(cnt);
  const int per = (kmax + W - 1) / W;
  const int k0 = min(wave * per, kmax);
  const int k1 = min(k0 + per, kmax);
  long cursor = wave_sum(min(cnt, k0));
  int w = 0;
  uint32_t word = 0;
  if (k0 < cnt) {
    word = read(0);
    int skip = k0;
    while (skip > 0) {
      const int pc = __popc(word);
      if (pc <= skip) {  // the k0-th entry lies in a later word
        skip -= pc;
        word = read(++w);
      } else {
        for (; skip > 0; --skip) word &= word - 1u;
      }
    }
  }
  for (int k = k0; k < k1; k += B) {
    int jv[B];
    long ev[B];
    bool act[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const bool active = k + q < k1 && k + q < cnt;
      const uint64_t M = wave_ballot(active);
      int jj = 0;
      if (active) {
        while (word == 0) word = read(++w);
        jj = w * 32 + __builtin_ctz(word);
        word &= word - 1u;
      }
      act[q] = active;
      ev[q] = base + (cursor + lanes_below(M)) * mult;
      cursor += __popcll(M);
      jv[q] = active ? a.neighbors[static_cast<long>(jj) * a.stride + i] : 0;
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      int jr = jv[q];
      asm volatile("" : "+v"(jr));  // the mask after the batch's loads, not inside each branch
      const int j = jr & kNeighMask;
      const long e = ev[q];
      if (act[q] && e + mult <= a.max_edges) {
        senders[e] = i;
        receivers[e] = j;
        mask[e] = 1;
        if (mult == 2) {
          senders[e + 1] = j;
          receivers[e + 1] = i;
          mask[e + 1] = 1;
        }
      }
    }
  }
}

__global__ __launch_bounds__(kPackWaves * kWave) void k_pack_write(PackArgs a, const int *__restrict__ tile_off,
                                                       int *__restrict__ senders,
                                                       int *__restrict__ receivers,
                                                       unsigned char *__restrict__ mask,
                                                       const StepResult *__restrict__ result,
                                                       const int *__restrict__ state,
                                                       int *__restrict__ counts_out)
{
  __shared__ uint32_t sbits[kCountWords][kWave];
  const int tile = tile_of_block();
  if (tile * kWave < a.num_rows)  // the whole block or none of it
    pack_write_tile(a, tile, tile_off, senders, receivers, mask, sbits);
  // ResetEdgeTailFunctor (cpp:157-173): slots past the new count that held the previous pack's
  // edges return to the padding (max_atoms, max_atoms, false); a grid-stride pass over every
  // block. Both bounds come from the scan pass, on the device.
  const long count = result->edge_count;
  const long reset_end = state[kPrevLive];
  if (counts_out && blockIdx.x == 0 && threadIdx.x == 0) {
    counts_out[0] = result->edge_count;
    counts_out[1] = result->edge_overflow;
  }
  for (long e = count + static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < reset_end;
       e += static_cast<long>(gridDim.x) * blockDim.x) {
    senders[e] = a.max_atoms;
    receivers[e] = a.max_atoms;
    mask[e] = 0;
  }
}

// CopyNeighborMatrixFunctor (cpp/pair_jax_kokkos.cpp:120-155): flat = slot * rows + row, atom
// fastest on both sides, so reads of the LayoutLeft list and writes of the matrix coalesce. Row i
// is atom i. The step result's edge count takes the widest row, its overflow flag a row longer
// than max_neighbors (that row is truncated).
__global__ void k_matrix_counts_reset(StepResult *r)
{
  if (threadIdx.x == 0) {
    r->edge_count = 0;
    r->edge_overflow = 0;
    r->ghost_sender = 0;
  }
}

__global__ __launch_bounds__(256) void k_copy_matrix(const int *__restrict__ numneigh,
                                                     const int *__restrict__ neighbors,
                                                     long stride, int num_rows, int rows,
                                                     int max_atoms, int max_neighbors,
                                                     int *__restrict__ matrix,
                                                     int *__restrict__ num_out, StepResult *r)
{
  const long flat = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (flat >= static_cast<long>(rows) * max_neighbors) return;
  const int slot = static_cast<int>(flat / rows);
  const int i = static_cast<int>(flat % rows);
  if (i >= num_rows) {
    matrix[flat] = max_atoms;
    if (slot == 0) num_out[i] = 0;
    return;
  }
  const int n = numneigh[i];
  if (slot == 0) {
    atomicMax(&r->edge_count, n);
    if (n > max_neighbors) r->edge_overflow = 1;
    num_out[i] = n < max_neighbors ? n : max_neighbors;
  }
  int j = max_atoms;
  if (slot < n) j = neighbors[static_cast<long>(slot) * stride + i] & kNeighMask;
  matrix[flat] = j < max_atoms ? j : max_atoms;
}

hipError_t launch_copy_matrix(Handle &h, hipStream_t s, const int *numneigh, const int *neighbors,
                              long stride, int num_rows)
{
  StageTimer timer(h, s, "copy_matrix");
  hipLaunchKernelGGL(k_matrix_counts_reset, dim3(1), dim3(64), 0, s, h.d_result);
  const long flat = static_cast<long>(h.matrix_rows) * h.contract.max_neighbors;
  const long blocks = (flat + 255) / 256;
  hipLaunchKernelGGL(k_copy_matrix, dim3(static_cast<unsigned>(blocks > 0 ? blocks : 1)),
                     dim3(256), 0, s, numneigh, neighbors, stride, num_rows, h.matrix_rows,
                     h.contract.max_atoms, h.contract.max_neighbors, h.d_matrix,
                     h.d_num_neighbors, h.d_result);
  return hipGetLastError();
}

__global__ void k_iota(int *p, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

hipError_t launch_iota(hipStream_t s, int *p, int n)
{
  hipLaunchKernelGGL(k_iota, dim3((n + 255) / 256 > 0 ? (n + 255) / 256 : 1), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_tile_scan(Handle &h, hipStream_t s, const int *tile_flags, int ntiles)
{
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, s, h.d_tile_count, tile_flags, ntiles,
                     h.contract.max_edges, h.d_tile_off, h.d_result, h.d_pack_state, -1);
  return hipGetLastError();
}

hipError_t launch_pack_atoms(Handle &h, hipStream_t s, const double *x, const int *type, int nall,
                             int *clear)
{
  const int span = nall < h.contract.max_atoms ? nall : h.contract.max_atoms;
  if (span <= 0 && !clear) return hipSuccess;
  const int blocks = span > 0 ? (span + 255) / 256 : 1;
  StageTimer timer(h, s, "pack_atoms");
  if (h.contract.precision == LK_FLOAT64)
    hipLaunchKernelGGL(k_pack_atoms<double>, dim3(blocks), dim3(256), 0, s, x, type, span,
                       static_cast<Atom4<double> *>(h.d_atoms), h.d_species, clear);
  else
    hipLaunchKernelGGL(k_pack_atoms<float>, dim3(blocks), dim3(256), 0, s, x, type, span,
                       static_cast<Atom4<float> *>(h.d_atoms), h.d_species, clear);
  return hipGetLastError();
}

PackArgs pack_args(Handle &h, const double *x, const int *ilist, const int *numneigh,
                   const int *neighbors, long stride, int num_rows, int maxneighs, int nlocal,
                   int duplicate, int half_edges, int unique_boundary)
{
  PackArgs a;
  a.x = x;
  a.ilist = ilist;
  a.numneigh = numneigh;
  a.neighbors = neighbors;
  a.stride = stride;
  a.num_rows = num_rows;
  a.maxneighs = maxneighs;
  a.max_atoms = h.contract.max_atoms;
  a.max_edges = h.contract.max_edges;
  a.nlocal = nlocal;
  a.cutsq = h.contract.cutoff * h.contract.cutoff;
  a.duplicate = duplicate;
  a.half_edges = half_edges;
  a.unique_boundary = unique_boundary;
  a.words = h.bits_words;
  a.pitch = h.contract.max_atoms;
  a.bits = h.d_bits;
  a.row_count = h.d_row_count;
  a.row_atom = h.d_row_atom;
  a.tile_count = h.d_tile_count;
  a.tile_flags = h.d_tile_count + (h.contract.max_atoms / kWave + 2);
  return a;
}

hipError_t launch_pack_write(Handle &h, hipStream_t s, const PackArgs &a)
{
  const int ntiles = (a.num_rows + kWave - 1) / kWave;
  // at least one block so the tail reset runs when the list is empty
  const int grid = tile_grid(ntiles > 0 ? ntiles : 1);
  StageTimer timer(h, s, "pack_write");
  hipLaunchKernelGGL(k_pack_write, dim3(grid), dim3(kPackWaves * kWave), 0, s, a, h.d_tile_off,
                     h.d_senders, h.d_receivers, h.d_mask, h.d_result, h.d_pack_state,
                     static_cast<int *>(nullptr));
  return hipGetLastError();
}

hipError_t launch_pack_edges(Handle &h, hipStream_t s, const double *x, const int *ilist,
                             const int *numneigh, const int *neighbors, long stride, int num_rows,
                             int maxneighs, int nlocal, int duplicate, int half_edges,
                             int unique_boundary)
{
  const PackArgs a = pack_args(h, x, ilist, numneigh, neighbors, stride, num_rows, maxneighs,
                               nlocal, duplicate, half_edges, unique_boundary);
  const int ntiles = (num_rows + kWave - 1) / kWave;
  h.packed_rows = num_rows;
  const int grid = tile_grid(ntiles);
  if (ntiles > 0) {
    StageTimer timer(h, s, "pack_count");
    hipLaunchKernelGGL(k_pack_count, dim3(grid), dim3(kPackWaves * kWave), 0, s, a);
  }
  {
    StageTimer timer(h, s, "tile_scan");
    hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, s, h.d_tile_count, a.tile_flags,
                       ntiles, h.contract.max_edges, h.d_tile_off, h.d_result, h.d_pack_state, -1);
  }
  hipError_t e = launch_pack_write(h, s, a);
  ++h.pack_serial;
  return e;
}

// ----------------------------------------------------------------------------------------------
// The pack without allocation (lk_pack_edges_noalloc). Its working memory (validity bits, row
// counts and row atoms, tile totals, flags and offsets, the scan's result and the slot counts)
// is `scratch`, a file-scope device array that every GPU the library runs on holds from the
// library's load to the end of the process: 24.2 MB. The caller owns the list and the packed
// arrays. Every call on a GPU shares that GPU's array and leaves its contents behind, so calls
// that overlap on one GPU race; each call writes every word it reads before reading it.
// ----------------------------------------------------------------------------------------------
namespace {

constexpr long kScratchTiles = kScratchRows / kWave + 2;
constexpr long kOffBits = 0;
constexpr long kOffRowCount = kOffBits + kScratchBitWords;
constexpr long kOffRowAtom = kOffRowCount + kScratchRows;
constexpr long kOffTileCount = kOffRowAtom + kScratchRows;
constexpr long kOffTileFlags = kOffTileCount + kScratchTiles;
constexpr long kOffTileOff = kOffTileFlags + kScratchTiles;
constexpr long kOffResult = ((kOffTileOff + kScratchTiles + 63) / 64) * 64;  // 256-byte aligned
constexpr long kOffState = kOffResult + 64;
constexpr long kScratchInts = kOffState + 64;
static_assert(sizeof(StepResult) <= 64 * sizeof(int), "step result slot");
static_assert(kPackStateWords <= 64, "pack state slot");

}  // namespace

static __device__ __align__(256) int scratch[kScratchInts];

namespace {

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
int *scratch_ptr[kMaxDevices] = {};

// The device address of this GPU's `scratch`: looked up once per device, with that device
// current, on the first call there (host code must not pass the array's own name to a kernel).
hipError_t scratch_address(int **out)
{
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    scratch_ptr[dev] = static_cast<int *>(p);
  }
  *out = scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace

hipError_t launch_pack_edges_noalloc(hipStream_t s, PackArgs a, int *senders, int *receivers,
                                     unsigned char *mask, int *counts_out, int prev_live)
{
  int *base = nullptr;
  if (hipError_t e = scratch_address(&base); e != hipSuccess) return e;
  a.pitch = a.num_rows > 0 ? a.num_rows : 1;
  a.words = (a.maxneighs + 31) / 32;
  a.bits = reinterpret_cast<uint32_t *>(base + kOffBits);
  a.row_count = base + kOffRowCount;
  a.row_atom = base + kOffRowAtom;
  a.tile_count = base + kOffTileCount;
  a.tile_flags = base + kOffTileFlags;
  int *tile_off = base + kOffTileOff;
  auto *result = reinterpret_cast<StepResult *>(base + kOffResult);
  int *state = base + kOffState;
  const int ntiles = (a.num_rows + kWave - 1) / kWave;
  if (ntiles > 0)
    hipLaunchKernelGGL(k_pack_count, dim3(tile_grid(ntiles)), dim3(kPackWaves * kWave), 0, s, a);
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, s, a.tile_count, a.tile_flags, ntiles,
                     a.max_edges, tile_off, result, state, prev_live);
  hipLaunchKernelGGL(k_pack_write, dim3(tile_grid(ntiles > 0 ? ntiles : 1)),
                     dim3(kPackWaves * kWave), 0, s, a, tile_off, senders, receivers, mask, result,
                     state, counts_out);
  return hipGetLastError();
}

}  // namespace lk
