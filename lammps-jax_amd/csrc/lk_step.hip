// The one-sided step in three launches: pack + EAM (or LJ) energy, forces and virial.
//
// What PairJaxKokkos::compute does per step (cpp/pair_jax_kokkos.cpp:989-1102) with the full-list
// row scheme of the model (eam_pallas.py:181-249, full list): pack_atoms, pack_neighbors and the
// tail reset (cpp:35-173, 794-874), the density and embedding (eam.py:298-321), the force and
// virial (eam.py:385-398, cpp:175-245).
//
//   K0 atoms:  atom records and species (lk_pack.hip); clears the pack's demand counter.
//   K1 pack:   per 64-row tile, the list walk with the cutoff filter (positions gathered from the
//              records, one load of 32 bytes, or of 16 in float32, per entry), validity bits and
//              row counts; on kept pairs the density of the row (float64: from the same r^2 the
//              filter formed); then F(rho), F'(rho), F' copied to the row's ghost images (the
//              forward comm of one rank) and the embedding energy of the tile. The tile then
//              claims its slot range with one atomic add on the demand counter (the reference's
//              packer claims slots the same way, per entry) and writes its edges in the
//              row-tile order while its list lines are still in cache.
//   K2 force:  the force sweep over the packed receivers (lk_eam.hip, lk_lj.hip); it also
//              resets the slots the previous step used past the new count, and its last block
//              reduces the tile partials in a fixed order into the step result.
// The packed arrays equal the reference's after canonical ordering; the tiles' order in them
// follows the atomic claims. Per-row sums never depend on it (each row's edges keep their order
// inside its tile), so energies, forces and virials are bitwise reproducible.

#include <cmath>
#include <limits>

#include "lk_eam_common.h"
#include "lk_pack.h"
#include "lk_tiles.h"

namespace lk {

// Inputs and pack outputs of the pack kernel besides the model arguments.
struct StepPack {
  const double *x;
  const int *type;
  const int *ilist;
  const int *numneigh;
  const int *neighbors;
  long stride;
  int num_rows;
  int maxneighs;
  int max_atoms;
  int max_edges;
  double cutsq;
  float cutsq_lo, cutsq_hi;  // cutsq rounded down and up to float
  int pitch;
  uint32_t *bits;
  int *row_count;
  int *row_atom;
  int *tile_base;
  int *state;  // pack state words (PackState): demand counter and ghost flag cleared by K0
  int *senders;
  int *receivers;
  unsigned char *mask;
  const int *ghost_off;
  const int *ghost_list;
  // float64 pack-only kernels of the fused two-sided step: the atom records of [0, records)
  // (PackAtomsFunctor), written here instead of by a launch of their own, or null; the filter
  // then reads x, since other blocks' records may not be written yet
  Atom4<double> *atoms_out;
  int *species_out;
  int records;
};

// The pack's filter, rsq <= cutsq with rsq formed in float64 from the engine's x without
// contraction (cpp:84-91), for float32 contracts, decided from float records where they decide
// it: xa and xo are the row's and the neighbour's records (x rounded to float), sa = |xa|_1. With
// u = 2^-24, l1 = |dx| + |dy| + |dz| of the float differences and s = l1 + |xa|_1 + |xo|_1, each
// float difference is within u (|d_c| + |x_a,c| + |x_o,c|) / (1 - u) of the float64 one, so the
// float r2 lies within u s (2 l1 + u s) / (1 - u)^2 + 3u r2 / (1 - 3u) of rsq; band, computed in
// float, is at least twice that and at least 8u r2, which also covers comparing r2 +- band with
// cutsq rounded down (up) to float. Only a slot inside the band reads the engine's float64
// position of its neighbour and forms rsq exactly as the float64 filter does.
__device__ __forceinline__ bool pack_keeps_f32(const StepPack &p, const Atom4<float> &xa,
                                               float sa, const Atom4<float> &xo, int j,
                                               double xi0, double xi1, double xi2)
{
  constexpr float u = 5.9604645e-8f;  // 2^-24
  float dx, dy, dz, r2;
  {
#pragma clang fp contract(off)
    dx = xo.x - xa.x;
    dy = xo.y - xa.y;
    dz = xo.z - xa.z;
    r2 = dx * dx + dy * dy + dz * dz;
  }
  const float l1 = fabsf(dx) + fabsf(dy) + fabsf(dz);
  const float s = l1 + sa + (fabsf(xo.x) + fabsf(xo.y) + fabsf(xo.z));
  const float band = 2.0f * u * (s * (2.0f * l1 + u * s) + 4.0f * r2);
  if (r2 + band <= p.cutsq_lo) return true;
  if (r2 - band > p.cutsq_hi) return false;
  double rsq;
  {
#pragma clang fp contract(off)
    const double ex = xi0 - p.x[3L * j + 0], ey = xi1 - p.x[3L * j + 1];
    const double ez = xi2 - p.x[3L * j + 2];
    rsq = ex * ex + ey * ey + ez * ez;
  }
  return !(rsq > p.cutsq);
}

// cutsq and its float bounds for the kernel arguments.
static void set_pack_cutoff(StepPack &p, double cutoff)
{
  p.cutsq = cutoff * cutoff;
  p.cutsq_lo = static_cast<float>(p.cutsq);
  p.cutsq_hi = p.cutsq_lo;
  if (static_cast<double>(p.cutsq_lo) > p.cutsq)
    p.cutsq_lo = std::nextafter(p.cutsq_lo, -std::numeric_limits<float>::infinity());
  if (static_cast<double>(p.cutsq_hi) < p.cutsq)
    p.cutsq_hi = std::nextafter(p.cutsq_hi, std::numeric_limits<float>::infinity());
}

constexpr int kStepWaves = 16;    // waves per block: kStepWaves / W tiles
constexpr int kStepLds = 3584;     // table window entries: 56 KB (two blocks per CU)
constexpr int kStepMaxWords = 8;   // validity words kept in LDS for the write (256 list slots)

// K1. Block-uniform control flow around every barrier: the group walk has the same trip count
// for all threads of a block, and fill_window is entered by all of them.
// MATRIX: the list is the neighbour matrix of a matrix bundle. No packer filter applies: an
// entry counts when the model's mask does (r^2 < cutoff^2 at the contract precision,
// eam_pallas.py list_pair), and only the internal receivers are written for the force sweep.
// Grid of K1. With the EAM table window to fill, blocks stay resident and walk several groups
// (two per CU), so the fill is paid once per block. Without it there is nothing to amortise: one
// group per block lets the dispatcher hand out groups as CUs free up, instead of a static share
// per block whose last round runs on a fraction of the blocks.
template <bool EAM>
static int step_pack_grid(int ngroups, int num_cus)
{
  if constexpr (EAM) return persistent_grid(ngroups, 2, num_cus);
  return ((ngroups + kXcds - 1) / kXcds) * kXcds;
}

template <typename S, bool EAM, bool MATRIX, int W>
__global__ __launch_bounds__(kStepWaves * kWave) __attribute__((amdgpu_waves_per_eu(8))) LK_EIGHT_WAVES
void k_step_pack(StepPack p, EamArgs<S> a, int ngroups)
{
  constexpr int TPB = kStepWaves / W;
  __shared__ LdsEntry<S> lds[EAM ? kStepLds : 1];
  __shared__ int cpart[TPB][W][kWave];
  __shared__ S rpart[TPB][W][kWave];
  __shared__ uint32_t sbits[TPB][kStepMaxWords][kWave];
  __shared__ int scnt[TPB][kWave];
  __shared__ int sbase[TPB];

  Window<S> win{};
  if constexpr (EAM) win = fill_window<S>(lds, kStepLds, a, a.n_el, W * TPB * kWave);
  if constexpr (!EAM && sizeof(S) == 8) {
    // the atom records for the sweeps (cpp:35-52: x as is, species = type - 1)
    if (p.atoms_out)
      for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < p.records;
           i += gridDim.x * blockDim.x) {
        const int sp = p.type[i] - 1;
        Atom4<double> r;
        r.x = p.x[3L * i + 0];
        r.y = p.x[3L * i + 1];
        r.z = p.x[3L * i + 2];
        r.w = static_cast<double>(sp);
        p.atoms_out[i] = r;
        p.species_out[i] = sp;
      }
  }
  const int sub = wave_in_block() / W;
  const int wave = wave_in_block() % W;
  const int lane = threadIdx.x & (kWave - 1);
  for (GroupWalk gw = group_walk(ngroups); gw.g < gw.g_end; gw.g += gw.step) {
    const int tile = gw.g * TPB + sub;
    const int ii = tile * kWave + lane;
    const bool row = ii < p.num_rows;
    int i = -1, nn = 0;
    if (row) {
      i = p.ilist[ii];
      if (i < p.max_atoms)
        nn = min(p.numneigh[i], p.maxneighs);
      else
        i = -1;  // cpp:84: rows past max_atoms pack nothing
    }
    double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0;
    Atom4<float> xa{0.0f, 0.0f, 0.0f, 0.0f};  // float32 pack-only: the row's record
    if (i >= 0) {
      xi0 = p.x[3L * i + 0];
      xi1 = p.x[3L * i + 1];
      xi2 = p.x[3L * i + 2];
      if constexpr (sizeof(S) == 4) xa = a.atoms[i];
    }
    const float sa = fabsf(xa.x) + fabsf(xa.y) + fabsf(xa.z);
    const int nn_max = wave_max_int(nn);
    const int nwords = (nn_max + 31) >> 5;
    const bool lds_bits = nwords <= kStepMaxWords;
    int cnt = 0;
    S rho = S(0);
    // The list entry of slot jj of this lane's row; past the row it reads element 0 (which
    // exists: the loops below only run when some row of the wave has a slot) and is unused.
    // The load is unconditional, so the compiler can count it exactly and wait for an earlier
    // load without waiting for this one.
    auto slot_entry = [&](int jj) -> int {
      return p.neighbors[jj < nn ? static_cast<long>(jj) * p.stride + i : 0L];
    };
    // One list slot of this lane's row (entry: its list entry) in the float64 model kernels: the
    // filter chain, and the density of a kept pair.
    auto visit = [&](int jj, int entry) -> bool {
      if constexpr (EAM && sizeof(S) == 8) {
        const int j = entry & kNeighMask;
        if (!(jj < nn && j < p.max_atoms)) return false;
        // one 32-byte gather (two 16-byte loads) brings x and species. The empty asm takes the
        // species where it arrives, so the compiler cannot defer it into an 8-byte gather of its
        // own behind the filter.
        const Atom4<double> rj = reinterpret_cast<const Atom4<double> *>(a.atoms)[j];
        asm volatile("" ::"v"(rj.w));
        double rsq;
        {
#pragma clang fp contract(off)
          const double dx = xi0 - rj.x, dy = xi1 - rj.y, dz = xi2 - rj.z;
          rsq = dx * dx + dy * dy + dz * dz;
        }
        if constexpr (MATRIX) {
          if (!(rsq < a.cutsq)) return false;
        } else {
          if (rsq > p.cutsq) return false;  // PackNeighborFunctor keeps rsq <= cutsq (cpp:91)
        }
        ++cnt;
        if (MATRIX || rsq < a.cutsq) {  // valid = mask & r_sq < cutoff_sq (eam.py:288)
          const double rr = rsq * rsqrt_nr(rsq);
          const Locator<double> L = locate_mul(rr, static_cast<double>(a.inv_dr), a.nr);
          rho += cvalue(rcoef(win, a, L.node, clamp_species(static_cast<int>(rj.w), a.n_el)), L.t);
        }
        return true;
      }
      return false;
    };
    // The float32 and the pack-only kernels walk the slots jj0, jj0 + step, ... < jj1 two at a
    // time: both entries are loaded one pair ahead, then both neighbour records gathered
    // together, so a pair costs one memory round trip. Every load
    // is unconditional (slots past the row read element 0 of the list and the record of atom 0,
    // which exist whenever the loop runs, and are unused), so the compiler counts them exactly
    // and waits for the gathers without waiting for the next pair's entries. The records are
    // this step's (K0 ran before, or the engine's lk_pack_atoms call): float64 ones hold x
    // exactly; float32 ones decide the filter through pack_keeps_f32 and give the model its r^2
    // and the neighbour's species (one 16-byte gather per slot in place of three 8-byte ones from
    // x and one from type: 104,284 atoms' matrix 83 -> 57 us, at eight waves per tile).
    auto walk32 = [&](int jj0, int jj1, int step, auto &&kept) {
      auto gather = [&](int jj, int entry) -> Atom4<float> {
        const int j = entry & kNeighMask;
        return reinterpret_cast<const Atom4<float> *>(a.atoms)[(jj < nn && j < p.max_atoms) ? j : 0];
      };
      auto test = [&](int jj, int entry, const Atom4<float> &xo) {
        const int j = entry & kNeighMask;
        if (!(jj < nn && j < p.max_atoms)) return;
        float r2 = 0.0f;
        if constexpr (EAM) {
#pragma clang fp contract(off)
          const float dx = xo.x - xa.x, dy = xo.y - xa.y, dz = xo.z - xa.z;
          r2 = dx * dx + dy * dy + dz * dz;
        }
        if constexpr (MATRIX) {
          if (!(r2 < a.cutsq)) return;
        } else {
          if (!pack_keeps_f32(p, xa, sa, xo, j, xi0, xi1, xi2)) return;
        }
        ++cnt;
        kept(jj);
        if constexpr (EAM && sizeof(S) == 4) {
          if (MATRIX || r2 < a.cutsq) {  // valid = mask & r_sq < cutoff_sq (eam.py:288)
            const float rr = r2 * rsqrt_nr(r2);
            const Locator<float> L = locate_mul(rr, a.inv_dr, a.nr);
            rho += cvalue(rcoef(win, a, L.node, clamp_species(static_cast<int>(xo.w), a.n_el)),
                          L.t);
          }
        }
      };
      int ea = slot_entry(jj0), eb = slot_entry(jj0 + step);
      for (int jj = jj0; jj < jj1; jj += 2 * step) {
        const int jb = jj + step;
        const Atom4<float> ra = gather(jj, ea), rb = gather(jb, eb);
        const int na = slot_entry(jj + 2 * step), nb = slot_entry(jj + 3 * step);
        test(jj, ea, ra);
        if (jb < jj1) test(jb, eb, rb);
        ea = na;
        eb = nb;
      }
    };
    auto walk = [&](int jj0, int jj1, int step, auto &&kept) {
      if constexpr (sizeof(S) == 4) {
        walk32(jj0, jj1, step, kept);
      } else {
        auto gather = [&](int jj, int entry, double &x0, double &x1, double &x2) {
          const int j = entry & kNeighMask;
          const long q = (jj < nn && j < p.max_atoms) ? j : 0;
          if (p.atoms_out) {  // this launch writes the records
            x0 = p.x[3 * q + 0];
            x1 = p.x[3 * q + 1];
            x2 = p.x[3 * q + 2];
          } else {
            const double2 h = reinterpret_cast<const double2 *>(a.atoms)[2 * q];
            x0 = h.x;
            x1 = h.y;
            x2 = reinterpret_cast<const double *>(a.atoms)[4 * q + 2];
          }
        };
        auto test = [&](int jj, int entry, double x0, double x1, double x2) {
          const int j = entry & kNeighMask;
          double rsq;
          {
#pragma clang fp contract(off)
            const double dx = xi0 - x0, dy = xi1 - x1, dz = xi2 - x2;
            rsq = dx * dx + dy * dy + dz * dz;
          }
          // PackNeighborFunctor keeps rsq <= cutsq (cpp:84-101)
          if (jj < nn && j < p.max_atoms && !(rsq > p.cutsq)) {
            ++cnt;
            kept(jj);
          }
        };
        int ea = slot_entry(jj0), eb = slot_entry(jj0 + step);
        for (int jj = jj0; jj < jj1; jj += 2 * step) {
          const int jb = jj + step;
          double a0, a1, a2, b0, b1, b2;
          gather(jj, ea, a0, a1, a2);
          gather(jb, eb, b0, b1, b2);
          const int na = slot_entry(jj + 2 * step), nb = slot_entry(jj + 3 * step);
          test(jj, ea, a0, a1, a2);
          if (jb < jj1) test(jb, eb, b0, b1, b2);
          ea = na;
          eb = nb;
        }
      }
    };
    // Each wave takes every W-th slot and ORs its bits into the tile's LDS words, which the first
    // barrier below completes (the global words are stored after it); rows of more words than
    // LDS holds go one word per wave at a time.
    if (lds_bits)
      for (int w = wave; w < nwords; w += W) sbits[sub][w][lane] = 0u;
    __syncthreads();
    if (lds_bits) {
      auto mark = [&](int jj) { atomicOr(&sbits[sub][jj >> 5][lane], 1u << (jj & 31)); };
      if constexpr (EAM && sizeof(S) == 8) {
        for (int jj = wave; jj < nn_max; jj += W)
          if (visit(jj, slot_entry(jj))) mark(jj);
      } else if (wave < nn_max) {
        walk(wave, nn_max, W, mark);
      }
    } else {
      for (int w = wave; w < nwords; w += W) {
        uint32_t word = 0;
        const int jj0 = w * 32;
        const int jj1 = min(jj0 + 32, nn_max);
        if constexpr (EAM && sizeof(S) == 8) {
          for (int jj = jj0; jj < jj1; ++jj)
            if (visit(jj, slot_entry(jj))) word |= 1u << (jj & 31);
        } else {
          walk(jj0, jj1, 1, [&](int jj) { word |= 1u << (jj & 31); });
        }
        if (row) p.bits[static_cast<long>(w) * p.pitch + ii] = word;
      }
    }
    cpart[sub][wave][lane] = cnt;
    if constexpr (EAM) rpart[sub][wave][lane] = rho;
    __syncthreads();
    if (lds_bits && row)
      for (int w = wave; w < nwords; w += W)
        p.bits[static_cast<long>(w) * p.pitch + ii] = sbits[sub][w][lane];
    if (wave == 0) {
      cnt = cpart[sub][0][lane];
      if constexpr (EAM) rho = rpart[sub][0][lane];
#pragma unroll
      for (int w = 1; w < W; ++w) {
        cnt += cpart[sub][w][lane];
        if constexpr (EAM) rho += rpart[sub][w][lane];
      }
      if (row) {
        p.row_count[ii] = cnt;
        p.row_atom[ii] = i;
      }
      scnt[sub][lane] = cnt;
      const int total = wave_sum(cnt);
      const uint64_t gmask = wave_ballot(i >= a.nlocal && cnt > 0);
      double e_own = 0.0;
      if constexpr (EAM) {
        if (i >= 0) {
          S F, Fp;
          embed(a, clamp_species(p.type[i] - 1, a.n_el), rho, F, Fp);
          a.fp[i] = Fp;
          if (a.rho) a.rho[i] = rho;
          if (i < a.nlocal) {
            e_own = static_cast<double>(F);
            if (p.ghost_off)
              for (int q = p.ghost_off[i]; q < p.ghost_off[i + 1]; ++q) a.fp[p.ghost_list[q]] = Fp;
          }
        }
      }
      const double esum = wave_sum(e_own);
      if (lane == 0 && tile * kWave < p.num_rows) {
        // the tile's slots [base, base + total): one claim per tile (cpp:102-110 claims per entry)
        const int base = atomicAdd(&p.state[kDemand], total);
        sbase[sub] = base;
        p.tile_base[tile] = base;
        if (gmask != 0) atomicOr(&p.state[kGhostFlag], 1);
        put_partial(a.partials + 8L * tile + 0, esum);
      }
    }
    __syncthreads();
    // Compacted write: ordinal k of every row (rows with more than k entries form the ballot M)
    // occupies popcount(M) consecutive slots after the slots of the ordinals below k. Wave w
    // writes one contiguous range of ordinals [k0, k1): its first slot is the sum over the rows
    // of min(count, k0); each lane skips its row's first k0 kept entries once, then pops them in
    // order. The list slot is read again from cache.
    {
      const int c = scnt[sub][lane];
      const long base = sbase[sub];
      const int kmax = wave_max_int(c);
      const int per = (kmax + W - 1) / W;
      const int k0 = min(wave * per, kmax);
      const int k1 = min(k0 + per, kmax);
      const long cursor0 = wave_sum(min(c, k0));
      // Writes ordinals [k0, k1), B at a time: the slot positions of a batch come from the
      // validity words alone (read(wd): word wd of this lane's row), so its list re-reads are
      // all in flight before its stores. The words come from LDS for rows of up to 256 slots
      // (batches of 4) and from memory past that (one ordinal at a time: a word loaded inside
      // the batch would make every re-read wait for it).
      auto write_ordinals = [&](auto read, auto batch) {
        constexpr int B = decltype(batch)::value;
        long cursor = cursor0;
        int wd = 0;
        uint32_t word = 0;
        if (k0 < c) {
          word = read(0);
          int skip = k0;
          while (skip > 0) {
            const int pc = __popc(word);
            if (pc <= skip) {  // the k0-th entry lies in a later word
              skip -= pc;
              word = read(++wd);
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
            const bool active = k + q < k1 && k + q < c;
            const uint64_t M = wave_ballot(active);
            int jj = 0;
            if (active) {
              while (word == 0) word = read(++wd);
              jj = wd * 32 + __builtin_ctz(word);
              word &= word - 1u;
            }
            act[q] = active;
            ev[q] = base + cursor + lanes_below(M);
            cursor += __popcll(M);
            jv[q] = active ? p.neighbors[static_cast<long>(jj) * p.stride + i] : 0;
          }
#pragma unroll
          for (int q = 0; q < B; ++q) {
            // the empty asm keeps the neighbour mask here, after the batch's loads have all gone
            // out (folded into each load's branch it would wait for each load in turn)
            int jr = jv[q];
            asm volatile("" : "+v"(jr));
            if (act[q] && ev[q] < p.max_edges) {  // past the capacity the count reports the demand
              p.receivers[ev[q]] = jr & kNeighMask;
              if constexpr (!MATRIX) {
                p.senders[ev[q]] = i;
                p.mask[ev[q]] = 1;
              }
            }
          }
        }
      };
      if (lds_bits)
        write_ordinals([&](int w) { return sbits[sub][w][lane]; }, std::integral_constant<int, 4>{});
      else
        write_ordinals([&](int w) { return p.bits[static_cast<long>(w) * p.pitch + ii]; },
                       std::integral_constant<int, 1>{});
    }
    __syncthreads();
  }
}

// The pack alone (two-sided and LJ steps; no model in the loop) of rows of up to 256 slots: one
// 64-row tile per block of eight waves, wave w walking the slots w, w + 8, ... of every row. What
// bounds it is the round trips of the walk (a list entry, then its neighbour's position), so four
// slots go at a time: their records gather together while the next four entries load, and every
// load is unconditional, so waiting for one never waits for a later one. The walked neighbours
// stay in LDS for the compacted write: read from memory again, each batch's loads wait for the
// stores of the batch before (one counter retires both in order). Blocks of one tile instead of
// four overlap one tile's walk with another's write, and small lists reach more CUs; eight waves
// against four halve the rounds of a tile. us before (k_step_pack's 4 tiles of 4 waves) and after:
//   1,024 atoms LJ float64 21 -> 9.8            1,048,576 atoms half list float32 292 -> 238
//   8,192 atoms half list float64 24 -> 10.7    262,144 atoms LJ with ghost rows float32 169 -> 131
//   131,072 atoms half list float64 53 -> 35    (about 2.5 TB/s of list and packed edges)
// Measured beside it: two slots at a time 254 and 140 (the last two float32 cases), sixteen waves
// 319 and 153, the edges compacted in LDS and stored 16 bytes at a time 238 and 131. Four waves take
// 226 and 147: rows of 48 slots (the half list) gain less by them than rows of 78 lose.
constexpr int kPackW = 8;      // waves per tile
constexpr int kPackU = 4;      // slots of a row in flight per wave
constexpr int kPackKeep = 128; // slots whose neighbours stay in LDS: 32 KB, four blocks per CU

template <typename S>
__global__ __launch_bounds__(kPackW * kWave) __attribute__((amdgpu_waves_per_eu(8))) LK_EIGHT_WAVES
void k_pack_rows(StepPack p, const Atom4<S> *__restrict__ atoms, int nlocal,
                 double *__restrict__ partials, int ntiles)
{
  constexpr int W = kPackW, U = kPackU, KEEP = kPackKeep;
  static_assert(32 % (W * U) == 0, "a round's slots lie in one validity word");
  __shared__ int sent[KEEP][kWave];  // the neighbours of the walked slots
  __shared__ uint32_t sbits[kStepMaxWords][kWave];
  __shared__ int sbase;
  if constexpr (sizeof(S) == 8) {
    // the atom records for the sweeps (cpp:35-52: x as is, species = type - 1)
    if (p.atoms_out)
      for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < p.records;
           i += gridDim.x * blockDim.x) {
        const int sp = p.type[i] - 1;
        Atom4<double> r;
        r.x = p.x[3L * i + 0];
        r.y = p.x[3L * i + 1];
        r.z = p.x[3L * i + 2];
        r.w = static_cast<double>(sp);
        p.atoms_out[i] = r;
        p.species_out[i] = sp;
      }
  }
  const int tile = tile_of_block();
  if (tile >= ntiles) return;  // whole block
  const int wave = wave_in_block();
  const int lane = threadIdx.x & (kWave - 1);
  const int ii = tile * kWave + lane;
  const bool row = ii < p.num_rows;
  int i = -1, nn = 0;
  if (row) {
    i = p.ilist[ii];
    if (i < p.max_atoms)
      nn = min(p.numneigh[i], p.maxneighs);
    else
      i = -1;  // cpp:84: rows past max_atoms pack nothing
  }
  const int nn_max = wave_max_int(nn);
  const int nwords = (nn_max + 31) >> 5;  // at most kStepMaxWords (launch_pack_rows)
  for (int w = wave; w < nwords; w += W) sbits[w][lane] = 0u;
  double xi0 = 0.0, xi1 = 0.0, xi2 = 0.0;
  Atom4<float> xa{0.0f, 0.0f, 0.0f, 0.0f};
  if (i >= 0) {
    xi0 = p.x[3L * i + 0];
    xi1 = p.x[3L * i + 1];
    xi2 = p.x[3L * i + 2];
    if constexpr (sizeof(S) == 4) xa = atoms[i];
  }
  const float sa = fabsf(xa.x) + fabsf(xa.y) + fabsf(xa.z);
  __syncthreads();
  if (wave < nn_max) {
    // The row of a lane whose slots reach nn_max: every slot below it exists there, so a lane
    // past its own row reads that one (unused) and the loads need no branch.
    const int longest = __shfl(i, __builtin_ctzll(wave_ballot(nn == nn_max)), kWave);
    auto slot_entry = [&](int jj) -> int {
      const int at = min(jj, nn_max - 1);  // uniform
      const int *col = p.neighbors + static_cast<long>(at) * p.stride;
      return col[static_cast<unsigned>(at < nn ? i : longest)] & kNeighMask;
    };
    struct Near {
      double x0, x1, x2;
    };
    using Rec = std::conditional_t<sizeof(S) == 4, Atom4<float>, Near>;
    auto gather = [&](int jj, int j) -> Rec {
      const long q = (jj < nn && j < p.max_atoms) ? j : 0;
      if constexpr (sizeof(S) == 4) {
        return atoms[q];
      } else {
        Near r;
        r.x0 = p.x[3 * q + 0];
        r.x1 = p.x[3 * q + 1];
        r.x2 = p.x[3 * q + 2];
        return r;
      }
    };
    int e[U];
#pragma unroll
    for (int q = 0; q < U; ++q) e[q] = slot_entry(wave + q * W);
    for (int jj = wave; jj < nn_max; jj += U * W) {
      Rec r[U];
      int ne[U];
#pragma unroll
      for (int q = 0; q < U; ++q) r[q] = gather(jj + q * W, e[q]);
#pragma unroll
      for (int q = 0; q < U; ++q) ne[q] = slot_entry(jj + (U + q) * W);
      uint32_t part = 0;
#pragma unroll
      for (int q = 0; q < U; ++q) {
        const int slot = jj + q * W, j = e[q];
        bool keep = slot < nn && j < p.max_atoms;
        if constexpr (sizeof(S) == 4) {
          if (keep) keep = pack_keeps_f32(p, xa, sa, r[q], j, xi0, xi1, xi2);
        } else {
#pragma clang fp contract(off)
          const double dx = xi0 - r[q].x0, dy = xi1 - r[q].x1, dz = xi2 - r[q].x2;
          // PackNeighborFunctor keeps rsq <= cutsq (cpp:84-101)
          keep = keep && !(dx * dx + dy * dy + dz * dz > p.cutsq);
        }
        part |= keep ? 1u << (slot & 31) : 0u;
        if (slot < KEEP) sent[slot][lane] = j;
        e[q] = ne[q];
      }
      if (part) atomicOr(&sbits[jj >> 5][lane], part);
    }
  }
  __syncthreads();
  int c = 0;
  for (int w = 0; w < nwords; ++w) c += __popc(sbits[w][lane]);
  const int total = wave_sum(c);
  if (wave == 0) {
    if (row) {
      p.row_count[ii] = c;
      p.row_atom[ii] = i;
    }
    const uint64_t gmask = wave_ballot(i >= nlocal && c > 0);
    if (lane == 0) {
      // the tile's slots [base, base + total): one claim per tile (cpp:102-110 claims per entry)
      const int base = atomicAdd(&p.state[kDemand], total);
      sbase = base;
      p.tile_base[tile] = base;
      if (gmask != 0) atomicOr(&p.state[kGhostFlag], 1);
      put_partial(partials + 8L * tile + 0, 0.0);
    }
  }
  if (row)
    for (int w = wave; w < nwords; w += W)
      p.bits[static_cast<long>(w) * p.pitch + ii] = sbits[w][lane];
  // Compacted write, as k_step_pack's: wave w writes one contiguous range of ordinals.
  const int kmax = wave_max_int(c);
  const int per = (kmax + W - 1) / W;
  const int k0 = min(wave * per, kmax);
  const int k1 = min(k0 + per, kmax);
  int cursor = wave_sum(min(c, k0));
  int wd = 0;
  uint32_t word = 0;
  if (k0 < c) {
    word = sbits[0][lane];
    int skip = k0;
    while (skip > 0) {
      const int pc = __popc(word);
      if (pc <= skip) {  // the k0-th entry lies in a later word
        skip -= pc;
        word = sbits[++wd][lane];
      } else {
        for (; skip > 0; --skip) word &= word - 1u;
      }
    }
  }
  __syncthreads();
  const int base = sbase;
  constexpr int B = 4;
  for (int k = k0; k < k1; k += B) {
    int jv[B], ev[B];
#pragma unroll
    for (int q = 0; q < B; ++q) {
      const bool active = k + q < k1 && k + q < c;
      const uint64_t M = wave_ballot(active);
      const int at = base + cursor + lanes_below(M);
      cursor += __popcll(M);
      ev[q] = active && at < p.max_edges ? at : -1;  // past the capacity the count is the demand
      jv[q] = 0;
      if (active) {
        while (word == 0) word = sbits[++wd][lane];
        const int jj = wd * 32 + __builtin_ctz(word);
        word &= word - 1u;
        jv[q] = jj < KEEP ? sent[jj][lane]
                          : p.neighbors[static_cast<long>(jj) * p.stride + i] & kNeighMask;
      }
    }
#pragma unroll
    for (int q = 0; q < B; ++q) {
      if (ev[q] >= 0) {
        p.receivers[ev[q]] = jv[q];
        p.senders[ev[q]] = i;
        p.mask[ev[q]] = 1;
      }
    }
  }
}

// Lists with room for more than 256 slots, whose validity words LDS might not hold, take k_step_pack
// at eight waves of dealt slots, also where their rows are shorter. LJ steps with such room, us, at
// four waves of whole words before and now: 1,024 atoms float64 36.7 -> 29.7, 32,000 float32
// 51.5 -> 45.4, 131,072 float64 124.7 -> 115.8 and float32 102.0 -> 95.2.
template <typename S>
static void launch_pack_rows(Handle &h, hipStream_t s, const StepPack &p, const EamArgs<S> &a,
                             int ntiles)
{
  if (p.maxneighs <= 32 * kStepMaxWords) {
    hipLaunchKernelGGL((k_pack_rows<S>), dim3(tile_grid(ntiles)), dim3(kPackW * kWave), 0, s, p,
                       a.atoms, a.nlocal, a.partials, ntiles);
    return;
  }
  constexpr int W = 8, TPB = kStepWaves / W;
  const int ngroups = (ntiles + TPB - 1) / TPB;
  hipLaunchKernelGGL((k_step_pack<S, false, false, W>),
                     dim3(step_pack_grid<false>(ngroups, h.num_cus)), dim3(kStepWaves * kWave), 0,
                     s, p, a, ngroups);
}

// Starts a pack without the atom records (matrix bundles, whose records come from a separate
// lk_pack_atoms): zeroes the demand count and the ghost-sender flag.
__global__ void k_clear_state(int *state)
{
  if (threadIdx.x == 0) {
    state[kDemand] = 0;
    state[kGhostFlag] = 0;
  }
}

// Starts a fused pack whose atom records another launch writes: what the atom-record launch does
// to the pack state (the live count of the previous pack bounds this one's tail reset; zero
// claims, no ghost sender).
__global__ void k_start_pack(int *state)
{
  if (threadIdx.x == 0) {
    state[kPrevLive] = state[kLive];
    state[kDemand] = 0;
    state[kGhostFlag] = 0;
  }
}

template <typename S, bool EAM, bool MATRIX>
static hipError_t step_onesided(Handle &h, hipStream_t s, const double *x, const int *type,
                                int nall, const int *ilist, const int *numneigh,
                                const int *neighbors, long stride, int num_rows, int maxneighs,
                                int nlocal, int nghost, int flags, double scale, double *f,
                                bool atoms, bool split = false)
{
  h.packed_rows = num_rows;
  EamArgs<S> a{};
  if constexpr (EAM) {
    a = eam_args<S>(h, nlocal, scale, f);
  } else {
    a.atoms = static_cast<const Atom4<S> *>(h.d_atoms);
    a.partials = h.d_partials;
    a.nlocal = nlocal;
  }
  StepPack p;
  p.x = x;
  p.type = type;
  p.ilist = ilist;
  p.numneigh = numneigh;
  p.neighbors = neighbors;
  p.stride = stride;
  p.num_rows = num_rows;
  p.maxneighs = maxneighs;
  p.max_atoms = h.contract.max_atoms;
  p.max_edges = h.contract.max_edges;
  set_pack_cutoff(p, h.contract.cutoff);
  p.pitch = h.contract.max_atoms;
  p.bits = h.d_bits;
  p.row_count = h.d_row_count;
  p.row_atom = h.d_row_atom;
  p.tile_base = h.d_tile_off;
  p.state = h.d_pack_state;
  p.senders = h.d_senders;
  p.receivers = h.d_receivers;
  p.mask = h.d_mask;
  // split: the engine's exchange of rho between the passes gives the ghost rows their F'
  p.ghost_off = nghost > 0 && !split ? h.d_ghost_off : nullptr;
  p.ghost_list = h.d_ghost_list;
  p.atoms_out = nullptr;
  p.species_out = nullptr;
  p.records = 0;
  const int ntiles = (num_rows + kWave - 1) / kWave;
  // float64 EAM over an engine list: the pack and density over tile lists (lk_tiles.hip)
  bool tiled = false;
  if constexpr (EAM && !MATRIX && sizeof(S) == 8) tiled = tile_step_eligible(h, num_rows, maxneighs);
  const int records = atoms ? (nall < h.contract.max_atoms ? nall : h.contract.max_atoms) : 0;
  const bool ready = h.pack_ready;
  h.pack_ready = false;  // until this step's force sweep is enqueued
  if (tiled && atoms) {
    // The tile kernel writes the atom records itself, and the last block of the previous fused
    // step left the pack state as the record launch would (h.pack_ready); a launch less per step.
    if (!ready) hipLaunchKernelGGL(k_start_pack, dim3(1), dim3(64), 0, s, h.d_pack_state);
  } else if (atoms) {
    // K0: atom records and species; zeroes the demand counter and the ghost-sender flag
    if (hipError_t e0 = launch_pack_atoms(h, s, x, type, nall, h.d_pack_state); e0 != hipSuccess)
      return e0;
  } else {
    // the records of a separate lk_pack_atoms call
    hipLaunchKernelGGL(k_clear_state, dim3(1), dim3(64), 0, s, h.d_pack_state);
  }
  const bool nonrows = EAM && h.nonrow_blocks > 0;  // the list misses owned atoms
  if (nonrows)
    if (hipError_t e = launch_mark_rows(h, s, ilist, num_rows, nlocal); e != hipSuccess) return e;
  if constexpr (EAM && !MATRIX && sizeof(S) == 8) {
    if (tiled)
      if (hipError_t e1 = launch_step_tiles(h, s, x, type, ilist, numneigh, neighbors, stride,
                                            num_rows, maxneighs, nlocal, nghost, a,
                                            tiled && atoms ? records : 0, !split);
          e1 != hipSuccess)
        return e1;
  }
  if (ntiles > 0 && !tiled) {
    StageTimer timer(h, s, "step_pack");
    if constexpr (!EAM) {
      launch_pack_rows<S>(h, s, p, a, ntiles);
    } else {
      auto launch = [&](auto waves) {
        constexpr int W = decltype(waves)::value, TPB = kStepWaves / W;
        const int groups = (ntiles + TPB - 1) / TPB;
        hipLaunchKernelGGL((k_step_pack<S, EAM, MATRIX, W>),
                           dim3(step_pack_grid<EAM>(groups, h.num_cus)), dim3(kStepWaves * kWave),
                           0, s, p, a, groups);
      };
      // float32: sixteen waves per tile while the tiles fill two blocks per CU, eight past that; us by
      // waves per tile 2, 4, 8, 16 (packed edges; four were used at every size before)
      //   16 tiles (1,008 atoms)  49, 33, 22, 17*   1,024 tiles (65,536)   68, 49, 41*, 45
      //   465 tiles (29,716)      58, 38, 28, 26*   2,048 tiles (131,072)  85, 75, 73*, 79
      // float64, whose walk is one slot at a time and so waits longer for each: sixteen at every
      // size; step in us by 8 and 16 (neighbour matrix; packed edges without a list epoch come
      // within 1.5 us of it)
      //   16 tiles (1,024 atoms)  46.7, 39.2*   1,024 tiles (65,536)    99.9, 98.7*
      //   128 tiles (8,192)       48.5, 41.6*   1,088 tiles (69,632)   133.5, 124.4*
      //   465 tiles (29,716)      61.2, 57.5*   2,048 tiles (131,072)  163.9, 159.3*
      // (four waves of whole 32-slot words before: 98, 102, 113, 132, 166 and 169).
      if constexpr (sizeof(S) == 8)
        launch(std::integral_constant<int, 16>{});
      else if (ntiles <= 2 * (h.num_cus > 0 ? h.num_cus : 256))
        launch(std::integral_constant<int, 16>{});
      else
        launch(std::integral_constant<int, 8>{});
    }
  }
  ++h.pack_serial;
  FusedPack fp;
  // matrix bundles keep the copy's widest row and overflow flag as the step's counts
  fp.state = MATRIX ? nullptr : h.d_pack_state;
  fp.senders = h.d_senders;
  fp.receivers = h.d_receivers;
  fp.mask = h.d_mask;
  fp.max_edges = h.contract.max_edges;
  fp.pad = h.contract.max_atoms;
  if constexpr (EAM) {
    if (nonrows)
      if (hipError_t e = launch_embed_nonrows(h, s, nlocal, nghost > 0 && !split);
          e != hipSuccess)
        return e;
    if (split) {  // the force pass (lk_model_force) finishes the pack
      h.split_pack = fp;
      return hipGetLastError();
    }
    a.pack = fp;
    hipError_t e = launch_eam_force(h, s, a, flags);
    // its last block resets the pack state for the next fused pack (finalize_last_block)
    h.pack_ready = e == hipSuccess && fp.state != nullptr;
    return e;
  }
  return launch_lj_onesided(h, s, nlocal, nghost, scale, f, flags, fp);
}

template <typename S>
static hipError_t pack_fused(Handle &h, hipStream_t s, const double *x, const int *type, int nall,
                             const int *ilist, const int *numneigh, const int *neighbors,
                             long stride, int num_rows, int maxneighs, int nlocal, FusedPack *out)
{
  h.packed_rows = num_rows;
  EamArgs<S> a{};
  a.atoms = static_cast<const Atom4<S> *>(h.d_atoms);
  a.partials = h.d_partials;
  a.nlocal = nlocal;
  StepPack p{};
  p.x = x;
  p.type = type;
  p.ilist = ilist;
  p.numneigh = numneigh;
  p.neighbors = neighbors;
  p.stride = stride;
  p.num_rows = num_rows;
  p.maxneighs = maxneighs;
  p.max_atoms = h.contract.max_atoms;
  p.max_edges = h.contract.max_edges;
  set_pack_cutoff(p, h.contract.cutoff);
  p.pitch = h.contract.max_atoms;
  p.bits = h.d_bits;
  p.row_count = h.d_row_count;
  p.row_atom = h.d_row_atom;
  p.tile_base = h.d_tile_off;
  p.state = h.d_pack_state;
  p.senders = h.d_senders;
  p.receivers = h.d_receivers;
  p.mask = h.d_mask;
  p.ghost_off = nullptr;  // no model: nothing to forward
  p.ghost_list = nullptr;
  const int ntiles = (num_rows + kWave - 1) / kWave;
  // float64: the pack kernel writes the atom records itself, and the previous fused step's last
  // block left the pack state as the record launch would (h.pack_ready), else one block resets
  // it. float32 filters from the records (pack_keeps_f32), so they come first.
  const bool ready = h.pack_ready;
  h.pack_ready = false;
  if (sizeof(S) == 8 && ntiles > 0) {
    if (!ready) hipLaunchKernelGGL(k_start_pack, dim3(1), dim3(64), 0, s, h.d_pack_state);
    p.atoms_out = static_cast<Atom4<double> *>(h.d_atoms);
    p.species_out = h.d_species;
    p.records = nall < h.contract.max_atoms ? nall : h.contract.max_atoms;
  } else if (hipError_t e0 = launch_pack_atoms(h, s, x, type, nall, h.d_pack_state);
             e0 != hipSuccess) {
    return e0;
  }
  if (ntiles > 0) {
    StageTimer timer(h, s, "step_pack");
    launch_pack_rows<S>(h, s, p, a, ntiles);
  }
  ++h.pack_serial;
  out->state = h.d_pack_state;
  out->senders = h.d_senders;
  out->receivers = h.d_receivers;
  out->mask = h.d_mask;
  out->max_edges = h.contract.max_edges;
  out->pad = h.contract.max_atoms;
  return hipGetLastError();
}

hipError_t launch_pack_fused(Handle &h, hipStream_t s, const double *x, const int *type, int nall,
                             const int *ilist, const int *numneigh, const int *neighbors,
                             long stride, int num_rows, int maxneighs, int nlocal,
                             FusedPack *out)
{
  if (h.contract.precision == LK_FLOAT64)
    return pack_fused<double>(h, s, x, type, nall, ilist, numneigh, neighbors, stride, num_rows,
                              maxneighs, nlocal, out);
  return pack_fused<float>(h, s, x, type, nall, ilist, numneigh, neighbors, stride, num_rows,
                           maxneighs, nlocal, out);
}

hipError_t launch_step_density(Handle &h, hipStream_t s, const double *x, const int *type,
                               int nall, const int *ilist, const int *numneigh,
                               const int *neighbors, long stride, int num_rows, int maxneighs,
                               int nlocal, int nghost)
{
  if (h.contract.precision == LK_FLOAT64)
    return step_onesided<double, true, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                              stride, num_rows, maxneighs, nlocal, nghost, 0, 1.0,
                                              nullptr, true, true);
  return step_onesided<float, true, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                           stride, num_rows, maxneighs, nlocal, nghost, 0, 1.0,
                                           nullptr, true, true);
}

hipError_t launch_step_onesided(Handle &h, hipStream_t s, const double *x, const int *type,
                                int nall, const int *ilist, const int *numneigh,
                                const int *neighbors, long stride, int num_rows, int maxneighs,
                                int nlocal, int nghost, int flags, double scale, double *f,
                                bool matrix, bool atoms)
{
  const bool f64 = h.contract.precision == LK_FLOAT64;
  const bool eam = h.model == 1;
  if (matrix) {  // the matrix bundles are EAM row models
    if (f64)
      return step_onesided<double, true, true>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                               stride, num_rows, maxneighs, nlocal, nghost, flags,
                                               scale, f, atoms);
    return step_onesided<float, true, true>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                            stride, num_rows, maxneighs, nlocal, nghost, flags,
                                            scale, f, atoms);
  }
  if (f64 && eam)
    return step_onesided<double, true, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                              stride, num_rows, maxneighs, nlocal, nghost, flags,
                                              scale, f, atoms);
  if (f64)
    return step_onesided<double, false, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                               stride, num_rows, maxneighs, nlocal, nghost, flags,
                                               scale, f, atoms);
  if (eam)
    return step_onesided<float, true, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                             stride, num_rows, maxneighs, nlocal, nghost, flags,
                                             scale, f, atoms);
  return step_onesided<float, false, false>(h, s, x, type, nall, ilist, numneigh, neighbors,
                                            stride, num_rows, maxneighs, nlocal, nghost, flags,
                                            scale, f, atoms);
}

}  // namespace lk
