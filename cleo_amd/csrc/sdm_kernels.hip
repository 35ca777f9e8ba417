// sdm_kernels.hip -- gfx950 kernels of the super-droplet step.
//
// Launch shapes: a thread per drop, or a wave64 per gridbox or few (with a capped grid each wave loops
// over gridboxes g, g + (waves in the grid), ...).  Drops of a gridbox are contiguous in the SoA store
// (sorted by sdgbxindex), so every per-drop load and store of a wave is a coalesced run.  No kernel
// uses atomics on drop data: sums keep the reference's sequential order and the sort is stable by
// construction.
#include <algorithm>
#include <cmath>

#include "kernels.hpp"
#include "sdm_kernels.hpp"

namespace cleo {

// ============================ per-gridbox sums ================================================
// A wave sums a tile of `gpt` consecutive gridboxes, one per lane (at most 64).  Its lanes add their
// gridboxes' values one after the other, so a tile takes the time of its drops' loads plus its longest
// sum; tiles of 64 gridboxes leave most of the chip idle below half a million gridboxes (sum_gpt).
__host__ __device__ __forceinline__ uint32_t sum_tiles(uint32_t ngbx, uint32_t gpt) { return (ngbx + gpt - 1) / gpt; }
// acc[c] + v[c][i0] + v[c][i0+1] + ... + v[c][i1-1] for N value sequences, each left to right.  Eight
// LDS reads of each are in flight while the eight before are added, and the sequences' adds alternate, so
// neither a read's 100 cycles nor an add's latency is waited for (one sequence after the other, with each
// eight reads waited for: k_cond_state 11.5 -> 10.5 us on 3750 gridboxes of 128 drops).
template <int N, class T>
__device__ __forceinline__ void add_in_order(T* acc, const T* const* v, uint32_t i0, uint32_t i1) {
  constexpr uint32_t kAhead = 8;
  const uint32_t full = (i1 - i0) / kAhead;
  T r[N][kAhead], next[N][kAhead];
  auto load = [&](uint32_t i, T(&to)[N][kAhead]) {
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j)
#pragma unroll
      for (int c = 0; c < N; ++c) to[c][j] = v[c][i + j];
  };
  auto add = [&](T(&from)[N][kAhead]) {
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j)
#pragma unroll
      for (int c = 0; c < N; ++c) acc[c] += from[c][j];
  };
  uint32_t i = i0;
  if (full) load(i, r);
  for (uint32_t k = 0; k < full; k += 2) {  // two eights per turn: no register moves
    if (k + 1 < full) load(i + kAhead, next);
    add(r);
    i += kAhead;
    if (k + 1 < full) {
      if (k + 2 < full) load(i + kAhead, r);
      add(next);
      i += kAhead;
    }
  }
  for (; i < i1; ++i)
#pragma unroll
    for (int c = 0; c < N; ++c) acc[c] += v[c][i];
}
// Drop-order sums of v(k) over [lo, lo + len) for the gridboxes of a tile (lane i passes its
// own gridbox's range and gets its sum).  The tile's drops [t_lo, t_hi) are staged through an LDS
// window of kSumWin values with coalesced loads (the next window's loads in flight while the current
// one is added); each lane then adds its gridbox's values left to right, exactly as a serial loop
// does (the reference's sums run in drop order under Serial).
template <class V>
__device__ __forceinline__ double tile_sum(double* win, uint32_t t_lo, uint32_t t_hi, uint32_t lo, uint32_t len, V v,
                                           int lane) {
  constexpr uint32_t kPer = kSumWin / kWave;
  double acc = 0.0;
  if (t_lo >= t_hi) return acc;
  // the next window's values are loaded into registers while the lanes add the current one's
  // (every lane loads, with indices clamped into the tile, so the loads stay in flight)
  double r[kPer];
  auto load = [&](uint32_t w) {
    for (uint32_t i = 0; i < kPer; ++i) r[i] = v(min(w + static_cast<uint32_t>(lane) + i * kWave, t_hi - 1u));
  };
  load(t_lo);
  for (uint32_t w = t_lo; w < t_hi; w += kSumWin) {
    const uint32_t we = min(w + kSumWin, t_hi);
    for (uint32_t i = 0; i < kPer; ++i) win[static_cast<uint32_t>(lane) + i * kWave] = r[i];
    wave_sync();
    if (we < t_hi) load(we);
    const uint32_t a0 = max(lo, w), a1 = min(lo + len, we);
    const double* const v1[1] = {win};
    if (a0 < a1) add_in_order<1>(&acc, v1, a0 - w, a1 - w);
    wave_sync();
  }
  return acc;
}
// The same for two value sequences at once (each summed left to right on its own): half the window
// each, one pass over the tile.
template <class V1, class V2>
__device__ __forceinline__ void tile_sum2(double* win, uint32_t t_lo, uint32_t t_hi, uint32_t lo, uint32_t len, V1 v1,
                                          V2 v2, int lane, double& s1, double& s2) {
  constexpr uint32_t kHalf = kSumWin / 2, kPer = kHalf / kWave;
  double acc[2] = {0.0, 0.0};
  s1 = s2 = 0.0;
  if (t_lo >= t_hi) return;
  // the next window's values are loaded into registers while the lanes add the current one's
  // (every lane loads, with indices clamped into the tile, so the loads stay in flight)
  double r1[kPer], r2[kPer];
  auto load = [&](uint32_t w) {
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t k = min(w + static_cast<uint32_t>(lane) + i * kWave, t_hi - 1u);
      r1[i] = v1(k);
      r2[i] = v2(k);
    }
  };
  load(t_lo);
  for (uint32_t w = t_lo; w < t_hi; w += kHalf) {
    const uint32_t we = min(w + kHalf, t_hi);
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t j = static_cast<uint32_t>(lane) + i * kWave;
      win[j] = r1[i];
      win[kHalf + j] = r2[i];
    }
    wave_sync();
    if (we < t_hi) load(we);
    const uint32_t b0 = max(lo, w), b1 = min(lo + len, we);
    const double* const v[2] = {win, win + kHalf};
    if (b0 < b1) add_in_order<2>(acc, v, b0 - w, b1 - w);
    wave_sync();
  }
  s1 = acc[0];
  s2 = acc[1];
}
// The same for N (one or two) value sequences and tiles of kRows gridboxes, with the next kRowLen values of
// every gridbox in the window at a time, so that all of the tile's lanes add.  A contiguous window holds
// the values of a gridbox or two once they have hundreds of drops, and LDS reads, which take the same time
// for two lanes as for 64, then bound the sums.  Rows of odd length keep the lanes' reads in different
// banks.
constexpr uint32_t kRows = 16;
template <int N, class V>
__device__ __forceinline__ void tile_rows_sum(double* win, uint32_t t_lo, uint32_t lo, uint32_t len, V v, int lane,
                                              double* acc) {
  constexpr uint32_t kHalf = kSumWin / 2, kRowLen = kHalf / kRows - 1, kPer = kHalf / kWave;
  static_assert(N <= 2 && kRowLen % 2 == 1 && kRows * kRowLen <= kHalf, "rows of the window");
  uint32_t most = len;
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), o)));
  if (most == 0) return;
  uint32_t first[kPer], left[kPer];  // this lane's items: the drop of the first window, the values from it on
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    const uint32_t j = static_cast<uint32_t>(lane) + i * kWave, row = min(j / kRowLen, kRows - 1u), at = j - row * kRowLen;
    const uint32_t n = static_cast<uint32_t>(__shfl(static_cast<int>(len), static_cast<int>(row)));
    first[i] = static_cast<uint32_t>(__shfl(static_cast<int>(lo), static_cast<int>(row))) + at;
    left[i] = at < kRowLen && at < n ? n - at : 0u;
  }
  double r[N][kPer];
  auto load = [&](uint32_t w) {  // every lane loads, from the tile's first drop where there is no value
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t k = w < left[i] ? first[i] + w : t_lo;
#pragma unroll
      for (int c = 0; c < N; ++c) r[c][i] = v(c, k);
    }
  };
  load(0u);
  for (uint32_t w = 0; w < most; w += kRowLen) {
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i)
#pragma unroll
      for (int c = 0; c < N; ++c) win[c * kHalf + static_cast<uint32_t>(lane) + i * kWave] = r[c][i];
    wave_sync();
    if (w + kRowLen < most) load(w + kRowLen);
    if (w < len) {
      const double* rows[N];
#pragma unroll
      for (int c = 0; c < N; ++c) rows[c] = win + c * kHalf + static_cast<uint32_t>(lane) * kRowLen;
      add_in_order<N>(acc, rows, 0u, min(kRowLen, len - w));
    }
    wave_sync();
  }
}
// condensed water of drop k (condensate_mass * xi, superdrop_attrs.hpp:207-216)
__device__ __forceinline__ double qcond_term(const SoA& s, const Solute& sol, DevCtl* ctl, uint32_t k) {
  bool bad = false;
  const double m = condensate_mass(s.r[k], s.msol[k], sol, &bad) * static_cast<double>(s.xi[k]);
  if (bad) set_error(ctl, CLEO_ERR_NEG_CONDENSATE, s.gbx[k], k);
  return m;
}

// ============================ qcond ===========================================================
// EffectOnHydrometeorStatesFunctor (movesupersindomain.hpp:95-136), standalone: 64 gridboxes per
// wave, drop-order sums of condensed mass, then one lane per gridbox for its qcond
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(4) k_qcond(QcondArgs a) {
  __shared__ double win_all[4][kSumWin];
  double* win = win_all[threadIdx.x >> 6];
  const int lane = lane_id();
  const uint32_t gpt = a.gpt, ntiles = sum_tiles(a.ngbx, gpt);
  for (uint32_t tile = wave_index(); tile < ntiles; tile += wave_count()) {
    const uint32_t g0 = tile * gpt, g = g0 + static_cast<uint32_t>(lane);
    const bool valid = static_cast<uint32_t>(lane) < gpt && g < a.ngbx;
    const uint32_t t_lo = a.off[g0], t_hi = a.off[min(g0 + gpt, a.ngbx)];
    const uint32_t lo = valid ? a.off[g] : t_hi, hi = valid ? a.off[g + 1] : t_hi;
    const double tot = tile_sum(win, t_lo, t_hi, lo, hi - lo, [&](uint32_t k) { return qcond_term(a.s, a.sol, a.ctl, k); },
                                lane);
    if (valid) {
      const double rho_cond = tot / a.st.vol[g] * dimless::R0cubed_VOL0;
      const double rho_dry = dry_air_density(a.st.press[g], a.st.temp[g], a.st.qv[g]);
      a.st.qc[g] = rho_cond / rho_dry;
    }
  }
}

// ============================ collisions ======================================================
// DoCollisions::do_collisions (collisions.hpp:140-278): Fisher-Yates shuffle of a gridbox's drops,
// pairs (2jj, 2jj+1) of the shuffled order, enactment, nulls moved behind the active drops
// (stable partition).  The drops stay where they are: the shuffled order is recorded in
// CollArgs::order (slot -> position) and only the attributes of enacted pairs are written, in
// place.  The reference moves every drop to its shuffled place; here the next sort moves each drop
// once, to its sorted place in that order.
// word t%4 of a block (selected without indexing the array by a lane-varying value)
__device__ __forceinline__ uint32_t rng_word(const uint32_t r4[4], uint32_t t) {
  const uint32_t w = t & 3u;
  return w == 0u ? r4[0] : (w == 1u ? r4[1] : (w == 2u ? r4[2] : r4[3]));
}
// uniform u32 -> index in [0, iter]
__device__ __forceinline__ uint32_t fy_scale(uint32_t u, uint32_t iter) {
  return static_cast<uint32_t>((static_cast<uint64_t>(u) * (iter + 1ull)) >> 32);
}
// The index j_t of Fisher-Yates swap t < n-1 of gridbox g is uniform in [0, iter], iter = n-1-t
// (shuffle.hpp:80-87): from the counter stream, word t%4 of the block for item t/4 (one block serves
// four consecutive swaps), or an injected index
__device__ __forceinline__ uint32_t inj_index(const CollArgs& a, uint32_t g, uint32_t base, uint32_t n, uint32_t t) {
  const uint32_t iter = n - 1 - t;
  uint32_t j = a.inj_j[a.inj_oj[g] + t];
  if (j > iter) {  // an injected index outside [0, iter] is an argument error
    set_error(a.ctl, CLEO_ERR_INJECTED_INDEX, g, base + iter);
    j = iter;
  }
  return j;
}

// position of the drop at slot `slot` of gridbox `base`'s logical order: through a pending order
// of an earlier event when there is one (the drops then stay where they are and the orders
// compose), else the slot itself
__device__ __forceinline__ uint32_t coll_pos(const CollArgs& a, uint32_t base, uint32_t slot) {
  return a.order_in ? a.order_in[base + slot] : base + slot;
}

// One collision pair (2jj, 2jj+1) of gridbox g (n active drops) from the drops at ka, kb
// (collisions.hpp:180-230): probability and enactment on (xi, r, msol) of both drops.
struct PairOut {
  DropAttrs A, B;  // the drops at ka and kb after the enactment
  bool nullA, nullB;
  bool enacted;
  int err;
};
template <bool Kinetic>
__device__ __forceinline__ PairOut coll_pair_eval(const CollArgs& a, uint32_t g, uint32_t n, uint32_t jj, uint32_t ka,
                                                  uint32_t kb, uint64_t event) {
  const uint32_t npairs = n / 2;
  const double scale_p = n * (n - 1.0) / (2.0 * npairs);
  const double VOLUME = a.vol[g] * dimless::VOL0;
  PairOut o{};
  const uint64_t xiA = a.s.xi[ka], xiB = a.s.xi[kb];
  const double rA = a.s.r[ka], rB = a.s.r[kb];
  const bool a_first = !(xiA < xiB);  // assign_drops (collisions.hpp:94-101)
  // d1 is the drop with the larger multiplicity; selected field by field (a reference picked by a
  // lane-varying flag would put both drops in scratch memory)
  DropAttrs d1{a_first ? xiA : xiB, a_first ? rA : rB, 0.0};
  DropAttrs d2{a_first ? xiB : xiA, a_first ? rB : rA, 0.0};
  const double prob_jk = pair_probability<Kinetic>(a.k, d1.r, d2.r, VOLUME);
  const double prob = scale_p * static_cast<double>(d1.xi) * prob_jk;
  double phi_coll, phi_out;
  if (a.inj_phi) {
    const uint64_t q = a.inj_op[g] + 2ull * jj;
    phi_coll = a.inj_phi[q];
    phi_out = a.inj_phi[q + 1];
  } else {
    uint32_t r4[4];
    rng_block(a.seed, event, 1u, g, jj, r4);
    phi_coll = u53(r4[0], r4[1]);
    phi_out = u53(r4[2], r4[3]);
  }
  // nothing happens to most pairs (fewer than 1e-4 of the coupled populations' are enacted, 3e-3 of the
  // Golovin box's): no conversions, no 64-bit division, and the solute masses are not read (k_coll_tiles on
  // 33.5M drops 299 -> 252 us, k_coll_team on 24679 gridboxes of 300 135 -> 125)
  if (prob >= 0.0 && prob < 1.0 && !(phi_coll < prob)) return o;
  const double mA = a.s.msol[ka], mB = a.s.msol[kb];
  d1.msol = a_first ? mA : mB;
  d2.msol = a_first ? mB : mA;
  const uint32_t res = enact_pair<Kinetic>(a.k, d1, d2, prob, phi_coll, phi_out, a.sol, o.err);
  o.enacted = (res >> 1) & 1u;
  o.nullA = (res & 1u) && a_first;
  o.nullB = (res & 1u) && !a_first;
  o.A = DropAttrs{a_first ? d1.xi : d2.xi, a_first ? d1.r : d2.r, a_first ? d1.msol : d2.msol};
  o.B = DropAttrs{a_first ? d2.xi : d1.xi, a_first ? d2.r : d1.r, a_first ? d2.msol : d1.msol};
  return o;
}
// the attributes of drop k after an enacted pair, in place; a null drop gets the out-of-domain key
__device__ __forceinline__ void coll_store(const CollArgs& a, uint32_t k, const DropAttrs& D, bool isnull) {
  a.s.xi[k] = D.xi;
  a.s.r[k] = D.r;
  a.s.msol[k] = D.msol;
  if (isnull) a.s.gbx[k] = kOOB;
}
// pair jj of the drops at ka, kb: the slots 2jj, 2jj+1 of the logical order, and the new attributes
// when it was enacted; true when one of the two became null; `events` counts enactments
template <bool Kinetic>
__device__ __forceinline__ bool coll_pair(const CollArgs& a, uint32_t g, uint32_t base, uint32_t n, uint32_t jj,
                                          uint32_t ka, uint32_t kb, uint64_t event, uint32_t& events) {
  const PairOut o = coll_pair_eval<Kinetic>(a, g, n, jj, ka, kb, event);
  if (o.err) set_error(a.ctl, o.err, g, base + 2 * jj);
  a.order[base + 2 * jj] = ka;
  a.order[base + 2 * jj + 1] = kb;
  if (o.enacted) {
    events += 1u;
    coll_store(a, ka, o.A, o.nullA);
    coll_store(a, kb, o.B, o.nullB);
  }
  return o.nullA || o.nullB;
}

// remove_null_supers (collisions.hpp:240-248) for gridbox g after its pairs: the reference's
// sort_team is restated as a stable partition of the gridbox's logical order (active drops first,
// nulls behind, each in order).  The partitioned order is staged in the gridbox's HBM scratch
// (2 u32 per drop from big + 2 base, free once the shuffle is done) and copied back.  Only this
// wave reads what it stored, so a workgroup-scope fence orders it (an agent-scope fence would
// write back the XCD's whole L2).
__device__ __forceinline__ void coll_order_nulls(const CollArgs& a, uint32_t g, uint32_t base, uint32_t n,
                                                 uint32_t nulls, int lane) {
  __threadfence_block();
  wave_sync();
  uint32_t* tmp = a.big + 2ull * base;
  const uint32_t nn = n - nulls;
  uint32_t run_nn = 0, run_null = 0;
  for (uint32_t c = 0; c < n; c += kWave) {
    const uint32_t k = c + lane;
    const bool act = k < n;
    const uint32_t pk = act ? a.order[base + k] : 0u;
    const bool isnull = act && a.s.xi[pk] == 0;
    const uint64_t mnull = __ballot(isnull);
    const uint64_t mnn = __ballot(act && !isnull);
    if (act) {
      const uint32_t pos = isnull ? nn + run_null + __popcll(mnull & lanemask_lt())
                                  : run_nn + __popcll(mnn & lanemask_lt());
      tmp[pos] = pk;
    }
    run_null += __popcll(mnull);
    run_nn += __popcll(mnn);
  }
  __threadfence_block();
  wave_sync();
  for (uint32_t k = lane; k < n; k += kWave) a.order[base + k] = tmp[k];
  if (lane == 0) {
    a.nact[g] = nn;
    a.ctl->resort_flag = 1u;
  }
}

// exclusive prefix of v over the wave's lanes, and its total
__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v, int lane, uint32_t& total) {
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  total = readlane_u32(x, kWave - 1);
  return x - v;
}
// exclusive prefix of v over the workgroup's threads, and its total (ws: a word per wave)
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* ws, uint32_t& total) {
  uint32_t wt;
  const uint32_t x = wave_excl_scan(v, lane_id(), wt);
  const uint32_t w = threadIdx.x / kWave, nw = blockDim.x / kWave;
  __syncthreads();  // the previous scan is done with ws
  if (lane_id() == 0) ws[w] = wt;
  __syncthreads();
  uint32_t pre = 0;
  total = 0;
  for (uint32_t i = 0; i < nw; ++i) {
    pre += i < w ? ws[i] : 0u;
    total += ws[i];
  }
  return pre + x;
}
// record p of src to position q of dst
__device__ __forceinline__ void copy_drop(const SoA& src, const SoA& dst, uint64_t p, uint64_t q) {
  dst.gbx[q] = src.gbx[p];
  dst.c3[q] = src.c3[p];
  dst.c1[q] = src.c1[p];
  dst.c2[q] = src.c2[p];
  dst.xi[q] = src.xi[p];
  dst.r[q] = src.r[p];
  dst.msol[q] = src.msol[p];
  dst.id[q] = src.id[p];
}
// the i < cnt with pre[i] <= f < pre[i+1] (pre[0] <= f < pre[cnt])
__device__ __forceinline__ uint32_t tile_owner(const uint32_t* pre, uint32_t cnt, uint32_t f) {
  uint32_t lo = 0, hi = cnt;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (pre[mid] <= f)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}
// ============================ re-sort after collisions ========================================
// When collisions left nulls, SDMMethods sorts again: the active drops of each gridbox move together
// and the nulls of all gridboxes, in order, go behind the domain (before the drops that were out of it
// already, which keep their positions).  Everything below ends at once when there are no nulls, so that
// a captured graph needs no host decision.  It usually does end at once, so what it costs is launches
// (2.3 us each in a graph): two for large domains (k_resort_gather, k_resort_back), one workgroup for
// all of it up to kResortOneDrops drops, and none for a single gridbox, whose last collision event
// closes the pass itself (step of one gridbox of 8192 drops 47 -> 26 us, 15 of them by the shares below).
//
// The re-sort also advances the event counter past the events of this microphysics pass.
//
// Two passes over the drops: the first puts them in their order into the spare buffer, each at its own
// slot, the second moves them back to their final places, `nulls before` places further down.  Beside the
// first, each of up to kResortSegs workgroups counts the nulls of one segment of the gridboxes, and the
// second sums those of the segments before.  Both walk the store with one window of 256 workgroups: 1.80 ms
// for 33.5M drops of 64^3 gridboxes and 1.75 of 256x128x128 (120 bytes a pass, 4.6 TB/s), and with 512 or
// 2048 workgroups, a segment of the store each, or every field loaded before the first is stored, 2.0 to
// 2.8.  (Each workgroup summing the active counts of all gridboxes before its own, with a wave per gridbox,
// took 2.21 and 5.97 ms.)
struct Resort {
  DevCtl* ctl;
  SoA src, dst;
  uint32_t *off, *nact;
  uint32_t* pre;    // scratch, a word per gridbox: the nulls before it in its segment
  uint32_t* order;  // the pending order, or null: the store is in its logical order (a condensation applied it)
  uint32_t ngbx;
  uint32_t* code;   // scratch, a word per drop: at a null's slot, the nulls before it in its segment
  uint32_t* part;   // scratch, two words per segment: its nulls and its first slot
  uint32_t shift;   // segment of gridbox g: g >> shift
};
__device__ __forceinline__ void resort_begin(const Resort& r, uint32_t events, uint32_t flag) {
  r.ctl->event += events;
  r.ctl->resort_go = flag;
  r.ctl->resort_nsrc = r.off[r.ngbx];
  if (flag) r.ctl->stats[ST_SORTS] += 1;
}
// pre and code of the gridboxes [lo, hi) by the B lanes of a workgroup; returns their nulls
template <int B>
__device__ __forceinline__ uint32_t resort_count(const Resort& r, uint32_t lo, uint32_t hi, uint32_t tid) {
  __shared__ uint32_t ws[B / kWave];
  uint32_t run = 0, all;
  for (uint32_t g0 = lo; g0 < hi; g0 += B) {
    const uint32_t g = g0 + tid;
    uint32_t o = 0, n = 0;
    if (g < hi) {
      o = r.off[g] + r.nact[g];
      n = r.off[g + 1] - o;
    }
    const uint32_t before = run + block_excl_scan(n, ws, all);
    if (g < hi) r.pre[g] = before;
    for (uint32_t k = 0; k < n; ++k) r.code[o + k] = before + k;
    run += all;
  }
  return run;
}
__device__ __forceinline__ void resort_take(const Resort& r, uint32_t nsrc, uint64_t first, uint64_t stride) {
  for (uint64_t s = first; s < nsrc; s += stride) {
    const uint64_t p = r.order ? r.order[s] : s;
    if (p < nsrc) copy_drop(r.src, r.dst, p, s);
  }
}
// before[i]: nulls of the segments before segment i, start[i]: its first slot
__device__ __forceinline__ void resort_put(const Resort& r, uint32_t nsrc, uint32_t nulls, const uint32_t* before,
                                           const uint32_t* start, uint32_t nseg, uint64_t first, uint64_t stride) {
  for (uint64_t s = first; s < nsrc; s += stride) {
    const uint32_t g = r.dst.gbx[s];
    const uint32_t q = g < r.ngbx ? static_cast<uint32_t>(s) - before[g >> r.shift] - r.pre[g]
                                  : nsrc - nulls + before[tile_owner(start, nseg, static_cast<uint32_t>(s))] + r.code[s];
    if (q >= nsrc) continue;
    copy_drop(r.dst, r.src, s, q);
    if (r.order) r.order[q] = q;
  }
  for (uint64_t g = first; g < r.ngbx; g += stride) r.off[g] -= before[g >> r.shift] + r.pre[g];  // the active counts stay
  if (first == 0) r.off[r.ngbx] = nsrc - nulls;
}
// all of it by one workgroup
template <int B>
__device__ __forceinline__ void resort_alone(const Resort& r, uint32_t events, uint32_t tid) {
  __shared__ uint32_t zero;
  const uint32_t flag = r.ctl->resort_flag;
  __syncthreads();
  if (tid == 0) {
    zero = 0u;
    resort_begin(r, events, flag);
    r.ctl->resort_flag = 0u;
  }
  if (!flag) return;
  const uint32_t nsrc = r.off[r.ngbx], nulls = resort_count<B>(r, 0u, r.ngbx, tid);
  resort_take(r, nsrc, tid, B);
  __syncthreads();
  resort_put(r, nsrc, nulls, &zero, &zero, 1u, tid, B);
}
__global__ void __launch_bounds__(1024) k_resort_one(Resort r, uint32_t events) { resort_alone<1024>(r, events, threadIdx.x); }
constexpr int kResortLanes = 1024;
__global__ void __launch_bounds__(kResortLanes) k_resort_gather(Resort r, uint32_t events) {
  const uint32_t flag = r.ctl->resort_flag, tid = threadIdx.x, b = blockIdx.x;  // cleared by k_resort_back
  if (b == 0 && tid == 0) resort_begin(r, events, flag);
  if (!flag) return;
  const uint32_t lo = b << r.shift, hi = min(r.ngbx, (b + 1u) << r.shift);
  if (b < kResortSegs && lo < r.ngbx) {
    const uint32_t nulls = resort_count<kResortLanes>(r, lo, hi, tid);
    if (tid == 0) {
      r.part[2u * b] = nulls;
      r.part[2u * b + 1u] = r.off[lo];
    }
  }
  resort_take(r, r.off[r.ngbx], b * static_cast<uint64_t>(kResortLanes) + tid, static_cast<uint64_t>(gridDim.x) * kResortLanes);
}
__global__ void __launch_bounds__(kResortLanes) k_resort_back(Resort r) {
  if (!r.ctl->resort_go) return;
  __shared__ uint32_t ws[kResortLanes / kWave], before[kResortSegs], start[kResortSegs];
  static_assert(kResortSegs <= kResortLanes, "a lane per segment");
  const uint32_t nsrc = r.ctl->resort_nsrc, tid = threadIdx.x, nseg = ((r.ngbx - 1u) >> r.shift) + 1u;
  if (blockIdx.x == 0 && tid == 0) r.ctl->resort_flag = 0u;
  uint32_t nulls;
  const uint32_t pre = block_excl_scan(tid < nseg ? r.part[2u * tid] : 0u, ws, nulls);
  if (tid < nseg) {
    before[tid] = pre;
    start[tid] = r.part[2u * tid + 1u];
  }
  __syncthreads();
  resort_put(r, nsrc, nulls, before, start, nseg, blockIdx.x * static_cast<uint64_t>(kResortLanes) + tid,
             static_cast<uint64_t>(gridDim.x) * kResortLanes);
}

__device__ __forceinline__ Resort coll_resort(const CollArgs& a) {
  return Resort{a.ctl, a.s, a.alt, a.off, a.nact, a.off_new, a.order, a.ngbx, a.big, nullptr, 31u};
}

// ---- Fisher-Yates without its serial chain -----------------------------------------------------
// Swap `iter` (iter = n-1 .. 1, with index j <= iter) moves the element at place j to place iter for
// good and the one at place iter to place j, so the shuffled order follows from the indices alone.
// With L(x) = { iter : j_iter = x } (all >= x), the element at place x just before swap x is
//   U(x) = x                          when L(x) \ {x} is empty,
//   U(x) = U(min(L(x) \ {x}))         otherwise (the last swap that put something there took it from
//                                     its own place), and
//   order[iter] = U(min{ e in L(j) : e > iter })   when there is such a swap,
//               = U(iter) when j = iter, else j;      order[0] = U(0).
// The lists L are built by all lanes at once with atomic exchanges on their heads; their walks (three
// entries long on average) only take minima, so the result does not depend on the order of the
// entries.  The chains of U are one hop long on average (11 at most in 8192 drops).  Serial swaps take
// one dependent memory round trip each: a gridbox of 8192 drops 1.68 ms for its collisions against
// 34 us here and 19 us in shares (below), 24679 gridboxes of 300 drops 4.9 ms against 0.13 ms.  What
// bounds it: LDS (about 30 accesses per 64 drops, with bank conflicts) and the latency of its four passes.
// (Injected indices may make lists and chains of any length: k_inj_long.)
//
// A team of B lanes (a wave, or a whole workgroup) shuffles the drops of one or more gridboxes, its
// items flattened over the lanes.  The lists of a team live in LDS as 16-bit places (kLdsIdx), or,
// for a gridbox above the team's LDS, in HBM scratch as 32-bit ones.
template <int B>
__device__ __forceinline__ void team_sync() {
  if constexpr (B == kWave) {
    __threadfence_block();  // lists in HBM scratch: this wave's stores before its loads
    wave_sync();
  } else {
    __syncthreads();
  }
}
// per item (drop): the list head of its place, the next swap in the list it is on, its index j and
// later the start of its chain, and the first hop of its place's chain
struct FyLds {
  using Idx = uint16_t;
  uint32_t* head;
  Idx *nxt, *jst, *hop;
  __device__ __forceinline__ uint32_t exch(uint32_t at, uint32_t v) const { return atomicExch(&head[at], v); }
  __device__ __forceinline__ uint32_t first(uint32_t at) const { return head[at]; }
};
struct FyHbm {
  using Idx = uint32_t;
  uint32_t* head;
  Idx *nxt, *jst, *hop;
  // the atomics act in L2, so the heads are read there too
  __device__ __forceinline__ uint32_t exch(uint32_t at, uint32_t v) const { return atomicExch(&head[at], v); }
  __device__ __forceinline__ uint32_t first(uint32_t at) const {
    return __hip_atomic_load(&head[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};
constexpr uint32_t kTeamMaxItems = 15360;  // 150 KB of lists
constexpr uint32_t kFyItemBytes = 10;  // LDS of one item: a 32-bit head and three 16-bit places
// gridboxes g0 .. g0 + cnt - 1 of a team: their drops, the prefixes of their active drops, of their
// blocks of four swaps and of their pairs
struct TeamGbx {
  uint32_t ipre[kWave + 1], qpre[kWave + 1], ppre[kWave + 1];
  uint32_t base[kWave], n[kWave], nfull[kWave], nulls[kWave];
};
// Shuffled order of the `cnt` gridboxes from entry i0 of T on, into M.nxt (gridbox i's from entry
// T.ipre[i] - T.ipre[i0] on).  Every lane of the team calls it.
template <int B, class Mem>
__device__ __forceinline__ void team_shuffle(const CollArgs& a, const Mem& M, const TeamGbx& T, uint32_t g0, uint32_t i0,
                                             uint32_t cnt, uint64_t event, uint32_t tid) {
  using Idx = typename Mem::Idx;
  constexpr uint32_t kNone = static_cast<uint32_t>(static_cast<Idx>(~Idx(0)));
  constexpr uint32_t kChain = kNone / 2u + 1u;  // top bit: the place to chase from, not the element
  const uint32_t off0 = T.ipre[i0], total = T.ipre[i0 + cnt] - off0;
  const uint32_t nquad = T.qpre[i0 + cnt] - T.qpre[i0];
  for (uint32_t f = tid; f < total; f += B) M.head[f] = kNone;
  team_sync<B>();
  // a lane draws one block of the counter stream and links its four swaps
  for (uint32_t f = tid; f < nquad; f += B) {
    const uint32_t i = i0 + tile_owner(T.qpre + i0, cnt, T.qpre[i0] + f);
    const uint32_t q = T.qpre[i0] + f - T.qpre[i], g = g0 + i, n = T.n[i], o = T.ipre[i] - off0;
    uint32_t r4[4] = {0u, 0u, 0u, 0u};
    if (!a.inj_j) rng_block(a.seed, event, 0u, g, q, r4);
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) {
      const uint32_t t = 4u * q + w;
      if (t + 1 < n) {
        const uint32_t iter = n - 1 - t;
        const uint32_t j = a.inj_j ? inj_index(a, g, T.base[i], n, t) : fy_scale(r4[w], iter);
        M.jst[o + iter] = static_cast<Idx>(j);
        M.nxt[o + iter] = static_cast<Idx>(M.exch(o + j, iter));
      }
    }
  }
  team_sync<B>();
  for (uint32_t f = tid; f < total; f += B) {
    const uint32_t i = i0 + tile_owner(T.ipre + i0, cnt, off0 + f);
    const uint32_t o = T.ipre[i] - off0, k = f - o;
    uint32_t m = kNone;  // min(L(k) \ {k})
    for (uint32_t e = M.first(f); e != kNone; e = M.nxt[o + e])
      if (e != k && e < m) m = e;
    M.hop[f] = static_cast<Idx>(m);
    uint32_t start = k | kChain;
    if (k > 0) {
      const uint32_t j = M.jst[f];
      if (j != k) {
        uint32_t s = kNone;  // min{ e in L(j) : e > k }
        for (uint32_t e = M.first(o + j); e != kNone; e = M.nxt[o + e])
          if (e > k && e < s) s = e;
        start = s != kNone ? (s | kChain) : j;
      }
    }
    M.jst[f] = static_cast<Idx>(start);
  }
  team_sync<B>();
  for (uint32_t f = tid; f < total; f += B) {
    const uint32_t i = i0 + tile_owner(T.ipre + i0, cnt, off0 + f);
    const uint32_t o = T.ipre[i] - off0, v = M.jst[f];
    uint32_t x = v & ~kChain;
    if (v & kChain)
      for (uint32_t h = M.hop[o + x]; h != kNone; h = M.hop[o + x]) x = h;
    M.nxt[f] = static_cast<Idx>(x);
  }
  team_sync<B>();
}

// Collisions of the `cnt` gridboxes from entry i0 of T on, by one team: the shuffle, the pairs
// flattened over the lanes, the unpaired drops, then the nulls.  lds: the lists are in L, else in
// the gridbox's HBM scratch (cnt is 1 then).
template <int B, bool Kinetic>
__device__ __forceinline__ void team_collide(const CollArgs& a, bool lds, const FyLds& L, TeamGbx& T, uint32_t g0,
                                             uint32_t i0, uint32_t cnt, uint64_t event, uint32_t tid, uint32_t& events) {
  FyHbm H{};
  if (lds) {
    team_shuffle<B>(a, L, T, g0, i0, cnt, event, tid);
  } else {
    // two words per drop of the collision scratch, two of the per-drop condensation scratch (free
    // during collisions)
    const uint64_t b2 = 2ull * T.base[i0];
    const uint32_t n = T.n[i0];
    H = FyHbm{a.big2 + b2, a.big + b2, a.big + b2 + n, a.big2 + b2 + n};
    team_shuffle<B>(a, H, T, g0, i0, cnt, event, tid);
  }
  const uint32_t off0 = T.ipre[i0], p0 = T.ppre[i0], npairs = T.ppre[i0 + cnt] - p0;
  auto place = [&](uint32_t f) -> uint32_t { return lds ? static_cast<uint32_t>(L.nxt[f]) : H.nxt[f]; };
  for (uint32_t f = tid; f < npairs; f += B) {
    const uint32_t i = i0 + tile_owner(T.ppre + i0, cnt, p0 + f);
    const uint32_t jj = p0 + f - T.ppre[i], o = T.ipre[i] - off0 + 2 * jj, bi = T.base[i];
    if (coll_pair<Kinetic>(a, g0 + i, bi, T.n[i], jj, coll_pos(a, bi, place(o)), coll_pos(a, bi, place(o + 1)), event,
                           events))
      atomicAdd(&T.nulls[i], 1u);
  }
  // unpaired last drop and the inactive tail (nulls of earlier sub-steps) keep their places
  auto tail = [&](uint32_t i, uint32_t k0, uint32_t step) {
    const uint32_t bi = T.base[i], n = T.n[i], o = T.ipre[i] - off0;
    for (uint32_t k = 2 * (n / 2) + k0; k < T.nfull[i]; k += step)
      a.order[bi + k] = coll_pos(a, bi, k < n ? place(o + k) : k);
  };
  if (cnt == 1)
    tail(i0, tid, B);
  else if (tid < cnt)
    tail(i0 + tid, 0u, 1u);
  team_sync<B>();
  for (uint32_t i = i0 + tid / kWave; i < i0 + cnt; i += B / kWave)
    if (T.nulls[i]) coll_order_nulls(a, g0 + i, T.base[i], T.n[i], T.nulls[i], lane_id());
}

// A team per workgroup of B lanes, `gpt` consecutive gridboxes at a time, whose lists fit `cap` items
// of LDS together, else one after the other (and through HBM scratch above cap drops).  For gridboxes
// of 512 drops or fewer its flat passes are faster than the chains of k_coll_split (one of 501 drops with
// kinetic energies 11.6 against 12.9 us), and so they are for many gridboxes up to 2048.
template <int B, bool Kinetic>
__global__ void __launch_bounds__(B) CLEO_OCCUPANCY(Kinetic && B <= 256 ? 3 : 4) k_coll_team(CollArgs a, uint32_t gpt, uint32_t cap) {
  extern __shared__ uint32_t lds_dyn[];
  __shared__ TeamGbx T;
  const uint32_t tid = threadIdx.x;
  uint16_t* half = reinterpret_cast<uint16_t*>(lds_dyn + cap);
  const FyLds L{lds_dyn, half, half + cap, half + 2 * cap};
  const uint64_t event = a.ctl->event + a.event_ofs;
  uint32_t pairs = 0, events = 0, nulls = 0;
  for (uint64_t g0 = static_cast<uint64_t>(blockIdx.x) * gpt; g0 < a.ngbx; g0 += static_cast<uint64_t>(gridDim.x) * gpt) {
    const uint32_t cnt = static_cast<uint32_t>(min(static_cast<uint64_t>(gpt), a.ngbx - g0));
    team_sync<B>();  // the previous gridboxes are done with T and L
    if (tid < kWave) {
      uint32_t base = 0, nfull = 0, n = 0;
      if (tid < cnt) {
        base = a.off[g0 + tid];
        nfull = a.off[g0 + tid + 1] - base;
        n = a.nact[g0 + tid];
      }
      uint32_t it, qt, pt;
      T.ipre[tid] = wave_excl_scan(n, static_cast<int>(tid), it);
      T.qpre[tid] = wave_excl_scan((n + 2u) / 4u, static_cast<int>(tid), qt);
      T.ppre[tid] = wave_excl_scan(n / 2u, static_cast<int>(tid), pt);
      if (tid == 0) {
        T.ipre[kWave] = it;
        T.qpre[kWave] = qt;
        T.ppre[kWave] = pt;
      }
      T.base[tid] = base;
      T.n[tid] = n;
      T.nfull[tid] = nfull;
      T.nulls[tid] = 0u;
    }
    team_sync<B>();
    const bool whole = T.ipre[cnt] <= cap;
    for (uint32_t i = 0; i < cnt;) {
      const uint32_t m = whole ? cnt : 1u;
      team_collide<B, Kinetic>(a, whole || T.n[i] <= cap, L, T, static_cast<uint32_t>(g0), i, m, event, tid, events);
      i += m;
      if (i < cnt) team_sync<B>();  // the lists are reused
    }
    if (tid < cnt) nulls += T.nulls[tid];
    if (tid == 0) pairs += T.ppre[cnt];
  }
  pairs = wave_sum_u32(pairs);
  events = wave_sum_u32(events);
  nulls = wave_sum_u32(nulls);
  if (lane_id() == 0) {
    put_stat(a.stat, ST_COLL_PAIRS, pairs);
    put_stat(a.stat, ST_COLL_EVENTS, events);
    put_stat(a.stat, ST_NULLS, nulls);
  }
  if (a.close) {
    team_sync<B>();
    resort_alone<B>(coll_resort(a), a.close, tid);
  }
}

// ---- large gridboxes: a workgroup, or one per share of the gridbox's pairs -----------------------
// Every workgroup builds the whole lists of its gridbox (draws and atomic exchanges, two draws of four
// swaps per lane for 8192 drops) and follows the chains only of the drops in its share of the pairs, so
// the shares need nothing from each other; a chain step takes the minimum of a place's list anew, and
// three passes over the lists with their barriers go.  What bounds it: the latency of the lists' two
// passes and of one pair per lane (k_coll_team's pairs of 8192 drops are four in series on one CU).
// The last share to finish orders the nulls; it needs the others' stores only then, but every share
// makes its own visible (one write-back of an L2 that holds this gridbox only).
constexpr uint32_t kSplitMaxItems = 19200;  // 150 KB of lists
constexpr uint32_t kSplitItemBytes = 8;     // LDS of one item: a 32-bit head and two 16-bit places
struct FySplitLds {
  uint32_t* head;
  uint16_t *nxt, *jst;
  using Idx = uint16_t;
  __device__ __forceinline__ uint32_t exch(uint32_t at, uint32_t v) const { return atomicExch(&head[at], v); }
  __device__ __forceinline__ uint32_t first(uint32_t at) const { return head[at]; }
};
template <int B, class Mem>
__device__ __forceinline__ void split_lists(const CollArgs& a, const Mem& M, uint32_t g, uint32_t base, uint32_t n,
                                            uint64_t event, uint32_t tid) {
  using Idx = typename Mem::Idx;
  constexpr uint32_t kNone = static_cast<uint32_t>(static_cast<Idx>(~Idx(0)));
  for (uint32_t f = tid; f < n; f += B) M.head[f] = kNone;
  __syncthreads();
  for (uint32_t q = tid; q < (n + 2u) / 4u; q += B) {
    uint32_t r4[4] = {0u, 0u, 0u, 0u};
    if (!a.inj_j) rng_block(a.seed, event, 0u, g, q, r4);
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) {
      const uint32_t t = 4u * q + w;
      if (t + 1 < n) {
        const uint32_t iter = n - 1 - t;
        const uint32_t j = a.inj_j ? inj_index(a, g, base, n, t) : fy_scale(r4[w], iter);
        M.jst[iter] = static_cast<Idx>(j);
        M.nxt[iter] = static_cast<Idx>(M.exch(j, iter));
      }
    }
  }
  __syncthreads();
}
// the shuffled order's entry k
template <class Mem>
__device__ __forceinline__ uint32_t split_place(const Mem& M, uint32_t k) {
  using Idx = typename Mem::Idx;
  constexpr uint32_t kNone = static_cast<uint32_t>(static_cast<Idx>(~Idx(0)));
  uint32_t x = k;
  if (k > 0) {
    const uint32_t j = M.jst[k];
    if (j != k) {
      x = kNone;  // min{ e in L(j) : e > k }
      for (uint32_t e = M.first(j); e != kNone; e = M.nxt[e])
        if (e > k && e < x) x = e;
      if (x == kNone) return j;
    }
  }
  for (;;) {
    uint32_t m = kNone;  // min(L(x) \ {x})
    for (uint32_t e = M.first(x); e != kNone; e = M.nxt[e])
      if (e != x && e < m) m = e;
    if (m == kNone) return x;
    x = m;
  }
}
template <int B, bool Kinetic>
__global__ void __launch_bounds__(B) CLEO_OCCUPANCY(Kinetic && B <= 512 ? 3 : 4) k_coll_split(CollArgs a, uint32_t split, uint32_t cap) {
  extern __shared__ uint32_t lds_dyn[];
  __shared__ uint32_t s_nulls, s_last;
  const uint32_t tid = threadIdx.x, g = blockIdx.x / split, part = blockIdx.x % split;
  const uint64_t event = a.ctl->event + a.event_ofs;
  const uint32_t base = a.off[g], nfull = a.off[g + 1] - base, n = a.nact[g];
  const bool lds = n <= cap;
  uint16_t* const half = reinterpret_cast<uint16_t*>(lds_dyn + cap);
  const FySplitLds L{lds_dyn, half, half + cap};
  // two words per drop of the collision scratch, two of the per-drop condensation scratch (free
  // during collisions)
  const uint64_t b2 = 2ull * base;
  const FyHbm H{a.big2 + b2, a.big + b2, a.big + b2 + n, nullptr};
  // the lists in HBM scratch are one workgroup's, and then all of the pairs
  const uint32_t shares = lds ? split : 1u;
  if (tid == 0) s_nulls = 0u;
  if (lds)
    split_lists<B>(a, L, g, base, n, event, tid);
  else if (part == 0)
    split_lists<B>(a, H, g, base, n, event, tid);
  auto place = [&](uint32_t k) -> uint32_t { return lds ? split_place(L, k) : split_place(H, k); };
  uint32_t events = 0, nulls = 0;
  const uint32_t npairs = n / 2, per = (npairs + shares - 1) / shares, hi = min(npairs, (part + 1) * per);
  if (part < shares) {
    for (uint32_t jj = part * per + tid; jj < hi; jj += B) {
      const uint32_t ka = coll_pos(a, base, place(2 * jj)), kb = coll_pos(a, base, place(2 * jj + 1));
      if (coll_pair<Kinetic>(a, g, base, n, jj, ka, kb, event, events)) ++nulls;
    }
    // unpaired last drop and the inactive tail (nulls of earlier sub-steps) keep their places
    if (part + 1 == shares)
      for (uint32_t k = 2 * npairs + tid; k < nfull; k += B) a.order[base + k] = coll_pos(a, base, k < n ? place(k) : k);
  }
  nulls = wave_sum_u32(nulls);
  events = wave_sum_u32(events);
  if (lane_id() == 0 && nulls) atomicAdd(&s_nulls, nulls);
  // this workgroup's stores are in L2 before its first wave makes them visible to the other shares
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const uint32_t mine = s_nulls;
    uint32_t all = mine, last = 1u;
    if (split > 1) {
      uint32_t* const share = a.share + 2u * g;  // nulls so far, shares done: zero between launches
      if (mine) atomicAdd(&share[0], mine);
      __threadfence();
      last = atomicAdd(&share[1], 1u) + 1u == split ? 1u : 0u;
      if (last) {
        __threadfence();
        all = atomicExch(&share[0], 0u);
        atomicExch(&share[1], 0u);
      }
    }
    s_nulls = all;
    s_last = last;
    if (part == 0) put_stat(a.stat, ST_COLL_PAIRS, n / 2);
    if (last) put_stat(a.stat, ST_NULLS, all);
  }
  if (lane_id() == 0) put_stat(a.stat, ST_COLL_EVENTS, events);
  __syncthreads();
  if (!s_last) return;
  if (s_nulls && tid < kWave) coll_order_nulls(a, g, base, n, s_nulls, static_cast<int>(tid));
  if (a.close) {
    __syncthreads();
    resort_alone<B>(coll_resort(a), a.close, tid);
  }
}

// ---- tiled collisions: 64 gridboxes per wave ---------------------------------------------------
// Lane i shuffles gridbox 64*tile + i: its permutation (one byte per drop) lives in the wave's LDS
// tile and the serial swaps of all 64 gridboxes run side by side.  The tile's pairs are then
// flattened over the lanes (a lane finds its gridbox by binary search over the prefix of per-gridbox
// pair counts), so every lane evaluates a pair whatever the gridbox sizes.  Gridboxes above kTileMaxN
// drops, or beyond the tile's LDS, follow one after the other with the whole wave as their team (64^3
// gridboxes of 128 drops, where a few of each tile overflow: 433 -> 316 us against their serial swaps in
// HBM scratch).  The constant-kinetics instantiation runs at four waves per SIMD (1.18 -> 1.07 ms on 134M
// drops against three), the kinetic-energy one at three.
struct CollTileLds {
  uint32_t perm32[kTilePermBytes / 4];  // byte permutations, gridbox i from byte loff[i]
  uint32_t ppre[kWave + 1];             // first pair of gridbox i among the tile's pairs
  uint32_t base[kWave];                 // first drop of gridbox i
  uint32_t loff[kWave];                 // kBigGbx: the gridbox is shuffled by the whole wave
  uint32_t n[kWave];
  uint32_t nulls[kWave];
};
static_assert(sizeof(CollTileLds) == kCollTileLdsBytes, "tile LDS size");
// drops of a large gridbox whose lists fit the tile's permutation bytes behind its TeamGbx
constexpr uint32_t kTileTeamCap = (kTilePermBytes - sizeof(TeamGbx)) / kFyItemBytes / 4u * 4u;

template <bool Kinetic>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(Kinetic ? 3 : 4) k_coll_tiles(CollArgs a) {
  extern __shared__ uint32_t lds_dyn[];
  const int lane = lane_id();
  CollTileLds& L = reinterpret_cast<CollTileLds*>(lds_dyn)[threadIdx.x >> 6];
  uint8_t* pb = reinterpret_cast<uint8_t*>(L.perm32);
  const uint64_t event = a.ctl->event + a.event_ofs;
  uint32_t pairs = 0, events = 0, nulls = 0;
  const uint32_t ntiles = (a.ngbx + kWave - 1) / kWave;
  for (uint32_t tile = wave_index(); tile < ntiles; tile += wave_count()) {
    wave_sync();  // the previous tile is done with L
    const uint32_t g = tile * kWave + static_cast<uint32_t>(lane);
    const bool valid = g < a.ngbx;
    uint32_t base = 0, nfull = 0, n = 0;
    if (valid) {
      base = a.off[g];
      nfull = a.off[g + 1] - base;
      n = a.nact[g];
    }
    const bool fits = valid && n <= kTileMaxN;
    uint32_t ltot;
    const uint32_t loff = wave_excl_scan(fits ? (n + 3u) & ~3u : 0u, lane, ltot);
    const bool small = fits && loff + n <= kTilePermBytes;
    // fisher_yates_shuffle (shuffle.hpp:80-87), one gridbox per lane
    if (small) {
      for (uint32_t k = 0; k < n; k += 4) L.perm32[(loff + k) >> 2] = k | ((k + 1) << 8) | ((k + 2) << 16) | ((k + 3) << 24);
      uint8_t* p = pb + loff;
      uint32_t r4[4] = {0u, 0u, 0u, 0u};
      for (uint32_t t = 0; t + 1 < n; ++t) {
        const uint32_t iter = n - 1 - t;
        uint32_t j;
        if (a.inj_j) {
          j = inj_index(a, g, base, n, t);
        } else {
          // t is the same for every lane still shuffling, so the block is drawn once per 4 swaps
          if ((t & 3u) == 0u) rng_block(a.seed, event, 0u, g, t >> 2, r4);
          j = fy_scale(rng_word(r4, t), iter);
        }
        const uint8_t pi = p[iter];
        p[iter] = p[j];
        p[j] = pi;
      }
    }
    const uint32_t np = small ? n / 2 : 0u;
    uint32_t ptot;
    const uint32_t pfirst = wave_excl_scan(np, lane, ptot);
    L.ppre[lane] = pfirst;
    if (lane == kWave - 1) L.ppre[kWave] = ptot;
    L.base[lane] = base;
    L.loff[lane] = small ? loff : kBigGbx;
    L.n[lane] = n;
    L.nulls[lane] = 0u;
    wave_sync();
    // the tile's pairs flattened over the lanes (pair f belongs to the gridbox i with
    // ppre[i] <= f < ppre[i+1]): each pair is evaluated once, by one lane, which records its two
    // slots of the logical order and stores the drops' new attributes when it was enacted
    for (uint32_t f = lane; f < ptot; f += kWave) {
      const uint32_t i = tile_owner(L.ppre, kWave, f);
      const uint32_t jj = f - L.ppre[i], bi = L.base[i];
      const uint8_t* pi = pb + L.loff[i];
      if (coll_pair<Kinetic>(a, tile * kWave + i, bi, L.n[i], jj, coll_pos(a, bi, pi[2 * jj]),
                             coll_pos(a, bi, pi[2 * jj + 1]), event, events))
        atomicAdd(&L.nulls[i], 1u);
    }
    // the unpaired last drop and the inactive tail of the lane's own gridbox keep their places
    if (small) {
      const uint8_t* p = pb + loff;
      for (uint32_t k = 2u * np; k < nfull; ++k)
        a.order[base + k] = coll_pos(a, base, k < n ? static_cast<uint32_t>(p[k]) : k);
    }
    wave_sync();
    const uint32_t mynulls = L.nulls[lane];
    pairs += np;
    nulls += mynulls;
    uint64_t m = __ballot(mynulls > 0u);
    while (m) {
      const int i = __ffsll(static_cast<unsigned long long>(m)) - 1;
      m &= m - 1;
      coll_order_nulls(a, tile * kWave + static_cast<uint32_t>(i), readlane_u32(base, i), readlane_u32(n, i),
                       readlane_u32(mynulls, i), lane);
    }
    // the gridboxes that are too large: one after the other by the whole wave, in the tile's LDS
    // (its permutations are done with) or HBM scratch
    TeamGbx& T = *reinterpret_cast<TeamGbx*>(L.perm32);
    uint32_t* head = L.perm32 + sizeof(TeamGbx) / 4;
    uint16_t* half = reinterpret_cast<uint16_t*>(head + kTileTeamCap);
    const FyLds lists{head, half, half + kTileTeamCap, half + 2 * kTileTeamCap};
    uint64_t mb = __ballot(valid && !small);
    while (mb) {
      const int i = __ffsll(static_cast<unsigned long long>(mb)) - 1;
      mb &= mb - 1;
      const uint32_t nb = readlane_u32(n, i), bb = readlane_u32(base, i), fb = readlane_u32(nfull, i);
      wave_sync();
      if (lane == 0) {
        T.ipre[0] = T.qpre[0] = T.ppre[0] = 0u;
        T.ipre[1] = nb;
        T.qpre[1] = (nb + 2u) / 4u;
        T.ppre[1] = nb / 2u;
        T.base[0] = bb;
        T.n[0] = nb;
        T.nfull[0] = fb;
        T.nulls[0] = 0u;
      }
      wave_sync();
      team_collide<kWave, Kinetic>(a, nb <= kTileTeamCap, lists, T, tile * kWave + static_cast<uint32_t>(i), 0u, 1u, event,
                                   static_cast<uint32_t>(lane), events);
      if (lane == 0) {
        pairs += nb / 2u;
        nulls += T.nulls[0];
      }
    }
  }
  pairs = wave_sum_u32(pairs);
  events = wave_sum_u32(events);
  nulls = wave_sum_u32(nulls);
  if (lane == 0) {
    put_stat(a.stat, ST_COLL_PAIRS, pairs);
    put_stat(a.stat, ST_COLL_EVENTS, events);
    put_stat(a.stat, ST_NULLS, nulls);
  }
}

// per-gridbox sizes of the injected stream: n-1 indices and 2*floor(n/2) phis
__global__ void k_inj_sizes(const uint32_t* nact, uint32_t ngbx, uint32_t* nj, uint32_t* np) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ngbx) return;
  const uint32_t n = nact[g];
  nj[g] = n >= 2 ? n - 1 : 0;
  np[g] = 2 * (n / 2);
}

// Injected indices may put any number of swaps on one list (all indices equal) or make a chain of any
// length (every index one below its swap's place), and the shuffle's passes would take n^2 steps: 1e12 in
// a gridbox of a million drops.  So before an injected event the lists of every gridbox of more than
// kFyBudget drops are looked over, and where a place's element is more than kFyBudget list entries away
// (drawn indices: 4 on average, at most 60 to 120 in 8192 to 200000 drops) one lane makes the swaps on the
// pending order itself and leaves indices that move nothing.
template <class Mem>
__device__ __forceinline__ bool fy_within_budget(const Mem& M, uint32_t k) {
  using Idx = typename Mem::Idx;
  constexpr uint32_t kNone = static_cast<uint32_t>(static_cast<Idx>(~Idx(0)));
  uint32_t x = k, steps = 0;
  if (k > 0 && M.jst[k] != k) {
    x = kNone;  // min{ e in L(j) : e > k }
    for (uint32_t e = M.first(M.jst[k]); e != kNone; e = M.nxt[e]) {
      if (++steps > kFyBudget) return false;
      if (e > k && e < x) x = e;
    }
  }
  while (x != kNone) {
    const uint32_t at = x;
    x = kNone;  // min(L(at) \ {at})
    for (uint32_t e = M.first(at); e != kNone; e = M.nxt[e]) {
      if (++steps > kFyBudget) return false;
      if (e != at && e < x) x = e;
    }
  }
  return true;
}
__global__ void __launch_bounds__(256) k_inj_long(CollArgs a, uint32_t* order, uint32_t* inj_j) {
  const uint32_t tid = threadIdx.x;
  for (uint32_t g = blockIdx.x; g < a.ngbx; g += gridDim.x) {
    const uint32_t base = a.off[g], n = a.nact[g], oj = a.inj_oj[g];
    if (n <= kFyBudget) continue;
    const uint64_t b2 = 2ull * base;
    const FyHbm M{a.big2 + b2, a.big + b2, a.big + b2 + n, nullptr};
    for (uint32_t k = tid; k < n; k += 256u) M.head[k] = ~0u;
    __syncthreads();
    for (uint32_t t = tid; t + 1 < n; t += 256u) {
      const uint32_t iter = n - 1 - t, j = min(inj_j[oj + t], iter);
      M.jst[iter] = j;
      M.nxt[iter] = M.exch(j, iter);
    }
    __syncthreads();
    bool within = true;
    for (uint32_t k = tid; k < n && within; k += 256u) within = fy_within_budget(M, k);
    if (__syncthreads_or(!within) && tid == 0) {
      for (uint32_t t = 0; t + 1 < n; ++t) {
        const uint32_t iter = n - 1 - t, j = inj_index(a, g, base, n, t);
        const uint32_t x = order[base + iter];
        order[base + iter] = order[base + j];
        order[base + j] = x;
        inj_j[oj + t] = iter;
      }
    }
    __syncthreads();
  }
}

// ============================ motion ==========================================================
// Source gridbox that reaches `d` by the neighbour step `s` (s = (dz+1) + 3(dx+1) + 9(dy+1)),
// or kOOB when the step would come from outside a finite axis.
__device__ __forceinline__ uint32_t source_of(const Grid& gr, uint32_t d, int s) {
  const int dz = s % 3 - 1, dx = (s / 3) % 3 - 1, dy = s / 9 - 1;
  int jz = static_cast<int>(d % gr.nz) - dz;
  int jx = static_cast<int>((d / gr.nz) % gr.nx) - dx;
  int jy = static_cast<int>(d / (gr.nz * gr.nx)) - dy;
  const int nz = static_cast<int>(gr.nz), nx = static_cast<int>(gr.nx), ny = static_cast<int>(gr.ny);
  if (jz < 0 || jz >= nz) {
    if (!gr.per[0]) return kOOB;
    jz = (jz + nz) % nz;
  }
  if (jx < 0 || jx >= nx) {
    if (!gr.per[1]) return kOOB;
    jx = (jx + nx) % nx;
  }
  if (jy < 0 || jy >= ny) {
    if (!gr.per[2]) return kOOB;
    jy = (jy + ny) % ny;
  }
  return static_cast<uint32_t>(jz + nz * (jx + nx * jy));
}

// gridbox reached from g by the step s (kOOB off a finite axis)
__device__ __forceinline__ uint32_t neighbour_of(const Grid& gr, uint32_t g, int s) { return source_of(gr, g, 26 - s); }


// wind at coordinate sd between the faces blo, bhi (predcorr.cpp:31-42).  inv_span = 1/(bhi - blo)
// of the gridbox, so the reference's alpha = (coord - blo) / (bhi - blo) is a product, within an
// ulp or two of the quotient.
__device__ __forceinline__ double interpolation(double blo, double bhi, double inv_span, double vlo, double vhi,
                                                double sd) {
  const double coord = fmin(bhi, fmax(blo, sd));
  const double alpha = (coord - blo) * inv_span;
  return alpha * vhi + (1 - alpha) * vlo;
}

// One axis of CartesianMaps::get_local_bounding_gridbox_index (cartesianmaps.cpp:68-286,
// domainboundaries.hpp:34-109): step to the backward/forward neighbour when the coordinate left
// [lower, upper) and wrap the coordinate at a periodic domain edge.  i is the drop's index along
// the axis, updated to the neighbour's.  Returns the step taken.
__device__ __forceinline__ int axis_step(uint32_t& idx, double& coord, uint32_t& i, uint32_t nd, uint32_t inc,
                                         bool periodic, const double* h) {
  const double lo = h[i], hi = h[i + 1];
  if (coord < lo) {
    if (i == 0) {
      if (periodic) {
        const uint32_t nb = idx + (nd - 1) * inc;
        coord = coord + h[nd] - lo;  // lim1 = upper bound of the backward neighbour
        idx = nb;
        i = nd - 1;
      } else {
        idx = kOOB;
      }
    } else {
      idx = idx - inc;
      i -= 1;
    }
    return -1;
  }
  if (coord >= hi) {
    if (i == nd - 1) {
      if (periodic) {
        const uint32_t nb = idx - (nd - 1) * inc;
        coord = coord + h[0] - hi;  // lim1 = lower bound of the forward neighbour
        idx = nb;
        i = 0;
      } else {
        idx = kOOB;
      }
    } else {
      idx = idx + inc;
      i += 1;
    }
    return 1;
  }
  return 0;
}

// bounds, reciprocal widths and face winds of gridbox g
struct GbxGeom {
  uint32_t iz, ix, iy;
  double zlo, zhi, xlo, xhi, ylo, yhi, wlo, whi, ulo, uhi, vlo, vhi;
  double inv_z, inv_x, inv_y;
};
__device__ __forceinline__ GbxGeom gbx_geom(const MotionArgs& a, uint32_t g) {
  const uint32_t nz = a.grid.nz, nx = a.grid.nx;
  GbxGeom G;
  G.iz = g % nz;
  G.ix = (g / nz) % nx;
  G.iy = g / (nz * nx);
  G.zlo = a.grid.zh[G.iz];
  G.zhi = a.grid.zh[G.iz + 1];
  G.xlo = a.grid.xh[G.ix];
  G.xhi = a.grid.xh[G.ix + 1];
  G.ylo = a.grid.yh[G.iy];
  G.yhi = a.grid.yh[G.iy + 1];
  G.wlo = a.st.wlo[g];
  G.whi = a.st.whi[g];
  G.ulo = a.st.ulo[g];
  G.uhi = a.st.uhi[g];
  G.vlo = a.st.vlo[g];
  G.vhi = a.st.vhi[g];
  G.inv_z = rcp_nr(G.zhi - G.zlo);
  G.inv_x = rcp_nr(G.xhi - G.xlo);
  G.inv_y = rcp_nr(G.yhi - G.ylo);
  return G;
}
// drop k of gridbox g after one predictor-corrector step: new coordinates, new gridbox (kOOB
// when it left the domain) and the step taken, dir = (dz+1) + 3(dx+1) + 9(dy+1), or 27 out of the
// domain.  PredCorr::delta_coord3/1/2 (predcorr.hpp:84-145), cfl_criteria (cfl_criteria.hpp:40-57),
// superdrop_gbx z, then x, then y (predcorrmotion.hpp:85-106) and CartesianCheckBounds
// (cartesian_motion.hpp:38-52); `report` records the CFL and bounds errors.
struct Moved {
  double c3, c1, c2;
  uint32_t idx;
  int dir;
};
// what the motion step reads of drop k
struct DropPos {
  double c3, c1, c2, r;
};
__device__ __forceinline__ DropPos drop_pos(const MotionArgs& a, uint64_t k) {
  return DropPos{a.s.c3[k], a.s.c1[k], a.s.c2[k], a.s.r[k]};
}
__device__ __forceinline__ DropPos drop_pos_nt(const MotionArgs& a, uint64_t k) {
  return DropPos{__builtin_nontemporal_load(&a.s.c3[k]), __builtin_nontemporal_load(&a.s.c1[k]),
                 __builtin_nontemporal_load(&a.s.c2[k]), __builtin_nontemporal_load(&a.s.r[k])};
}
__device__ __forceinline__ Moved move_drop(const MotionArgs& a, uint32_t g, const GbxGeom& G, const DropPos& P,
                                           uint64_t k, bool report) {
  const uint32_t nz = a.grid.nz, nx = a.grid.nx, ny = a.grid.ny;
  const double delt = a.delt;
  const double c3_0 = P.c3, c1_0 = P.c1, c2_0 = P.c2;
  double coord3 = c3_0;
  const double terminal = terminal_velocity(a.tv, P.r);
  double vel3 = interpolation(G.zlo, G.zhi, G.inv_z, G.wlo, G.whi, coord3);
  vel3 -= terminal;
  coord3 += vel3 * delt;
  double corrvel3 = interpolation(G.zlo, G.zhi, G.inv_z, G.wlo, G.whi, coord3);
  corrvel3 -= terminal;
  const double delta3 = (vel3 + corrvel3) * (delt / 2);
  double coord1 = c1_0;
  const double vel1 = interpolation(G.xlo, G.xhi, G.inv_x, G.ulo, G.uhi, coord1);
  coord1 += vel1 * delt;
  const double corrvel1 = interpolation(G.xlo, G.xhi, G.inv_x, G.ulo, G.uhi, coord1);
  const double delta1 = (vel1 + corrvel1) * (delt / 2);
  double coord2 = c2_0;
  const double vel2 = interpolation(G.ylo, G.yhi, G.inv_y, G.vlo, G.vhi, coord2);
  coord2 += vel2 * delt;
  const double corrvel2 = interpolation(G.ylo, G.yhi, G.inv_y, G.vlo, G.vhi, coord2);
  const double delta2 = (vel2 + corrvel2) * (delt / 2);
  bool cfl = (fabs(delta3) <= fabs(G.zhi - G.zlo));
  cfl = (fabs(delta1) <= fabs(G.xhi - G.xlo)) && cfl;
  cfl = (fabs(delta2) <= fabs(G.yhi - G.ylo)) && cfl;
  if (report && !cfl) set_error(a.ctl, CLEO_ERR_CFL, g, k);
  Moved M;
  M.c3 = c3_0 + delta3;
  M.c1 = c1_0 + delta1;
  M.c2 = c2_0 + delta2;
  uint32_t idx = g, jz = G.iz, jx = G.ix, jy = G.iy;
  const int dz = axis_step(idx, M.c3, jz, nz, 1u, a.grid.per[0] != 0, a.grid.zh);
  int dx = 0, dy = 0;
  if (idx != kOOB) dx = axis_step(idx, M.c1, jx, nx, nz, a.grid.per[1] != 0, a.grid.xh);
  if (idx != kOOB) dy = axis_step(idx, M.c2, jy, ny, nz * nx, a.grid.per[2] != 0, a.grid.yh);
  M.idx = idx;
  M.dir = 27;
  if (idx != kOOB) {
    const bool bad = (M.c3 < a.grid.zh[jz]) | (M.c3 >= a.grid.zh[jz + 1]) | (M.c1 < a.grid.xh[jx]) |
                     (M.c1 >= a.grid.xh[jx + 1]) | (M.c2 < a.grid.yh[jy]) | (M.c2 >= a.grid.yh[jy + 1]);
    if (report && bad) set_error(a.ctl, CLEO_ERR_BOUNDS, g, k);
    // on a periodic axis of one or two gridboxes several steps lead to one neighbour; the step is then
    // the change of the index, so that drops with the same source and destination have the same step
    // (the sort places drops by their step)
    const int sz = nz <= 2 ? static_cast<int>(jz) - static_cast<int>(G.iz) : dz;
    const int sx = nx <= 2 ? static_cast<int>(jx) - static_cast<int>(G.ix) : dx;
    const int sy = ny <= 2 ? static_cast<int>(jy) - static_cast<int>(G.iy) : dy;
    M.dir = (sz + 1) + 3 * (sx + 1) + 9 * (sy + 1);
  }
  return M;
}
__device__ __forceinline__ Moved move_drop(const MotionArgs& a, uint32_t g, const GbxGeom& G, uint64_t k, bool report) {
  return move_drop(a, g, G, drop_pos(a, k), k, report);
}

// ============================ neighbour sort ==================================================

// the condensation inputs of a gridbox (condensation.cpp:44-56)
__device__ __forceinline__ void gbx_thermo(const GState& st, uint32_t g, double* gs) {
  const double temp = st.temp[g], press = st.press[g];
  const double psat = saturation_pressure(temp);
  gs[kGsStride * g] = supersaturation_ratio(press, st.qv[g], psat);
  gs[kGsStride * g + 1] = diffusion_factor(press, temp, psat);
  const double akoh = kohler_a(temp);
  gs[kGsStride * g + 2] = akoh;
  gs[kGsStride * g + 3] = rcp_nr(akoh);
}

// Per destination d (thread per d): the drops arriving in d, and for each step s the drops that
// reach d from source gridboxes of lower index than the source of s (the stable order puts them
// first).  The counts are destination-major (row d, column s: arrivals at d by the step s), read as
// one row and, on small domains, left zero for the next motion (counts_stay_clear).  The run offsets are
// written source-major into `runs` (row g, column s: the offset of g's drops taking the step s), so the
// rank pass reads its gridbox's 27 offsets as one contiguous row.  Every entry of `runs` belongs to one
// destination (g + step s): no two threads write the same entry.  Only the entries of steps that some drop
// takes are written (a source off a finite axis has none); the others keep older values that no pass reads.
// The arrivals and the drops that leave the domain are scanned here within the block of gridboxes, into the
// new refs and the out-of-domain prefix; k_nsort_apply adds what the blocks before have.  (Separate
// launches for the fill of the counts, two three-level scans, the refs, the active counts and the
// condensation inputs, with the same for the re-sort after collisions, made 34 launches of a coupled step,
// nine now: 409 -> 349 us on 32^3 gridboxes of 64 drops with eleven of them.)  kThermo: the gridboxes'
// condensation inputs too, for a condensation in the sort's gather (the State is that of before the sort),
// by workgroups of their own from number nblk on: both are serial chains of a few us (one after the other
// in each thread: 10.3 us on 3750 gridboxes, 7.4 on 20; now 7.8 and 5.0).
template <bool kThermo>
__global__ void __launch_bounds__(kTabBlock) k_nsort_tot(NsortArgs a, GState st, double* gs) {
  __shared__ uint32_t ws[kTabBlock / kWave];
  if (kThermo && blockIdx.x >= a.nblk) {
    const uint32_t g = (blockIdx.x - a.nblk) * kTabBlock + threadIdx.x;
    if (g < a.grid.ngbx) {
      if (st.temp[g] <= 0) set_error(a.ctl, CLEO_ERR_TEMP_NONPOSITIVE, g, a.off[g]);
      gbx_thermo(st, g, gs);
    }
    return;
  }
  const uint32_t d = blockIdx.x * kTabBlock + threadIdx.x;
  uint32_t t = 0, gone = 0;
  if (d < a.grid.ngbx) {
    uint4* row = reinterpret_cast<uint4*>(a.cnt + 28ull * d);
    uint32_t cnt[28];
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      const uint4 v = row[i];
      cnt[4 * i] = v.x;
      cnt[4 * i + 1] = v.y;
      cnt[4 * i + 2] = v.z;
      cnt[4 * i + 3] = v.w;
    }
    if (a.clear) {
#pragma unroll
      for (int i = 0; i < 7; ++i) row[i] = uint4{0u, 0u, 0u, 0u};
    }
    gone = cnt[27];
#pragma unroll
    for (int s = 0; s < 27; ++s) t += cnt[s];
    const Grid& gr = a.grid;
    const int nz = static_cast<int>(gr.nz), nx = static_cast<int>(gr.nx), ny = static_cast<int>(gr.ny);
    const int gz = static_cast<int>(d % gr.nz), gx = static_cast<int>((d / gr.nz) % gr.nx),
              gy = static_cast<int>(d / (gr.nz * gr.nx));
    auto axis = [](int i, int dd, int n, bool per) {
      int j = i - dd;
      if (j < 0) j = per ? j + n : -1;
      if (j >= n) j = per ? j - n : -1;
      return j;
    };
    uint32_t src[27];  // the source of each step (kOOB: off a finite axis, no drops)
#pragma unroll
    for (int s = 0; s < 27; ++s) {
      const int jz = axis(gz, s % 3 - 1, nz, gr.per[0] != 0), jx = axis(gx, (s / 3) % 3 - 1, nx, gr.per[1] != 0),
                jy = axis(gy, s / 9 - 1, ny, gr.per[2] != 0);
      src[s] = (jz >= 0 && jx >= 0 && jy >= 0) ? static_cast<uint32_t>(jz + nz * (jx + nx * jy)) : kOOB;
    }
    const bool wraps = (gr.per[0] && (gz == 0 || gz + 1 == nz)) || (gr.per[1] && (gx == 0 || gx + 1 == nx)) ||
                       (gr.per[2] && (gy == 0 || gy + 1 == ny));
    if (!wraps) {
      // no step wraps: the source of step s is d - (dz + nz dx + nz nx dy), so the sources in index
      // order are the steps in decreasing order
      uint32_t before = 0;
#pragma unroll
      for (int s = 26; s >= 0; --s) {
        if (cnt[s] > 0u && src[s] != kOOB) a.runs[28ull * src[s] + static_cast<uint32_t>(s)] = before;
        before += cnt[s];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 27; ++s) {
        uint32_t before = 0;
#pragma unroll
        for (int q = 0; q < 27; ++q) before += src[q] < src[s] ? cnt[q] : 0u;
        if (cnt[s] > 0u && src[s] != kOOB) a.runs[28ull * src[s] + static_cast<uint32_t>(s)] = before;
      }
    }
    a.nact[d] = t;
  }
  uint32_t tsum, gsum;
  const uint32_t tpre = block_excl_scan(t, ws, tsum), gpre = block_excl_scan(gone, ws, gsum);
  if (d < a.grid.ngbx) {
    a.off_new[d] = tpre;
    a.oobpre[d] = gpre;
  }
  if (threadIdx.x == 0) {
    a.part[2u * blockIdx.x] = tsum;
    a.part[2u * blockIdx.x + 1u] = gsum;
    if (a.nblk == 1) a.off_new[a.grid.ngbx] = tsum;  // no k_nsort_apply follows
    if (blockIdx.x == 0) a.ctl->stats[ST_SORTS] += 1;
  }
}
// kTabBlock blocks' totals to their prefixes (one workgroup), for domains of many blocks
__global__ void __launch_bounds__(1024) k_nsort_part(uint32_t* part, uint32_t nblk) {
  __shared__ uint32_t ws[16];
  uint32_t t0 = 0, g0 = 0;
  for (uint32_t b0 = 0; b0 < nblk; b0 += 1024u) {
    const uint32_t b = b0 + threadIdx.x;
    const uint32_t t = b < nblk ? part[2u * b] : 0u, g = b < nblk ? part[2u * b + 1u] : 0u;
    uint32_t ts, gs;
    const uint32_t tp = block_excl_scan(t, ws, ts), gp = block_excl_scan(g, ws, gs);
    if (b < nblk) {
      part[2u * b] = t0 + tp;
      part[2u * b + 1u] = g0 + gp;
    }
    t0 += ts;
    g0 += gs;
  }
  if (threadIdx.x == 0) part[2u * nblk] = t0;
}
// Adds the totals of the blocks before to the prefixes of block blockIdx.x: the prefixes themselves
// (kScanned: k_nsort_part ran), or the sum of those blocks' totals, which up to kApplyBlocks blocks is
// cheaper than a launch that scans them.
template <bool kScanned>
__global__ void __launch_bounds__(kTabBlock) k_nsort_apply(NsortArgs a) {
  uint32_t t0 = 0, g0 = 0;
  if constexpr (kScanned) {
    t0 = a.part[2u * blockIdx.x];
    g0 = a.part[2u * blockIdx.x + 1u];
  } else {
    __shared__ uint32_t ws[kTabBlock / kWave];
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kTabBlock) {
      t0 += a.part[2u * b];
      g0 += a.part[2u * b + 1u];
    }
    uint32_t all;
    block_excl_scan(t0, ws, all);
    t0 = all;
    block_excl_scan(g0, ws, all);
    g0 = all;
  }
  const uint32_t d = blockIdx.x * kTabBlock + threadIdx.x;
  if (d < a.grid.ngbx) {
    a.off_new[d] += t0;
    a.oobpre[d] += g0;
  }
  if (threadIdx.x == 0 && blockIdx.x + 1 == gridDim.x)
    a.off_new[a.grid.ngbx] = kScanned ? a.part[2u * a.nblk] : t0 + a.part[2u * blockIdx.x];
}

// Stable scatter (sortsupers.hpp:63-76,167-193 under Serial): drop p of source gridbox g with
// key d lands at  base[d] + (drops reaching d from gridboxes < g) + (earlier drops of g with key d);
// the middle term is entry (g, step g -> d) of the `runs` table k_nsort_tot writes, so the 27
// run offsets of g are its own contiguous row.  The 27 run starts of g (one per step, with base[d])
// and the start of its out-of-domain run are loaded by lanes 0..27 together with the keys (one
// round trip; loading only the steps that occur costs a second one), so the ranking below touches
// no memory.  The destination of each drop is
// recorded as perm[dest] = p; k_nsort_gather then moves the records, so that each cache line of the
// sorted store is written whole by one wave (runs scattered from many source gridboxes into one
// line cost HBM read-modify-writes).
// The ranking of a gridbox is split in four stages so that a wave works on four gridboxes at once,
// each stage reading what the previous one loaded an iteration earlier: the head (range and run
// starts), the positions of the first two chunks of slots, the keys of those drops, then the
// ranking itself.  Every load of a stage is issued by all lanes, with indices clamped into the
// arrays, so the number of loads in flight is the same on every path and the waits of the ranking
// leave the younger stages' loads outstanding.
//
// head of gridbox g: its range of positions and, in lane s < 27, the next place of its drops that
// take step s (lane 27: of those leaving).  The neighbour reached by step s = (dz+1) + 3(dx+1) +
// 9(dy+1) is g + noff away from the edges, else wrapped on periodic axes (the same gridbox as
// neighbour_of, without a division per lane).  A g past the last gridbox gives an empty head.
struct RankHead {
  uint32_t g, sbase, nfull, trun;
};
__device__ __forceinline__ RankHead rank_head(const NsortArgs& a, uint64_t g, int gz, int gx, int gy, int32_t noff,
                                              int lane) {
  const uint32_t ngbx = a.grid.ngbx;
  const int nz = static_cast<int>(a.grid.nz), nx = static_cast<int>(a.grid.nx), ny = static_cast<int>(a.grid.ny);
  const bool valid = g < ngbx;
  const uint32_t gc = valid ? static_cast<uint32_t>(g) : ngbx - 1u;
  RankHead h{gc, 0u, 0u, 0u};
  const uint32_t lo = a.off[gc], hi = a.off[gc + 1];
  h.sbase = lo;
  h.nfull = valid ? hi - lo : 0u;
  uint32_t d = ngbx;  // lanes 27..63: the out-of-domain run (off_new[ngbx] + oobpre[g])
  bool ok = valid && lane == 27;
  if (lane < 27 && !valid) {
    d = 0u;  // no gridbox: a harmless load, discarded
  } else if (lane < 27) {
    const bool interior = gz > 0 && gz + 1 < nz && gx > 0 && gx + 1 < nx && gy > 0 && gy + 1 < ny;
    d = gc + static_cast<uint32_t>(noff);
    ok = true;
    if (!interior) {
      auto axis = [](int i, int dd, int n, bool per) {
        int j = i + dd;
        if (j < 0) j = per ? j + n : -1;
        if (j >= n) j = per ? j - n : -1;
        return j;
      };
      const int jz = axis(gz, lane % 3 - 1, nz, a.grid.per[0] != 0);
      const int jx = axis(gx, (lane / 3) % 3 - 1, nx, a.grid.per[1] != 0);
      const int jy = axis(gy, lane / 9 - 1, ny, a.grid.per[2] != 0);
      ok = jz >= 0 && jx >= 0 && jy >= 0;
      d = ok ? static_cast<uint32_t>(jz + nz * (jx + nx * jy)) : 0u;
    }
  }
  const uint32_t b = a.off_new[d];
  const uint32_t extra = lane < 27 ? a.runs[28ull * gc + static_cast<uint32_t>(lane)] : a.oobpre[gc];
  h.trun = ok ? b + extra : 0u;
  return h;
}
// positions held by slots lane and lane + 64 of the gridbox's logical order (the order collisions
// left, or the store's own order); kOOB past the gridbox
struct RankSlots {
  uint32_t p0, p1;
};
template <bool kOrder>
__device__ __forceinline__ RankSlots rank_slots(const NsortArgs& a, const RankHead& h, uint32_t nsrc, int lane) {
  const uint32_t i0 = static_cast<uint32_t>(lane), i1 = i0 + kWave;
  const uint32_t q0 = min(h.sbase + i0, nsrc - 1u), q1 = min(h.sbase + i1, nsrc - 1u);
  uint32_t p0 = q0, p1 = q1;
  if constexpr (kOrder) {
    p0 = a.order[q0];
    p1 = a.order[q1];
  }
  return RankSlots{i0 < h.nfull ? p0 : kOOB, i1 < h.nfull ? p1 : kOOB};
}
// the step recorded for each of those drops
struct RankKeys {
  uint32_t k0, k1;
};
__device__ __forceinline__ RankKeys rank_keys(const NsortArgs& a, const RankSlots& s, uint32_t nsrc) {
  const uint32_t c0 = s.p0 < nsrc ? s.p0 : 0u, c1 = s.p1 < nsrc ? s.p1 : 0u;
  return RankKeys{a.step[c0], a.step[c1]};
}
// ranks the drops of the head's gridbox and records perm[dest] = p (stable scatter above); the
// first two chunks use the preloaded positions and keys, later chunks load their own
template <bool kOrder>
__device__ __forceinline__ void rank_gbx(const NsortArgs& a, const RankHead& h, const RankSlots& s, const RankKeys& k,
                                         uint32_t nsrc, int lane) {
  const uint32_t g = h.g, sbase = h.sbase, nfull = h.nfull;
  uint32_t trun = h.trun;
  // chunk c of 64 slots: the drop of slot sbase + c + lane is at position p with key kv
  auto chunk = [&](uint32_t c, uint32_t p, uint32_t kv) {
    const uint32_t q = sbase + c + lane;
    const bool act = c + lane < nfull;
    // the step motion recorded (27: out of the domain); another value, or a position outside the
    // domain, is an error
    int sv = 27;
    bool ok = act;
    if (act && p >= nsrc) {
      set_error(a.ctl, CLEO_ERR_SORT_NONLOCAL, g, q);
      ok = false;
    }
    if (ok) {
      sv = static_cast<int>(kv);
      if (sv > 27) {
        set_error(a.ctl, CLEO_ERR_SORT_NONLOCAL, g, p);
        ok = false;
      }
    }
    // one round per distinct step in the chunk: its lanes take consecutive places from the run's
    // next place (held by lane v), in lane order
    uint32_t dest = 0;
    const uint64_t okm = ballot(ok);
    uint64_t mask = okm;
    while (mask) {
      const int leader = __ffsll(static_cast<unsigned long long>(mask)) - 1;
      const int v = static_cast<int>(readlane_u32(static_cast<uint32_t>(sv), leader));
      const uint64_t m = ballot(sv == v) & okm;
      const uint32_t start = readlane_u32(trun, v);
      const uint32_t here = start + lanes_below(m);
      dest = (ok && sv == v) ? here : dest;
      trun = lane == v ? start + static_cast<uint32_t>(__popcll(m)) : trun;
      mask &= ~m;
    }
    if (ok && dest >= a.ntot) {  // counts inconsistent with keys: never write out of range
      set_error(a.ctl, CLEO_ERR_SORT_NONLOCAL, g, p);
    } else if (ok) {
      a.perm[dest] = p;
    }
  };
  // the first two chunks from the preloaded positions and keys, straight-line; larger gridboxes
  // (rare at these sizes) load the rest as they go
  if (nfull > 0) chunk(0u, s.p0, k.k0);
  if (nfull > kWave) chunk(kWave, s.p1, k.k1);
  for (uint32_t c = 2 * kWave; c < nfull; c += kWave) {
    const bool act = c + lane < nfull;
    const uint32_t q = sbase + c + lane;
    const uint32_t p = act ? (kOrder ? a.order[q] : q) : kOOB;
    const uint32_t kv = (act && p < nsrc) ? a.step[p] : 0u;
    chunk(c, p, kv);
  }
}
// first pass of the neighbour sort: the destination of every drop of the domain, as perm[dest] = p.
// Gridboxes go to waves through xcd_wave_index(), so each XCD sweeps one contiguous range and the
// count-table rows that neighbouring gridboxes share are fetched into one L2.  The gridbox's
// (z, x, y) advance by the stride's with carries (no division per gridbox).
template <bool kOrder>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(6) k_nsort_perm(NsortArgs a) {
  const int lane = lane_id();
  const uint32_t nz = a.grid.nz, nx = a.grid.nx;
  const uint64_t ngbx = a.grid.ngbx;
  const uint32_t g0 = xcd_wave_index(), stride = wave_count();
  const uint32_t nsrc = a.off[ngbx];
  if (g0 >= ngbx || nsrc == 0) return;
  uint32_t gz = g0 % nz, gx = (g0 / nz) % nx, gy = g0 / (nz * nx);
  const uint32_t sz = stride % nz, sx = (stride / nz) % nx, sy = stride / (nz * nx);
  const int32_t noff = (lane % 3 - 1) + static_cast<int32_t>(nz) * ((lane / 3) % 3 - 1) +
                       static_cast<int32_t>(nz * nx) * (lane / 9 - 1);
  uint64_t gh = g0;  // next gridbox whose head is loaded
  auto next_head = [&]() {
    const RankHead h = rank_head(a, gh, static_cast<int>(gz), static_cast<int>(gx), static_cast<int>(gy), noff, lane);
    gh += stride;
    gz += sz;
    uint32_t carry = gz >= nz ? 1u : 0u;
    gz -= carry * nz;
    gx += sx + carry;
    carry = gx >= nx ? 1u : 0u;
    gx -= carry * nx;
    gy += sy + carry;
    return h;
  };
  // rings of four per stage, rotated by name over a four-fold unrolled loop: no register moves
  // between iterations, which would wait for the loads in flight
  RankHead H0 = next_head(), H1 = next_head(), H2, H3;
  RankSlots S0 = rank_slots<kOrder>(a, H0, nsrc, lane), S1, S2, S3;
  H2 = next_head();
  S1 = rank_slots<kOrder>(a, H1, nsrc, lane);
  RankKeys K0 = rank_keys(a, S0, nsrc), K1, K2, K3;
  // gridbox i: loads the head of i + 3, the slots of i + 2, the keys of i + 1, then ranks i
  auto stage = [&](const RankHead& hu, RankHead& hl, const RankHead& hs, const RankSlots& su, RankSlots& sl,
                   const RankSlots& sk, const RankKeys& ku, RankKeys& kl) {
    hl = next_head();
    sl = rank_slots<kOrder>(a, hs, nsrc, lane);
    kl = rank_keys(a, sk, nsrc);
    rank_gbx<kOrder>(a, hu, su, ku, nsrc, lane);
  };
  for (uint64_t g = g0;;) {
    stage(H0, H3, H2, S0, S2, S1, K0, K1);
    if ((g += stride) >= ngbx) break;
    stage(H1, H0, H3, S1, S3, S2, K1, K2);
    if ((g += stride) >= ngbx) break;
    stage(H2, H1, H0, S2, S0, S3, K2, K3);
    if ((g += stride) >= ngbx) break;
    stage(H3, H2, H1, S3, S1, S0, K3, K0);
    if ((g += stride) >= ngbx) break;
  }
}

// The drops that were out of the domain before (positions nsrc on) follow the newly out-of-domain
// ones; the domain's drops fill the first nsrc positions of the sorted store either way, so they keep
// their positions.
__device__ __forceinline__ void copy_oob(const NsortArgs& a, uint64_t nsrc) {
  for (uint64_t p = nsrc + blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; p < a.ntot;
       p += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    copy_drop(a.src, a.dst, p, p);
}

// Second pass: destination position q takes the record at source position perm[q].  Consecutive
// threads write consecutive positions, so each cache line of the sorted store is written whole by
// one wave; the reads follow the runs of the source order.  Two positions per thread, all loads of
// both issued before the stores.  A position whose perm entry is not a source position of the
// domain (counts inconsistent with the keys) is reported and skipped, so no read leaves the store.
__global__ void __launch_bounds__(256) k_nsort_gather(NsortArgs a) {
  const uint64_t nsrc = a.off[a.grid.ngbx];
  for (uint64_t q0 = 2ull * blockIdx.x * blockDim.x; q0 < nsrc; q0 += 2ull * gridDim.x * blockDim.x) {
    const uint64_t qa = q0 + threadIdx.x, qb = qa + blockDim.x;
    const uint32_t pa = qa < nsrc ? a.perm[qa] : 0u, pb = qb < nsrc ? a.perm[qb] : 0u;
    const bool oka = qa < nsrc && pa < nsrc, okb = qb < nsrc && pb < nsrc;
    if (qa < nsrc && !oka) set_error(a.ctl, CLEO_ERR_SORT_NONLOCAL, kOOB, qa);
    if (qb < nsrc && !okb) set_error(a.ctl, CLEO_ERR_SORT_NONLOCAL, kOOB, qb);
    const uint32_t sa = oka ? pa : 0u, sb = okb ? pb : 0u;
    const uint32_t ga = a.src.gbx[sa], gb = a.src.gbx[sb];
    const double c3a = a.src.c3[sa], c3b = a.src.c3[sb];
    const double c1a = a.src.c1[sa], c1b = a.src.c1[sb];
    const double c2a = a.src.c2[sa], c2b = a.src.c2[sb];
    const uint64_t xia = a.src.xi[sa], xib = a.src.xi[sb];
    const double ra = a.src.r[sa], rb = a.src.r[sb];
    const double ma = a.src.msol[sa], mb = a.src.msol[sb];
    const uint64_t ida = a.src.id[sa], idb = a.src.id[sb];
    if (oka) {
      a.dst.gbx[qa] = ga;
      a.dst.c3[qa] = c3a;
      a.dst.c1[qa] = c1a;
      a.dst.c2[qa] = c2a;
      a.dst.xi[qa] = xia;
      a.dst.r[qa] = ra;
      a.dst.msol[qa] = ma;
      a.dst.id[qa] = ida;
    }
    if (okb) {
      a.dst.gbx[qb] = gb;
      a.dst.c3[qb] = c3b;
      a.dst.c1[qb] = c1b;
      a.dst.c2[qb] = c2b;
      a.dst.xi[qb] = xib;
      a.dst.r[qb] = rb;
      a.dst.msol[qb] = mb;
      a.dst.id[qb] = idb;
    }
  }
  copy_oob(a, nsrc);
}

// Second pass of the fused motion + sort (the first is k_motion_drops<false>): the drops of
// gridbox g move again, with the arithmetic of the counting pass, and go with their new coordinates
// and gridbox straight to their place in the sorted store.  The place is the start of the
// (destination, step) run left in the count table by k_nsort_tot plus the drop's rank among this
// gridbox's drops that took the same step -- the stable order of the scatter above.
__device__ __forceinline__ void motion_scatter_gbx(const MotionArgs& a, const NsortArgs& n, uint32_t g, int lane) {
  const uint32_t base = a.off[g];
  const uint32_t nfull = a.off[g + 1] - base;
  const GbxGeom G = gbx_geom(a, g);
  uint32_t run = 0;   // lane L < 28: next position of the drops of step L
  uint32_t have = 0;  // bit L: the run of step L has its start
  for (uint32_t c = 0; c < nfull; c += kWave) {
    const uint32_t k = base + c + lane;
    const bool act = c + lane < nfull;
    Moved M{0.0, 0.0, 0.0, 0u, 0};
    if (act) M = move_drop(a, g, G, k, false);
    const int dir = act ? M.dir : -1;
    // the steps present in this chunk; the runs they open get their starts in one round of loads
    uint32_t present = 0;
    uint64_t mask = __ballot(act);
    while (mask) {
      const int leader = __ffsll(static_cast<unsigned long long>(mask)) - 1;
      const int v = static_cast<int>(readlane_u32(static_cast<uint32_t>(dir), leader));
      present |= 1u << v;
      mask &= ~__ballot(act && dir == v);
    }
    const uint32_t need = present & ~have;
    if (lane < 28 && ((need >> lane) & 1u)) {
      if (lane == 27) {
        run = n.off_new[a.grid.ngbx] + n.oobpre[g];
      } else {
        const uint32_t d = neighbour_of(a.grid, g, lane);
        run = n.off_new[d] + n.runs[28ull * g + lane];
      }
    }
    have |= need;
    uint32_t dest = 0;
    mask = __ballot(act);
    while (mask) {
      const int leader = __ffsll(static_cast<unsigned long long>(mask)) - 1;
      const int v = static_cast<int>(readlane_u32(static_cast<uint32_t>(dir), leader));
      const uint64_t m = __ballot(act && dir == v);
      const uint32_t start = readlane_u32(run, v);
      if ((m >> lane) & 1ull) dest = start + static_cast<uint32_t>(__popcll(m & lanemask_lt()));
      if (lane == v) run += static_cast<uint32_t>(__popcll(m));
      mask &= ~m;
    }
    if (act && dest >= n.ntot) {  // counts inconsistent with the moves: never write out of range
      set_error(n.ctl, CLEO_ERR_SORT_NONLOCAL, g, k);
    } else if (act) {
      n.dst.gbx[dest] = M.idx;
      n.dst.c3[dest] = M.c3;
      n.dst.c1[dest] = M.c1;
      n.dst.c2[dest] = M.c2;
      n.dst.xi[dest] = a.s.xi[k];
      n.dst.r[dest] = a.s.r[k];
      n.dst.msol[dest] = a.s.msol[k];
      n.dst.id[dest] = a.s.id[k];
    }
  }
}
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(4) k_motion_scatter(MotionArgs a, NsortArgs n) {
  const int lane = lane_id();
  for (uint32_t g = wave_index(); g < a.grid.ngbx; g += wave_count()) motion_scatter_gbx(a, n, g, lane);
  copy_oob(n, n.off[a.grid.ngbx]);
}

__global__ void k_set_nact(const uint32_t* off, uint32_t ngbx, uint32_t* nact, DevCtl* ctl, bool upload) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < ngbx) nact[g] = off[g + 1] - off[g];
  if (g == 0) ctl->stats[ST_SORTS] = upload ? 0 : ctl->stats[ST_SORTS] + 1;
}
__global__ void k_publish_ctl(const DevCtl* ctl, const uint32_t* off, uint32_t ngbx, HostCtl* out) {
  constexpr uint32_t kWords = sizeof(DevCtl) / 4;
  static_assert(kWords <= kWave, "one word per lane");
  if (threadIdx.x < kWords) reinterpret_cast<uint32_t*>(&out->ctl)[threadIdx.x] = reinterpret_cast<const uint32_t*>(ctl)[threadIdx.x];
  if (threadIdx.x == 0) out->ndomain = off[ngbx];
}
__global__ void k_set_event(DevCtl* ctl, uint64_t event) { ctl->event = event; }

// ============================ generic stable radix sort =======================================
// LSD radix sort of (key, position) with digits of up to 8 bits, three launches per pass: digit counts
// of every tile of kRsTile keys, their prefixes along each digit's row of tiles, and the scatter.  A
// wave takes its keys 64 at a time in order; lanes with equal digits find each other with one ballot
// per bit, so the rank of a key among its tile's equal digits needs no atomics and is stable.  (4-bit
// digits with a three-level scan of the counts took twice the passes and 20 launches; 1M drops of
// 32768 gridboxes in random order: 245 us, now 122.)
constexpr uint32_t kRsItems = 8, kRsTile = 256 * kRsItems, kRsDigits = 256;
static_assert(kRsTile == kRadixTile, "tile of the radix sort");
// the digit's key: the drop's gridbox, or ngbx behind all gridboxes (_get_count_position,
// sortsupers.hpp:44-48)
template <bool kFirst>
__device__ __forceinline__ uint32_t rs_key(const uint32_t* key, uint64_t p, uint32_t ngbx) {
  const uint32_t k = key[p];
  return kFirst && k >= ngbx ? ngbx : k;
}
// the active lanes whose digit (`bits` wide) equals this lane's
__device__ __forceinline__ uint64_t rs_match(uint32_t digit, int bits, bool act) {
  uint64_t m = ballot(act);
  for (int b = 0; b < bits; ++b) {
    const uint64_t x = ballot((digit >> b) & 1u);
    m &= ((digit >> b) & 1u) ? x : ~x;
  }
  return m;
}
// a drop as one 64-byte row, for the gather of drops in random order
struct alignas(16) DropRow {
  double c3, c1, c2, r, msol;
  uint64_t xi, id;
  uint32_t gbx, pad;
};
static_assert(sizeof(DropRow) == 4u * kDropRowWords, "row of a drop");

// first pass (kFirst): `key` is the drops' gridbox field, and with `rows` the drops are also laid out
// as rows there
template <bool kFirst>
__global__ void __launch_bounds__(256) k_rs_count(const uint32_t* key, uint64_t n, uint32_t ngbx, int shift, int bits,
                                                  uint32_t ntiles, uint32_t* cnt, SoA src, DropRow* rows) {
  __shared__ uint32_t cw[4][kRsDigits];
  const uint32_t w = threadIdx.x >> 6, nd = 1u << bits;
  const int lane = lane_id();
  for (uint32_t d = threadIdx.x; d < 4u * kRsDigits; d += 256u) (&cw[0][0])[d] = 0u;
  __syncthreads();
  const uint64_t p0 = static_cast<uint64_t>(blockIdx.x) * kRsTile + w * (kRsTile / 4u) + static_cast<uint32_t>(lane);
  uint32_t k[kRsItems];
#pragma unroll
  for (uint32_t i = 0; i < kRsItems; ++i) k[i] = p0 + i * kWave < n ? rs_key<kFirst>(key, p0 + i * kWave, ngbx) : 0u;
#pragma unroll
  for (uint32_t i = 0; i < kRsItems; ++i) {
    const bool act = p0 + i * kWave < n;
    const uint32_t d = (k[i] >> shift) & (nd - 1u);
    const uint64_t m = rs_match(d, bits, act);
    if (act && lanes_below(m) == 0u) cw[w][d] += static_cast<uint32_t>(__popcll(m));
    wave_sync();
  }
  if (kFirst && rows) {
    for (uint32_t i = 0; i < kRsItems; ++i) {
      const uint64_t p = p0 + i * kWave;
      if (p < n)
        rows[p] = DropRow{src.c3[p], src.c1[p], src.c2[p], src.r[p], src.msol[p], src.xi[p], src.id[p], src.gbx[p], 0u};
    }
  }
  __syncthreads();
  if (threadIdx.x < nd) {
    const uint32_t d = threadIdx.x;
    cnt[static_cast<uint64_t>(d) * ntiles + blockIdx.x] = cw[0][d] + cw[1][d] + cw[2][d] + cw[3][d];
  }
}
// row blockIdx.x of the counts to its exclusive prefix, its total to totals[blockIdx.x]
__global__ void __launch_bounds__(1024) k_rs_rows(uint32_t* cnt, uint32_t ntiles, uint32_t* totals) {
  __shared__ uint32_t ws[16];
  uint32_t* row = cnt + static_cast<uint64_t>(blockIdx.x) * ntiles;
  uint32_t run = 0;
  for (uint32_t t0 = 0; t0 < ntiles; t0 += 4096u) {
    const uint32_t t = t0 + 4u * threadIdx.x;
    uint32_t v[4], sum = 0, all;
    for (uint32_t i = 0; i < 4; ++i) {
      v[i] = t + i < ntiles ? row[t + i] : 0u;
      sum += v[i];
    }
    uint32_t at = run + block_excl_scan(sum, ws, all);
    for (uint32_t i = 0; i < 4; ++i) {
      if (t + i < ntiles) row[t + i] = at;
      at += v[i];
    }
    run += all;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = run;
}
template <bool kFirst>
__global__ void __launch_bounds__(256) k_rs_scatter(const uint32_t* key, const uint32_t* idx, uint64_t n, uint32_t ngbx,
                                                    int shift, int bits, uint32_t ntiles, const uint32_t* cnt,
                                                    const uint32_t* totals, uint32_t* key2, uint32_t* idx2) {
  __shared__ uint32_t cw[4][kRsDigits], ws[4];
  const uint32_t w = threadIdx.x >> 6, nd = 1u << bits;
  const int lane = lane_id();
  for (uint32_t d = threadIdx.x; d < 4u * kRsDigits; d += 256u) (&cw[0][0])[d] = 0u;
  // first place of each digit: those of the lower digits, then those of earlier tiles
  const uint32_t mine = threadIdx.x < nd ? totals[threadIdx.x] : 0u;
  const uint32_t before = threadIdx.x < nd ? cnt[static_cast<uint64_t>(threadIdx.x) * ntiles + blockIdx.x] : 0u;
  const uint64_t p0 = static_cast<uint64_t>(blockIdx.x) * kRsTile + w * (kRsTile / 4u) + static_cast<uint32_t>(lane);
  uint32_t k[kRsItems], at[kRsItems], rank[kRsItems];
#pragma unroll
  for (uint32_t i = 0; i < kRsItems; ++i) {
    const uint64_t p = p0 + i * kWave;
    k[i] = p < n ? rs_key<kFirst>(key, p, ngbx) : 0u;
    at[i] = kFirst ? static_cast<uint32_t>(p) : (p < n ? idx[p] : 0u);
  }
  uint32_t all;
  const uint32_t base = block_excl_scan(mine, ws, all) + before;  // (synchronises: cw is zero)
#pragma unroll
  for (uint32_t i = 0; i < kRsItems; ++i) {
    const bool act = p0 + i * kWave < n;
    const uint32_t d = (k[i] >> shift) & (nd - 1u);
    const uint64_t m = rs_match(d, bits, act);
    const uint32_t below = lanes_below(m), old = cw[w][d];
    rank[i] = old + below;
    wave_sync();
    if (act && below == 0u) cw[w][d] = old + static_cast<uint32_t>(__popcll(m));
    wave_sync();
  }
  __syncthreads();
  if (threadIdx.x < nd) {
    uint32_t a = base;
    for (uint32_t v = 0; v < 4; ++v) {
      const uint32_t c = cw[v][threadIdx.x];
      cw[v][threadIdx.x] = a;
      a += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kRsItems; ++i) {
    if (p0 + i * kWave < n) {
      const uint32_t dst = cw[w][(k[i] >> shift) & (nd - 1u)] + rank[i];
      if (dst < n) {
        key2[dst] = k[i];
        idx2[dst] = at[i];
      }
    }
  }
}

// The sorted drops to dst, from the store, or from their rows (each drop then touches one line instead
// of eight: 143 -> 32 us on 1M drops in random order, for 23 us more in the first count), and off[b] =
// first position with key >= b, b = 0..ngbx (find_refs / find_domainrefs, findrefs.hpp), by bisection of
// the sorted keys.
__global__ void __launch_bounds__(256) k_rs_gather(SoA src, const DropRow* rows, SoA dst, const uint32_t* key,
                                                   const uint32_t* idx, uint64_t n, uint32_t ngbx, uint32_t* off) {
  const uint64_t first = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x,
                 stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  if (rows) {
    for (uint64_t p = first; p < n; p += stride) {
      const DropRow d = rows[idx[p]];
      dst.gbx[p] = d.gbx;
      dst.c3[p] = d.c3;
      dst.c1[p] = d.c1;
      dst.c2[p] = d.c2;
      dst.xi[p] = d.xi;
      dst.r[p] = d.r;
      dst.msol[p] = d.msol;
      dst.id[p] = d.id;
    }
  } else {
    for (uint64_t p = first; p < n; p += stride) copy_drop(src, dst, idx[p], p);
  }
  for (uint64_t b = first; b <= ngbx; b += stride) {
    uint64_t lo = 0, hi = n;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) / 2;
      if (key[mid] < b)
        lo = mid + 1;
      else
        hi = mid;
    }
    off[b] = static_cast<uint32_t>(lo);
  }
}

// ============================ scan (exclusive, u32) ===========================================
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ uint32_t load_in(const uint32_t* in, uint64_t i, uint32_t stride, uint32_t offset,
                                            uint64_t len) {
  return i < len ? in[i * stride + offset] : 0u;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(const uint32_t* in, uint64_t len, uint32_t stride,
                                                              uint32_t offset, uint32_t* partial) {
  __shared__ uint32_t ws[4];
  const uint64_t t0 = static_cast<uint64_t>(blockIdx.x) * kScanTile;
  uint32_t s = 0;
  for (int i = 0; i < kScanItems; ++i) s += load_in(in, t0 + i * kScanThreads + threadIdx.x, stride, offset, len);
  s = wave_sum_u32(s);
  if (lane_id() == 0) ws[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ void __launch_bounds__(kScanThreads) k_scan_apply(const uint32_t* in, uint64_t len, uint32_t stride,
                                                             uint32_t offset, const uint32_t* block_off,
                                                             uint32_t* out) {
  __shared__ uint32_t ws[4];
  const uint64_t t0 = static_cast<uint64_t>(blockIdx.x) * kScanTile;
  // each thread owns kScanItems consecutive items
  uint32_t v[kScanItems];
  uint32_t s = 0;
  for (int i = 0; i < kScanItems; ++i) {
    v[i] = load_in(in, t0 + static_cast<uint64_t>(threadIdx.x) * kScanItems + i, stride, offset, len);
    s += v[i];
  }
  // inclusive wave scan of per-thread sums
  const int lane = lane_id();
  uint32_t incl = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o);
    if (lane >= o) incl += y;
  }
  if (lane == 63) ws[threadIdx.x >> 6] = incl;
  __syncthreads();
  uint32_t pre = block_off ? block_off[blockIdx.x] : 0u;
  for (int ww = 0; ww < static_cast<int>(threadIdx.x >> 6); ++ww) pre += ws[ww];
  uint32_t run = pre + incl - s;
  for (int i = 0; i < kScanItems; ++i) {
    const uint64_t idx = t0 + static_cast<uint64_t>(threadIdx.x) * kScanItems + i;
    if (idx < len) out[idx] = run;
    run += v[i];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanThreads - 1) out[len] = run;
}

}  // namespace cleo

// ============================ host-side launchers =============================================
namespace cleo {

static inline unsigned nblocks(uint64_t n, uint64_t per) {
  const uint64_t b = (n + per - 1) / per;
  return static_cast<unsigned>(b == 0 ? 1 : b);
}
__global__ void k_iota_u32(uint32_t* p, uint64_t n);
template <bool kWrite>
static void launch_motion_drops(cleo_ctx* c, const MotionArgs& a, unsigned nb);
static void launch_gather_move(cleo_ctx* c, const NsortArgs& n, const MotionArgs& m);
// blocks of the motion drop loop (two drops per thread), capped at `grid_waves` waves when non-zero
static inline unsigned motion_blocks(uint64_t n, uint32_t grid_waves) {
  const unsigned b = nblocks(n, 512);
  return grid_waves ? std::min<unsigned>(b, std::max<unsigned>(1u, grid_waves / 4)) : b;
}

// events around the main kernel of a stage (stage timing), recorded only while kev_on is set
static inline void kev_mark(cleo_ctx* c, int i) {
  if (c->kev_on) (void)hipEventRecord(c->kev[i], c->stream);
}
// blocks of a gridbox loop: one wave per gridbox, capped at `grid_waves` waves when non-zero
static inline unsigned gbx_blocks(uint64_t ngbx, uint32_t wpb, uint32_t grid_waves) {
  const unsigned b = nblocks(ngbx, wpb);
  return grid_waves ? std::min<unsigned>(b, std::max<unsigned>(1u, grid_waves / wpb)) : b;
}
// blocks of 256 threads of a drop loop: one thread per drop, capped at `grid_waves` waves
static inline unsigned drop_blocks(uint64_t n, uint32_t grid_waves) {
  const unsigned b = nblocks(n, 256);
  return grid_waves ? std::min<unsigned>(b, std::max<unsigned>(1u, grid_waves / 4)) : b;
}
static void launch_nsort_perm(cleo_ctx* c, const NsortArgs& a, uint32_t ngbx) {
  const dim3 grid(gbx_blocks(ngbx, a.wpb, c->tiles.motion_grid_waves)), block(64 * a.wpb);
  if (a.order)
    hipLaunchKernelGGL(k_nsort_perm<true>, grid, block, 0, c->stream, a);
  else
    hipLaunchKernelGGL(k_nsort_perm<false>, grid, block, 0, c->stream, a);
}
static inline unsigned stride_blocks(uint64_t n) {
  const uint64_t b = (n + 255) / 256;
  return static_cast<unsigned>(b == 0 ? 1 : (b > 65536 ? 65536 : b));
}
// blocks of a grid-stride loop that usually has nothing to do (the re-sort after collisions).
// 2048 blocks of 256 threads still fill every CU when the work is there; a launch of many
// thousands of blocks that exit at once costs tens of microseconds.
static inline unsigned sparse_blocks(uint64_t n) { return std::min<unsigned>(stride_blocks(n), 2048u); }

__global__ void k_set_u32(uint32_t* out, uint32_t v) { *out = v; }

// Gridboxes per tile of the per-gridbox sums: as many as leave 8192 waves, but at least the 512 drops
// of a window.  Mass moments with 64 / by this rule / 1 gridbox per tile: 32^3 gridboxes of 64 drops
// 41 / 17 / 51 us, 24679 of 300 drops 478 (at 256 waves) / 96 / 115 us, 3750 of 128 drops 160 / 12 /
// 14 us; from 64^3 gridboxes on the passes are bound by HBM at any width (134M drops: 0.59 ms).
static uint32_t sum_gpt(const cleo_ctx* c) {
  const uint64_t ngbx = c->grid.ngbx, mean = std::max<uint64_t>(1, c->ntot / ngbx);
  return static_cast<uint32_t>(std::min<uint64_t>(kWave, std::max<uint64_t>({1, ngbx / 8192, 512 / mean})));
}
static unsigned sum_blocks(const cleo_ctx* c, uint32_t grid_waves) {
  return gbx_blocks(sum_tiles(c->grid.ngbx, sum_gpt(c)), 4, grid_waves);
}
void launch_qcond(cleo_ctx* c, const QcondArgs& args) {
  if (args.ngbx == 0) return;
  QcondArgs a = args;
  a.gpt = sum_gpt(c);
  hipLaunchKernelGGL(k_qcond, dim3(sum_blocks(c, c->tiles.cond_grid_waves)), dim3(256), 0, c->stream, a);
}
template <int B, bool Kinetic>
static void launch_coll_team_k(cleo_ctx* c, const CollArgs& a, unsigned nb, uint32_t gpt, uint32_t cap) {
  const size_t lds = static_cast<size_t>(cap) * kFyItemBytes;
  kev_mark(c, 0);
  hipLaunchKernelGGL((k_coll_team<B, Kinetic>), dim3(nb), dim3(B), lds, c->stream, a, gpt, cap);
  kev_mark(c, 1);
}
template <int B>
static void launch_coll_team(cleo_ctx* c, const CollArgs& args, uint32_t gpt, uint64_t items) {
  CollArgs a = args;
  const uint32_t cap = static_cast<uint32_t>(std::min<uint64_t>(kTeamMaxItems, (items + 63) / 64 * 64));
  const unsigned nb = gbx_blocks(a.ngbx, gpt, 0);
  a.stat = stat_slots(c);
  if (coll_is_kinetic(a.k))
    launch_coll_team_k<B, true>(c, a, nb, gpt, cap);
  else
    launch_coll_team_k<B, false>(c, a, nb, gpt, cap);
}
template <int B>
static void launch_coll_split(cleo_ctx* c, const CollArgs& args, uint32_t split, uint64_t items) {
  CollArgs a = args;
  const uint32_t cap = static_cast<uint32_t>(std::min<uint64_t>(kSplitMaxItems, (items + 63) / 64 * 64));
  a.stat = stat_slots(c);
  a.share = c->coll_share;
  kev_mark(c, 0);
  if (coll_is_kinetic(a.k))
    hipLaunchKernelGGL((k_coll_split<B, true>), dim3(a.ngbx * split), dim3(B), cap * kSplitItemBytes, c->stream, a, split, cap);
  else
    hipLaunchKernelGGL((k_coll_split<B, false>), dim3(a.ngbx * split), dim3(B), cap * kSplitItemBytes, c->stream, a, split, cap);
  kev_mark(c, 1);
}
// Tiles give the least work per drop (33.5M drops: 0.25 ms, teams 0.56), but a wave walks through its 64
// gridboxes' swaps and pairs in about 1.2 us per drop of the mean, so they need enough gridboxes to fill
// the chip (32^3 gridboxes of 64: 81 us against 45 us; the lines cross near 75,000 gridboxes at any mean)
// whose drops fit a tile's 8 KB of permutations.
bool coll_takes_tiles(const cleo_ctx* c) {
  const uint64_t ngbx = c->grid.ngbx;
  return ngbx >= kTileMinGbx && c->ntot / ngbx <= kTilePermBytes / kWave + 4;
}
void launch_collisions(cleo_ctx* c, const CollArgs& args) {
  if (args.ngbx == 0) return;
  CollArgs a = args;
  const uint64_t mean = std::max<uint64_t>(1, c->ntot / a.ngbx);
  if (coll_takes_tiles(c)) {
    const unsigned nb = gbx_blocks((a.ngbx + kWave - 1) / kWave, a.wpb, c->tiles.coll_grid_waves);
    a.stat = stat_slots(c);
    kev_mark(c, 0);
    if (coll_is_kinetic(a.k))
      hipLaunchKernelGGL(k_coll_tiles<true>, dim3(nb), dim3(64 * a.wpb), a.wpb * kCollTileLdsBytes, c->stream, a);
    else
      hipLaunchKernelGGL(k_coll_tiles<false>, dim3(nb), dim3(64 * a.wpb), a.wpb * kCollTileLdsBytes, c->stream, a);
    kev_mark(c, 1);
    return;
  }
  // Teams, one workgroup each.  A wave takes as many gridboxes as make 512 drops (128 to 1024 tried:
  // 55, 49, 45, 68 us on 32^3 gridboxes of 64), but no more than leave 4096 teams (3750 gridboxes of
  // 128: 18 us with one each, 33 us with four).  With few gridboxes, or larger ones, a workgroup takes
  // the pairs of one gridbox.
  if (mean <= 512 && (mean <= 96 || a.ngbx > 512)) {
    const uint64_t gpt = std::min<uint64_t>(kWave, std::max<uint64_t>(1, std::min<uint64_t>(512 / mean, a.ngbx / 4096)));
    const double items = static_cast<double>(gpt * mean);
    launch_coll_team<kWave>(c, a, static_cast<uint32_t>(gpt), static_cast<uint64_t>(items + 6.0 * std::sqrt(items)) + 128);
  } else if (mean <= 512 || (mean <= 2048 && a.ngbx > kSplitGbx)) {
    launch_coll_team<256>(c, a, 1u, 2 * mean);
  } else {
    // Large gridboxes: as many lanes as the chip has room for, and one more workgroup per 1024 drops
    // of a gridbox while 128 of them stay free of each other (us by team / 512 lanes / 1024 lanes /
    // 1024 lanes in shares; 1 gridbox of 1000 drops 16.1 / 13.6 / 13.8 / 14.8, of 2000 26.9 / 19.7 /
    // 16.6 / 18.2, of 8192 39.7 / 45.1 / 31.9 / 20.7, of 14000 62.8 / 71.4 / 48.6 / 23.2; 64 of 5000
    // 29.3 / 37.0 / 25.9 / 25.7; 512 of 1500 27.3 / 22.6 / 30.4; 400 of 3000 38.9 / 32.3 / 37.4).
    if (a.ngbx <= 256 && mean > 1024)
      launch_coll_split<1024>(c, a, static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(mean / 1024, 128 / a.ngbx))), 2 * mean);
    else
      launch_coll_split<512>(c, a, 1u, 2 * mean);
  }
}
StatSlots stat_slots(cleo_ctx* c) { return StatSlots{c->sp}; }
// (their own status, as hipGetLastError may hold an error that another call of the thread left)
hipError_t launch_publish_ctl(cleo_ctx* c) {
  const DevCtl* ctl = c->ctl;
  const uint32_t* off = c->off;
  uint32_t ngbx = c->grid.ngbx;
  HostCtl* out = c->h_ctl;
  void* args[] = {&ctl, &off, &ngbx, &out};
  return hipLaunchKernel(reinterpret_cast<const void*>(k_publish_ctl), dim3(1), dim3(64), args, 0, c->stream);
}
hipError_t launch_set_event(cleo_ctx* c, uint64_t event) {
  void* args[] = {&c->ctl, &event};
  return hipLaunchKernel(reinterpret_cast<const void*>(k_set_event), dim3(1), dim3(1), args, 0, c->stream);
}
void launch_inj_sizes(cleo_ctx* c, uint32_t* nj, uint32_t* np) {
  hipLaunchKernelGGL(k_inj_sizes, dim3(nblocks(c->grid.ngbx, 256)), dim3(256), 0, c->stream, c->nact, c->grid.ngbx, nj, np);
}

void launch_inj_long(cleo_ctx* c, const CollArgs& a) {
  hipLaunchKernelGGL(k_inj_long, dim3(std::min<uint32_t>(a.ngbx, 4096u)), dim3(256), 0, c->stream, a, c->order, c->inj_j);
}

static size_t scan_words_rec(uint64_t len) {
  const uint64_t nb = (len + kScanTile - 1) / kScanTile;
  if (nb <= 1) return 0;
  return nb + (nb + 1) + scan_words_rec(nb);
}
size_t scan_tmp_words(uint64_t len) { return scan_words_rec(len) + 16; }

static void scan_rec(hipStream_t stream, const uint32_t* in, uint64_t len, uint32_t stride, uint32_t offset,
                     uint32_t* out, uint32_t* tmp) {
  if (len == 0) {
    hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(1), 0, stream, out, 0u);
    return;
  }
  const uint64_t nb = (len + kScanTile - 1) / kScanTile;
  if (nb == 1) {
    hipLaunchKernelGGL(k_scan_apply, dim3(1), dim3(kScanThreads), 0, stream, in, len, stride, offset,
                       static_cast<const uint32_t*>(nullptr), out);
    return;
  }
  uint32_t* partial = tmp;
  uint32_t* pscan = tmp + nb;
  hipLaunchKernelGGL(k_scan_reduce, dim3(static_cast<unsigned>(nb)), dim3(kScanThreads), 0, stream, in, len, stride,
                     offset, partial);
  scan_rec(stream, partial, nb, 1u, 0u, pscan, tmp + nb + nb + 1);
  hipLaunchKernelGGL(k_scan_apply, dim3(static_cast<unsigned>(nb)), dim3(kScanThreads), 0, stream, in, len, stride,
                     offset, static_cast<const uint32_t*>(pscan), out);
}
void scan_u32(cleo_ctx* c, const uint32_t* in, uint64_t len, uint32_t stride, uint32_t offset, uint32_t* out) {
  scan_rec(c->stream, in, len, stride, offset, out, c->scan_tmp);
}

// Whether the count table is left zero by the sort that reads it, rather than filled before motion: a
// launch less, but on large domains motion's atomics then find the table in HBM and not in a cache that
// a fill has just written (524288 gridboxes: motion 515 us against 478 us and 16 us for the fill).
static bool counts_stay_clear(const cleo_ctx* c) { return c->grid.ngbx <= 65536u; }
__global__ void __launch_bounds__(256) k_fill_u32x4(uint4* p, uint64_t n) {
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    p[i] = uint4{0u, 0u, 0u, 0u};
}
// the counts of the next motion start from zero
static void clear_counts(cleo_ctx* c) {
  if (counts_stay_clear(c)) return;
  const uint64_t n = 7ull * c->grid.ngbx;
  hipLaunchKernelGGL(k_fill_u32x4, dim3(stride_blocks(n)), dim3(256), 0, c->stream, reinterpret_cast<uint4*>(c->cnt), n);
}
// argument block of the neighbour-sort kernels reading `src` and writing `dst`
static NsortArgs nsort_args(cleo_ctx* c, const SoA& src, const SoA& dst) {
  NsortArgs a{};
  a.src = src;
  a.dst = dst;
  a.off = c->off;
  a.off_new = c->off_alt;
  a.nact = c->nact;
  a.cnt = c->cnt;
  a.runs = c->cnt + 28ull * c->grid.ngbx;
  a.oobpre = c->oobpre;
  a.part = c->part;
  a.nblk = nblocks(c->grid.ngbx, kTabBlock);
  a.clear = counts_stay_clear(c) ? 1u : 0u;
  a.grid = c->grid;
  a.wpb = c->tiles.motion_waves_per_block ? c->tiles.motion_waves_per_block : 1;
  a.ctl = c->ctl;
  a.ntot = c->ntot;
  a.perm = c->perm;
  a.order = c->order_live ? c->order : nullptr;
  return a;
}
// totals per destination, run offsets and the prefixes they start from; with `gs`, the condensation
// inputs of every gridbox too
static void nsort_tables(cleo_ctx* c, const NsortArgs& a, double* gs = nullptr) {
  if (gs)
    hipLaunchKernelGGL(k_nsort_tot<true>, dim3(2 * a.nblk), dim3(kTabBlock), 0, c->stream, a, c->st, gs);
  else
    hipLaunchKernelGGL(k_nsort_tot<false>, dim3(a.nblk), dim3(kTabBlock), 0, c->stream, a, GState{}, gs);
  if (a.nblk > kApplyBlocks) {
    hipLaunchKernelGGL(k_nsort_part, dim3(1), dim3(1024), 0, c->stream, a.part, a.nblk);
    hipLaunchKernelGGL(k_nsort_apply<true>, dim3(a.nblk), dim3(kTabBlock), 0, c->stream, a);
  } else if (a.nblk > 1) {
    hipLaunchKernelGGL(k_nsort_apply<false>, dim3(a.nblk), dim3(kTabBlock), 0, c->stream, a);
  }
}
// the sorted store in buffer `dst` becomes current, with the refs its sort wrote
static void nsort_commit(cleo_ctx* c, int dst) {
  c->cur = dst;
  c->order_live = false;  // the sorted store is in its logical order
  std::swap(c->off, c->off_alt);
}

void neighbour_sort_to(cleo_ctx* c, const SoA& src, const SoA& dst, int commit_dst, const uint8_t* step) {
  NsortArgs a = nsort_args(c, src, dst);
  a.step = step;
  nsort_tables(c, a);
  launch_nsort_perm(c, a, c->grid.ngbx);
  // streaming copy: one pair of positions per thread (measured faster than a capped grid)
  hipLaunchKernelGGL(k_nsort_gather, dim3(motion_blocks(c->ntot, 0)), dim3(256), 0, c->stream, a);
  if (commit_dst >= 0) nsort_commit(c, commit_dst);
}

void resort_nulls(cleo_ctx* c, uint32_t events) {
  const uint32_t ngbx = c->grid.ngbx;
  const bool one = c->ntot <= kResortOneDrops && ngbx <= kResortOneDrops;
  uint32_t shift = one ? 31u : 0u;
  while (((ngbx - 1u) >> shift) >= kResortSegs) ++shift;
  // the condensation inputs are free at the end of a pass: eight words per gridbox, two taken per segment
  const Resort r{c->ctl, c->buf[c->cur], c->buf[1 - c->cur], c->off, c->nact, c->off_alt,
                 c->order_live ? c->order : nullptr, ngbx, c->big_scratch, reinterpret_cast<uint32_t*>(c->gs), shift};
  if (one) {
    hipLaunchKernelGGL(k_resort_one, dim3(1), dim3(1024), 0, c->stream, r, events);
    return;
  }
  hipLaunchKernelGGL(k_resort_gather, dim3(kResortBlocks), dim3(kResortLanes), 0, c->stream, r, events);
  hipLaunchKernelGGL(k_resort_back, dim3(kResortBlocks), dim3(kResortLanes), 0, c->stream, r);
}

// the store as it is, with the identity as its pending order
void pending_identity_order(cleo_ctx* c) {
  hipLaunchKernelGGL(k_iota_u32, dim3(stride_blocks(c->ntot)), dim3(256), 0, c->stream, c->order, c->ntot);
  c->order_live = true;
}
// A pending collision order applied: the domain's drops are gathered into the other buffer in
// their logical order (the out-of-domain drops are copied as they are) and that buffer becomes
// current.  Nothing happens when the store is already in order.
void materialize_order(cleo_ctx* c) {
  if (!c->order_live) return;
  const int src = c->cur, dst = 1 - c->cur;
  NsortArgs a = nsort_args(c, c->buf[src], c->buf[dst]);
  a.perm = c->order;
  hipLaunchKernelGGL(k_nsort_gather, dim3(motion_blocks(c->ntot, 0)), dim3(256), 0, c->stream, a);
  c->cur = dst;
  c->order_live = false;
}

// Motion + neighbour sort in two passes over the drops: count the moves, build the tables, then
// move again and write each drop to its sorted place in `dst` (src is left unchanged).
// commit_dst >= 0: that buffer becomes current.
void motion_sort_fused(cleo_ctx* c, const MotionArgs& args, const SoA& dst, int commit_dst) {
  const uint32_t ngbx = c->grid.ngbx;
  MotionArgs a = args;
  const unsigned nb = motion_blocks(c->ntot, c->tiles.motion_grid_waves);
  a.stat = stat_slots(c);
  launch_motion_drops<false>(c, a, nb);
  NsortArgs n = nsort_args(c, a.s, dst);
  nsort_tables(c, n);
  kev_mark(c, 0);
  hipLaunchKernelGGL(k_motion_scatter, dim3(gbx_blocks(ngbx, n.wpb, c->tiles.motion_grid_waves)), dim3(64 * n.wpb), 0,
                     c->stream, a, n);
  kev_mark(c, 1);
  if (commit_dst >= 0) nsort_commit(c, commit_dst);
}

// Motion + neighbour sort with the motion arithmetic in the gather (motion_flat 3): a counting
// pass records each drop's step (nothing of the store changes), the tables and the rank pass
// follow, and the gather moves each drop again as it writes it to its sorted place in `dst`.
// commit_dst >= 0: that buffer becomes current.
void motion_sort_gather(cleo_ctx* c, const MotionArgs& args, const SoA& dst, int commit_dst) {
  const uint32_t ngbx = c->grid.ngbx;
  if (ngbx == 0) return;
  MotionArgs a = args;
  a.step = c->dstep;
  const unsigned nb = motion_blocks(c->ntot, c->tiles.motion_grid_waves);
  a.stat = stat_slots(c);
  kev_mark(c, 0);
  launch_motion_drops<false>(c, a, nb);
  kev_mark(c, 1);
  NsortArgs n = nsort_args(c, a.s, dst);
  n.step = c->dstep;
  nsort_tables(c, n);
  launch_nsort_perm(c, n, ngbx);
  launch_gather_move(c, n, a);
  if (commit_dst >= 0) nsort_commit(c, commit_dst);
}

RadixScratch radix_scratch_at(uint32_t* base, uint64_t n) {
  RadixScratch sc{};
  sc.rows = base;
  sc.key[0] = base + kDropRowWords * n;
  sc.key[1] = sc.key[0] + n;
  sc.idx[0] = sc.key[1] + n;
  sc.idx[1] = sc.idx[0] + n;
  sc.cnt = sc.idx[1] + n;
  return sc;
}

// stable LSD radix sort of the drops of `src` by sdgbxindex (keys >= ngbx in one bucket after every
// gridbox, as _get_count_position, sortsupers.hpp:44-48), gathered into `dst`, with off[0..ngbx]
// the first position of each bucket (find_refs, findrefs.hpp)
void radix_sort_soa(hipStream_t stream, const SoA& src, const SoA& dst, uint64_t n, uint32_t ngbx, uint32_t* off,
                    const RadixScratch& sc) {
  const uint32_t ntiles = static_cast<uint32_t>((n + kRsTile - 1) / kRsTile);
  DropRow* rows = reinterpret_cast<DropRow*>(sc.rows);
  int bits = 1;
  while (bits < 32 && (ngbx >> bits) != 0) ++bits;
  const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
  uint32_t* totals = sc.cnt + static_cast<uint64_t>(kRsDigits) * ntiles;
  int cur = 0;
  for (int p = 0; p < passes && n > 0; ++p) {
    const int shift = p * width;
    if (p == 0)
      hipLaunchKernelGGL(k_rs_count<true>, dim3(ntiles), dim3(256), 0, stream, static_cast<const uint32_t*>(src.gbx), n,
                         ngbx, shift, width, ntiles, sc.cnt, src, rows);
    else
      hipLaunchKernelGGL(k_rs_count<false>, dim3(ntiles), dim3(256), 0, stream,
                         static_cast<const uint32_t*>(sc.key[cur]), n, ngbx, shift, width, ntiles, sc.cnt, SoA{},
                         static_cast<DropRow*>(nullptr));
    hipLaunchKernelGGL(k_rs_rows, dim3(1u << width), dim3(1024), 0, stream, sc.cnt, ntiles, totals);
    if (p == 0)
      hipLaunchKernelGGL(k_rs_scatter<true>, dim3(ntiles), dim3(256), 0, stream, static_cast<const uint32_t*>(src.gbx),
                         static_cast<const uint32_t*>(nullptr), n, ngbx, shift, width, ntiles, sc.cnt, totals, sc.key[0],
                         sc.idx[0]);
    else
      hipLaunchKernelGGL(k_rs_scatter<false>, dim3(ntiles), dim3(256), 0, stream, sc.key[cur], sc.idx[cur], n, ngbx,
                         shift, width, ntiles, sc.cnt, totals, sc.key[1 - cur], sc.idx[1 - cur]);
    if (p > 0) cur = 1 - cur;
  }
  hipLaunchKernelGGL(k_rs_gather, dim3(stride_blocks(std::max<uint64_t>(n, ngbx + 1ull))), dim3(256), 0, stream, src, rows,
                     dst, sc.key[cur], sc.idx[cur], n, ngbx, off);
}

void generic_sort(cleo_ctx* c, const SoA& src, bool upload) {
  const uint64_t n = c->ntot;
  const uint32_t ngbx = c->grid.ngbx;
  const int dst = 1 - c->cur;
  RadixScratch sc{};
  for (int i = 0; i < 2; ++i) {
    sc.key[i] = c->rs_key[i];
    sc.idx[i] = c->rs_idx[i];
  }
  sc.cnt = c->rs_cnt;  // no rows: the drops of an upload mostly come in order
  radix_sort_soa(c->stream, src, c->buf[dst], n, ngbx, c->off, sc);
  if (n > 0) c->cur = dst;
  hipLaunchKernelGGL(k_set_nact, dim3(nblocks(ngbx, 256)), dim3(256), 0, c->stream, c->off, ngbx, c->nact, c->ctl, upload);
}

}  // namespace cleo

// ============================ flat (thread-per-drop) variants =================================
namespace cleo {

// per gridbox: optional qcond recompute (ordered, before any radius changes), then the
// saturation ratio and diffusion factor condensation uses (condensation.cpp:44-56)
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(4) k_cond_prep(CondFlatArgs a) {
  __shared__ double win_all[4][kSumWin];
  double* win = win_all[threadIdx.x >> 6];
  const int lane = lane_id();
  const uint32_t gpt = a.gpt, ntiles = sum_tiles(a.ngbx, gpt);
  for (uint32_t tile = wave_index(); tile < ntiles; tile += wave_count()) {
    const uint32_t g0 = tile * gpt, g = g0 + static_cast<uint32_t>(lane);
    const bool valid = static_cast<uint32_t>(lane) < gpt && g < a.ngbx;
    double tot = 0.0;
    const bool qcond_here = a.fuse_qcond && !a.qm;  // else k_cond_state recomputes it from qm
    if (qcond_here) {
      const uint32_t t_lo = a.off[g0], t_hi = a.off[min(g0 + gpt, a.ngbx)];
      const uint32_t lo = valid ? a.off[g] : t_hi, hi = valid ? a.off[g + 1] : t_hi;
      tot = tile_sum(win, t_lo, t_hi, lo, hi - lo, [&](uint32_t k) { return qcond_term(a.s, a.sol, a.ctl, k); }, lane);
    }
    if (valid) {
      const double temp = a.st.temp[g], press = a.st.press[g], qv = a.st.qv[g];
      if (qcond_here) {
        const double rho_cond = tot / a.st.vol[g] * dimless::R0cubed_VOL0;
        a.st.qc[g] = rho_cond / dry_air_density(press, temp, qv);
      }
      if (temp <= 0) set_error(a.ctl, CLEO_ERR_TEMP_NONPOSITIVE, g, a.off[g]);
      gbx_thermo(a.st, g, a.gs);
    }
  }
}

// One active drop k of gridbox g: Koehler factors, Newton solve, radius update, mass change * xi
// into dm[k] (condensation.cpp:44-125).  With cfg.budget the solve may give up (returns false,
// nothing written) so that the drop is solved again, without a budget, by solve_listed.
struct CondStats {
  uint32_t solved, iters, subs, restarts;
};
// The solve of one active drop of gridbox g from its radius r and solute mass msol: Koehler
// factors, Newton, new radius rnew, condensed-mass change * xi (dm) and condensed mass * xi before
// the solve (qm, the drop's term of the qcond recompute).  Errors and the iteration count are
// recorded under position k; xi() gives the multiplicity (read after the solve).  Returns false,
// with nothing recorded, when cfg.budget ran out: the drop is solved again later from the same r.
template <class Xi>
__device__ __forceinline__ bool cond_solve(const CondFlatArgs& a, const NewtonCfg& cfg, uint32_t g, uint64_t k, double r,
                                           double msol, Xi xi_of, double warm, CondStats& st, double& rnew, double& dm,
                                           double& qm) {
  const double s_ratio = a.gs[kGsStride * g], ffactor = a.gs[kGsStride * g + 1];
  const double akoh = a.gs[kGsStride * g + 2], bkoh = kohler_b(msol, a.sol);
  SolveOut o{0, false, false, false, false};
  const double newr =
      solve_condensation(cfg, s_ratio, akoh, bkoh, a.gs[kGsStride * g + 3], ffactor, r, warm, a.warm_limit, o);
  if (o.deferred) return false;
  bool bad = false;
  const double old_m = condensate_mass(r, msol, a.sol, &bad);
  const double xi = static_cast<double>(xi_of());
  qm = old_m * xi;
  rnew = at_least_dry(newr, msol, a.sol);
  dm = (condensate_mass(rnew, msol, a.sol, &bad) - old_m) * xi;
  if (bad) set_error(a.ctl, CLEO_ERR_NEG_CONDENSATE, g, k);
  if (o.maxed) set_error(a.ctl, CLEO_ERR_NEWTON_MAXITERS, g, k);
  if (a.niters) a.niters[k] = o.iters;
  st.iters += o.iters;
  st.subs += o.substep ? 1u : 0u;
  st.restarts += o.restarted ? 1u : 0u;
  st.solved += 1;
  return true;
}
// drop k of the store: its solve, the new radius in place, dm[k] and qm[k]
__device__ __forceinline__ bool cond_drop(const CondFlatArgs& a, const NewtonCfg& cfg, uint32_t g, uint64_t k,
                                          double warm, CondStats& st) {
  double rnew, dm, qm;
  if (!cond_solve(a, cfg, g, k, a.s.r[k], a.s.msol[k], [&] { return a.s.xi[k]; }, warm, st, rnew, dm, qm))
    return false;
  a.s.r[k] = rnew;
  a.dm[k] = dm;
  if (a.qm) a.qm[k] = qm;
  return true;
}
__device__ __forceinline__ void put_cond_stats(const StatSlots& sl, CondStats st) {
  st.solved = wave_sum_u32(st.solved);
  st.iters = wave_sum_u32(st.iters);
  st.subs = wave_sum_u32(st.subs);
  st.restarts = wave_sum_u32(st.restarts);
  if (lane_id() == 0) {
    put_stat(sl, ST_COND_DROPS, st.solved);
    put_stat(sl, ST_NEWTON_ITERS, st.iters);
    put_stat(sl, ST_SUBSTEP_DROPS, st.subs);
    put_stat(sl, ST_WARM_RESTARTS, st.restarts);
  }
}

// the learned guess z = r^2 exp(2 y) of every in-domain drop into a.warm_buf (NaN for inactive
// drops; also into a.guess_out when recording), 64 drops per network pass; it runs after
// k_cond_prep, whose saturation ratio it reads
__global__ void __launch_bounds__(256) k_cond_guess(CondFlatArgs a) {
  __shared__ InferConst K;
  infer_const_load(K, a.W.p);
  __syncthreads();
  const InferFrags F = infer_frags(a.W);
  const uint32_t ndom = a.off[a.ngbx];
  // wave-uniform loop: every lane of a wave runs the network on each chunk of 64 drops
  for (uint64_t k0 = static_cast<uint64_t>(blockIdx.x) * blockDim.x + (threadIdx.x & ~63u); k0 < ndom;
       k0 += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint64_t k = k0 + lane_id();
    bool valid = false;
    uint32_t g = 0;
    float f[kIn] = {0, 0, 0, 0, 0, 0};
    double r = 0.0;
    if (k < ndom) {
      g = a.s.gbx[k];
      valid = g < a.ngbx && (a.unsorted || k < a.off[g] + a.nact[g]);
      if (valid) {
        r = a.s.r[k];
        drop_features(r, a.s.msol[k], a.gs[kGsStride * g], a.st.temp[g], a.st.press[g], a.cfg.delt, f);
      }
    }
    float xn[kIn];
    infer_normalise(K, f, valid, xn);
    const float yn = mlp_infer(F, K, xn);
    if (k < ndom) {
      const double z = valid ? learned_z(K, r, yn) : __longlong_as_double(0x7FF8000000000000ll);
      a.warm_buf[k] = z;
      if (a.guess_out && valid) a.guess_out[k] = z;
    }
  }
}

// Drops whose solve outlives cfg.budget iterations (a few per cent; their lanes would hold the other
// 63 of the wave) are set aside by their workgroup and solved later, without a budget, packed into
// whole waves.  A workgroup takes a contiguous range of drops and lists its deferred ones in that range
// of a.dlist, so there is room for all of them, and counts them in LDS.  (One list for all workgroups,
// with an atomic per wave on its counter, took 238 us for the gather with the solves on 2.1M drops,
// 591 us on 8.4M, and 18 and 31 us more for a launch that solved the list; same-address atomics take
// about 5 ns each.)  Who solves them:
// - kTail: the workgroup itself at the end of its range, about 60 drops of 2048, while others fill the
//   CU: no further launch (2.1M drops: 104 us against 110; 91 with the solves as they are now).
// - else k_cond_deferred, which packs the lists of several workgroups and keeps the second copy of
//   the solve, with its registers, out of the main loop (33.5M drops: 1155 us against 1209, 134M:
//   4.44 ms against 4.64; equal at 8.4M; 1053 us and 4.0 ms with the solves as they are now).
__device__ __forceinline__ void defer_drop(uint32_t* ndef, uint32_t* list, bool deferred, uint32_t q) {
  const uint64_t m = ballot(deferred);
  if (!m) return;
  uint32_t base = 0;
  const int leader = __ffsll(static_cast<unsigned long long>(m)) - 1;
  if (lane_id() == leader) base = atomicAdd(ndef, static_cast<uint32_t>(__popcll(m)));
  base = readlane_u32(base, leader);
  if (deferred) list[base + lanes_below(m)] = q;
}
// the workgroup's range of n drops: whole chunks of its threads, consecutive ranges on one XCD
__device__ __forceinline__ uint64_t block_span(uint64_t n, uint32_t blocks, uint32_t threads) {
  return ((n + blocks - 1) / blocks + threads - 1) / threads * threads;
}
__device__ __forceinline__ void block_range(uint64_t n, uint64_t& lo, uint64_t& hi) {
  const uint64_t per = block_span(n, gridDim.x, blockDim.x);
  lo = min(static_cast<uint64_t>(xcd_block()) * per, n);
  hi = min(lo + per, n);
}

__device__ __forceinline__ void solve_listed(const CondFlatArgs& a, uint32_t k, CondStats& st) {
  NewtonCfg nobudget = a.cfg;
  nobudget.budget = 0;
  const double warm =
      a.warm ? a.warm[a.warm_perm ? a.warm_perm[k] : k] : __longlong_as_double(0x7FF8000000000000ll);
  cond_drop(a, nobudget, a.s.gbx[k], k, warm, st);
}
// Every thread of the workgroup calls it, after its last defer_drop.
template <bool kTail>
__device__ __forceinline__ void finish_deferred(const CondFlatArgs& a, const uint32_t* ndef, const uint32_t* list,
                                                CondStats& st) {
  __syncthreads();  // the entries, and the drops' records, were written by the workgroup's other waves
  const uint32_t n = *ndef;
  if constexpr (kTail) {
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) solve_listed(a, list[i], st);
  } else {
    if (threadIdx.x == 0) a.dcount[xcd_block()] = n;
  }
}

// The kernel's arguments where the launch put them: Args has the kernel's parameters as its members, all
// of 8-byte alignment.  After reread_args the compiler reads them again (scalar loads): arguments used
// throughout a long loop body otherwise move out of the loop, into more scalar registers than there
// are, and come back one v_readlane at a time, 75 to 100 per 64 drops of the gather with the solves
// (2.1M drops: 99 -> 94 us; 33M coupled 178 -> 172 ms in 60 steps).
template <class Args>
__device__ __forceinline__ const Args* kernel_args() {
  return reinterpret_cast<const Args*>((const void*)__builtin_amdgcn_kernarg_segment_ptr());
}
template <class Args>
__device__ __forceinline__ void reread_args(const Args*& args) {
  const __attribute__((address_space(4))) Args* p = (const __attribute__((address_space(4))) Args*)args;
  asm volatile("" : "+s"(p));
  args = (const Args*)p;
}
// per active drop, one thread each
template <bool kTail>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(5) k_cond_drops(CondFlatArgs) {
  struct Args {
    CondFlatArgs a;
  };
  auto args = kernel_args<Args>();
  const CondFlatArgs& a = args->a;
  __shared__ uint32_t ndef;
  if (threadIdx.x == 0) ndef = 0u;
  __syncthreads();
  CondStats st{0, 0, 0, 0};
  uint64_t k_lo, k_hi;
  block_range(a.off[a.ngbx], k_lo, k_hi);
  for (uint64_t k0 = k_lo; k0 < k_hi; k0 += blockDim.x) {
    reread_args(args);
    const CondFlatArgs& a = args->a;
    const uint64_t k = k0 + threadIdx.x;
    bool active = false;
    uint32_t g = 0;
    if (k < k_hi) {
      g = a.s.gbx[k];
      active = g < a.ngbx && k < a.off[g] + a.nact[g];
    }
    double warm = __longlong_as_double(0x7FF8000000000000ll);
    if (active && a.warm) warm = a.warm[k];
    bool deferred = false;
    if (active) deferred = !cond_drop(a, a.cfg, g, k, warm, st);
    defer_drop(&ndef, a.dlist + k_lo, deferred, static_cast<uint32_t>(k));
  }
  finish_deferred<kTail>(a, &ndef, a.dlist + k_lo, st);
  put_cond_stats(a.stat, st);
}

// The deferred drops of a solving pass of `nlists` workgroups over n drops, kListsPerBlock lists
// flattened over a workgroup's threads.
constexpr uint32_t kListsPerBlock = 8;
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(5) k_cond_deferred(CondFlatArgs a, uint32_t nlists) {
  __shared__ uint32_t pre[kListsPerBlock + 1];
  CondStats st{0, 0, 0, 0};
  const uint64_t per = block_span(a.off[a.ngbx], nlists, 256u);
  for (uint32_t l0 = blockIdx.x * kListsPerBlock; l0 < nlists; l0 += gridDim.x * kListsPerBlock) {
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t t = 0;
      for (uint32_t i = 0; i < kListsPerBlock; ++i) {
        pre[i] = t;
        t += l0 + i < nlists ? a.dcount[l0 + i] : 0u;
      }
      pre[kListsPerBlock] = t;
    }
    __syncthreads();
    for (uint32_t f = threadIdx.x; f < pre[kListsPerBlock]; f += blockDim.x) {
      const uint32_t i = tile_owner(pre, kListsPerBlock, f);
      solve_listed(a, a.dlist[(l0 + i) * per + f - pre[i]], st);
    }
  }
  put_cond_stats(a.stat, st);
}

// Condensation in the sort's gather, for a condensation that follows motion at once: destination
// q takes the drop at position perm[q] of the unsorted store and, when it stays in the domain,
// solves it before writing its record (with the new radius) and dm[q], qm[q] to the sorted store.
// The solve does not depend on the order of the drops; the per-gridbox sums run afterwards on the
// sorted store (k_cond_state).  Drops that outlive cfg.budget iterations are written unsolved and
// set aside, as in k_cond_drops.  The memory traffic of
// the gather and the FP64 arithmetic of the solves overlap in one pass.
// kMove: the unsorted store holds the drops before motion (the counting pass k_motion_drops<false>
// only recorded their steps); each drop moves here, with the same arithmetic, before its solve in
// the gridbox it reaches, so motion writes nothing of its own.  kLds: the coordinate bounds are read
// from an LDS copy (dynamic shared memory of nz + nx + ny + 3 doubles).
template <bool kMove, bool kLds, bool kTail>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(kMove ? 4 : 5) k_sort_gather_cond(NsortArgs, CondFlatArgs, MotionArgs) {
  struct Args {
    NsortArgs n;
    CondFlatArgs a;
    MotionArgs m;
  };
  static_assert(sizeof(Args) == sizeof(NsortArgs) + sizeof(CondFlatArgs) + sizeof(MotionArgs) && alignof(Args) == 8, "layout");
  auto args = kernel_args<Args>();
  const NsortArgs& n = args->n;
  const CondFlatArgs& a = args->a;
  const MotionArgs& m = args->m;
  extern __shared__ double bounds_lds[];
  MotionArgs b = m;
  if constexpr (kMove && kLds) {
    const uint32_t nzh = m.grid.nz + 1, nxh = m.grid.nx + 1, nyh = m.grid.ny + 1;
    for (uint32_t i = threadIdx.x; i < nzh + nxh + nyh; i += blockDim.x)
      bounds_lds[i] = i < nzh ? m.grid.zh[i] : (i < nzh + nxh ? m.grid.xh[i - nzh] : m.grid.yh[i - nzh - nxh]);
    __syncthreads();
    b.grid.zh = bounds_lds;
    b.grid.xh = bounds_lds + nzh;
    b.grid.yh = bounds_lds + nzh + nxh;
  }
  __shared__ uint32_t ndef;
  if (threadIdx.x == 0) ndef = 0u;
  __syncthreads();
  const uint64_t nsrc = n.off[n.grid.ngbx];
  CondStats st{0, 0, 0, 0};
  const double nowarm = __longlong_as_double(0x7FF8000000000000ll);
  // Each block takes one contiguous range of destinations, in block-uniform chunks (every wave
  // of the block stays in the loop for the ballots below).  A drop that changed gridbox is read
  // from lines that the neighbouring destinations' drops also read; with contiguous ranges those
  // readers run on the same CU at about the same time, and with the ranges in xcd_block() order
  // the neighbouring ranges run on the same XCD, behind one L2 (measured 4.82 -> 4.61 -> 4.49 ms
  // against chunks strided over the grid).
  uint64_t q_lo, q_hi;
  block_range(nsrc, q_lo, q_hi);
  for (uint64_t q0 = q_lo; q0 < q_hi; q0 += blockDim.x) {
    if constexpr (!kMove) reread_args(args);
    const NsortArgs& n = args->n;
    const CondFlatArgs& a = args->a;
    const uint64_t q = q0 + threadIdx.x;
    const bool inq = q < q_hi;
    const uint32_t p = inq ? n.perm[q] : 0u;
    const bool okp = inq && p < nsrc;
    if (inq && !okp) set_error(n.ctl, CLEO_ERR_SORT_NONLOCAL, kOOB, q);
    const uint32_t sp = okp ? p : 0u;
    uint32_t g = n.src.gbx[sp];
    double c3 = n.src.c3[sp], c1 = n.src.c1[sp], c2 = n.src.c2[sp];
    const uint64_t xi = n.src.xi[sp], id = n.src.id[sp];
    const double r = n.src.r[sp], msol = n.src.msol[sp];
    if constexpr (kMove) {
      // an in-domain drop's gridbox is below ngbx; the guard keeps a corrupted one from indexing
      const uint32_t gg = g < n.grid.ngbx ? g : 0u;
      const GbxGeom G = gbx_geom(b, gg);
      const Moved M = move_drop(b, gg, G, DropPos{c3, c1, c2, r}, sp, false);
      c3 = M.c3;
      c1 = M.c1;
      c2 = M.c2;
      g = M.idx;
    }
    const bool active = okp && g < a.ngbx;
    const double warm = a.warm ? a.warm[sp] : nowarm;  // learned guesses by source position
    // non-temporal stores: the sorted store and dm, qm are read back only after the whole pass,
    // from HBM either way, and streaming them past the L2 leaves it to the source lines that
    // neighbouring destinations still read (5.31 -> 5.11 ms).  Every field but the radius is
    // final before the solve and is written first, so its registers are free during the solve.
    if (okp) {
      __builtin_nontemporal_store(g, &n.dst.gbx[q]);
      __builtin_nontemporal_store(c3, &n.dst.c3[q]);
      __builtin_nontemporal_store(c1, &n.dst.c1[q]);
      __builtin_nontemporal_store(c2, &n.dst.c2[q]);
      __builtin_nontemporal_store(xi, &n.dst.xi[q]);
      __builtin_nontemporal_store(msol, &n.dst.msol[q]);
      __builtin_nontemporal_store(id, &n.dst.id[q]);
    }
    double rnew = r, dm = 0.0, qm = 0.0;
    bool solved = false;
    if (active) solved = cond_solve(a, a.cfg, g, q, r, msol, [&] { return xi; }, warm, st, rnew, dm, qm);
    defer_drop(&ndef, a.dlist + q_lo, active && !solved, static_cast<uint32_t>(q));
    if (okp) __builtin_nontemporal_store(solved ? rnew : r, &n.dst.r[q]);
    if (solved) {
      __builtin_nontemporal_store(dm, &a.dm[q]);
      if (a.qm) __builtin_nontemporal_store(qm, &a.qm[q]);
    }
  }
  finish_deferred<kTail>(a, &ndef, a.dlist + q_lo, st);
  copy_oob(n, nsrc);
  put_cond_stats(a.stat, st);
}

// ---- condensation with a per-wave task ring ------------------------------------------------------
// Newton iteration counts differ from drop to drop (2 for about a quarter, 5-6 for most, tens for
// a few), so 64 drops solved in lockstep leave most lanes idle.  Here each lane runs the solve of
// its drop as a state machine, one g-evaluation per tick, and a lane whose drop is done takes the
// next prepared task from a ring in LDS; a setup pass prepares 64 drops at a time whenever fewer
// than 64 tasks wait.  Every drop goes through exactly the operations of solve_condensation
// (initial evaluation, two iterations, restart until converged, sub-steps, learned guess), so the
// result does not depend on the scheduling.
struct CondRing {
  double s_ratio[kRing], akoh[kRing], bkoh[kRing], inv_ffv[kRing], r0[kRing], zplain[kRing], zwarm[kRing],
      mindelt[kRing], dryr[kRing], oldm[kRing], msol[kRing];
  uint64_t xi[kRing];
  uint32_t k[kRing], unique[kRing];
};
static_assert(sizeof(CondRing) == kCondRingBytes, "ring size");

enum : uint32_t { PH_EVAL = 0, PH_FIRST = 1, PH_SECOND = 2, PH_UNTIL = 3 };
enum : uint32_t { MODE_PLAIN = 0, MODE_WARM = 1, MODE_SUB = 2 };

__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(3) k_cond_queue(CondFlatArgs a) {
  extern __shared__ uint32_t lds_dyn[];
  CondRing& R = reinterpret_cast<CondRing*>(lds_dyn)[threadIdx.x >> 6];
  const int lane = lane_id();
  const NewtonCfg cfg = a.cfg;
  const uint64_t ndom = a.off[a.ngbx];
  const uint64_t nw = wave_count(), w = wave_index();
  const uint64_t k_hi = ndom * (w + 1) / nw;
  uint64_t next = ndom * w / nw;  // first drop not yet prepared (wave-uniform)
  uint32_t head = 0, tail = 0;    // ring positions handed out / prepared (wave-uniform)
  // lane state
  bool busy = false, restarted = false, maxed = false;
  uint32_t k = 0, phase = PH_EVAL, mode = MODE_PLAIN, niter = 0, limit = 0, iters = 0;
  ODEConsts c{0, 0, 0, 0, 0, 0, 0};
  double rprev = 0, r0 = 0, subdelt = 0, remdelt = 0, mindelt = 0, zplain = 0;
  double z = 0, gz = 0, dgz = 0, z0 = 0, g0 = 0, dg0 = 0, dryr = 0, oldm = 0, msol = 0;
  uint64_t xi = 0;
  uint32_t st_solved = 0, st_iters = 0, st_subs = 0, st_restarts = 0;
  while (true) {
    if (tail - head < static_cast<uint32_t>(kWave) && next < k_hi) {
      // setup pass: Koehler factors, ventilation, initial guess and uniqueness criteria of the next
      // 64 drops (condensation.cpp:44-56, impliciteuler.cpp:35-54)
      const uint64_t kk = next + static_cast<uint64_t>(lane);
      bool act = false;
      uint32_t g = 0;
      if (kk < k_hi) {
        g = a.s.gbx[kk];
        act = g < a.ngbx && kk < a.off[g] + a.nact[g];
      }
      const uint64_t m = __ballot(act);
      if (act) {
        const uint32_t slot = (tail + static_cast<uint32_t>(__popcll(m & lanemask_lt()))) % kRing;
        const double s_ratio = a.gs[kGsStride * g], ffactor = a.gs[kGsStride * g + 1];
        const double r = a.s.r[kk], ms = a.s.msol[kk];
        bool bad = false;
        const double om = condensate_mass(r, ms, a.sol, &bad);
        if (bad) set_error(a.ctl, CLEO_ERR_NEG_CONDENSATE, g, kk);
        const double akoh = a.gs[kGsStride * g + 2], bkoh = kohler_b(ms, a.sol);
        ODEConsts cc{s_ratio, akoh, bkoh, 0.0, 0.0, 0.0, a.gs[kGsStride * g + 3]};
        ffactor_over_vent(ffactor, r, cc.ffv_num, cc.ffv_den, cc.inv_ffv);
        double zg;
        bool uniq;
        ode_setup(cc, r, cfg.delt, zg, uniq);
        const double critdelt = uniq ? 0.0 : critical_timestep(cc);
        R.s_ratio[slot] = s_ratio;
        R.akoh[slot] = akoh;
        R.bkoh[slot] = bkoh;
        R.inv_ffv[slot] = cc.inv_ffv;
        R.r0[slot] = r;
        R.zplain[slot] = zg;
        double zw = a.warm ? a.warm[kk] : __longlong_as_double(0x7FF8000000000000ll);
        if (uniq && zw == zw) {  // the learned path starts from the plain guess where that is the root
          double gp, dg;       // to the tolerance (solve_condensation)
          ode_g_dg<true>(ode_run(cc, cfg.delt, r), zg, gp, dg);
          if (fabs(gp) < cfg.atol) zw = zg;
        }
        R.zwarm[slot] = zw;
        R.mindelt[slot] = uniq ? 0.0 : fmax(critdelt, cfg.minsubdelt);
        R.dryr[slot] = dryradius(ms, a.sol);
        R.oldm[slot] = om;
        R.msol[slot] = ms;
        R.xi[slot] = a.s.xi[kk];
        R.k[slot] = static_cast<uint32_t>(kk);
        R.unique[slot] = uniq ? 1u : 0u;
      }
      tail += static_cast<uint32_t>(__popcll(m));
      next += kWave;
      wave_sync();
    }
    // hand the waiting tasks to idle lanes
    const uint64_t midle = __ballot(!busy);
    const uint32_t avail = tail - head;
    if (!busy) {
      const uint32_t rank = static_cast<uint32_t>(__popcll(midle & lanemask_lt()));
      if (rank < avail) {
        const uint32_t slot = (head + rank) % kRing;
        c = ODEConsts{R.s_ratio[slot], R.akoh[slot], R.bkoh[slot], 0.0, 0.0, R.inv_ffv[slot], 0.0};
        r0 = R.r0[slot];
        zplain = R.zplain[slot];
        mindelt = R.mindelt[slot];
        dryr = R.dryr[slot];
        oldm = R.oldm[slot];
        msol = R.msol[slot];
        xi = R.xi[slot];
        k = R.k[slot];
        const double zw = R.zwarm[slot];
        rprev = r0;
        iters = 0;
        restarted = maxed = false;
        if (R.unique[slot]) {
          subdelt = cfg.delt;
          if (zw == zw) {
            mode = MODE_WARM;
            limit = a.warm_limit;
            z = zw;
          } else {
            mode = MODE_PLAIN;
            limit = cfg.maxniters;
            z = zplain;
          }
        } else {
          mode = MODE_SUB;
          limit = cfg.maxniters;
          remdelt = cfg.delt;
          subdelt = fmin(mindelt, remdelt);
          z = zplain;
        }
        phase = PH_EVAL;
        busy = true;
      }
    }
    head += min(static_cast<uint32_t>(__popcll(midle)), avail);
    wave_sync();
    if (!__any(busy)) {
      if (next >= k_hi && head == tail) break;
      continue;
    }
    if (busy) {
      // one evaluation of g: the initial state of a segment, or a Newton iteration
      // (newton_iterate, impliciteuler.cpp:240-255)
      double zn = z;
      if (phase != PH_EVAL) zn = newton_next(z, gz, dgz);
      double g1, dg1;
      ode_g_dg<true>(ode_run(c, subdelt, rprev), zn, g1, dg1);
      bool segok = false, segfail = false;
      if (phase == PH_EVAL) {
        z0 = z = zn;
        g0 = gz = g1;
        dg0 = dgz = dg1;
        if (mode == MODE_WARM) {  // from the learned guess: iterate until converged at once
          phase = PH_UNTIL;
          niter = 1;
          segfail = niter > limit;
        } else {
          phase = PH_FIRST;
        }
      } else {
        ++iters;
        const bool conv = newton_converged(cfg, g1, gz);
        z = zn;
        gz = g1;
        dgz = dg1;
        if (phase == PH_FIRST) {
          phase = PH_SECOND;
        } else if (phase == PH_SECOND) {  // integrate_condensation_ode: restart unless converged
          if (conv) {
            segok = true;
          } else {
            z = z0;
            gz = g0;
            dgz = dg0;
            phase = PH_UNTIL;
            niter = 1;
            segfail = niter > limit;
          }
        } else {  // newtonraphson_untilconverged (impliciteuler.cpp:207-227)
          ++niter;
          if (conv)
            segok = true;
          else
            segfail = niter > limit;
        }
      }
      if (segfail) {
        if (mode == MODE_WARM) {  // the learned guess failed: the reference path from its guess
          restarted = true;
          mode = MODE_PLAIN;
          limit = cfg.maxniters;
          subdelt = cfg.delt;
          rprev = r0;
          z = zplain;
          phase = PH_EVAL;
        } else {
          maxed = true;
          segok = true;
        }
      }
      if (segok) {
        bool done = true;
        if (mode == MODE_SUB) {  // substepping loop of solve_condensation
          rprev = sqrt(z);
          remdelt -= subdelt;
          if (remdelt > 0.0) {
            subdelt = fmin(mindelt, remdelt);
            phase = PH_EVAL;
            done = false;
            if (!(subdelt > 0.0)) {  // no progress possible: stop with the reference's substep error
              set_error(a.ctl, CLEO_ERR_SUBSTEP, a.s.gbx[k], k);
              done = true;
            }
          }
        }
        if (done) {
          const double rnew = fmax(sqrt(z), dryr);  // change_radius (superdrop_attrs.cpp:35-45)
          a.s.r[k] = rnew;
          bool bad = false;
          a.dm[k] = (condensate_mass(rnew, msol, a.sol, &bad) - oldm) * static_cast<double>(xi);
          if (bad) set_error(a.ctl, CLEO_ERR_NEG_CONDENSATE, a.s.gbx[k], k);
          if (maxed) set_error(a.ctl, CLEO_ERR_NEWTON_MAXITERS, a.s.gbx[k], k);
          if (a.niters) a.niters[k] = iters;
          st_solved += 1;
          st_iters += iters;
          st_subs += mode == MODE_SUB ? 1u : 0u;
          st_restarts += restarted ? 1u : 0u;
          busy = false;
        }
      }
    }
  }
  st_solved = wave_sum_u32(st_solved);
  st_iters = wave_sum_u32(st_iters);
  st_subs = wave_sum_u32(st_subs);
  st_restarts = wave_sum_u32(st_restarts);
  if (lane == 0) {
    put_stat(a.stat, ST_COND_DROPS, st_solved);
    put_stat(a.stat, ST_NEWTON_ITERS, st_iters);
    put_stat(a.stat, ST_SUBSTEP_DROPS, st_subs);
    put_stat(a.stat, ST_WARM_RESTARTS, st_restarts);
  }
}

// per gridbox: Σ dm in drop order and the thermodynamic feedback (condensation.cpp:126-137); kByRows:
// the sums by tile_rows_sum, tiles of kRows gridboxes.
// With a.qm, first the qcond recompute after motion from the drops' terms before the solve (the
// same ordered sum and formula as k_cond_prep's; State is unchanged until here).
template <bool kByRows>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(4) k_cond_state(CondFlatArgs a) {
  __shared__ double win_all[4][kSumWin];
  double* win = win_all[threadIdx.x >> 6];
  const int lane = lane_id();
  const uint32_t gpt = a.gpt, ntiles = sum_tiles(a.ngbx, gpt);
  for (uint32_t tile = wave_index(); tile < ntiles; tile += wave_count()) {
    const uint32_t g0 = tile * gpt, g = g0 + static_cast<uint32_t>(lane);
    const bool valid = static_cast<uint32_t>(lane) < gpt && g < a.ngbx;
    const uint32_t t_lo = a.off[g0], t_hi = a.off[min(g0 + gpt, a.ngbx)];
    const uint32_t lo = valid ? a.off[g] : t_hi, n = valid ? a.nact[g] : 0u;
    double qc_new = 0.0, tot = 0.0;
    if (a.qm) {
      double totq = 0.0;
      if constexpr (kByRows) {
        double both[2] = {0.0, 0.0};
        tile_rows_sum<2>(win, t_lo, lo, n, [&](int c, uint32_t k) { return c == 0 ? a.qm[k] : a.dm[k]; }, lane, both);
        totq = both[0];
        tot = both[1];
      } else {
        tile_sum2(win, t_lo, t_hi, lo, n, [&](uint32_t k) { return a.qm[k]; }, [&](uint32_t k) { return a.dm[k]; },
                  lane, totq, tot);
      }
      if (valid) {
        const double rho_cond = totq / a.st.vol[g] * dimless::R0cubed_VOL0;
        qc_new = rho_cond / dry_air_density(a.st.press[g], a.st.temp[g], a.st.qv[g]);
        if (!a.alter) a.st.qc[g] = qc_new;
      }
    } else {
      if constexpr (kByRows)
        tile_rows_sum<1>(win, t_lo, lo, n, [&](int, uint32_t k) { return a.dm[k]; }, lane, &tot);
      else
        tot = tile_sum(win, t_lo, t_hi, lo, n, [&](uint32_t k) { return a.dm[k]; }, lane);
    }
    if (valid && a.alter) {
      const double temp = a.st.temp[g], press = a.st.press[g];
      double qv = a.st.qv[g], qc = a.qm ? qc_new : a.st.qc[g];
      const double totrho = tot / a.st.vol[g] * dimless::R0cubed_VOL0;
      const double dq = totrho / dry_air_density(press, temp, qv);
      qv -= dq;
      qc += dq;
      a.st.temp[g] = temp + (dimless::Latent_v / moist_specific_heat(qv, qc)) * dq;
      a.st.qv[g] = qv;
      a.st.qc[g] = qc;
    }
  }
}

// ============================ coupling ========================================================
// FromFileComms::update_gridbox_state for every gridbox (fromfilecomms.cpp:51-62): thermodynamics
// at the gridbox, winds at its lower and upper faces (fromfile_cartesian_dynamics.cpp:150-215)
__global__ void k_receive_dynamics(GState st, Grid gr, cleo_dynamics_step dyn) {
  const uint32_t nz = gr.nz, nx = gr.nx, ngbx = gr.ngbx;
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < ngbx; g += gridDim.x * blockDim.x) {
    const uint32_t k = g % nz, i = (g / nz) % nx, j = g / (nz * nx);
    st.press[g] = dyn.press[g];
    st.temp[g] = dyn.temp[g];
    st.qv[g] = dyn.qvap[g];
    st.qc[g] = dyn.qcond[g];
    double wl = 0.0, wh = 0.0, ul = 0.0, uh = 0.0, vl = 0.0, vh = 0.0;
    if (dyn.wvel_zfaces) {
      const uint64_t l = static_cast<uint64_t>(nx) * (nz + 1) * j + static_cast<uint64_t>(nz + 1) * i + k;
      wl = dyn.wvel_zfaces[l];
      wh = dyn.wvel_zfaces[l + 1];
    }
    if (dyn.uvel_xfaces) {
      const uint64_t l = static_cast<uint64_t>(nx + 1) * nz * j + static_cast<uint64_t>(nz) * i + k;
      ul = dyn.uvel_xfaces[l];
      uh = dyn.uvel_xfaces[l + nz];
    }
    if (dyn.vvel_yfaces) {
      vl = dyn.vvel_yfaces[g];
      vh = dyn.vvel_yfaces[static_cast<uint64_t>(g) + static_cast<uint64_t>(nx) * nz];
    }
    st.wlo[g] = wl;
    st.whi[g] = wh;
    st.ulo[g] = ul;
    st.uhi[g] = uh;
    st.vlo[g] = vl;
    st.vhi[g] = vh;
  }
}
void launch_receive_dynamics(cleo_ctx* c, const cleo_dynamics_step& dyn) {
  if (c->grid.ngbx == 0) return;
  hipLaunchKernelGGL(k_receive_dynamics, dim3(stride_blocks(c->grid.ngbx)), dim3(256), 0, c->stream, c->st, c->grid,
                     dyn);
}

// ============================ observers =======================================================
// Mass moments per gridbox (observers/massmoments_observer.cpp:23-73): one lane per gridbox of a
// tile.  The tile's drops pass through an LDS window with coalesced loads (the next
// window's loads in flight while the current one is added); the loading lane turns each drop into
// its three terms (xi; (float)(xi m); (float)(xi m m), m the drop mass,
// zero for a drop below the raindrop radius when kRain), and each lane then adds its gridbox's
// terms left to right, so the float sums are the reference's serial ones.
constexpr uint32_t kMomWin = 512;
template <bool kRain>
__global__ void __launch_bounds__(256) k_mass_moments(SoA s, const uint32_t* off, uint32_t ngbx, uint32_t gpt,
                                                      Solute sol, DevCtl* ctl, uint64_t* mom0, float* mom1, float* mom2) {
  __shared__ uint64_t w0_all[4][kMomWin];
  __shared__ float w1_all[4][kMomWin], w2_all[4][kMomWin];
  const uint32_t wv = threadIdx.x >> 6;
  uint64_t* w0 = w0_all[wv];
  float* w1 = w1_all[wv];
  float* w2 = w2_all[wv];
  const int lane = lane_id();
  constexpr double rlim(40e-6 / dimless::R0);  // calculate_rainmassmoments: raindrop radius
  const uint32_t ntiles = sum_tiles(ngbx, gpt);
  for (uint32_t tile = wave_index(); tile < ntiles; tile += wave_count()) {
    const uint32_t g0 = tile * gpt, g = g0 + static_cast<uint32_t>(lane);
    const bool valid = static_cast<uint32_t>(lane) < gpt && g < ngbx;
    const uint32_t t_lo = off[g0], t_hi = off[min(g0 + gpt, ngbx)];
    const uint32_t lo = valid ? off[g] : t_hi, hi = valid ? off[g + 1] : t_hi;
    uint64_t m0 = 0;
    float m12[2] = {0.f, 0.f};
    if (t_lo >= t_hi) {
      if (valid) {
        mom0[g] = 0;
        mom1[g] = 0.f;
        mom2[g] = 0.f;
      }
      continue;
    }
    // the next window's drops are loaded into registers while the lanes add the current window
    // (every lane loads, with indices clamped into the tile, so the loads stay in flight)
    constexpr uint32_t kPer = kMomWin / kWave;
    uint64_t rx[kPer];
    double rr[kPer], rm[kPer];
    auto load = [&](uint32_t w) {
      for (uint32_t i = 0; i < kPer; ++i) {
        const uint32_t k = min(w + static_cast<uint32_t>(lane) + i * kWave, t_hi - 1u);
        rx[i] = __builtin_nontemporal_load(&s.xi[k]);  // read once (0.63 -> 0.60 ms)
        rr[i] = __builtin_nontemporal_load(&s.r[k]);
        rm[i] = __builtin_nontemporal_load(&s.msol[k]);
      }
    };
    load(t_lo);
    for (uint32_t w = t_lo; w < t_hi; w += kMomWin) {
      const uint32_t we = min(w + kMomWin, t_hi);
      for (uint32_t i = 0; i < kPer; ++i) {
        const uint32_t j = static_cast<uint32_t>(lane) + i * kWave;
        const uint64_t xi = rx[i];
        const double r = rr[i];
        if (j < we - w && xi == ~0ull) set_error(ctl, CLEO_ERR_XI_OVERFLOW, s.gbx[w + j], w + j);
        const bool in = !kRain || r >= rlim;
        const double m = drop_mass(r, rm[i], sol);
        const double xm = static_cast<double>(xi) * m;
        w0[j] = in ? xi : 0ull;
        w1[j] = in ? static_cast<float>(xm) : 0.f;
        w2[j] = in ? static_cast<float>(xm * m) : 0.f;
      }
      wave_sync();
      if (we < t_hi) load(we);
      const uint32_t b0 = max(lo, w), b1 = min(hi, we);
      if (b0 < b1) {
        const uint64_t* const v0[1] = {w0};
        const float* const v12[2] = {w1, w2};
        add_in_order<1>(&m0, v0, b0 - w, b1 - w);
        add_in_order<2>(m12, v12, b0 - w, b1 - w);
      }
      wave_sync();
    }
    if (valid) {
      mom0[g] = m0;
      mom1[g] = m12[0];
      mom2[g] = m12[1];
    }
  }
}
void launch_mass_moments(cleo_ctx* c, bool rain, uint64_t* mom0, float* mom1, float* mom2) {
  const uint32_t ngbx = c->grid.ngbx;
  if (ngbx == 0) return;
  materialize_order(c);  // the sums follow the drops' logical order
  const uint32_t gpt = sum_gpt(c);
  const unsigned nb = sum_blocks(c, 0);
  if (rain)
    hipLaunchKernelGGL(k_mass_moments<true>, dim3(nb), dim3(256), 0, c->stream, c->buf[c->cur], c->off, ngbx, gpt,
                       c->solute, c->ctl, mom0, mom1, mom2);
  else
    hipLaunchKernelGGL(k_mass_moments<false>, dim3(nb), dim3(256), 0, c->stream, c->buf[c->cur], c->off, ngbx, gpt,
                       c->solute, c->ctl, mom0, mom1, mom2);
}

// the thermodynamic functions of the condensation (gbx_thermo) at n states, thread per state
__global__ void k_thermo_eval(uint64_t n, const double* temp, const double* press, const double* qvap,
                              double* psat, double* s_ratio, double* ffactor) {
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const double ps = saturation_pressure(temp[i]);
    psat[i] = ps;
    s_ratio[i] = supersaturation_ratio(press[i], qvap[i], ps);
    ffactor[i] = diffusion_factor(press[i], temp[i], ps);
  }
}
void launch_thermo_eval(cleo_ctx* c, uint64_t n, const double* temp, const double* press, const double* qvap,
                        double* psat, double* s_ratio, double* ffactor) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_thermo_eval, dim3(stride_blocks(n)), dim3(256), 0, c->stream, n, temp, press, qvap, psat,
                     s_ratio, ffactor);
}

// p[i] = i for i < n
__global__ void k_iota_u32(uint32_t* p, uint64_t n) {
  for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    p[i] = static_cast<uint32_t>(i);
}

// count-table key of a moved drop: 28*d + step for destination d, 28*g + 27 when it left the domain
__device__ __forceinline__ uint32_t motion_key(const Moved& M, uint32_t g) {
  return M.idx != kOOB ? 28u * M.idx + static_cast<uint32_t>(M.dir) : 28u * g + 27u;
}
// adds the wave's drops per distinct key to the count table (every lane of the wave calls it)
__device__ __forceinline__ void count_keys(uint32_t* cnt, uint32_t key, bool act, int lane) {
  uint64_t mask = __ballot(act);
  while (mask) {
    const int leader = __ffsll(static_cast<unsigned long long>(mask)) - 1;
    const uint32_t v = readlane_u32(key, leader);
    const uint64_t m = __ballot(act && key == v);
    if (lane == leader) atomicAdd(&cnt[v], static_cast<uint32_t>(__popcll(m)));
    mask &= ~m;
  }
}
// largest coordinate-bound table (zh, xh, yh together) that the motion kernels stage in LDS
constexpr uint32_t kMotionLdsBounds = 2048;

// MoveSupersInGridboxesFunctor per drop, two drops per thread and iteration with every load of
// both issued before the arithmetic; the destination-major counts are aggregated per wave, then
// added with atomics, and the step of each drop goes to a.step when that is set.  kLds: the
// coordinate bounds are read from an LDS copy (dynamic shared memory of (nz + nx + ny + 3)
// doubles).  Without kWrite this is the counting pass of a fused motion + sort: the drops' new
// coordinates and gridboxes are not stored (the second pass computes them again).
template <bool kWrite, bool kLds>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(3) k_motion_drops(MotionArgs a) {
  extern __shared__ double bounds_lds[];
  const int lane = lane_id();
  MotionArgs b = a;
  if constexpr (kLds) {
    const uint32_t nzh = a.grid.nz + 1, nxh = a.grid.nx + 1, nyh = a.grid.ny + 1;
    for (uint32_t i = threadIdx.x; i < nzh + nxh + nyh; i += blockDim.x)
      bounds_lds[i] = i < nzh ? a.grid.zh[i] : (i < nzh + nxh ? a.grid.xh[i - nzh] : a.grid.yh[i - nzh - nxh]);
    __syncthreads();
    b.grid.zh = bounds_lds;
    b.grid.xh = bounds_lds + nzh;
    b.grid.yh = bounds_lds + nzh + nxh;
  }
  const uint32_t ndom = a.off[a.grid.ngbx];
  // block-uniform chunks of 512 drops keep every wave in the loop together for the ballots
  for (uint64_t k0 = 2ull * blockIdx.x * blockDim.x; k0 < ndom; k0 += 2ull * gridDim.x * blockDim.x) {
    const uint64_t ka = k0 + threadIdx.x, kb = ka + blockDim.x;
    const bool acta = ka < ndom, actb = kb < ndom;
    // past the end a lane reads drop k0 (in the domain) and discards the result
    const uint64_t la = acta ? ka : k0, lb = actb ? kb : k0;
    // non-temporal loads: each drop's fields are read once here (2.21 -> 1.94 ms)
    const uint32_t ga = __builtin_nontemporal_load(&a.s.gbx[la]), gb = __builtin_nontemporal_load(&a.s.gbx[lb]);
    const DropPos pa = drop_pos_nt(a, la), pb = drop_pos_nt(a, lb);
    const GbxGeom Ga = gbx_geom(b, ga), Gb = gbx_geom(b, gb);
    const Moved Ma = move_drop(b, ga, Ga, pa, la, acta);
    const Moved Mb = move_drop(b, gb, Gb, pb, lb, actb);
    // non-temporal stores: the moved coordinates and steps are read back by the sort's passes,
    // after the whole launch (2.27 -> 2.23 ms)
    if (kWrite && acta) {
      __builtin_nontemporal_store(Ma.c3, &a.s.c3[ka]);
      __builtin_nontemporal_store(Ma.c1, &a.s.c1[ka]);
      __builtin_nontemporal_store(Ma.c2, &a.s.c2[ka]);
      __builtin_nontemporal_store(Ma.idx, &a.s.gbx[ka]);
    }
    if (kWrite && actb) {
      __builtin_nontemporal_store(Mb.c3, &a.s.c3[kb]);
      __builtin_nontemporal_store(Mb.c1, &a.s.c1[kb]);
      __builtin_nontemporal_store(Mb.c2, &a.s.c2[kb]);
      __builtin_nontemporal_store(Mb.idx, &a.s.gbx[kb]);
    }
    if (a.step && acta) __builtin_nontemporal_store(static_cast<uint8_t>(Ma.dir), &a.step[ka]);
    if (a.step && actb) __builtin_nontemporal_store(static_cast<uint8_t>(Mb.dir), &a.step[kb]);
    count_keys(a.cnt, motion_key(Ma, ga), acta, lane);
    count_keys(a.cnt, motion_key(Mb, gb), actb, lane);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) put_stat(a.stat, ST_MOTION_DROPS, ndom);  // each drop of the domain
}

// launches k_motion_drops with the bounds in LDS when they fit
template <bool kWrite>
static void launch_motion_drops(cleo_ctx* c, const MotionArgs& a, unsigned nb) {
  clear_counts(c);
  const uint32_t nb_ = a.grid.nz + a.grid.nx + a.grid.ny + 3;
  if (nb_ <= kMotionLdsBounds)
    hipLaunchKernelGGL((k_motion_drops<kWrite, true>), dim3(nb), dim3(256), nb_ * sizeof(double), c->stream, a);
  else
    hipLaunchKernelGGL((k_motion_drops<kWrite, false>), dim3(nb), dim3(256), 0, c->stream, a);
}

// Motion fused into the sort's gather (motion_flat 3): destination q takes the drop at position
// perm[q] of the unmoved store, moved by the same predictor-corrector step the counting pass
// computed for it (the arithmetic is deterministic, so the new gridbox is the key the drop was
// ranked by); the new coordinates and gridbox go straight to q.  One position per thread and
// iteration (two would spill); bounds from LDS when kLds.  A perm entry that is not a position of
// the domain is reported and skipped.
template <bool kLds>
__global__ void __launch_bounds__(256) CLEO_OCCUPANCY(4) k_nsort_gather_move(NsortArgs n, MotionArgs m) {
  extern __shared__ double bounds_lds[];
  MotionArgs b = m;
  if constexpr (kLds) {
    const uint32_t nzh = m.grid.nz + 1, nxh = m.grid.nx + 1, nyh = m.grid.ny + 1;
    for (uint32_t i = threadIdx.x; i < nzh + nxh + nyh; i += blockDim.x)
      bounds_lds[i] = i < nzh ? m.grid.zh[i] : (i < nzh + nxh ? m.grid.xh[i - nzh] : m.grid.yh[i - nzh - nxh]);
    __syncthreads();
    b.grid.zh = bounds_lds;
    b.grid.xh = bounds_lds + nzh;
    b.grid.yh = bounds_lds + nzh + nxh;
  }
  const uint64_t nsrc = n.off[n.grid.ngbx];
  for (uint64_t q = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; q < nsrc;
       q += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint32_t p = n.perm[q];
    if (p >= nsrc) {
      set_error(n.ctl, CLEO_ERR_SORT_NONLOCAL, kOOB, q);
      continue;
    }
    const uint32_t g = n.src.gbx[p];
    const DropPos P = drop_pos(b, p);
    // an in-domain drop's gridbox is below ngbx; the guard keeps a corrupted one from indexing
    const uint32_t gg = g < n.grid.ngbx ? g : 0u;
    const GbxGeom G = gbx_geom(b, gg);
    const Moved M = move_drop(b, gg, G, P, p, false);
    n.dst.gbx[q] = M.idx;
    n.dst.c3[q] = M.c3;
    n.dst.c1[q] = M.c1;
    n.dst.c2[q] = M.c2;
    n.dst.xi[q] = n.src.xi[p];
    n.dst.r[q] = P.r;
    n.dst.msol[q] = n.src.msol[p];
    n.dst.id[q] = n.src.id[p];
  }
  copy_oob(n, nsrc);
}
static void launch_gather_move(cleo_ctx* c, const NsortArgs& n, const MotionArgs& m) {
  const uint32_t nb_ = m.grid.nz + m.grid.nx + m.grid.ny + 3;
  const unsigned nb = drop_blocks(c->ntot, 0);
  if (nb_ <= kMotionLdsBounds)
    hipLaunchKernelGGL(k_nsort_gather_move<true>, dim3(nb), dim3(256), nb_ * sizeof(double), c->stream, n, m);
  else
    hipLaunchKernelGGL(k_nsort_gather_move<false>, dim3(nb), dim3(256), 0, c->stream, n, m);
}

// the gather with the solves; with m, the drops also move in it (k_sort_gather_cond<true, ...>)
template <bool kTail>
static void launch_gather_cond(cleo_ctx* c, const NsortArgs& n, const CondFlatArgs& a, const MotionArgs* m,
                               unsigned nb) {
  if (!m) {
    hipLaunchKernelGGL((k_sort_gather_cond<false, false, kTail>), dim3(nb), dim3(256), 0, c->stream, n, a, MotionArgs{});
    return;
  }
  const uint32_t nb_ = m->grid.nz + m->grid.nx + m->grid.ny + 3;
  if (nb_ <= kMotionLdsBounds)
    hipLaunchKernelGGL((k_sort_gather_cond<true, true, kTail>), dim3(nb), dim3(256), nb_ * sizeof(double), c->stream, n,
                       a, *m);
  else
    hipLaunchKernelGGL((k_sort_gather_cond<true, false, kTail>), dim3(nb), dim3(256), 0, c->stream, n, a, *m);
}
static void launch_deferred(cleo_ctx* c, CondFlatArgs a, unsigned nlists) {
  const unsigned nb = nblocks(nlists, kListsPerBlock);
  a.stat = stat_slots(c);
  hipLaunchKernelGGL(k_cond_deferred, dim3(nb), dim3(256), 0, c->stream, a, nlists);
}

// whether the workgroups of a solving pass solve their deferred drops themselves (finish_deferred)
static bool tail_solves(const cleo_ctx* c, uint32_t budget) { return budget == 0 || c->ntot < 6000000u; }
// Blocks of a solving pass: ranges of 8 to 16 chunks of 256 drops, long enough to pack the deferred
// drops, short enough to balance (33.5M drops in ranges of 4 / 8 / 16 / 32 chunks: 1190 / 1155 / 1181 /
// 1277 us; 134M: 4.69 / 4.58 / 4.44 / 4.60 ms), but never fewer than fill the chip at five workgroups
// per CU; at most grid_waves waves when that is set.
static unsigned solve_blocks(const cleo_ctx* c, uint32_t grid_waves) {
  const uint64_t chunks = std::max<uint64_t>(1, (c->ntot + 255) / 256);
  const uint64_t per = std::min<uint64_t>(16, std::max<uint64_t>(8, chunks / 16384));
  const uint64_t nb = std::min(chunks, std::max<uint64_t>(5ull * c->num_cu, (chunks + per - 1) / per));
  return static_cast<unsigned>(grid_waves ? std::min<uint64_t>(nb, std::max<uint32_t>(1u, grid_waves / 4)) : nb);
}

// Whether the State pass sums by rows: from as many drops per gridbox on as make the windows' reads for a
// lane or two dearer than the rows' extra work, and from 256 tiles of 16 gridboxes that fill the chip.
// Two sums (after motion) gain from 128 drops on, few gridboxes from 160 (us, windows / rows: 4096 of 128
// drops 11.1 / 13.5, of 170 14.8 / 14.0; 8192 of 128 13.2 / 13.2; 24679 of 300 93 / 41; 64^3 of 128
// 169 / 152, of 250 503 / 280).  One sum loses on few gridboxes, and on many, where the windows are near
// the bandwidth (64^3 of 128 65 / 77, of 150 79 / 86, of 190 105 / 105, of 230 140 / 125; 1M of 130
// 240 / 292; 8192 of 128 7.1 / 8.3, of 190 11.1 / 10.2; 4096 of 230 9.5 / 11.0; between them 32768 of 128
// 15.9 / 13.2, 65536 of 128 21.8 / 22.2, of 150 30 / 24, 8000 of 400 30 / 16).
static bool sums_by_rows(uint64_t ngbx, uint64_t mean, bool two) {
  if (ngbx < 256 * kRows) return false;
  if (two) return mean >= (ngbx < 8192 ? 160u : 128u);
  return mean >= (ngbx < 8192 ? 256u : ngbx < 16384 || ngbx > 65536 ? 192u : 128u);
}
static void launch_cond_state(cleo_ctx* c, CondFlatArgs a, uint32_t gw) {
  if (sums_by_rows(a.ngbx, c->ntot / a.ngbx, a.qm != nullptr)) {
    a.gpt = kRows;
    hipLaunchKernelGGL(k_cond_state<true>, dim3(gbx_blocks(sum_tiles(a.ngbx, kRows), 4, gw)), dim3(256), 0, c->stream, a);
  } else {
    hipLaunchKernelGGL(k_cond_state<false>, dim3(sum_blocks(c, gw)), dim3(256), 0, c->stream, a);
  }
}

// The deferral budget in counted iterations: the two that a restart repeats count for the drop but are
// not made again (8 that are made: 33M drops coupled 2.43 -> 2.39 ms a step against 8 counted; 6 to 16
// counted: 2.63, 2.43, 2.39, 2.39, 2.40 ms for 6, 8, 10, 12, 16).
static uint32_t counted_budget(uint32_t budget) { return budget ? std::min(budget, 0xfffffffdu) + 2u : 0u; }

void launch_condensation_flat(cleo_ctx* c, const CondFlatArgs& args) {
  if (args.ngbx == 0) return;
  CondFlatArgs a = args;
  // the thread-per-drop solve records each drop's qcond term, so the qcond recompute after motion
  // joins k_cond_state (the task ring keeps it in k_cond_prep)
  a.qm = (a.fuse_qcond && c->cond_variant() == 1) ? c->qm : nullptr;
  const uint32_t gw = c->tiles.cond_grid_waves;
  a.gpt = sum_gpt(c);
  const uint32_t budget = c->cond_variant() == 2 ? 0u : c->defer_budget();
  a.cfg.budget = counted_budget(budget);
  a.dlist = c->dlist;
  a.dcount = c->dcount;
  hipLaunchKernelGGL(k_cond_prep, dim3(sum_blocks(c, gw)), dim3(256), 0, c->stream, a);
  if (c->cond_variant() == 2) {
    // task-ring kernel: waves of 4 per block; by default as many waves as fit on the device at once
    const uint64_t waves = gw ? gw : static_cast<uint64_t>(c->num_cu) * kCondQueueWavesPerCu;
    const unsigned nb = static_cast<unsigned>(std::max<uint64_t>(1, std::min<uint64_t>(waves / 4, (c->ntot + 255) / 256)));
    a.stat = stat_slots(c);
    kev_mark(c, 0);
    hipLaunchKernelGGL(k_cond_queue, dim3(nb), dim3(256), 4 * kCondRingBytes, c->stream, a);
    kev_mark(c, 1);
  } else {
    const unsigned nb = solve_blocks(c, gw);
    a.stat = stat_slots(c);
    if (a.mlp_inline) {  // the learned guesses, from the saturation ratios k_cond_prep left
      hipLaunchKernelGGL(k_cond_guess, dim3(drop_blocks(c->ntot, gw ? gw : 32768)), dim3(256), 0, c->stream, a);
      a.warm = a.warm_buf;
    }
    kev_mark(c, 0);
    const bool tail = tail_solves(c, budget);
    if (tail)
      hipLaunchKernelGGL(k_cond_drops<true>, dim3(nb), dim3(256), 0, c->stream, a);
    else
      hipLaunchKernelGGL(k_cond_drops<false>, dim3(nb), dim3(256), 0, c->stream, a);
    if (!tail) launch_deferred(c, a, nb);
    kev_mark(c, 1);
  }
  launch_cond_state(c, a, gw);
}

// Motion, the neighbour sort and a condensation that follows at once, with the condensation solve
// in the sort's gather (k_sort_gather_cond): motion (thread per drop), the sort tables and ranks,
// the saturation ratios (State only), the gather with the solves, the commit of the sorted store,
// the deferred drops, then the ordered sums and the State update (with the qcond recompute).
// margs.s is the store motion reads, `dst` the sorted store; commit_dst >= 0: that buffer becomes
// current (else, for timing, the context's refs stay those of the unsorted store).
void motion_sort_condense(cleo_ctx* c, const MotionArgs& margs, const CondFlatArgs& cond, const SoA& dst,
                          int commit_dst) {
  const uint32_t ngbx = c->grid.ngbx;
  if (ngbx == 0) return;
  MotionArgs m = margs;
  m.step = c->dstep;
  // motion variant 3: the drops move inside the gather (the counting pass writes only the steps);
  // not with learned guesses, which are evaluated on the moved store before the gather
  const bool move_in_gather = c->motion_variant() == 3 && !cond.mlp_inline && !cond.warm;
  const bool on = c->kev_on;
  c->kev_on = false;  // the main kernel of this sequence is the gather with the solves
  if (move_in_gather) {
    const unsigned mb = motion_blocks(c->ntot, c->tiles.motion_grid_waves);
    m.stat = stat_slots(c);
    launch_motion_drops<false>(c, m, mb);
  } else {
    launch_motion_flat(c, m);
  }
  c->kev_on = on;
  NsortArgs n = nsort_args(c, m.s, dst);
  n.step = c->dstep;
  nsort_tables(c, n, cond.gs);
  launch_nsort_perm(c, n, ngbx);
  CondFlatArgs a = cond;
  a.s = dst;
  a.qm = c->qm;  // the qcond recompute joins k_cond_state
  const uint32_t gw = c->tiles.cond_grid_waves;
  a.gpt = sum_gpt(c);
  const uint32_t budget = c->defer_budget();
  a.cfg.budget = counted_budget(budget);
  a.dlist = c->dlist;
  a.dcount = c->dcount;
  if (a.mlp_inline) {  // learned guesses of the drops where motion left them
    CondFlatArgs ga = a;
    ga.s = m.s;
    ga.unsorted = 1;
    ga.guess_out = nullptr;
    hipLaunchKernelGGL(k_cond_guess, dim3(drop_blocks(c->ntot, gw ? gw : 32768)), dim3(256), 0, c->stream, ga);
    a.warm = a.warm_buf;
    a.warm_perm = n.perm;
  }
  const unsigned nb = solve_blocks(c, gw);
  a.stat = stat_slots(c);
  kev_mark(c, 0);
  const bool tail = tail_solves(c, budget);
  if (tail)
    launch_gather_cond<true>(c, n, a, move_in_gather ? &m : nullptr, nb);
  else
    launch_gather_cond<false>(c, n, a, move_in_gather ? &m : nullptr, nb);
  kev_mark(c, 1);
  if (!tail) launch_deferred(c, a, nb);
  if (commit_dst >= 0) nsort_commit(c, commit_dst);
  a.off = n.off_new;  // the sorted store's refs, of the same sort as its active counts
  launch_cond_state(c, a, gw);
}

void launch_motion_flat(cleo_ctx* c, const MotionArgs& args) {
  if (args.grid.ngbx == 0) return;
  MotionArgs a = args;
  const unsigned nb = motion_blocks(c->ntot, c->tiles.motion_grid_waves);
  a.stat = stat_slots(c);
  kev_mark(c, 0);
  launch_motion_drops<true>(c, a, nb);
  kev_mark(c, 1);
}

}  // namespace cleo
