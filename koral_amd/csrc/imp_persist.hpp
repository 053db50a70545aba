// The implicit-source solve of many cells as six passes, one per attempt of
// solve_implicit_lab's fallback chain (rad.c:1389-1464: energy LAB, energy
// FF, swapped LAB, swapped FF, entropy LAB, entropy swapped).
//
// Pass a works on the cells still unsolved after a - 1 attempts, held in two
// lists by the primitives attempt a iterates on (MHD or RAD).  One launch
// solves both lists, the MHD list first, each by code specialised at compile
// time for the attempt's (primitives, equation, frame), so the lanes of a
// wave run the same branch of the residual; a block whose share of the first
// list is done goes on to the second, so an attempt waits once for its
// slowest cells.  The kernels are persistent: a lane owns one cell at a time
// and advances it by one evaluation of the residual per trip of its loop
// (imp_lane_trip); idle lanes take the next list entries from a work counter
// (the wave ballots its idle lanes, one lane claims that many entries with
// one atomic add, each idle lane takes its rank).  A cell that fails the
// attempt is appended, by the same ballot/prefix-count scheme, to the list of
// the next attempt.  Cells need 1 to 51 iterations per attempt, so no lane
// waits for the slowest cell of its wave.  The solved cells' entropies and
// conserved states are formed by one pass over all cells at the end
// (k_imp_finish).
//
// A batch with few cells runs one launch in which a wave takes a cell through
// its whole chain (k_imp_wave).
//
// With a learned initial guess a first pass runs before the chain: the
// energy-equation lab-frame solve from a start given per cell.  With a
// radiation guess the learned classification takes the primitives of the
// chain's attempt 0 (the old state's E^ < RADIMPLICITTHRESHOLD u choice,
// rad.c:1381): the radiation primitives from the radiation network's guess
// (the gas part from the gas guess), or the gas primitives from the gas
// guess; without a radiation guess every cell takes the gas primitives.
// Iterations on the gas primitives are much cheaper (no inner gas inversion
// per residual), so a cell whose old state favours them tries them first
// even where it will need the radiation primitives.  With both guesses a
// cell the first learned try does not solve within its iteration budget
// tries the other primitive set from its guess (as the plain chain falls
// back between primitive sets).  A cell the learned tries do not solve enters
// attempt 0 of the plain chain unchanged, so the guess can change the
// iteration count but not what the chain would do without it.  A cell
// solved by a learned try reports attempt 6.
//
// Src provides, for a cell index c:
//   time()                         global time of the solve (device side)
//   load(c, uu00, pp00, g, dt)     inputs of the solve
//   init(c)                        before the first attempt
//   add_iters(c, it)               after every attempt
//   done_ok(c, pp, it, attempt, whichprim, whicheq, whichframe)   the solved
//                                  primitives but the entropy, and the flags
//   done_fail(c)                   after the sixth failed attempt
//   solved(c)                      whether done_ok was called for the cell
//   load_p(c, pp, g)               its primitives and metric
//   finish(c, pp, uu)              the entropy pp[5] and the conserved state
#pragma once
#include "dev_implicit.hpp"
#include "capi_util.hpp"

namespace kd {

// Device buffers of the passes: two list pairs (ping-pong, each n entries per
// primitive kind) and IMP_NCTR counters.  Counter 4 a + k: k = 0, 1 the list
// lengths for attempt a (MHD, RAD); k = 2, 3 the work counters of its two
// lists.  The first learned try reads list pair 1 (free until attempt 0
// writes its failures there) with lengths IMP_LEARN_LEN + k and work
// counters IMP_LEARN_Q + k; the second try reads the lists second[k] with
// lengths IMP_SECOND_LEN + k and work counters IMP_SECOND_Q + k (counters
// 24-27 are otherwise unused: attempt 5 appends nothing).
constexpr int IMP_NCTR = 33;
constexpr int IMP_SECOND_LEN = 24;
constexpr int IMP_SECOND_Q = 26;
constexpr int IMP_LEARN_LEN = 28;
constexpr int IMP_LEARN_Q = 30;
constexpr int IMP_ASYM = 32;  // set once a cell of the batch has a metric that is not symmetric
constexpr int IMP_LEARNED_ATTEMPT = 6;
struct ImpBufs {
  unsigned *list[2][2];
  unsigned *second[2];  // lists of the second learned try (learned solves only)
  unsigned *ctr;
};

// Batches of at most this many cells run the wave-per-cell chain: a cell's
// chain is about four times as fast by a wave as by a lane, but the chip then
// holds 2048 cells at a time instead of 65536 (measured: 3000 cells 7.9 ms
// against 24.5 ms by the passes, 10 000 cells 18.4 against 25.3 ms, 20 000
// cells 28.6 against 26.1 ms).
constexpr long IMP_WAVE_CELLS = 1L << 14;
// the line of the kernels without scratch (implicit_passes), which hold half
// the waves at a time: 12 288 cells 22.5 ms by waves, 12 289 cells 25.0 by the
// passes, 16 384 cells 28 by the passes
constexpr long IMP_WAVE_CELLS_NOSCRATCH = 3L << 12;

// pass modes of k_imp_pass
enum { IMP_CHAIN = 0, IMP_LEARN1 = 1, IMP_LEARN2 = 2 };

KD_INL int imp_other(int wp) { return wp == P_RAD ? P_MHD : P_RAD; }

// primitives of attempt a + 1 for a cell iterating on wp in attempt a
KD_INL int imp_next_wp(int a, int wp)
{
  const bool swapped = (a == 2 || a == 3 || a == 5);
  const int startwith = swapped ? imp_other(wp) : wp;
  const bool swapped_next = (a + 1 == 2 || a + 1 == 3 || a + 1 == 5);
  return swapped_next ? imp_other(startwith) : startwith;
}

KD_INL bool symmetric(const Geom &g)
{
  bool s = true;
#pragma unroll
  for (int i = 1; i < 4; i++)
#pragma unroll
    for (int j = 0; j < i; j++) s = s && g.g[i][j] == g.g[j][i] && g.G[i][j] == g.G[j][i];
  return s;
}

// sorts the n cells into the two attempt-0 lists by the primitives the
// chain starts with
template <int MAG, int RAD, class Src>
__global__ void __launch_bounds__(256) k_imp_classify(koral_params P, Src src, long n, ImpBufs b)
{
  constexpr int NV = Lay<MAG, RAD>::NV;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int wp = 0;
  if (c < n) {
    src.init(c);
    double uu00[NV], pp00[NV], dt;
    Geom g;
    src.load(c, uu00, pp00, g, dt);
    wp = imp_startwith<MAG, RAD>(P, pp00, g);
    if (!symmetric(g)) b.ctr[IMP_ASYM] = 1u;
  }
  append_index(wp == P_MHD, (unsigned)c, b.list[0][0], &b.ctr[0]);
  append_index(wp == P_RAD, (unsigned)c, b.list[0][1], &b.ctr[1]);
}

// learned classification: the primitive kind of every cell's first learned
// try (see above), or, for a cell whose gas start gxg is NaN, of its first
// chain attempt; gxr may be null
template <int MAG, class Src>
__global__ void __launch_bounds__(256) k_imp_learned_classify(koral_params P, Src src, long n, ImpBufs b,
                                                              const double *__restrict__ gxg,
                                                              const double *__restrict__ gxr)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int wp = 0;
  bool skip = false;  // no learned try: a NaN gas start (gated out)
  if (c < n) {
    src.init(c);
    wp = P_MHD;
    skip = isnan(gxg[c]);
    double uu00[NV], pp00[NV], dt;
    Geom g;
    src.load(c, uu00, pp00, g, dt);
    if (gxr || skip) wp = imp_startwith<MAG, 1>(P, pp00, g);
    if (!symmetric(g)) b.ctr[IMP_ASYM] = 1u;
  }
  // a skipped cell joins attempt 0 of the chain as a failed learned try does
  append_index(skip && wp == P_MHD, (unsigned)c, b.list[0][0], &b.ctr[0]);
  append_index(skip && wp == P_RAD, (unsigned)c, b.list[0][1], &b.ctr[1]);
  append_index(!skip && wp == P_MHD, (unsigned)c, b.list[1][0], &b.ctr[IMP_LEARN_LEN]);
  append_index(!skip && wp == P_RAD, (unsigned)c, b.list[1][1], &b.ctr[IMP_LEARN_LEN + 1]);
}

// lanes of a wave that wait, idle, until so many can take new cells at once:
// reading a cell holds the whole wave for a gather of 67 values
constexpr int IMP_REFILL = 8;

// A lane's LDS column (256 lanes a block): conserved state, the two 4x4
// metrics, gdet, alpha, gttpert, dt, the old u and E^.  SYM: the metrics of
// every cell are symmetric to the last bit (the usual case, found by the
// classification), ten numbers each: 39 doubles, so two blocks of four waves
// share a CU.  Otherwise, be it one cell of the batch, sixteen each for all of
// them and one block a CU: a table whose halves differ by rounding gives what
// reading both halves gives (2^22 cells 228 ms against 162).
template <int MAG, bool SYM>
struct LaneCol {
  static constexpr int NV = Lay<MAG, 1>::NV, M = SYM ? 10 : 16;
  static constexpr int G = NV, GDET = G + 2 * M, DT = GDET + 3, U0 = DT + 1, E0 = U0 + 1, N = E0 + 1;
};
template <bool SYM>
KD_INL constexpr int metric_index(int i, int j)
{
  return !SYM ? 4 * i + j : (i <= j ? i * 4 - i * (i - 1) / 2 + (j - i) : j * 4 - j * (j - 1) / 2 + (i - j));
}
// views of a column with the interface of a state vector and of Geom; an
// element is read where it is used, so none has to stay in registers
struct LaneVec {
  const double *p;
  KD_INL double operator[](int i) const { return p[i * 256]; }
};
template <bool SYM>
struct LaneMat {
  const double *p;
  struct Row {
    const double *p;
    int i;
    KD_INL double operator[](int j) const { return p[metric_index<SYM>(i, j) * 256]; }
  };
  KD_INL Row operator[](int i) const { return Row{p, i}; }
};
template <bool SYM>
struct LaneGeom {
  LaneMat<SYM> g, G;
  double gdet, alpha, gttpert;
};

// Attempt a on the cells of one list, all iterating on primitives WP with
// equation WE in frame WF.  Bound by FP64 issue, about 2000 FP64 instruction
// slots per evaluation, at the two waves per SIMD (SYM; one without) that the
// LDS columns allow.
template <int MAG, bool SYM, int WP, int WE, int WF, int MODE, class Src>
KD_INL void imp_pass_list(const koral_params &P, const Src &src, int a, const ImpBufs &b, int *counts,
                          const double *gxg, const double *gxr, long n_all, double (*keep)[256])
{
  constexpr int NV = Lay<MAG, 1>::NV;
  constexpr int EE = Lay<MAG, 1>::EE;
  using LC = LaneCol<MAG, SYM>;
  const double global_time = src.time();
  const int lane = threadIdx.x & 63;
  const int kind = (WP == P_MHD) ? 0 : 1;
  // the learned tries take lists of their own and hand failures to attempt 0;
  // attempt a takes its list and hands failures to attempt a + 1
  constexpr bool LEARN = MODE != IMP_CHAIN;
  // the first learned try hands failures to the second try on the other
  // primitives when there is one (b.second set), else to attempt 0; the
  // second try hands them to attempt 0; attempt a hands them to a + 1
  const bool to_second = MODE == IMP_LEARN1 && b.second[0] != nullptr;
  const unsigned *list = MODE == IMP_LEARN1 ? b.list[1][kind] : (MODE == IMP_LEARN2 ? b.second[kind] : b.list[a & 1][kind]);
  unsigned *out0 = to_second ? b.second[0] : (LEARN ? b.list[0][0] : b.list[(a + 1) & 1][0]);
  unsigned *out1 = to_second ? b.second[1] : (LEARN ? b.list[0][1] : b.list[(a + 1) & 1][1]);
  const long n = MODE == IMP_LEARN1 ? (long)b.ctr[IMP_LEARN_LEN + kind]
                                    : (MODE == IMP_LEARN2 ? (long)b.ctr[IMP_SECOND_LEN + kind] : (long)b.ctr[4 * a + kind]);
  unsigned *queue = MODE == IMP_LEARN1 ? &b.ctr[IMP_LEARN_Q + kind]
                                       : (MODE == IMP_LEARN2 ? &b.ctr[IMP_SECOND_Q + kind] : &b.ctr[4 * a + 2 + kind]);
  unsigned *out_len = to_second ? &b.ctr[IMP_SECOND_LEN] : (LEARN ? &b.ctr[0] : &b.ctr[4 * (a + 1)]);
  int next_kind = to_second ? 1 - kind : (LEARN ? 0 : ((imp_next_wp(a, WP) == P_MHD) ? 0 : 1));
  bool active = false, fresh = false, exhausted = n == 0;
  unsigned c = 0, c_push = 0;
  bool push = false;
  int n_ok = 0, n_it = 0, n_bad = 0;
  double pp[NV], J[16];
  ImpLane s;
  // The inputs of a lane's current cell, copied once when the lane takes the
  // cell: the lanes of a wave hold unrelated cells, so reloading them from
  // the cell arrays every trip would touch one cache line per lane and
  // value.  Column threadIdx.x belongs to this lane alone (no barrier).
  const int me = threadIdx.x;
  for (;;) {
    // failures of the last trip go to the next attempt's list
    append_index(push && next_kind == 0, c_push, out0, &out_len[0]);
    append_index(push && next_kind == 1, c_push, out1, &out_len[1]);
    push = false;
    const unsigned long long need = __ballot(!active);
    if (!exhausted) {
      const int cnt = __popcll(need);
      if (cnt >= IMP_REFILL) {
        const int leader = __ffsll((unsigned long long)need) - 1;
        unsigned base = 0;
        if (lane == leader) base = atomicAdd(queue, (unsigned)cnt);
        base = __shfl(base, leader);
        if ((long)base + cnt >= n) exhausted = true;
        if (!active) {
          const long k = (long)base + __popcll(need & ((1ull << lane) - 1ull));
          if (k < n) {
            c = list[k];
            active = true;
            fresh = true;
          }
        }
      }
    } else if (need == ~0ull) {
      break;
    }
    if (fresh) {
      fresh = false;
      double uu00[NV], dt;
      Geom g;
      src.load(c, uu00, pp, g, dt);
#pragma unroll
      for (int i = 0; i < NV; i++) keep[i][me] = uu00[i];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = SYM ? i : 0; j < 4; j++) {
          keep[LC::G + metric_index<SYM>(i, j)][me] = g.g[i][j];
          keep[LC::G + LC::M + metric_index<SYM>(i, j)][me] = g.G[i][j];
        }
      keep[LC::GDET][me] = g.gdet;
      keep[LC::GDET + 1][me] = g.alpha;
      keep[LC::GDET + 2][me] = g.gttpert;
      keep[LC::DT][me] = dt;
      keep[LC::U0][me] = pp[1];
      keep[LC::E0][me] = WF == FF ? -ff_Rtt<MAG, 1>(pp, g, nullptr) : 0.;
      if (LEARN) {
        if (!to_second) next_kind = (imp_startwith<MAG, 1>(P, pp, g) == P_MHD) ? 0 : 1;
        // the gas guess also starts the gas inversion of a radiation-primitive attempt
#pragma unroll
        for (int i = 0; i < 4; i++) pp[1 + i] = gxg[i * n_all + c];
        if (WP == P_RAD) {
#pragma unroll
          for (int i = 0; i < 4; i++) pp[EE + i] = gxr[i * n_all + c];
        }
      }
      imp_lane_start<WP, EE>(s, pp);
    }
    // On the gas primitives (few repeated trials) the wave runs the lanes of
    // one column, or those at the iterate, per trip: the part most of them
    // are at.  A lane that took an extra trial waits for the others to come
    // round, and the parts' own work (the inverse Jacobian above all) runs
    // with the wave full instead of in every trip for a fifth of its lanes.
    // Radiation primitives repeat trials too often to wait.
    bool run = active;
    if (WP == P_MHD) {
      const int part = s.stage > 4 ? 0 : s.stage;
      int best = 0, most = -1;
#pragma unroll
      for (int q = 0; q < 5; q++) {
        const int cnt = __popcll(__ballot(active && part == q));
        if (cnt > most) {
          most = cnt;
          best = q;
        }
      }
      run = active && part == best;
    }
    if (run) {
      const LaneGeom<SYM> g{LaneMat<SYM>{&keep[LC::G][me]}, LaneMat<SYM>{&keep[LC::G + LC::M][me]},
                            keep[LC::GDET][me], keep[LC::GDET + 1][me], keep[LC::GDET + 2][me]};
      const int st = imp_lane_trip<MAG, WP, WE, WF>(P, s, pp, LaneVec{&keep[0][me]}, keep[LC::U0][me],
                                                    keep[LC::E0][me], keep[LC::DT][me], g, global_time,
                                                    P.radimpmaxiter, [&](int i) -> double & { return J[i]; });
      if (st != IMP_CONT) {
        src.add_iters(c, s.iter);
        if (st == IMP_OK) {
          src.done_ok(c, pp, s.iter, LEARN ? IMP_LEARNED_ATTEMPT : a, WP, WE, WF);
          n_ok++;
          n_it += s.iter;
        } else if (!LEARN && a == 5) {
          src.done_fail(c);
          n_bad++;
        } else {
          push = true;
          c_push = c;
        }
        active = false;
      }
    }
  }
  if (counts) {
    for (int off = 32; off > 0; off >>= 1) {
      n_ok += __shfl_xor(n_ok, off);
      n_it += __shfl_xor(n_it, off);
      n_bad += __shfl_xor(n_bad, off);
    }
    if (lane == 0) {
      if (n_ok) atomicAdd(&counts[0], n_ok);
      if (n_it) atomicAdd(&counts[1], n_it);
      if (n_bad) atomicAdd(&counts[2], n_bad);
    }
  }
}

// attempt a on both lists; both variants are launched, and the one the
// classification did not find to apply ends at once
template <int MAG, bool SYM, int WE, int WF, int MODE, class Src>
__global__ void __launch_bounds__(256, SYM ? 2 : 1) k_imp_pass(koral_params P, Src src, int a, ImpBufs b, int *counts,
                                                               const double *gxg, const double *gxr, long n_all)
{
  __shared__ double keep[LaneCol<MAG, SYM>::N][256];
  if ((b.ctr[IMP_ASYM] == 0) != SYM) return;
  imp_pass_list<MAG, SYM, P_MHD, WE, WF, MODE>(P, src, a, b, counts, gxg, gxr, n_all, keep);
  imp_pass_list<MAG, SYM, P_RAD, WE, WF, MODE>(P, src, a, b, counts, gxg, gxr, n_all, keep);
}

// entropy and conserved state of the solved cells
template <int MAG, class Src>
__global__ void __launch_bounds__(256) k_imp_finish(koral_params P, Src src, long n)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n || !src.solved(c)) return;
  double pp[NV], uu[NV];
  Geom g;
  src.load_p(c, pp, g);
  imp_finish<MAG>(P, pp, uu, g);
  src.finish(c, pp, uu);
}

// The whole chain of n cells, a wave per cell: a cell's attempts follow one
// another in its wave, so the time of a launch with few cells is one cell's
// chain.  Two waves per SIMD (WPS) spill 430 bytes a lane and are still faster
// than one without spills (7.4 against 9.7 ms for 3001 cells).
template <int MAG, int WPS, class Src>
__global__ void __launch_bounds__(256, WPS) k_imp_wave(koral_params P, Src src, int *counts, const double *gxg,
                                                     const double *gxr, long n, int learned_maxiter)
{
  constexpr int NV = Lay<MAG, 1>::NV;
  constexpr int EE = Lay<MAG, 1>::EE;
  __shared__ WaveCell<MAG> cells[4];
  WaveCell<MAG> &w = cells[threadIdx.x >> 6];
  const double gt = src.time();
  const int lane = threadIdx.x & 63;
  const long nw = (long)gridDim.x * (blockDim.x >> 6);
  int n_ok = 0, n_it = 0, n_bad = 0;
  for (long k = (long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); k < n; k += nw) {
    const unsigned c = (unsigned)k;
    int at = 0;
    {
      // every lane stores the same values to its own wave's copy
      double uu00[NV], pp00[NV], dt;
      Geom g;
      src.load(c, uu00, pp00, g, dt);
      wave_sync();
#pragma unroll
      for (int i = 0; i < NV; i++) {
        w.uu[i] = uu00[i];
        w.pp00[i] = pp00[i];
      }
      w.g = g;
      w.dt = dt;
      w.Ehat0 = -ff_Rtt<MAG, 1>(pp00, g, nullptr);
      wave_sync();
    }
    const double Ehat0 = w.Ehat0;
    const int start = (Ehat0 < P.radimplicitthreshold * w.pp00[1]) ? P_RAD : P_MHD;  // imp_startwith
    if (lane == 0) src.init(c);
    // a NaN gas start has no learned try
    if (gxg && !isnan(gxg[c])) at = IMP_LEARNED_ATTEMPT;
    for (;;) {
      const bool learn = at >= IMP_LEARNED_ATTEMPT;
      const int second = at - IMP_LEARNED_ATTEMPT;
      ImpKind kd;
      if (learn) {
        // without a radiation guess every learned try takes the gas primitives
        kd = ImpKind{gxr ? (second ? imp_other(start) : start) : P_MHD, ENERGYEQ, LAB};
      } else {
        imp_attempt(at, start, kd.wp, kd.we, kd.wf);
      }
      // (a vector value even where it is uniform: the attempt takes scalars)
      kd.wp = __builtin_amdgcn_readfirstlane(kd.wp);
      kd.we = __builtin_amdgcn_readfirstlane(kd.we);
      kd.wf = __builtin_amdgcn_readfirstlane(kd.wf);
      wave_sync();
#pragma unroll
      for (int i = 0; i < NV; i++) w.pp[i] = w.pp00[i];
      if (learn) {
#pragma unroll
        for (int i = 0; i < 4; i++) w.pp[1 + i] = gxg[i * n + c];
        if (kd.wp == P_RAD) {
#pragma unroll
          for (int i = 0; i < 4; i++) w.pp[EE + i] = gxr[i * n + c];
        }
      }
      wave_sync();
      int iter = 0;
      const int st = imp_wave_attempt<MAG>(P, kd, w, gt, learn ? learned_maxiter : P.radimpmaxiter, iter);
      if (lane == 0) src.add_iters(c, iter);
      if (st == IMP_OK) {
        double uu[NV], pp[NV];
#pragma unroll
        for (int i = 0; i < NV; i++) pp[i] = w.pp[i];
        imp_finish<MAG>(P, pp, uu, w.g);
        if (lane == 0) {
          src.finish(c, pp, uu);
          src.done_ok(c, pp, iter, learn ? IMP_LEARNED_ATTEMPT : at, kd.wp, kd.we, kd.wf);
        }
        n_ok++;
        n_it += iter;
        break;
      }
      if (at == 5) {
        if (lane == 0) src.done_fail(c);
        n_bad++;
        break;
      }
      at = learn ? ((gxr && second == 0) ? at + 1 : 0) : at + 1;
    }
  }
  if (counts && lane == 0) {
    if (n_ok) atomicAdd(&counts[0], n_ok);
    if (n_it) atomicAdd(&counts[1], n_it);
    if (n_bad) atomicAdd(&counts[2], n_bad);
  }
}

// clears n (<= 64) counters on the launching stream (a kernel, so the clear
// can sit inside a captured graph), and sets counter one (>= 0) to 1
static __global__ void k_zero_u32(unsigned *q, int n, int one)
{
  if ((int)threadIdx.x < n) q[threadIdx.x] = (int)threadIdx.x == one ? 1u : 0u;
}

// Blocks of bs threads that fill every CU at the kernel's occupancy (never
// more than the n work items need).
template <class K>
int resident_blocks(K kernel, int bs, long n, unsigned *blocks)
{
  int dev = 0, cus = 0, per = 0;
  int rc = check_hip(hipGetDevice(&dev), "hipGetDevice");
  if (!rc) rc = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "CU count");
  if (!rc) rc = check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, bs, 0), "occupancy");
  if (rc) return rc;
  if (per < 1) per = 1;
  long want = (long)cus * per;
  long need = (n + bs - 1) / bs;
  if (need < 1) need = 1;
  *blocks = (unsigned)(want < need ? want : need);
  return 0;
}

// Two blocks a CU where the lanes have several cells each; fewer cells finish
// sooner with the SIMDs to themselves (measured: 262 144 cells 37.1 against
// 38.9 ms, 2^20 cells 75.2 against 65.0 ms with one and two blocks a CU).
constexpr long IMP_TWO_BLOCKS = 1L << 19;
template <int MAG, bool SCRATCH, int WE, int WF, int MODE = IMP_CHAIN, class Src>
int imp_launch_pass(const koral_params &P, const Src &src, long n, int a, const ImpBufs &b, int *counts,
                    hipStream_t s, const double *gxg = nullptr, const double *gxr = nullptr)
{
  unsigned two = 0, one = 0;
  int rc = resident_blocks(k_imp_pass<MAG, false, WE, WF, MODE, Src>, 256, n, &one);
  if constexpr (SCRATCH) {
    if (!rc) rc = resident_blocks(k_imp_pass<MAG, true, WE, WF, MODE, Src>, 256, n, &two);
    if (n < IMP_TWO_BLOCKS && two > one) two = one;
    if (!rc) k_imp_pass<MAG, true, WE, WF, MODE, Src><<<two, 256, 0, s>>>(P, src, a, b, counts, gxg, gxr, n);
  }
  if (rc) return rc;
  k_imp_pass<MAG, false, WE, WF, MODE, Src><<<one, 256, 0, s>>>(P, src, a, b, counts, gxg, gxr, n);
  return 0;
}

// all passes for n cells (asynchronous on s); counts may be null.  With a
// learned guess, gxg [4][n] is the gas start (u, u~^1..3) and gxr [4][n] (may
// be null) the radiation start (E, F~^1..3); the learned pass stops a cell
// after learned_maxiter iterations when that is positive and below
// RADIMPMAXITER.
//
// SCRATCH false: kernels that need no scratch memory alone, for a caller that
// cannot have device memory taken (the runtime sets scratch aside when a queue
// first runs a kernel that spills: 216 MiB for the wave kernel, 26 for the
// passes).  These are the wave kernel at one wave per SIMD and the passes'
// general variant, at one block a CU.
template <int MAG, bool SCRATCH = true, class Src>
int implicit_passes(const koral_params &P, const Src &src, long n, const ImpBufs &b, int *counts, hipStream_t s, const double *gxg = nullptr, const double *gxr = nullptr, int learned_maxiter = 0)
{
  const unsigned nb = (unsigned)((n + 255) / 256);
  koral_params Pl = P;
  if (learned_maxiter > 0 && learned_maxiter < Pl.radimpmaxiter) Pl.radimpmaxiter = learned_maxiter;
  int rc = 0;
  if (n <= (SCRATCH ? IMP_WAVE_CELLS : IMP_WAVE_CELLS_NOSCRATCH)) {
    constexpr int WPS = SCRATCH ? 2 : 1;
    unsigned blocks = 0;
    rc = resident_blocks(k_imp_wave<MAG, WPS, Src>, 256, 64 * n, &blocks);
    if (!rc) k_imp_wave<MAG, WPS, Src><<<blocks, 256, 0, s>>>(P, src, counts, gxg, gxr, n, Pl.radimpmaxiter);
    return rc;
  }
  k_zero_u32<<<1, 64, 0, s>>>(b.ctr, IMP_NCTR, SCRATCH ? -1 : IMP_ASYM);
  if (gxg) {
    k_imp_learned_classify<MAG, Src><<<nb, 256, 0, s>>>(P, src, n, b, gxg, gxr);
    // without a radiation guess there is no second try: b.second must then be null
    ImpBufs bl = b;
    if (!gxr) bl.second[0] = bl.second[1] = nullptr;
    rc = imp_launch_pass<MAG, SCRATCH, ENERGYEQ, LAB, IMP_LEARN1>(Pl, src, n, 0, bl, counts, s, gxg, gxr);
    if (!rc && bl.second[0]) rc = imp_launch_pass<MAG, SCRATCH, ENERGYEQ, LAB, IMP_LEARN2>(Pl, src, n, 0, bl, counts, s, gxg, gxr);
  } else {
    k_imp_classify<MAG, 1, Src><<<nb, 256, 0, s>>>(P, src, n, b);
  }
  for (int a = 0; a < 6 && !rc; a++) {
    if (a >= 4)
      rc = imp_launch_pass<MAG, SCRATCH, ENTROPYEQ, LAB>(P, src, n, a, b, counts, s);
    else if (a == 1 || a == 3)
      rc = imp_launch_pass<MAG, SCRATCH, ENERGYEQ, FF>(P, src, n, a, b, counts, s);
    else
      rc = imp_launch_pass<MAG, SCRATCH, ENERGYEQ, LAB>(P, src, n, a, b, counts, s);
  }
  if (!rc) k_imp_finish<MAG, Src><<<nb, 256, 0, s>>>(P, src, n);
  return rc;
}

}  // namespace kd
