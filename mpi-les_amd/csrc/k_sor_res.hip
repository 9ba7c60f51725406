// The red-black SOR of press (press.f95:89-122) as one launch per solve: the
// iterates and the right-hand side stay in the registers of the whole GPU
// from the first iteration to the last.
//
// A domain is cut into nb boxes of pairs x rows x levels, one per block, with
// one block or two per compute unit (kResClass).  A thread owns one (pair, row) column
// of its box -- red and black cell of each level, their rhs, in registers --
// so the k neighbours are its own values; the in-plane neighbours come from
// one LDS copy of the colour last updated, with a ring of halo cells around
// it.  After each colour sweep the blocks exchange the cells on their box
// faces through memory as 8-byte {value, tag} words (relaxed agent-scope
// atomics: a word whose tag is the expected sweep carries the value, so no
// flag, fence or second round trip is needed).  Every update is k_sor_pair's
// expression on the same operands, so the iterates have the same bits.
//
// What bounds it: the exchange on small domains (one word crosses between two
// compute units in 1 us, and a solve of 50 iterations waits for 100 of them
// in a row); on large ones the vector ALU (37 lane-instructions per cell and
// iteration, 377 of the 656 us of a solve at 300x300x90) and the words (2.7 GB
// of memory traffic there, 4 TB/s, for 0.13 GB of fields).  The
// launches per two iterations it replaces where a domain fits (k_sor_pair)
// cost 8 us each on the smallest domains and recompute a four-cell ring and
// six extra levels per block on large ones (0.37 of their lane-steps are
// useful at 300x300x90).  Microseconds of a 50-iteration solve, before and
// now: 24x20x16 455 and 163, 96x96x64 498 and 232, 150x150x90 675 and 319,
// 203x117x61 878 and 318 (odd jm: one iteration per launch before), 256x256x64
// 898 and 385, 300x300x90 1130 and 656.
//
// Waiting on other blocks is safe only while all of them run.  The blocks
// first count themselves in (res_arrive, res_enter).  When all have arrived, none can be
// left unscheduled and the waits always end.  When they have not within
// kEnterTicks (another process's blocks hold the compute units; the steps of
// this one are in order, turns.h), the launch
// falls back to sweeps over memory handed out by a ticket counter
// (res_ticket): a sweep waits only for tickets taken earlier, which running
// blocks hold, so that needs no co-residency at all.  It takes 8 to 10 times
// as long as the launch-per-iterations kernels, so the host, told by a counter,
// goes over to those for some steps (res_review).
#include <algorithm>
#include <type_traits>

#include "les_kernels.h"

namespace les {

namespace {

typedef unsigned long long u64;
// Two kernels: one block per compute unit with 256 registers a thread, and two
// blocks per unit with 128.  With two, one box computes while the other waits
// for its halo; with one, the box is larger (fewer faces) and the loads of four
// levels are in flight at a time.  per: blocks per unit; plane: floats per
// level of the LDS copy (a box and its halo ring, and a cell nothing reads),
// at most; words: in-plane halo words per thread, at most; levels: of a box
// (two to four registers each), at most; group: levels fetched together.
constexpr int kResNT = 512;  // threads per block, at most
struct ResClass {
  int per, plane, words, levels, group;
};
constexpr ResClass kResClass[2] = {{1, 832, 8, 40, 4}, {2, 640, 4, 24, 2}};
// Levels whose black rhs lies in LDS beside the copy instead of in registers.
constexpr int res_lds_rhs(int cls, int bk) {
  const int room = (163840 / kResClass[cls].per - 512 - 4 * bk * kResClass[cls].plane) / (4 * kResNT);
  return cls == 0 ? 0 : room < bk ? room : bk;
}
constexpr long long kEnterTicks = 1000000;  // 10 ms of the 100 MHz wall clock
constexpr int kEnterShift = 6;  // ... and 0.16 after as many solves in a row by tickets
constexpr int kTickets = 128;   // pieces a sweep is handed out in, at most
constexpr int kSpinMax = 1 << 22;  // polls of one word before the solve is given up (seconds)

__device__ __forceinline__ int rcix(const SplitGrid& s, int t, int j, int k) {
  return t + (j - 1) * s.cp + (k - 1) * s.cplane;
}

template <class T>
__device__ __forceinline__ T ald(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void ast(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 word(unsigned tag, float v) { return ((u64)tag << 32) | __float_as_uint(v); }
__device__ __forceinline__ unsigned wtag(u64 w) { return (unsigned)(w >> 32); }
__device__ __forceinline__ float wval(u64 w) { return __uint_as_float((unsigned)w); }
// A table no kernel running beside this one writes: uniform reads of it are
// scalar loads whatever the kernel stores in between.
typedef const __attribute__((address_space(4))) float* ConstF;
__device__ __forceinline__ ConstF constf(const float* p) { return (ConstF)(unsigned long long)p; }

// The solve's arguments, read again where they are used (scalar loads from
// the scalar cache): held over the solve they would take most of the scalar
// registers, and the rest would spill into vector ones.
typedef const __attribute__((address_space(4))) ResArgs* ConstArgs;
__device__ __forceinline__ ConstArgs again(ConstArgs a) {
  asm volatile("" : "+s"(a));
  return a;
}

// The sum of v over the wave, in its last lane (row shifts and broadcasts of
// the vector ALU: no LDS latency).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_sum_last(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  return dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}

// The sum of v over the block, in thread 0, the waves' totals in wave order.
__device__ __forceinline__ double res_block_sum(double v, int tid, int nthr, double* lds) {
  for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  if (tid % kWave == 0) lds[tid / kWave] = v;
  __syncthreads();
  double s = 0.0;
  if (tid == 0)
    for (int w = 0; w < nthr / kWave; w++) s += lds[w];
  __syncthreads();
  return s;
}

// The mean of the rhs, in every thread: the partial sums added in the order of
// k_finalize_head's 256 threads.
__device__ __forceinline__ double res_mean(ConstArgs a, int tid, int nthr, double* lds) {
  const int n = a->nred, lane = tid % kWave;
  const double* const part = a->rpart;
  for (int w = tid / kWave; w < 256 / kWave; w += nthr / kWave) {
    double s = 0.0;
    for (int b = w * kWave + lane; b < n; b += 256) s += part[b];
    for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
    if (lane == 0) lds[w] = s;
  }
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < 256 / kWave; w++) s += lds[w];
  __syncthreads();
  return s / a->area;
}

// Records iteration l's sum of reltmp^2 and returns whether it stops the
// loop (press.f95:119-121, or a non-finite sum).
__device__ __forceinline__ bool res_record(Ctrl* ctrl, int l, double s, float pjuge, bool writer) {
  const bool bad = !(s == s) || s > 1.0e300;
  const bool stop = s < (double)pjuge || bad;
  if (writer) {
    if (l <= kSorHist) ctrl->sor_hist[l - 1] = s;
    ctrl->sor_iters = l;
    if (bad) ctrl->nonfinite = 1;
    if (stop) ctrl->sor_done = l;
  }
  return stop;
}

// The block after the boxes: the stop test of every iteration (press.f95:
// 119-121), off the boxes' way.  Adds each iteration's partial sums in a fixed
// order, records the total and publishes one word: its tag that of the sums,
// its value 1 where the loop stops.
__device__ __forceinline__ void res_monitor(ConstArgs a, int nb, unsigned tag, int tid, int nthr, double* lds) {
  const int np = nb * (nthr / kWave);  // one partial sum per wave
  for (int l = 1; l <= a->nmaxp; l++) {
    const unsigned pt = tag + 2 * l;
    double x = 0.0;
    for (int b = tid; b < np; b += nthr) {
      const u64* const pw = a->parts + ((size_t)(l & 3) * np + b) * 2;
      u64 h = ald(pw), lo = ald(pw + 1);
      for (int spin = 0; wtag(h) != pt || wtag(lo) != pt;) {
        h = ald(pw);
        lo = ald(pw + 1);
        if (++spin > kSpinMax) return;  // cannot happen while every block runs
      }
      x += __longlong_as_double((long long)((h << 32) | (lo & 0xffffffffull)));
    }
    x = res_block_sum(x, tid, nthr, lds);
    if (tid == 0) {
      const bool stop = res_record(a->ctrl, l, x, a->pjuge, true);
      ast(a->parts + 8 * (size_t)np + (l & 3), ((u64)pt << 32) | (stop ? 1u : 0u));
      lds[0] = stop ? 1.0 : 0.0;
    }
    __syncthreads();
    const bool stop = lds[0] != 0.0;
    __syncthreads();
    if (stop) return;
  }
}

// Iteration l's word of the monitor: 1 where the loop stops.
__device__ __forceinline__ int res_verdict(ConstArgs a, int np, int l, unsigned pt, int* dead) {
  const u64* const pw = a->parts + 8 * (size_t)np + (l & 3);
  u64 w = ald(pw);
  for (int spin = 0; wtag(w) != pt;) {
    w = ald(pw);
    if (++spin > kSpinMax) {
      *dead = 1;
      break;
    }
  }
  return (int)(w & 1u);
}

// 1: every block of the launch is resident; 2: they are not, and the launch
// runs by tickets.  Thread 0 of each block; the last block to arrive decides
// 1, a block that waited kEnterTicks decides 2, whichever comes first.  Where
// the launches before went by tickets the wait is shorter, for work that holds
// the device mostly goes on holding it: steps enqueued ahead would pay it each.
__device__ __forceinline__ void res_arrive(Ctrl* ctrl, int nb) {
  const int n = __hip_atomic_fetch_add(&ctrl->res_arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (n == nb - 1) {
    int want = 0;
    __hip_atomic_compare_exchange_strong(&ctrl->res_state, &want, 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  }
}
__device__ __forceinline__ int res_enter(Ctrl* ctrl, int* note) {
  const long long t0 = wall_clock64();
  for (;;) {
    const int st = ald(&ctrl->res_state);
    if (st != 0) return st;
    const long long t = wall_clock64() - t0;
    if (t > (kEnterTicks >> kEnterShift) && t > (kEnterTicks >> min(ald(&ctrl->res_short), kEnterShift))) {
      int want = 0;
      if (__hip_atomic_compare_exchange_strong(&ctrl->res_state, &want, 2, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)) {
        ast(&ctrl->res_short, ald(&ctrl->res_short) + 1);
        // the solves of a domain follow each other: one writer at a time
        const int n = __hip_atomic_load(note, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(note, n + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      return ald(&ctrl->res_state);
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

// The solve without co-residency: colour sweeps over the split arrays (sets 0
// and 1 by iteration parity, as k_sweep), each cut into tickets taken in
// order.  A sweep starts when the one before is complete; its tickets were
// taken before and are held by running blocks.
__device__ __forceinline__ void res_ticket(ConstArgs a0, float* lds_f, double av) {
  double* const lds = (double*)lds_f;
  int* const sh = (int*)(lds_f + 2 * (kResNT / kWave));
  const int tid = threadIdx.x, nthr = blockDim.x;
  const ConstArgs a = a0;
  const Grid g = {a->g.im, a->g.jm, a->g.km, a->g.sj, a->g.sk};
  const SplitGrid s = {a->s.nt, a->s.cp, a->s.cplane};
  Ctrl* ctrl = a->ctrl;
  const int im = g.im, jm = g.jm, km = g.km, nt = s.nt;
  if (a->nred > 0 && blockIdx.x == 0 && tid == 0) ctrl->rhsav = av;
  const int npr = nt * jm;                          // pairs per level
  const int chunks = (npr + nthr - 1) / nthr;      // pieces of a level, a pair to each thread
  const int items = chunks * km;
  // pieces per ticket: kTickets tickets per sweep.  Each costs its place in two
  // counters and the fences that carry a sweep from one block to another: a
  // step of 300x300x90 took 170 ms with a ticket per piece (7920 per sweep), 34
  // with 990, 14.1 with 256, 12.7 with 128 and 17.5 with 64; 96x96x64 17.7, 9.7, 4.2,
  // 4.3 and 4.3.
  const int span = (items + kTickets - 1) / kTickets;
  const int per = (items + span - 1) / span;        // tickets per sweep
  for (;;) {
    __syncthreads();
    if (tid == 0)
      sh[0] = __hip_atomic_fetch_add(&ctrl->tk_next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tk = sh[0];
    // sweep 0 is the copy of the start iterate into set 0, sweep 2l-1 red of
    // iteration l, 2l its black
    const int sweep = tk / per, it = tk % per;
    if (sweep > 2 * a->nmaxp) return;
    if (tid == 0) {
      sh[1] = 0;
      for (int spin = 0; ald(&ctrl->tk_phase) < sweep; spin++) {
        __builtin_amdgcn_s_sleep(2);
        if (spin > kSpinMax) {  // cannot happen: the tickets waited for are held by running blocks
          ctrl->nonfinite = 1;
          sh[1] = 1;
          break;
        }
      }
      if (ald(&ctrl->sor_done) != 0) sh[1] = 1;
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (sh[1] != 0) return;
    const int l = (sweep + 1) / 2, col = sweep & 1;  // col 1 = red
    const int src = (l - 1) & 1, dst = l & 1;
    double acc = 0.0;
    for (int m = it * span; m < min(items, (it + 1) * span); m++) {
      const int x = (m % chunks) * nthr + tid, k = 1 + m / chunks;
      if (x >= npr) continue;
      const int t = x % nt, j = 1 + x / nt;
      const int q = rcix(s, t, j, k);
      if (sweep == 0) {
        for (int c = 0; c < 2; c++) {
          const int i = 2 * t + 1 + ((1 + j + k + c) & 1);
          a->sb.p[0][c][q] = (a->zero || i > im) ? 0.0f : a->pent[ix(g, i, j, k)];
          if (a->nred > 0) a->sb.rhs[c][q] = (float)((double)a->rhsr[c][q] - av);
        }
      } else {
        const int pos = (1 + j + k + col) & 1, i = 2 * t + 1 + pos;
        if (i <= im) {
          const float* own_ = a->sb.p[src][col];
          const float* oth = a->sb.p[col ? src : dst][col ^ 1];
          const float own = own_[q];
          const bool ent = l == 1 && !a->zero;  // iteration 1 reads the ghosts p had on entry
          // i ghosts mirror the cell; j wraps (the cell's own colour when jm is odd); k ghosts mirror
          float lo = (i == 1) ? own : oth[q - 1 + pos];
          float hi = (i == im) ? own : oth[q + pos];
          const float* wr = (jm & 1) ? own_ : oth;
          float pjm = (j == 1) ? wr[rcix(s, t, jm, k)] : oth[q - s.cp];
          float pjp = (j == jm) ? wr[rcix(s, t, 1, k)] : oth[q + s.cp];
          float pkm = (k == 1) ? own : oth[q - s.cplane];
          float pkp = (k == km) ? own : oth[q + s.cplane];
          if (ent) {
            if (col == 1) {
              if (i == 1) lo = a->pent[ix(g, 0, j, k)];
              if (i == im) hi = a->pent[ix(g, im + 1, j, k)];
              if (j == 1) pjm = a->pent[ix(g, i, 0, k)];
              if (j == jm) pjp = a->pent[ix(g, i, jm + 1, k)];
            }
            if (k == 1) pkm = a->pent[ix(g, i, j, 0)];
            if (k == km) pkp = a->pent[ix(g, i, j, km + 1)];
          }
          const float rel = a->omega * (a->m.lev4[4 * k + 2] * (a->c2 * hi + a->c2 * lo + a->c3 * pjp + a->c3 * pjm +
                                                          M1(a->m.cn4l, k) * pkp + M1(a->m.cn4s, k) * pkm -
                                                          a->sb.rhs[col][q]) -
                                       own);
          a->sb.p[dst][col][q] = own + rel;
          acc += (double)rel * (double)rel;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const double bsum = res_block_sum(acc, tid, nthr, lds);  // its barriers: every store of the block is released
    if (tid == 0) {
      ast((u64*)&a->tparts[(size_t)(sweep & 3) * per + it], (u64)__double_as_longlong(bsum));
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      sh[0] = __hip_atomic_fetch_add(&ctrl->tk_done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    if (sh[0] != (sweep + 1) * per - 1) continue;
    // the sweep's last ticket: iteration l's sum after its black sweep, then the next sweep
    double tot = 0.0;
    if (sweep > 0 && col == 0) {
      for (int b = tid; b < per; b += nthr) {
        tot += __longlong_as_double((long long)ald((u64*)&a->tparts[(size_t)((sweep - 1) & 3) * per + b]));
        tot += __longlong_as_double((long long)ald((u64*)&a->tparts[(size_t)(sweep & 3) * per + b]));
      }
      tot = res_block_sum(tot, tid, nthr, lds);
    }
    if (tid == 0) {
      bool stop = false;
      if (sweep > 0 && col == 0) {
        stop = res_record(ctrl, l, tot, a->pjuge, true);
        ctrl->p_final = l & 1;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      // a stop ends every wait: the tickets of later sweeps find sor_done
      ast(&ctrl->tk_phase, stop ? 0x7fffffff : sweep + 1);
    }
  }
}

// The resident solve of one box.  CLS: the kernel (kResClass); a block is
// launched with as many waves as its largest box has columns or halo words
// for.  BK: the most levels of a box, of which a box has BK-4 to BK.  OM1:
// omega == 1 (1*y is y: the multiplication is dropped).  ODD: im is odd, so
// the last pair of a row has one cell.
template <int CLS, int BK, bool OM1, bool ODD>
__device__ __forceinline__ void res_block(ConstArgs a0, const int bid) {
  constexpr int PLANE = kResClass[CLS].plane, NW = kResClass[CLS].words, G = kResClass[CLS].group;
  constexpr int NG = (BK + G - 1) / G, NT = kResNT, RL = res_lds_rhs(CLS, BK);
  __shared__ float S[BK * PLANE];
  __shared__ float RB[RL > 0 ? RL * NT : 1];  // rhs of the black cells of levels below RL, by thread
  __shared__ double wsum[NT / kWave], av_s;
  __shared__ int sh[3];  // mode; a wait that gave up; the monitor's verdict
  const int tid = threadIdx.x, nthr = blockDim.x, nwav = nthr / kWave;
  const int nb = a0->nb;
  // sor_done set on entry (a finished defect correction): nothing to solve
  const bool skip = a0->ctrl->sor_done != 0;  // (no block passes res_enter, to change it, before all have read it)
  if (tid == 0 && !skip && !a0->force_ticket) res_arrive(a0->ctrl, nb + 1 + a0->missing);
  const double av = a0->nred > 0 ? res_mean(again(a0), tid, nthr, wsum) : 0.0;  // while the others arrive
  if (tid == 0) {
    sh[0] = skip ? 0 : a0->force_ticket ? 2 : res_enter(a0->ctrl, a0->note);
    sh[1] = 0;
    av_s = av;  // read where the rhs is
  }
  __syncthreads();
  const int mode = sh[0];
  if (mode == 0) return;
  if (mode == 2) {
    res_ticket(a0, S, av);
    return;
  }
  if (bid == nb) {
    if (tid == 0) ast(&a0->ctrl->res_short, 0);
    res_monitor(again(a0), nb, (unsigned)a0->ctrl->res_epoch * 8192u, tid, nthr, wsum);
    return;
  }
  const int W = a0->tp + 2;  // LDS row pitch; halo columns 0 and tpn+1, halo rows 0 and tjn+1
  const bool oddj = (a0->g.jm & 1) != 0;
  // balanced cuts: box sizes differ by at most one in each direction
  const int bx = bid % a0->ntx, by = (bid / a0->ntx) % a0->nty, bz = bid / (a0->ntx * a0->nty);
  const int k0 = 1 + bz * a0->g.km / a0->ntz, nlev = (bz + 1) * a0->g.km / a0->ntz + 1 - k0;
  const bool kbot = bz == 0, ktop = bz == a0->ntz - 1;
  int cent, side, rowd = 0;
  bool act, wl[2], inv[2], wrl, wrh;
  unsigned wsd[NW], wto[NW];  // S source | S destination; word in the inboxes | destination by colour << 31
  {
    const ConstArgs a = again(a0);
    const int nt = a->s.nt, jm = a->g.jm, im = a->g.im;
    const int t0 = bx * nt / a->ntx, tpn = (bx + 1) * nt / a->ntx - t0;
    const int j0 = 1 + by * jm / a->nty, tjn = (by + 1) * jm / a->nty + 1 - j0;
    const int row = tid / tpn, t = tid % tpn;
    act = row < tjn;
    const int tg = t0 + t;
    const int par = (j0 + row + k0) & 1;  // position (i = 2t+1+position) of the red cell at the first level
    const bool wlo = tg == 0, whi = tg == nt - 1;
    // a cell at position 0 has its other in-row neighbour in pair t-1, at
    // position 1 in pair t+1; red of level kk takes side kk & 1, black the
    // other.  Threads without a column read cell 0 and write nothing.
    cent = act ? (row + 1) * W + t + 1 : W + 1;
    side = par ? 1 : -1;
    wl[0] = par ? whi : wlo;  // the side lies beyond a wall
    wl[1] = par ? wlo : whi;
    const bool lastp = ODD && whi && (im & 1);  // the pair with one cell (position 0)
    inv[0] = lastp && par == 1;                 // the cell using that side does not exist
    inv[1] = lastp && par == 0;
    // odd jm: across the periodic boundary the neighbour has the cell's own
    // colour and keeps its previous iterate: rows tj+2 + 2c + side hold it
    wrl = oddj && by == 0 && row == 0;
    wrh = oddj && by == a->nty - 1 && row == tjn - 1;
    rowd = (a->tj + 1 - row) * W;
    // in-plane halo words e = tid + q*nthr, sent after every sweep of either
    // colour: ranges i-lo, i-hi (row, level), j-lo, j-hi (level, pair).  A box
    // sends word e to the next box up (lo) or down (hi) the direction, whose
    // halo its range is, and receives its own word e.  No branch on what a
    // word holds: the boxes form a ring in i too, where the word that crosses
    // the walls goes to the last cell of the plane, as the words of rows,
    // pairs or levels a box does not have; a face of which only the other
    // colour has cells in a row is sent as well, into a halo cell not read then.
    const int kl = a->kl, NI = a->ntx > 1 ? a->tj * kl : 0, NJ = a->tp * kl, IW = a->iw;
#pragma unroll
    for (int q = 0; q < NW; q++) {
      const int e = tid + q * nthr;
      unsigned so = 0, de = PLANE - 1, wrap = 0;
      int to = bid;
      if (e < 2 * NI) {
        const int hi = e >= NI, x = hi ? e - NI : e, r = x / kl, kk = x % kl;
        to = bid - bx + (hi ? bx + a->ntx - 1 : bx + 1) % a->ntx;
        if (r < tjn && kk < nlev) {
          so = kk * PLANE + (r + 1) * W + (hi ? 1 : tpn);
          if (hi ? bx < a->ntx - 1 : bx > 0) de = kk * PLANE + (r + 1) * W + (hi ? tpn + 1 : 0);
        }
      } else if (e < 2 * NI + 2 * NJ) {
        const int f = e - 2 * NI, hi = f >= NJ, x = hi ? f - NJ : f, kk = x / a->tp, p = x % a->tp;
        to = bx + a->ntx * ((hi ? by + a->nty - 1 : by + 1) % a->nty + a->nty * bz);
        if (p < tpn && kk < nlev) {
          so = kk * PLANE + (hi ? 1 : tjn) * W + p + 1;
          wrap = oddj && (hi ? by == a->nty - 1 : by == 0);  // kept by colour
          de = kk * PLANE + (wrap ? a->tj + 2 + hi : hi ? tjn + 1 : 0) * W + p + 1;
        }
      }
      wsd[q] = so | (de << 16);
      wto[q] = (unsigned)(to * IW + e) | (wrap << 31);
    }
  }
  const int nq = a0->nq;                    // halo words per thread
  const unsigned nw0 = (unsigned)(nq * nthr);  // the k words follow the in-plane ones
  const unsigned tag0 = (unsigned)a0->ctrl->res_epoch * 8192u;
  const bool writer = bid == 0 && tid == 0;
  float v[2][BK], rh[2][BK];  // [0] black, [1] red: iterate and rhs by level
  float hlo[2], hhi[2];       // the k neighbours of colour c outside the box
  int limit = a0->nmaxp;
  bool dead = false;
  const float c2 = a0->c2, c3 = a0->c3, omega = a0->omega;
  // per level: cn4l, cn4s, cn1; those of the first group are kept
  const ConstF lv0 = constf(a0->m.lev4 + 4 * k0);
  float cu0[G], cl0[G], cn0[G];
#pragma unroll
  for (int u = 0; u < G; u++) {
    cu0[u] = lv0[4 * u];
    cl0[u] = lv0[4 * u + 1];
    cn0[u] = lv0[4 * u + 2];
  }
  const bool zero0 = a0->zero != 0;

  for (int pass = 0; pass < 2; pass++) {
    const unsigned tag = tag0 + pass * 4096u;
    __syncthreads();
    // ---- the start iterate and its halo (the padded field holds the ghosts
    // p had on entry, which iteration 1 reads)
    {
      const ConstArgs a = again(a0);
      int ce = cent;
      asm volatile("" : "+v"(ce));  // addresses made here, not held over the solve
      const Grid g = {a->g.im, a->g.jm, a->g.km, a->g.sj, a->g.sk};
      const SplitGrid s = {a->s.nt, a->s.cp, a->s.cplane};
      const float* const pent = a->pent;
      const bool zero = a->zero != 0;
      const int t0 = bx * s.nt / a->ntx, tpn = (bx + 1) * s.nt / a->ntx - t0;
      const int j0 = 1 + by * g.jm / a->nty, tjn = (by + 1) * g.jm / a->nty + 1 - j0;
      const int tg = t0 + ce % W - 1, j = j0 + ce / W - 1;
      {
        const bool mean = a->nred > 0;
        const double av = av_s;
        const int rq = rcix(s, tg, j, k0);
        const float* r0 = (mean ? a->rhsr[0] : a->sb.rhs[0]) + rq;
        const float* r1 = (mean ? a->rhsr[1] : a->sb.rhs[1]) + rq;
        float* w0 = a->sb.rhs[0] + rq;
        float* w1 = a->sb.rhs[1] + rq;
        const float* pp = pent + ix(g, 2 * tg + 1, j, k0);  // i = 1 is 256-byte aligned
#pragma unroll
        for (int kk = 0; kk < BK; kk++) {
          v[0][kk] = v[1][kk] = rh[0][kk] = rh[1][kk] = 0.0f;
          if (kk < BK - 4 || kk < nlev) {
            float x0 = *r0, x1 = *r1;
            if (mean) {  // press.f95:81-87, the subtraction in FP64 as in k_rhs_sub
              x0 = (float)((double)x0 - av);
              x1 = (float)((double)x1 - av);
              if (act) {
                *w0 = x0;
                *w1 = x1;
              }
              w0 += s.cplane;
              w1 += s.cplane;
            }
            if (kk < RL)
              RB[kk * NT + tid] = x0;
            else
              rh[0][kk] = x0;
            rh[1][kk] = x1;
            if (!zero) {
              const float2 x = *(const float2*)pp;
              const bool pr = (side > 0) != ((kk & 1) != 0);  // red at position 1
              v[1][kk] = pr ? x.y : x.x;
              v[0][kk] = pr ? x.x : x.y;
            }
            r0 += s.cplane;
            r1 += s.cplane;
            pp += g.sk;
          }
        }
      }
      for (int c = 0; c < 2; c++) hlo[c] = hhi[c] = 0.0f;
      if (!zero) {
        for (int c = 0; c < 2; c++) {  // colour c at level k sits where the other colour does at k -+ 1
          hlo[c] = pent[ix(g, 2 * tg + 1 + ((1 + j + k0 + c) & 1), j, k0 - 1)];
          const int k1 = k0 + nlev - 1;
          hhi[c] = pent[ix(g, 2 * tg + 1 + ((1 + j + k1 + c) & 1), j, k1 + 1)];
        }
      }
      // the black cells and the in-plane halo the first red sweep reads
      if (act) {
#pragma unroll
        for (int kk = 0; kk < BK; kk++)
          if (kk < BK - 4 || kk < nlev) S[kk * PLANE + ce] = v[0][kk];
      }
      for (int x = tid; x < (tpn + tjn) * 2 * nlev; x += nthr) {
        const int kk = x / (2 * (tpn + tjn)), y = x % (2 * (tpn + tjn)), k = k0 + kk;
        if (y < 2 * tpn) {
          const int hi = y >= tpn, p = hi ? y - tpn : y, tt = t0 + p;
          const int je = hi ? j0 + tjn - 1 : j0, jn = hi ? je + 1 : je - 1;  // edge row and the row beyond
          const int i = 2 * tt + 1 + ((1 + je + k + 1) & 1);                 // red of the edge row
          const float x0 = zero ? 0.0f : pent[ix(g, i, jn, k)];
          if (oddj && (hi ? je == g.jm : je == 1)) {
            S[kk * PLANE + (a->tj + 4 + hi) * W + p + 1] = x0;  // red
            const int ib = 2 * tt + 1 + ((1 + je + k) & 1);     // black of the edge row: the wrapped row itself
            S[kk * PLANE + (a->tj + 2 + hi) * W + p + 1] =
                (zero || ib > g.im) ? 0.0f : pent[ix(g, ib, hi ? 1 : g.jm, k)];
          } else {
            S[kk * PLANE + (hi ? tjn + 1 : 0) * W + p + 1] = x0;
          }
        } else {
          const int z = y - 2 * tpn, hi = z >= tjn, r = hi ? z - tjn : z;
          const int i = hi ? 2 * (t0 + tpn) + 1 : 2 * t0;
          S[kk * PLANE + (r + 1) * W + (hi ? tpn + 1 : 0)] = zero ? 0.0f : pent[ix(g, i, j0 + r, k)];
        }
      }
    }
    __syncthreads();

    int stop_at = 0;
    for (int l = 1; l <= limit; l++) {
      double acc = 0.0;
#pragma unroll
      for (int cc = 1; cc >= 0; cc--) {
        const int c = cc;  // 1 red, 0 black
        const unsigned wt = tag + 2 * l + c;
        const bool later = l > 1 || zero0;  // walls mirror (a zero start has zero ghosts either way)
        // ---- the colour sweep
        {
          float below_v = hlo[c];
          if (kbot && later) below_v = v[c][0];
          const bool mir = later || c == 0;
          const bool wall0 = wl[c ^ 1] && mir, wall1 = wl[c] && mir;
          const bool own_top = ktop && later;
          // the LDS address of every access is an immediate offset from these
          // four (as loop invariants the compiler would hold one per access)
          asm volatile("" : "+v"(cent));
          const int al[2] = {cent + side, cent - side};
          int au = cent - W, ad = cent + W;
          if (oddj) {
            const int xr = cent + rowd + 2 * c * W;
            au = wrl ? xr : au;
            ad = wrh ? xr + W : ad;
          }
          int tr = tid;
          asm volatile("" : "+v"(tr));
          ConstF lv = lv0;
          asm volatile("" : "+s"(lv));
          // groups of G levels; a group's operands are fetched while the one
          // before is computed
          float lat[2][G], pjm[2][G], pjp[2][G], rb[2][G], cu[2][G], cl[2][G], cn[2][G];
          auto fetch = [&](auto gi) {
            constexpr int g0 = decltype(gi)::value, b = g0 & 1;
#pragma unroll
            for (int u = 0; u < G; u++) {
              const int kk = g0 * G + u;
              if (kk < BK) {
                const float* P = S + kk * PLANE;
                lat[b][u] = P[al[(kk & 1) ^ (c ^ 1)]];
                pjm[b][u] = P[au];
                pjp[b][u] = P[ad];
                rb[b][u] = (c == 0 && kk < RL) ? RB[kk * NT + tr] : rh[c][kk];
                cu[b][u] = g0 == 0 ? cu0[u] : lv[4 * kk];
                cl[b][u] = g0 == 0 ? cl0[u] : lv[4 * kk + 1];
                cn[b][u] = g0 == 0 ? cn0[u] : lv[4 * kk + 2];
              }
            }
          };
          auto ready = [&](auto gi) {  // wait for the group here, before the next one's loads are issued
            constexpr int g0 = decltype(gi)::value, b = g0 & 1;
#pragma unroll
            for (int u = 0; u < G; u++)
              if (g0 * G + u < BK) {
                const float x0 = lat[b][u], x1 = pjm[b][u], x2 = pjp[b][u], x3 = rb[b][u], y0 = cu[b][u], y1 = cl[b][u], y2 = cn[b][u];
                asm volatile("" ::"v"(x0), "v"(x1), "v"(x2), "v"(x3), "s"(y0), "s"(y1), "s"(y2));
              }
          };
          auto compute = [&](auto gi) {
            constexpr int g0 = decltype(gi)::value, b = g0 & 1;
#pragma unroll
            for (int u = 0; u < G; u++) {
              const int kk = g0 * G + u;
              if (kk < BK && (kk < BK - 4 || kk < nlev)) {
                const int ai = (kk & 1) ^ (c ^ 1);
                const float own = v[c][kk];
                float oth = v[c ^ 1][kk];
                const float la = ((kk & 1) ? wall1 : wall0) ? own : lat[b][u];
                if (ODD) oth = (inv[ai ^ 1] && mir) ? own : oth;  // the pair's other cell is the ghost at im+1
                const float pkm = kk == 0 ? below_v : v[c ^ 1][kk > 0 ? kk - 1 : 0];
                float pkp = v[c ^ 1][kk < BK - 1 ? kk + 1 : kk];
                if (kk >= BK - 5) {
                  if (kk == nlev - 1) pkp = own_top ? own : hhi[c];
                }
                const float x = c2 * la + c2 * oth + c3 * pjp[b][u] + c3 * pjm[b][u] + cu[b][u] * pkp +
                                cl[b][u] * pkm - rb[b][u];
                float rel = cn[b][u] * x - own;
                if (!OM1) rel = omega * rel;
                if (ODD) rel = inv[ai] ? 0.0f : rel;
                acc = __builtin_fma((double)rel, (double)rel, acc);
                v[c][kk] = own + rel;
              }
            }
          };
          auto run = [&](auto self, auto gi) {
            constexpr int g0 = decltype(gi)::value;
            if constexpr (g0 < NG) {
              ready(gi);
              if constexpr (g0 + 1 < NG) fetch(std::integral_constant<int, g0 + 1>{});
              __builtin_amdgcn_sched_barrier(0);
              compute(gi);
              __builtin_amdgcn_sched_barrier(0);
              self(self, std::integral_constant<int, g0 + 1>{});
            }
          };
          fetch(std::integral_constant<int, 0>{});
          run(run, std::integral_constant<int, 0>{});
        }
        const ConstArgs a = again(a0);
        u64* const inb = a->slots + (c ? (unsigned)nb * (unsigned)a->iw : 0u);  // red inboxes after the black ones
        // (nothing derived from these is to be held over the loop)
        unsigned tx = tid;
        int nl = nlev, nqo = nq;
        asm volatile("" : "+v"(tx), "+s"(nl), "+s"(nqo));
#pragma unroll
        for (int q = 0; q < NW; q++) asm volatile("" : "+v"(wsd[q]), "+v"(wto[q]));
        // the k faces: my first level is the box below's k-hi, my last the
        // box above's k-lo (the same columns, so the same threads, without
        // one the same too)
        if (!kbot) ast(inb + (unsigned)((bid - a->ntx * a->nty) * a->iw) + nw0 + NT + tx, word(wt, v[c][0]));
        if (!ktop) {
          float vtop = v[c][BK - 1];
#pragma unroll
          for (int kk = BK > 5 ? BK - 5 : 0; kk < BK - 1; kk++) vtop = kk == nl - 1 ? v[c][kk] : vtop;
          ast(inb + (unsigned)((bid + a->ntx * a->nty) * a->iw) + nw0 + tx, word(wt, vtop));
        }
        __syncthreads();  // every read of the other colour's copy is done
        if (act) {
#pragma unroll
          for (int kk = 0; kk < BK; kk++) S[kk * PLANE + cent] = v[c][kk];  // levels from nlev on are not read
        }
        __syncthreads();  // the copy holds colour c
        // ---- send the in-plane faces
        const int cw = 2 * c * W;
        if (nb == 1) {  // a box that is its own neighbour
#pragma unroll
          for (int q = 0; q < NW; q++)
            if (q < nqo) S[(wsd[q] >> 16) + ((wto[q] >> 31) ? cw : 0)] = S[wsd[q] & 0xffffu];
        } else {
          float x[NW];
#pragma unroll
          for (int q = 0; q < NW; q++)
            if (q < nqo) x[q] = S[wsd[q] & 0xffffu];
#pragma unroll
          for (int q = 0; q < NW; q++)
            if (q < nqo) ast(inb + (wto[q] & 0x7fffffffu), word(wt, x[q]));
        }
        if (c == 0 && pass == 0) {  // the iteration's sum of reltmp^2, wave by wave (while the words cross)
          const double x = wave_sum_last(act ? acc : 0.0);
          if (tid % kWave == kWave - 1) {
            const u64 bits = (u64)__double_as_longlong(x), wq = (u64)wt << 32;
            u64* const pw = a->parts + ((size_t)(l & 3) * (nb * nwav) + (bid * nwav + tid / kWave)) * 2;
            ast(pw, wq | (bits >> 32));
            ast(pw + 1, wq | (bits & 0xffffffffull));
          }
        }
        // ---- receive the halo, and the verdict on iteration l-2, published
        // during l-1 (asked for first: a look of its own takes as long as the
        // exchange, 677 us instead of 657 per solve at 300x300x90)
        const bool ask = c == 0 && pass == 0 && l > 2 && tid == 0;
        u64 said = 0;
        if (ask) said = ald(a->parts + 8 * (size_t)(nb * nwav) + ((l - 2) & 3));
        if (nb > 1) {
          const u64* const me = inb + (unsigned)(bid * a->iw);
          u64 w[NW], wk[2] = {0, 0};
          for (int spin = 0;; spin++) {
            unsigned miss = 0;
            if (!kbot) wk[0] = ald(me + nw0 + tx);
            if (!ktop) wk[1] = ald(me + nw0 + NT + tx);
#pragma unroll
            for (int q = 0; q < NW; q++)
              if (q < nqo) w[q] = ald(me + tx + q * nthr);
            if (!kbot) miss |= wtag(wk[0]) ^ wt;
            if (!ktop) miss |= wtag(wk[1]) ^ wt;
#pragma unroll
            for (int q = 0; q < NW; q++)
              if (q < nqo) miss |= wtag(w[q]) ^ wt;
            if (miss == 0) break;
            if (spin > kSpinMax) {  // cannot happen while every block runs
              sh[1] = 1;
              break;
            }
          }
          if (!kbot) hlo[c ^ 1] = wval(wk[0]);
          if (!ktop) hhi[c ^ 1] = wval(wk[1]);
#pragma unroll
          for (int q = 0; q < NW; q++)
            if (q < nqo) S[(wsd[q] >> 16) + ((wto[q] >> 31) ? cw : 0)] = wval(w[q]);
        }
        if (ask) {
          const unsigned pt = tag + 2 * (l - 2);
          sh[2] = wtag(said) == pt ? (int)(said & 1u) : res_verdict(a, nb * nwav, l - 2, pt, &sh[1]);
        }
        __syncthreads();  // the halo is in place
        if (sh[1]) {
          dead = true;
          break;
        }
      }
      if (dead) break;
      if (pass == 0 && l > 2 && sh[2]) {
        stop_at = l - 2;
        break;
      }
    }
    if (dead) {
      if (tid == 0) a0->ctrl->nonfinite = 1;
      break;
    }
    if (pass == 1) break;
    if (stop_at == 0) {  // the verdicts not yet seen
      __syncthreads();
      if (tid == 0) {
        const ConstArgs a = again(a0);
        int at = 0;
        for (int l = max(1, limit - 1); l <= limit && at == 0; l++)
          if (res_verdict(a, nb * nwav, l, tag + 2 * l, &sh[1])) at = l;
        sh[2] = at;
      }
      __syncthreads();
      stop_at = sh[2];
      if (stop_at == 0 || stop_at == limit) break;  // the registers hold iterate `limit`
    }
    // the loop ran past the iteration that stopped it: run again from the
    // start, which the solve has not changed, to exactly that one
    limit = stop_at;
  }
  {
    const ConstArgs a = again(a0);
    const int t0 = bx * a->s.nt / a->ntx, j0 = 1 + by * a->g.jm / a->nty;
    const int q0 = rcix({a->s.nt, a->s.cp, a->s.cplane}, t0 + cent % W - 1, j0 + cent / W - 1, k0), cpl = a->s.cplane;
    float* const b = a->sb.p[1][0] + q0;
    float* const r = a->sb.p[1][1] + q0;
    if (act) {
#pragma unroll
      for (int kk = 0; kk < BK; kk++)
        if (kk < BK - 4 || kk < nlev) {
          b[kk * cpl] = v[0][kk];
          r[kk * cpl] = v[1][kk];
        }
    }
    if (writer) {
      a->ctrl->p_final = 1;
      if (a->nred > 0) a->ctrl->rhsav = av_s;
    }
  }
}

// One solve, of the arguments a, or (nd > 0) those of a batch: domain e's
// arguments are tab[e] and its blocks start at b0[e].  The domains of a batch
// share the device side by side, each with boxes of its own and a handshake of
// its own: 9 domains of 96..160 x 96..160 x 64 solve 50
// iterations in 880 us (two launches; 1165 in one, with boxes of 22 levels), one
// iteration of all of them per launch took 2090.
template <int CLS, int BK, bool OM1, bool ODD>
__global__ __launch_bounds__(kResNT, 2 * kResClass[CLS].per) void k_sor_res(ResArgs a,
                                                                             const ResArgs* __restrict__ tab,
                                                                             const int* __restrict__ b0, int nd) {
  (void)a;  // the kernel argument segment starts with it
  ConstArgs at = (ConstArgs)__builtin_amdgcn_kernarg_segment_ptr();
  int bid = (int)blockIdx.x;
  if (nd > 0) {
    int e = 0;
    for (int r = 1; r < nd; r++)
      if ((int)blockIdx.x >= b0[r]) e = r;
    at = (ConstArgs)(unsigned long long)(tab + e);
    bid -= b0[e];
  }
  res_block<CLS, BK, OM1, ODD>(at, bid);
}

}  // namespace

// Microseconds of one sweep of a cut, as a model: the sweep of a unit's boxes
// (80 cycles per level and wave of a SIMD, no less than the latency of a wave
// alone), the exchange (latency, and words per unit), and what a box of two
// hides of it.  on: boxes on the fullest unit.  The tallest boxes of each class
// spill registers: a sweep of 18 levels in class 1 takes 6.8 us at 300x300x90
// where the rest of the model gives 5.4, one of 22 levels 9.7 for 6.0.  The last
// terms are fits: 48x40x24 takes 171 us per solve with 180 boxes of class 1, 206
// with 504 and 200 with 252 of class 0, 24x20x16 170 with 16 boxes, 200 with one.
static double res_cost(const ResShape& h, int words, int on) {
  const int waves = h.nthr / kWave, kl = h.kl, over = kl - (h.cls == 0 ? 32 : 16);
  const double slow = over <= 0 ? 1.0 : over <= 2 ? 1.25 : over <= 4 ? 1.4 : over <= 6 ? 1.65 : 2.0;
  const double sweep = std::max(0.034 * ((on * waves + 3) / 4), 0.055) * kl + 0.3 + 0.05 * waves * on;
  const double cross = 1.5 + 0.35 * on * words / 1024;
  if (h.nb == 1) return sweep + 0.6;
  if (on == 1) return slow * (sweep + cross) - (h.cls == 1 ? 0.35 : 0.0);
  return slow * std::max(sweep, 0.6 * sweep + cross);
}

static int up(int a, int b) { return (a + b - 1) / b; }
static int res_face_words(const ResShape& h) { return 2 * (h.ntx > 1 ? h.tj * h.kl : 0) + 2 * h.tp * h.kl; }
// The threads a launch has: whole waves.
static void res_threads(ResShape* h, int nthr) {
  h->nthr = nthr;
  h->nq = up(res_face_words(*h), nthr);
  h->iw = h->nq * nthr + 2 * kResNT;
}

// Calls f(shape, halo words) for every cut of a domain into at most nmax boxes
// of class cls with klo < levels <= khi.
template <class F>
static void res_cuts(const Grid& g, const SplitGrid& s, int cls, int nmax, int klo, int khi, F f) {
  const ResClass C = kResClass[cls];
  for (int ntz = std::max(1, up(g.km, khi)); ntz <= std::min(g.km, nmax); ntz++) {
    const int kl = up(g.km, ntz);
    if (kl <= klo) break;
    if (kl > khi || (ntz > 1 && kl == up(g.km, ntz - 1))) continue;
    for (int ntx = 1; ntx <= s.nt && ntx * ntz <= nmax; ntx++) {
      const int tp = up(s.nt, ntx);
      if (tp > kResNT || (ntx > 1 && tp == up(s.nt, ntx - 1))) continue;
      for (int nty = std::max(1, up(g.jm, kResNT / tp)); nty <= g.jm && ntx * nty * ntz <= nmax; nty++) {
        const int tj = up(g.jm, nty);
        if (tp * tj > kResNT || (nty > 1 && tj == up(g.jm, nty - 1))) continue;
        if ((tp + 2) * (tj + 2 + ((g.jm & 1) ? 4 : 0)) >= C.plane) continue;
        ResShape h{ntx, nty, ntz, tp, tj, kl, ntx * nty * ntz, 0, 0, cls, 0};
        // enough waves for the columns and for the halo words
        const int wds = res_face_words(h);
        const int nthr = up(std::max(tp * tj, up(wds, C.words)), kWave) * kWave;
        if (nthr > kResNT) continue;
        res_threads(&h, nthr);
        f(h, wds + (ntz > 1 ? 2 * nthr : 0));
      }
    }
  }
}

// The cut of a domain into boxes with the least modelled time.  False when
// no cut fits (about 12 million cells on 256 units).
bool res_shape(const Grid& g, const SplitGrid& s, int units, ResShape* out) {
  double best = -1.0;
  for (int cls = 0; cls < 2; cls++)  // one block runs the monitor
    res_cuts(g, s, cls, kResClass[cls].per * units - 1, 0, kResClass[cls].levels, [&](const ResShape& h, int wds) {
      const double c = res_cost(h, wds, h.nb > units ? 2 : 1);
      if (best < 0.0 || c < best) {
        best = c;
        *out = h;
      }
    });
  return best >= 0.0;
}

// One launch for the domains ds (indices into all): the kernel (class and
// levels) and one cut of each, such that all boxes run at once, with the least
// modelled time of the slowest domain.  From its fewest boxes each domain takes
// more while it is the slowest and they fit.  Returns the time, negative when
// no kernel holds them all.
struct Cut {
  ResShape h;
  double cost;
};
// A domain's cuts by class and levels / 4, made when first asked for.
struct Cuts {
  std::vector<Cut> v[2][16];
  bool have[2][16] = {};
};
static double res_batch_cut(const DevDomain* const* all, const std::vector<int>& ds, int units, ResShape* shapes,
                            std::vector<Cuts>& memo) {
  double best = -1.0;
  for (int cls = 0; cls < 2; cls++) {
    const int cap = kResClass[cls].per * units;
    for (int bk = 4; bk <= kResClass[cls].levels; bk += 4) {
      std::vector<std::vector<Cut>> cuts(ds.size());  // of rising boxes and falling time
      long total = 0;
      bool ok = true;
      for (size_t q = 0; q < ds.size() && ok; q++) {
        const DevDomain& d = *all[ds[q]];
        Cuts& mm = memo[ds[q]];
        if (mm.have[cls][bk / 4]) {
          cuts[q] = mm.v[cls][bk / 4];
          ok = !cuts[q].empty();
          if (ok) total += cuts[q][0].h.nb + 1;
          continue;
        }
        std::vector<Cut> v;
        res_cuts(d.g, d.sg, cls, cap - 1, bk - 4, bk, [&](const ResShape& h, int wds) {
          v.push_back({h, res_cost(h, wds, cls == 1 ? 2 : 1)});
        });
        std::stable_sort(v.begin(), v.end(), [](const Cut& a, const Cut& b) { return a.h.nb < b.h.nb; });
        for (const Cut& c : v) {
          auto& w = cuts[q];
          if (!w.empty() && c.cost >= w.back().cost) continue;
          if (!w.empty() && c.h.nb == w.back().h.nb)
            w.back() = c;
          else
            w.push_back(c);
        }
        mm.v[cls][bk / 4] = cuts[q];
        mm.have[cls][bk / 4] = true;
        ok = !cuts[q].empty();
        if (ok) total += cuts[q][0].h.nb + 1;
      }
      if (!ok || total > cap) continue;
      std::vector<size_t> at(ds.size(), 0);
      double slow;
      for (;;) {
        size_t m = 0;
        for (size_t q = 1; q < ds.size(); q++)
          if (cuts[q][at[q]].cost > cuts[m][at[m]].cost) m = q;
        slow = cuts[m][at[m]].cost;
        if (at[m] + 1 == cuts[m].size()) break;
        const long more = cuts[m][at[m] + 1].h.nb - cuts[m][at[m]].h.nb;
        if (total + more > cap) break;
        total += more;
        at[m]++;
      }
      if (best >= 0.0 && slow >= best) continue;
      best = slow;
      int nthr = 0;
      for (size_t q = 0; q < ds.size(); q++) nthr = std::max(nthr, cuts[q][at[q]].h.nthr);
      for (size_t q = 0; q < ds.size(); q++) {
        shapes[ds[q]] = cuts[q][at[q]].h;
        res_threads(&shapes[ds[q]], nthr);
      }
    }
  }
  return best;
}

double res_batch_plan(const DevDomain* const* ds, int n, int units, ResShape* shapes, std::vector<int>* group) {
  std::vector<int> by(n);  // largest first
  for (int q = 0; q < n; q++) by[q] = q;
  const auto cells = [&](int q) { return (long)ds[q]->g.im * ds[q]->g.jm * ds[q]->g.km; };
  std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return cells(a) > cells(b); });
  // as few launches as hold them, or more while that is faster
  double best = -1.0;
  std::vector<ResShape> sh(n);
  std::vector<Cuts> memo(n);
  for (int ng = 1; ng <= n; ng++) {
    std::vector<std::vector<int>> in(ng);  // dealt out there and back
    for (int r = 0; r < n; r++) in[(r / ng) & 1 ? ng - 1 - r % ng : r % ng].push_back(by[r]);
    double sum = 0.0;
    for (const auto& v : in) {
      const double c = res_batch_cut(ds, v, units, sh.data(), memo);
      if (c < 0.0) {
        sum = -1.0;
        break;
      }
      sum += c;
    }
    if (sum < 0.0) continue;
    if (best >= 0.0 && sum >= best) break;
    best = sum;
    std::copy(sh.begin(), sh.end(), shapes);
    group->assign(n, 0);
    for (int q = 0; q < ng; q++)
      for (int r : in[q]) (*group)[r] = q;
  }
  return best;
}

// 8-byte words of the workspace: inboxes of both colours, the partial sums
// of four iterations (two words each) and their verdicts, and the partial sums of the ticket
// sweeps.
long res_words(const ResShape& h) {
  return 2L * h.nb * h.iw + 8L * h.nb * (h.nthr / kWave) + 8 + 4 * kTickets;
}

ResArgs res_args(const DevDomain& d, const ResShape& h, unsigned long long* mem, const SplitBufs& sb, int nmaxp,
                 float pjuge, float omega, bool zero) {
  ResArgs a{};
  a.g = d.g;
  a.s = d.sg;
  a.m = d.m;
  a.sb = sb;
  a.ctrl = d.ctrl;
  a.pent = d.F.p;
  a.slots = mem;
  a.parts = mem + 2L * h.nb * h.iw;
  a.tparts = (double*)(a.parts + 8L * h.nb * (h.nthr / kWave) + 8);
  a.c2 = d.res_c2;
  a.c3 = d.res_c3;
  a.omega = omega;
  a.pjuge = pjuge;
  a.nmaxp = nmaxp;
  a.zero = zero;
  a.force_ticket = d.res_on == 2;
  a.missing = d.res_on == 3 || (d.res_on == 4 && __atomic_load_n(d.res_note, __ATOMIC_RELAXED) == 0);
  a.note = d.res_note;
  a.ntx = h.ntx;
  a.nty = h.nty;
  a.ntz = h.ntz;
  a.tp = h.tp;
  a.tj = h.tj;
  a.kl = h.kl;
  a.nb = h.nb;
  a.iw = h.iw;
  a.nq = h.nq;
  return a;
}

struct ResGrid {
  int blocks, nthr, kl;
  hipStream_t stream;
  const ResArgs* tab;
  const int* b0;
  int nd;
};

template <int CLS, bool OM1, bool ODD>
static void launch_res(const ResGrid& r, const ResArgs& a) {
#define RES(BK)                                                                                                   \
  if (r.kl <= BK) {                                                                                               \
    hipLaunchKernelGGL((k_sor_res<CLS, BK, OM1, ODD>), dim3(r.blocks), dim3(r.nthr), 0, r.stream, a, r.tab, r.b0, \
                       r.nd);                                                                                     \
    return;                                                                                                       \
  }
  RES(4)
  RES(8)
  RES(12)
  RES(16)
  // (every two levels where registers spill: 300x300x90, boxes of 18 levels,
  // took 680 us per solve, in the kernel for 20 levels 760)
  if constexpr (CLS == 1) RES(18)
  RES(20)
  if constexpr (CLS == 1) RES(22)
  RES(24)
  if constexpr (CLS == 0) {
    RES(28)
    RES(32)
    RES(36)
    RES(40)
  }
#undef RES
}

static void launch_res(const ResGrid& r, const ResArgs& a, int cls, bool om1, bool odd) {
  if (cls == 0) {
    if (!om1)
      launch_res<0, false, true>(r, a);
    else if (odd)
      launch_res<0, true, true>(r, a);
    else
      launch_res<0, true, false>(r, a);
  } else {
    if (!om1)
      launch_res<1, false, true>(r, a);
    else if (odd)
      launch_res<1, true, true>(r, a);
    else
      launch_res<1, true, false>(r, a);
  }
}

void launch_sor_res(const DevDomain& d, const SplitBufs& sb, int nmaxp, float pjuge, float omega, bool zero,
                    int nred) {
  const ResShape& h = d.res;
  ResArgs a = res_args(d, h, d.res_mem, sb, nmaxp, pjuge, omega, zero);
  a.rhsr[0] = sb.rhsr[0];
  a.rhsr[1] = sb.rhsr[1];
  a.rpart = d.partials;
  a.nred = nred;
  a.area = d.area;
  const ResGrid r{h.nb + 1, h.nthr, h.kl, d.stream, nullptr, nullptr, 0};
  TIMED(d, KC_SOR, launch_res(r, a, h.cls, omega == 1.0f, (d.g.im & 1) != 0));
}

void launch_sor_res_batch(const ResBatch& b, hipStream_t stream) {
  const ResGrid r{b.blocks, b.nthr, b.kl, stream, b.tab, b.b0, b.nd};
  launch_res(r, ResArgs{}, b.cls, b.om1, b.odd);
}

}  // namespace les
