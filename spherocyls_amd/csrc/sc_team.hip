// Many steps in one launch: teams of workgroups.
//
// A step of a packing of a few hundred to a few ten thousand particles is two
// small kernels whose time is launch gaps and chains of dependent loads, not
// bandwidth or arithmetic (N = 16384: force pass 9.5 us and update 13.8 us per
// FIRE iteration for 0.6 us of memory traffic).  Here the workgroups of a
// packing (its team) stay resident and run the steps themselves.  Each member
// owns a run of consecutive particles of the cell-sorted bank and keeps their
// state in registers and LDS; the particles around them (its halo) are copied
// into LDS once per force pass, so the pair loop reads LDS only.
//
// Exchange between members.  Every XCD has its own L2, so members exchange
// through 8-byte words written and read with relaxed agent-scope atomics
// (write-through stores, loads that bypass the caches); no fence, which would
// write back and invalidate a whole L2, is needed:
//   * positions: a record of 4 words per particle in one of four buffers.  A
//     word no position can have (kEmpty, a NaN with a payload no operation
//     yields) marks a word not written yet, so a reader polls the data
//     itself: one trip instead of flag-then-data.  A member waits for its
//     halo only, not for the whole team;
//   * sums (minimisers): four words per member and update wavefront in one of
//     three slots, empty-marked like the positions; every member adds up all
//     sums in the same order and takes the same decision;
//   * flags (Heun): one word per member and pass, (sequence number << 8 |
//     bits), in four slots; a reader waits for the pass's number.
// Rebuilds.  Rows hold while no particle has moved half the skin from its
// position at the last rebuild.  Minimisers evaluate a pass on the old rows
// and a member that has moved too far says so in place of its sums: the team
// then rebuilds from the same positions and repeats the pass, so the common
// pass has no exchange for it.  Heun steps have no team-wide exchange to
// carry that: a member asks at 0.6 of the limit, all read the flags one pass
// late, when they have long arrived, and a particle that reached the limit
// before the rebuild makes the launch end at the start of the step whose forces
// it missed, which every member still holds (the host goes on from there with
// the launches per step).
// Buffer reuse.  Positions of a pass are marked empty once every member is
// known to have read them: in a minimiser when all sums of the pass are in, in
// Heun two passes later, when all flags of the pass in between are in.  The
// marks are waited for before the member's next sums or flags go out, which
// everyone who will poll the buffer's next positions reads first.  Sum slots
// follow the same rule with the sums themselves.
//
// Every wait is bounded.  The first pass's rebuild doubles as the roll call: a
// member that is not resident within a.roll_call (another process's kernels
// hold the CUs) makes the others leave without having written anything, and the
// host goes on with the launches per step, for some time without another try.
// The host launches at most as many members of teams of several as are resident
// at once.  A packing that is a single member waits for nobody: any number of
// them go in one launch, behind the others.
//
// Measured, all-gather of 4 words by G workgroups over all XCDs: 1.05 us (G = 2),
// 1.5 (16), 1.8 (64), 2.0 (128), 2.8 (256); an empty kernel in a captured graph
// takes 1.65 us.  Against the launches per step, wall time of a long
// call over its steps: two-point FIRE from a random start to convergence, 16384
// particles 24.1 -> 12.4 us an iteration, 700 22.9 -> 9.7, 128 20.9 -> 8.2; sheared
// steps of a relaxed packing of 16384 23.5 -> 10.6 us, of 512 and 700 21.3 -> 10.1;
// descent of 1000 20.9 -> 8.0.
// Where a FIRE iteration of 16384 goes in a compression step, which rebuilds less
// often (10.9 us, 26k cycles): gathering the sums 7.6k, pair math 3.0k, rebuilds
// 3.2k (22 in 381 passes; 4.4k when every member looked at every particle), new
// positions 1.9k, halo 1.7k, row tests 1.3k, sums 0.9k, decision 0.7k (1.8k by one
// thread on the whole record of scalars).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "sc_internal.h"
#include "sc_physics.h"

namespace sc {

namespace {

typedef unsigned long long u64;
constexpr u64 kEmpty = 0x7ff8deadbeef0001ull;
// In place of a sum: the rows no longer hold; a coordinate is not finite.
constexpr u64 kNeedMark = 0x7ff8deadbeef0002ull, kStopMark = 0x7ff8deadbeef0003ull;
constexpr int kBufs = 4;  // position buffers
constexpr int kWaves = kTeamThreads / 64;
constexpr int kRowStride = kTeamRow + 2;  // odd word stride: rows start in different banks

__device__ __forceinline__ u64 word_load(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void word_store(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 bits_of(double v) { return (u64)__double_as_longlong(v); }
__device__ __forceinline__ double from_bits(u64 v) { return __longlong_as_double((long long)v); }

// All of this wavefront's stores have reached the coherence point.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The value, opaque to the optimiser: addresses formed from it are computed
// where they are used instead of being hoisted out of the step loop, where the
// two dozen arrays' addresses would fill the registers the pair math needs.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A wait that ends: over() is true once `limit` ticks (100 MHz) have passed
// since its first call (at once for a limit of 0), or, after 0.1 ms, when a
// member of the team has reported that it gave up.  One serves all words of a
// stage, so a stage ends at its limit however many words are missing.  (The
// clock is not read while words arrive at the first look.)
struct Wait {
  u64 t0 = 0;
  __device__ __forceinline__ bool over(u64 limit, const int* status) {
    const u64 t = wall_clock64();
    if (t0 == 0) {
      t0 = t;
      return limit == 0;
    }
    return t - t0 > limit ||
           (t - t0 > 10000 &&
            (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
             (kTeamAbsent | kTeamStalled)));
  }
};

// LDS of a member of up to OWN particles, OWN + halo <= CAP.  Compile-time sizes
// put every array at a constant offset, so an access is one index register and
// an immediate.  The cell marks of a rebuild follow (dynamic, by the packing's
// grid).
template <int OWN, int CAP>
struct TeamLds {
  double x[CAP], y[CAP], nx[CAP], ny[CAP], R[CAP], A[CAP];  // own particles, then the halo
  double fx[OWN], fy[OWN], tq[OWN];                         // own particles: forces
  double phi[OWN], vx[OWN], vy[OWN], vp[OWN];  // ... angle; FIRE velocity, Heun predictor velocity
  double xb[OWN], yb[OWN];                     // ... position at the last rebuild
  double m[OWN];                               // ... FIRE 1 / sqrt(I), GD and Heun I
  double ox[OWN], oy[OWN], op[OWN], rc[OWN];   // ... Heun: state the step starts from, RC
  int id[CAP];
  int halo[CAP];                               // storage index of halo entry e
  union {
    unsigned short row[OWN * kRowStride];      // partners (local indices)
    struct {                                   // rebuild, by runs of 64 particles
      u64 hit[8 * OWN];                        // particles in the halo
      int run[8 * OWN], at[8 * OWN];           // runs looked at; their first halo entry
    } scan;
  };
  unsigned cells[4];                           // rebuild: marked cells (dynamic)
};

}  // namespace

// Bytes of dynamic LDS of a launch of shape `shape` over grids of up to
// cell_words * 32 cells.
size_t team_lds_bytes(int shape, int cell_words) {
  const size_t fixed = shape == 0   ? sizeof(TeamLds<kTeamOwn[0], kTeamCap[0]>)
                       : shape == 1 ? sizeof(TeamLds<kTeamOwn[1], kTeamCap[1]>)
                                    : sizeof(TeamLds<kTeamOwn[2], kTeamCap[2]>);
  return fixed + (size_t)cell_words * sizeof(unsigned);
}

// Empty marks for every word a launch polls, zero flags.  (A launch of single
// members polls none, and needs none of it.)
__global__ void k_team_clear(TeamArgs a) {
  const size_t np = (size_t)kBufs * a.ntot * 4, ns = (size_t)3 * a.nseats * 4 * kTeamUpdWaves,
               nf = (size_t)kTeamFlagSlots * a.nseats, nc = (size_t)a.nseats * 4 * kTeamUpdWaves;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < np + ns + nf + nc;
       i += stride) {
    if (i < np) a.pos[i] = kEmpty;
    else if (i < np + ns) a.sums[i - np] = kEmpty;
    else if (i < np + ns + nf) a.flags[i - np - ns] = 0;
    else a.chunks[i - np - ns - nf] = 0;
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.nseats; i += (int)stride) a.status[i] = 0;
}

// Stress and energy records of a launch (one packing): a workgroup adds up a
// record's partial sums and normalises them as k_reduce does.  kRecordRuns runs
// of members are added in member order and then the runs, so a thread waits for
// a 28th of the members' loads (9 records of 256 members: 45 us by nine threads
// alone, now 5.8).
constexpr int kRecordRuns = 28;
// pack_sum keeps the last record of a state that the launch has left behind (of
// the state it ended at the host goes on to record, or to take again).
__global__ void __launch_bounds__(256)
    k_team_records(TeamArgs a, int team, double* out, double* pack_sum) {
  __shared__ double s_run[kRecordRuns * kNSe];
  const int r = blockIdx.x, t = threadIdx.x;
  const int run = t / kNSe, i = t - run * kNSe, per = (team + kRecordRuns - 1) / kRecordRuns;
  if (run < kRecordRuns) {
    double v = 0.0;
    for (int m = run * per; m < min(team, (run + 1) * per); ++m)
      v += a.se_part[((size_t)r * team + m) * kNSe + i];
    s_run[t] = v;
  }
  __syncthreads();
  if (t >= kNSe) return;
  const PackInfo& P = a.packs[0];
  const PackScal& S = a.scal[0];
  double v = 0.0;
  for (int k = 0; k < kRecordRuns; ++k) v += s_run[k * kNSe + t];
  if (t == kSeE) v *= P.inv_2n;
  else if (t != kSeNc) v /= S.Lx * S.Ly;
  out[(size_t)r * kNSe + t] = v;
  const int at = ((a.step0 + a.se_every - a.se_first) / a.se_every + r) * a.se_every;
  if (at < S.step && at + a.se_every >= S.step) pack_sum[t] = v;
}

// MODE kTeamFire / kTeamGd: minimiser iterations (force pass, sums and
// decision, update) until the packing has finished or a.max_steps have run.
// MODE kTeamHeun / kTeamHeunSe: a.max_steps sheared Heun steps (predictor and
// corrector passes); kTeamHeunSe also records stress and energy, FP64 only.
// The formulas, the rows' selection rule and the FIRE state machine are those
// of k_list and k_update; sums run in another order.
template <int MODE, bool TWO_POINT, bool MIXED, int SHAPE>
__global__ void __launch_bounds__(kTeamThreads) __attribute__((amdgpu_waves_per_eu(4)))
k_team(TeamArgs a) {
#pragma clang fp contract(off)
  constexpr bool kHeun = MODE == kTeamHeun || MODE == kTeamHeunSe;
  constexpr bool kFire = MODE == kTeamFire, kGd = MODE == kTeamGd;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ double s_part[kWaves * kNSe];
  __shared__ int s_count[kWaves];
  // Raised and read in phases separated by barriers, so that all threads leave
  // a loop together: s_need (own particles ask for a rebuild), s_bits (flags
  // gathered from the team), s_fail (a wait ran out), s_over (halo or row
  // overflow), s_next (what the minimiser does next).  s_stop, of
  // a single member: kFlagStop for this (the next) pass; by turns, since one
  // update wavefront may be at the new positions before the other has looked.
  __shared__ int s_need, s_bits, s_fail, s_over, s_next, s_stop[2];
  enum : int { kGoOn = 0, kDone = 1, kAgain = 2 };
  // A minimiser's state of iteration k in slot k & 1: thread 0 writes the next
  // iteration's while others still read this one's.
  __shared__ MinState s_m[2];
  __shared__ double s_frms;
  __shared__ int s_end;                     // MinStep::end; -1: stopped on such a coordinate
  __shared__ PackScal s_S;                  // thread 0's: Heun strain, and what goes back
  __shared__ double s_gamma0, s_total0;     // thread 0's: Heun strain at the start of the step
  __shared__ u64 s_near[2];                 // rebuild: rows, columns of cells around own particles
  const int tid0 = threadIdx.x, lane64 = tid0 & 63, wave = tid0 >> 6;
  int tid = tid0;
  const TeamSeat seat = a.seats[blockIdx.x];
  const int pk = seat.pack, T = seat.team, me = seat.member;
  const PackInfo P = a.packs[pk];
  if (T == 1 && tid0 == 0) a.status[seat.base] = 0;
  if (!kHeun && a.scal[pk].converged) return;  // the whole team
  const Bank& b = a.b;
  const int own = seat.count, first = seat.first;
  const int cell_words = (P.rows * P.cols + 31) >> 5;
  constexpr int kCap = kTeamCap[SHAPE];
  TeamLds<kTeamOwn[SHAPE], kCap>& l = *reinterpret_cast<TeamLds<kTeamOwn[SHAPE], kCap>*>(lds_raw);
  double* const lpos = reinterpret_cast<double*>(lds_raw);  // l.x, l.y, l.nx, l.ny, kCap each
  int* const status = a.status + seat.base;  // the team's
  u64* const flags = a.flags + seat.base;    // [slot][member]: slots nseats apart
  u64* const sums = a.sums + (size_t)seat.base * 4 * kTeamUpdWaves;

  // force mapping: L lanes per own particle; update mapping: thread t moves
  // own particle t (the first wavefronts)
  int L = 1, lg = 0;
  while (L < 8 && own * 2 * L <= kTeamThreads) {
    L *= 2;
    ++lg;
  }
  const int lane = tid & (L - 1), p0 = tid >> lg;
  const bool act = p0 < own;
  const int glane = lane64 & ~(L - 1);  // first lane of the particle's group in the wavefront
  const bool upd = tid < own;
  const int nuw = (seat.most + 63) >> 6;  // update wavefronts of the team's largest member
  const int nsum = T > 1 ? T * nuw : 1;   // published sums
  int gu = first + (upd ? tid : 0);

  if (upd) {
    l.x[tid] = b.x[gu];
    l.y[tid] = b.y[gu];
    l.nx[tid] = b.nx[gu];
    l.ny[tid] = b.ny[gu];
    l.R[tid] = b.R[gu];
    l.A[tid] = b.A[gu];
    l.id[tid] = b.id[gu];
    l.phi[tid] = b.phi[gu];
    l.m[tid] = kFire ? 1.0 / sqrt(b.I[gu]) : b.I[gu];
    if (kFire) {
      l.vx[tid] = b.vx[gu];
      l.vy[tid] = b.vy[gu];
      l.vp[tid] = b.vpsi[gu];
    }
    if (kHeun) l.rc[tid] = b.RC[gu];
  }
  if (tid == 0) {
    s_need = s_bits = s_fail = s_over = s_next = s_end = s_stop[0] = s_stop[1] = 0;
    s_S = a.scal[pk];
    s_m[0] = min_state(s_S);
  }
  const double Lx = a.scal[pk].Lx, Ly = a.scal[pk].Ly;
  const double le_ratio = Lx / Ly;
  const double skin = P.pad, sx = fmax(1.5, 1.0 + 0.5 * Lx / Ly) * P.pad, hs = 0.5 * P.pad;
  double gam = a.scal[pk].gamma, gam_eval = gam, center = gam;
  const double window = kHeun ? a.gamma_window : 0.0;
  const u64 kStall = 500000000ull;  // 5 s
  u64 limit = a.roll_call;          // of a rebuild's waits
  int missed = kTeamAbsent;         // what one that runs out means

  auto record_of = [&](int j, int g) {
    return a.pos + ((size_t)(j & (kBufs - 1)) * a.ntot + g) * 4;
  };
  // Large teams move records word by word with four lanes to a record, so that
  // an instruction touches 16 whole records (512 bytes in a row) and not one
  // word of 64: all members' words are under way at once.  Small teams wait for
  // one trip, which the way through LDS and the further rounds lengthen.  Record
  // by record and word by word, ms: 200 sheared steps of 8192 particles (128
  // members) 2.28 and 2.41, of 20000 (313) 3.33 and 3.33, of 24000 (375) 3.74
  // and 3.46, of 32700 (511) 4.09 and 3.62; with 128 particles a member of 33000
  // (258 members) 3.85 and 4.23, of 40000 (313) 4.44 and 4.39, of 60001 (469)
  // 5.11 and 4.71.  150 steps of descent of 16384 (256) 1.51 and 1.54, of 24000
  // 2.06 and 1.96.  FIRE, whose members all wait for all sums, gains earlier: 400
  // iterations of 1000 (16) 4.51 and 4.54, of 8192 (128) 5.81 and 5.72, of 32700
  // 9.25 and 8.58.
  const bool wide = T >= (kFire ? 128 : 320);
  // publish this wavefront's own positions, which it has written to LDS, as
  // pass j's
  auto publish = [&](int j) {
    if (T > 1 && !wide) {
      if (upd) {
        u64* r = record_of(j, gu);
        word_store(r, bits_of(l.x[tid]));
        word_store(r + 1, bits_of(l.y[tid]));
        word_store(r + 2, bits_of(l.nx[tid]));
        word_store(r + 3, bits_of(l.ny[tid]));
      }
    } else if (T > 1) {
      // (x, y, nx, ny lie kCap apart in LDS)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = wave * 64 + k * 16 + (lane64 >> 2), w = tid & 3;
        if (i < own) word_store(record_of(j, first + i) + w, bits_of(lpos[w * kCap + i]));
      }
    }
  };
  auto mark_empty = [&](int j) {  // the first nuw wavefronts
    if (T > 1) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = wave * 64 + k * 16 + (lane64 >> 2);
        if (i < own) word_store(record_of(j, first + i) + (tid & 3), kEmpty);
      }
    }
  };
  // halo entries' positions of pass j into LDS
  auto fetch_halo = [&](int j, int H, u64 limit) {
    Wait wait;
    if (!wide) {
      for (int e = tid; e < H; e += kTeamThreads) {
        const u64* r = record_of(j, l.halo[e]);
        u64 v[4];
        while (true) {
#pragma unroll
          for (int k = 0; k < 4; ++k) v[k] = word_load(r + k);
          if (v[0] != kEmpty && v[1] != kEmpty && v[2] != kEmpty && v[3] != kEmpty) break;
          if (wait.over(limit, status)) {
            s_fail = 1;
            break;
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) lpos[k * kCap + own + e] = from_bits(v[k]);
      }
      return;
    }
    constexpr int kAhead = 4;
    const int w = tid & 3, n4 = 4 * H;
    for (int i0 = tid; i0 < n4; i0 += kAhead * kTeamThreads) {
      const u64* r[kAhead];
      u64 v[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k)
        if (i0 + k * kTeamThreads < n4) r[k] = record_of(j, l.halo[(i0 + k * kTeamThreads) >> 2]) + w;
      while (true) {
        bool all = true;
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
          v[k] = 0;
          if (i0 + k * kTeamThreads < n4) v[k] = word_load(r[k]);
        }
#pragma unroll
        for (int k = 0; k < kAhead; ++k) all = all && v[k] != kEmpty;
        if (all) break;
        if (wait.over(limit, status)) {
          s_fail = 1;
          break;
        }
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int i = i0 + k * kTeamThreads;
        if (i < n4) lpos[w * kCap + own + (i >> 2)] = from_bits(v[k]);
      }
    }
  };
  // every member's flag word numbered seq in slot `slot`, ORed into s_bits
  auto gather_flags = [&](int slot, unsigned seq, u64 limit) {
    const u64* f = flags + (size_t)slot * a.nseats;
    Wait wait;
    for (int m = tid; m < T; m += kTeamThreads) {
      u64 v;
      while (((v = word_load(f + m)) >> 8) != seq)
        if (wait.over(limit, status)) {
          s_fail = 1;
          break;
        }
      if ((v >> 8) == seq && (v & 0xff)) atomicOr(&s_bits, (int)(v & 0xff));
    }
  };
  auto put_flag = [&](int slot, unsigned seq, int bits) {  // one thread
    word_store(flags + (size_t)slot * a.nseats + me, ((u64)seq << 8) | (u64)bits);
  };
  // a member that comes up after the others have left at the roll call finds
  // their report and leaves as absent too
  auto give_up = [&](int why) {
    if (why == kTeamStalled &&
        (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kTeamAbsent))
      return;
    atomicOr(status, why);   // (for the team)
    atomicOr(a.err + 1, why);  // (for the host)
  };

  int H = 0;    // halo entries
  int cnt = 0;  // row length of the force mapping's particle (same in its L lanes)
  int steps = 0, pass = 0, xch = 0, nrec = 0;
  unsigned rebuilds = 0;
  bool build = true;       // this pass starts with new rows (uniform over the team)
  bool was_built = false;  // Heun: the previous pass did
  bool predicted = false;  // Heun: the positions are a step's predicted ones
  bool outran = false;     // Heun: the last pass's positions had outrun the rows
  if (wave < nuw) publish(0);
  if (kHeun && T > 1 && tid == 0) put_flag(0, 1, 0);
  __syncthreads();

  while (true) {
    tid = opaque(tid0);
    gu = first + (upd ? tid : 0);
    const int p = opaque(p0);
    // ---- positions of this pass
    if (T > 1) {
      if (kHeun && pass > 0) gather_flags((pass - 1) & 3, (unsigned)pass, kStall);
      if (!build) fetch_halo(pass, H, kStall);  // (the first pass builds)
    }
    __syncthreads();
    if (s_fail) {
      if (tid == 0) give_up(kTeamStalled);
      return;
    }
    if (kHeun) {
      const int bits = T > 1 ? s_bits : s_need;
      if (bits & kFlagStop) break;  // a non-finite coordinate: the error word says so
      if (T > 1) {
        outran = (bits & kFlagFast) && !was_built;
        if (outran) break;
        build = build || ((bits & kFlagRebuild) && !was_built);
        if (pass >= 2 && wave < nuw) mark_empty(pass - 2);
      } else {
        build = build || (bits & kFlagRebuild);
      }
    } else if (T == 1) {
      build = build || (s_need & kFlagRebuild);
    }
    // ---- halo and rows from the positions of this pass
    const bool built = build;
    if (build) {
      center = gam_eval;
      const double glo = gam_eval - window, ghi = gam_eval + window;
      __syncthreads();  // s_need and s_bits read by all
      if (tid == 0) s_need = s_bits = 0;
      if (upd) {
        l.xb[tid] = l.x[tid];
        l.yb[tid] = l.y[tid];
      }
      H = 0;
      if (T > 1) {
        ++rebuilds;
        // Cells within one of an own particle's; and for each run of 64 own
        // particles the rows and columns of cells (modulo 64) it lies in, for
        // the other members.
        for (int w = tid; w < cell_words; w += kTeamThreads) l.cells[w] = 0;
        if (tid < 2) s_near[tid] = 0;
        __syncthreads();
        if (wave < nuw) {
          u64 at_row = 0, at_col = 0, near_row = 0, near_col = 0;
          if (upd) {
            double xw = l.x[tid], yw = l.y[tid];
            wrap_coord(xw, Lx);
            wrap_coord(yw, Ly);
            int col, row;
            cell_col_row(xw, yw, Lx, Ly, P, col, row);
            at_row = 1ull << (row & 63);
            at_col = 1ull << (col & 63);
            for (int d = -1; d <= 1; ++d) {
              const int r = (row + d + P.rows) % P.rows, c = (col + d + P.cols) % P.cols;
              near_row |= 1ull << (r & 63);
              near_col |= 1ull << (c & 63);
              for (int e = -1; e <= 1; ++e) {
                const int q = r * P.cols + (col + e + P.cols) % P.cols;
                atomicOr(&l.cells[q >> 5], 1u << (q & 31));
              }
            }
          }
          at_row = wave_or(at_row);
          at_col = wave_or(at_col);
          near_row = wave_or(near_row);
          near_col = wave_or(near_col);
          if (lane64 == 63) {
            u64* c = a.chunks + ((size_t)blockIdx.x * kTeamUpdWaves + wave) * 4;
            word_store(c, at_row);
            word_store(c + 1, at_col);
            stores_done();
            word_store(c + 2, rebuilds);
            atomicOr(&s_near[0], near_row);
            atomicOr(&s_near[1], near_col);
          }
        }
        __syncthreads();
        // the runs of 64 particles that may reach into those cells, in storage
        // order (s_count: each wavefront's number of them)
        const u64 near_row = s_near[0], near_col = s_near[1];
        int nrun = 0;
        Wait come;
        for (int c0 = 0; c0 < T * nuw; c0 += kTeamThreads) {
          const int c = c0 + tid, m = c / nuw, part = c - m * nuw;
          bool look = false;
          if (c < T * nuw && part * 64 < min(seat.most, P.n - m * seat.most)) {
            const u64* w = a.chunks + ((size_t)(seat.base + m) * kTeamUpdWaves + part) * 4;
            while (word_load(w + 2) != rebuilds)
              if (come.over(limit, status)) {
                s_fail = 1;
                break;
              }
            look = m != me && (word_load(w) & near_row) && (word_load(w + 1) & near_col);
          }
          const u64 looks = __ballot(look);
          if (lane64 == 0) s_count[wave] = __popcll(looks);
          __syncthreads();
          int to = nrun;
          for (int w = 0; w < kWaves; ++w) {
            if (w < wave) to += s_count[w];
            nrun += s_count[w];
          }
          if (look) l.scan.run[to + __popcll(looks & ((1ull << lane64) - 1ull))] = c;
          __syncthreads();
        }
        // their particles in marked cells
        constexpr int kAhead = 4;
        auto run_at = [&](int k, int& count) {  // first particle of the packing, and how many
          const int c = l.scan.run[k], m = c / nuw, part = c - m * nuw;
          count = min(64, min(seat.most, P.n - m * seat.most) - part * 64);
          return m * seat.most + part * 64;
        };
        Wait wait;
        for (int k0 = wave; k0 < nrun; k0 += kWaves * kAhead) {
          u64 wx[kAhead], wy[kAhead];
          while (true) {
            bool all = true;
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
              wx[k] = wy[k] = 0;
              if (k0 + k * kWaves >= nrun) continue;
              int count;
              const int i = run_at(k0 + k * kWaves, count);
              const u64* r = record_of(pass, P.poff + i + min(lane64, count - 1));
              wx[k] = word_load(r);
              wy[k] = word_load(r + 1);
            }
#pragma unroll
            for (int k = 0; k < kAhead; ++k) all = all && wx[k] != kEmpty && wy[k] != kEmpty;
            if (all) break;
            if (wait.over(limit, status)) {
              s_fail = 1;
              break;
            }
          }
#pragma unroll
          for (int k = 0; k < kAhead; ++k) {
            if (k0 + k * kWaves >= nrun) break;
            int count;
            run_at(k0 + k * kWaves, count);
            double xw = from_bits(wx[k]), yw = from_bits(wy[k]);
            wrap_coord(xw, Lx);
            wrap_coord(yw, Ly);
            int col, row;
            cell_col_row(xw, yw, Lx, Ly, P, col, row);
            const int c = row * P.cols + col;
            const u64 m = __ballot(lane64 < count && ((l.cells[c >> 5] >> (c & 31)) & 1u));
            if (lane64 == 0) l.scan.hit[k0 + k * kWaves] = m;
          }
        }
        __syncthreads();
        if (wave == 0) {  // first halo entry of each run
          int at = 0;
          for (int k0 = 0; k0 < nrun; k0 += 64) {
            const int k = k0 + lane64, v = k < nrun ? __popcll(l.scan.hit[k]) : 0;
            int incl = v;
            for (int off = 1; off < 64; off <<= 1) {
              const int t = __shfl_up(incl, off);
              if (lane64 >= off) incl += t;
            }
            if (k < nrun) l.scan.at[k] = at + incl - v;
            at += __shfl(incl, 63);
          }
          if (lane64 == 0) s_count[0] = at;
        }
        __syncthreads();
        H = s_count[0];
        if (own + H <= kCap) {
          for (int k = wave; k < nrun; k += kWaves) {
            const u64 m = l.scan.hit[k];
            int count;
            const int i = run_at(k, count);
            if ((m >> lane64) & 1ull)
              l.halo[l.scan.at[k] + __popcll(m & ((1ull << lane64) - 1ull))] =
                  P.poff + i + lane64;
          }
        } else {
          H = 0;
          if (tid == 0) s_over = 1;
        }
        __syncthreads();
        fetch_halo(pass, H, limit);
        for (int e = tid; e < H; e += kTeamThreads) {
          const int g = l.halo[e];
          l.R[own + e] = b.R[g];
          l.A[own + e] = b.A[g];
          l.id[own + e] = b.id[g];
        }
      }
      __syncthreads();
      // rows: the list kernels' selection rule, a ballot placing the hits in
      // increasing local index
      cnt = 0;
      {
        const int pp = act ? p : 0, M = own + H;
        const double xp = l.x[pp], yp = l.y[pp], reach_p = l.R[pp] + l.A[pp];
        for (int base = 0; base < M; base += L) {
          const int q = base + lane;
          bool hit = false;
          if (act && q < M && q != p) {
            const double reach = reach_p + l.R[q] + l.A[q];
            const double dy = min_image(yp - l.y[q], Ly);
            if (fabs(dy) < reach + skin) {
              const double dx = min_image(xp - l.x[q], Lx);
              hit = fabs(dx + glo * dy) < reach + sx || fabs(dx + ghi * dy) < reach + sx;
            }
          }
          const u64 hits = (__ballot(hit) >> glane) & ((1ull << L) - 1ull);
          const int pos = cnt + __popcll(hits & ((1ull << lane) - 1ull));
          if (hit && pos < kTeamRow) l.row[p * kRowStride + pos] = (unsigned short)q;
          cnt += __popcll(hits);
        }
        if (cnt > kTeamRow) s_over = 2;
      }
      __syncthreads();
      // The team goes on only if every member's halo and rows fit.  A member one of
      // whose waits above ran out leaves here, without a flag that the others
      // would go on from.  (Leaving at each wait instead, three more ways out of
      // the step loop, cost 5% of every FIRE pass: 8 packings of 8000, 300
      // iterations, 10.6 and 11.2 ms.)
      bool over = s_over != 0;
      if (T > 1) {
        const bool missing = s_fail != 0;
        if (tid == 0 && !missing) put_flag(4 + (rebuilds & 1), rebuilds, over ? kFlagOver : 0);
        if (!missing) gather_flags(4 + (rebuilds & 1), rebuilds, limit);
        __syncthreads();
        over = (s_bits & kFlagOver) != 0;
        if (s_fail) {
          if (tid == 0) give_up(missed);
          return;
        }
      }
      if (over) {
        if (tid == 0) atomicOr(a.err + 1, kTeamOver);
        break;  // the state of this pass is written back
      }
      build = false;
    }

    // ---- forces (force mapping): the bounding-circle hits of the particle's
    // row as a bit mask, the same in its L lanes, which then take them in turn,
    // so a wavefront runs the pair math (two-point: about 470 FP64
    // instructions) as often as its busiest particle has L hits
    const bool fp64 = !MIXED || s_m[kHeun ? 0 : steps & 1].prec == kFP64;
    const bool record = MODE == kTeamHeunSe && !predicted && (steps > 0 || a.se_first) &&
                        (a.step0 + steps) % a.se_every == 0;
    double Fx = 0.0, Fy = 0.0, Tq = 0.0;
    double acc[kNSum] = {};
    if (act) {
      const double xp = l.x[p], yp = l.y[p], nxp = l.nx[p], nyp = l.ny[p];
      const double Rp = l.R[p], Ap = l.A[p], reach_p = Rp + Ap;
      const int idp = l.id[p];
      const unsigned short* row = l.row + p * kRowStride;
      u64 mask = 0;
      for (int base = 0; base < cnt; base += L) {
        bool hit = false;
        if (base + lane < cnt) {
          const int q = row[base + lane];
          double dx = min_image(xp - l.x[q], Lx);
          const double dy = min_image(yp - l.y[q], Ly);
          dx += gam_eval * dy;
          const double reach = reach_p + l.R[q] + l.A[q];
          hit = dx * dx + dy * dy < reach * reach * (1.0 + 1e-10);
        }
        mask |= ((__ballot(hit) >> glane) & ((1ull << L) - 1ull)) << base;
      }
      for (int k = 0; k < lane; ++k) mask &= mask - 1;  // this lane's first hit
      while (mask) {
        const int q = row[__ffsll((long long)mask) - 1];
        pair_into<kGd || MODE == kTeamHeunSe, TWO_POINT>(
            xp, yp, nxp, nyp, Rp, Ap, idp, l.x[q], l.y[q], l.nx[q], l.ny[q], l.R[q], l.A[q],
            l.id[q], Lx, Ly, gam_eval, fp64, kGd || record, Fx, Fy, Tq, acc);
        for (int k = 0; k < L; ++k) mask &= mask - 1;  // its next one
      }
    }
    double F[3] = {Fx, Fy, Tq};
    group_sum(F, L);
    if (act && lane == 0) {
      l.fx[p] = F[0];
      l.fy[p] = F[1];
      l.tq[p] = F[2];
    }
    if (kGd) {  // energy of this wavefront's pairs
      const double e = wave_sum(acc[kSeE]);
      if (lane64 == 63) s_part[wave] = e;
    }
    if (MODE == kTeamHeunSe && record) {
#pragma unroll
      for (int k = 0; k < kNSe; ++k) {
        const double v = wave_sum(acc[k]);
        if (lane64 == 63) s_part[wave * kNSe + k] = v;
      }
    }
    __syncthreads();  // forces visible to the update mapping
    tid = opaque(tid0);
    if (MODE == kTeamHeunSe && record) {
      if (tid < kNSe) {
        double v = 0.0;
        for (int w = 0; w < kWaves; ++w) v += s_part[w * kNSe + tid];
        a.se_part[((size_t)nrec * T + me) * kNSe + tid] = v;
      }
      ++nrec;
    }
    double x = 0.0, y = 0.0, phi = 0.0;  // the particle's new state (update mapping)
    bool moved = kHeun;                  // uniform over a wavefront
    if (kHeun) {
      // ---- predictor or corrector (sheared steps, as k_list)
      if (tid == 0) s_bits = s_need = 0;
      const double dt = P.dt, gd = P.strain_rate;
      if (upd) {
        const double fx = l.fx[tid], fy = l.fy[tid], tq = l.tq[tid], Iu = l.m[tid];
        const double iso = gd * iso_rot_seg(l.rc[tid], l.nx[tid], l.ny[tid], l.A[tid]);
        if (!predicted) {
          const double ox = l.x[tid], oy = l.y[tid], op = l.phi[tid];
          const double vx = fx - gam * fy, vy = fy, vp = tq / Iu - iso;
          l.ox[tid] = ox;
          l.oy[tid] = oy;
          l.op[tid] = op;
          l.vx[tid] = vx;
          l.vy[tid] = vy;
          l.vp[tid] = vp;
          x = ox + dt * vx;
          y = oy + dt * vy;
          phi = op + dt * vp;
        } else {
          x = l.ox[tid] + 0.5 * dt * (l.vx[tid] + (fx - gam_eval * fy));
          y = l.oy[tid] + 0.5 * dt * (l.vy[tid] + fy);
          phi = l.op[tid] + 0.5 * dt * (l.vp[tid] + (tq / Iu - iso));
        }
      }
      if (!predicted) {
        gam_eval = gam + dt * gd;  // the corrector's strain
        build = fabs(gam_eval - center) >= window;
      } else {
        double g2 = gam + gd * dt;
        if (g2 >= 0.5 * le_ratio) {
          if (upd) {
            if (y < 0) y += Ly;
            else if (y > Ly) y -= Ly;
            x += le_ratio * y;
            if (x < 0) x += Lx;
            else {
              int guard = 0;
              while (x > Lx && guard++ < 8) x -= Lx;
            }
          }
          g2 -= le_ratio;
          build = true;
        }
        if (tid == 0) {
          double gt = s_S.gamma_total + gd * dt;
          if (build && le_ratio == 1.0) gt = (double)(int)(gt + 1) + g2;
          s_gamma0 = s_S.gamma;
          s_total0 = s_S.gamma_total;
          s_S.gamma = g2;
          s_S.gamma_total = gt;
          s_S.step = s_S.step + 1;
        }
        gam = gam_eval = g2;
        build = build || fabs(gam - center) >= window;
        ++steps;
      }
      predicted = !predicted;
      __syncthreads();  // s_need cleared
    }
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    if (!kHeun && wave < nuw) {
      // ---- sums and decision: every update wavefront of every member publishes
      // its sums, adds up all of them in the same order and decides the same
      if (kGd) {
        if (wave == 0 && lane64 < kWaves) s0 = s_part[lane64];
      } else if (upd) {
        const double fx = l.fx[tid], fy = l.fy[tid], tq = l.tq[tid], gp = tq * l.m[tid];
        const double vx = l.vx[tid], vy = l.vy[tid], vp = l.vp[tid];
        const double f2 = fx * fx + fy * fy;
        s0 = f2 + tq * tq;
        s1 = fx * vx + fy * vy + gp * vp;
        s2 = f2 + gp * gp;
        s3 = vx * vx + vy * vy + vp * vp;
      }
      // FIRE: value i of the sums in lanes 12 + i
      s0 = kFire ? four_sums(s0, s1, s2, s3) : wave_sum(s0);
      if (T == 1 && kFire && (lane64 >> 2) == 3) s_part[wave * 4 + (lane64 & 3)] = s0;
    }
    if (T == 1 && kFire && nuw > 1) __syncthreads();
    if (!kHeun && wave < nuw) {
      if (T == 1 && nuw > 1) {  // several update wavefronts of one member: through LDS
        if (kFire) {
          s0 = s_part[lane64 & 3];
          for (int w = 1; w < nuw; ++w) s0 += s_part[4 * w + (lane64 & 3)];
        } else {
          s0 = 0.0;
          for (int w = 0; w < kWaves; ++w) s0 += s_part[w];
        }
      }
      const int need = *(T > 1 ? &s_need : &s_stop[pass & 1]);
      bool again = false, stop = (need & kFlagStop) != 0;
      if (nsum > 1) {
        u64* const cur = sums + (size_t)(xch % 3) * a.nseats * 4 * kTeamUpdWaves;
        stores_done();  // empty marks of the last pass
        const bool first_word = kFire ? lane64 == 12 : lane64 == 63;
        if (first_word || (kFire && (lane64 >> 2) == 3))
          word_store(cur + (me * nuw + wave) * 4 + (kFire ? lane64 & 3 : 0),
                     !first_word ? bits_of(s0)
                     : stop      ? kStopMark
                     : (need & kFlagRebuild) ? kNeedMark : bits_of(s0));
        // every wavefront's sums, a word to a lane (FIRE: four lanes to a record)
        constexpr int kRecords = kFire ? 16 : 64;  // of a load
        s0 = 0.0;
        auto collect = [&](int k0, auto ahead) {
          constexpr int kAhead = decltype(ahead)::value;
          u64 v[kAhead];
          const int r0 = k0 + (kFire ? lane64 >> 2 : lane64), w = kFire ? lane64 & 3 : 0;
          Wait wait;
          while (true) {
            bool all = true;
#pragma unroll
            for (int k = 0; k < kAhead; ++k)
              v[k] = word_load(cur + min(r0 + k * kRecords, nsum - 1) * 4 + w);
#pragma unroll
            for (int k = 0; k < kAhead; ++k) all = all && v[k] != kEmpty;
            if (all) break;
            if (wait.over(kStall, status)) {
              s_fail = 1;
              break;
            }
          }
#pragma unroll
          for (int k = 0; k < kAhead; ++k)
            if (r0 + k * kRecords < nsum) {
              again = again || v[k] == kNeedMark;
              stop = stop || v[k] == kStopMark;
              s0 += from_bits(v[k]);
            }
        };
        if (nsum <= kRecords) collect(0, std::integral_constant<int, 1>{});
        else if (nsum <= 4 * kRecords) collect(0, std::integral_constant<int, 4>{});
        else
          for (int k0 = 0; k0 < nsum; k0 += 16 * kRecords)
            collect(k0, std::integral_constant<int, 16>{});
        again = __any(again);
        stop = __any(stop);
        s0 = kFire ? quad_sum(s0) : wave_sum(s0);
      }
      if (stop || again) {
        if (tid == 0) {
          s_next = stop ? kDone : kAgain;
          if (stop) s_end = -1;
        }
      } else {
        mark_empty(pass);  // all have read this pass's positions
        const MinState S0 = s_m[steps & 1];
        const MinStep S =
            kFire ? minimiser_step(a.fire, true, P.n, P.inv_2n, S0, lane_value(s0, 12),
                                   lane_value(s0, 13), lane_value(s0, 14), lane_value(s0, 15), 0.0,
                                   false)
                  : minimiser_step(a.fire, false, P.n, P.inv_2n, S0, 0.0, 0.0, 0.0, 0.0,
                                   lane_value(s0, 63), false);
        moved = S.end == 0;
        if (tid == 0) {
          s_m[(steps + 1) & 1] = after(S0, S);
          s_end = S.end;
          s_frms = S.frms;
          s_next = S.end ? kDone : kGoOn;
        }
        // ---- update (update mapping); nothing moves once finished
        if (upd && moved) {
          const double fx = l.fx[tid], fy = l.fy[tid], tq = l.tq[tid];
          x = l.x[tid];
          y = l.y[tid];
          phi = l.phi[tid];
          if (kGd) {
            x += P.dt * fx;
            y += P.dt * fy;
            phi += P.dt * tq / l.m[tid];
          } else {
            const double isq = l.m[tid], gp = tq * isq;
            const double vx = l.vx[tid], vy = l.vy[tid], vp = l.vp[tid];
            double ux, uy, up;
            if (S.mix) {
              ux = S.c_keep * vx + S.c_force * fx;
              uy = S.c_keep * vy + S.c_force * fy;
              up = S.c_keep * vp + S.c_force * gp;
            } else {
              x -= 0.5 * S.dt_old * vx;
              y -= 0.5 * S.dt_old * vy;
              phi -= 0.5 * S.dt_old * vp * isq;
              ux = uy = up = 0.0;
            }
            const double dt = S.dt;
            ux += dt * fx;
            uy += dt * fy;
            up += dt * gp;
            l.vx[tid] = ux;
            l.vy[tid] = uy;
            l.vp[tid] = up;
            double mx = dt * ux, my = dt * uy;
            const double m2 = mx * mx + my * my;
            if (m2 > a.fire.max_move * a.fire.max_move) {
              const double sc = a.fire.max_move / sqrt(m2);
              mx *= sc;
              my *= sc;
            }
            x += mx;
            y += my;
            phi += dt * up * isq;
          }
        }
      }
      // the sum slot after next (its sums have been read by all: those of the
      // exchange before this one are in)
      if (nsum > 1 && lane64 < 4)
        word_store(sums + ((size_t)((xch + 2) % 3) * a.nseats * kTeamUpdWaves + me * nuw + wave) * 4 +
                       lane64,
                   kEmpty);
    }
    // ---- the new positions
    if (upd && moved) {
      double wx = x, wy = y;
      const bool okx = wrap_coord(wx, Lx), oky = wrap_coord(wy, Ly);
      int need = 0;
      if (!okx || !oky || !isfinite(phi)) {
        atomicOr(a.err, kErrNonFinite);
        need = kFlagStop;
        s_stop[(pass + 1) & 1] = kFlagStop;
      }
      if (!(kHeun && predicted)) {  // a predicted state stays unwrapped
        x = wx;
        y = wy;
      }
      double sn, cs;
      rod_sincos(phi, &sn, &cs);
      if (kHeun && !wide) {  // from registers: the others wait for this alone
        stores_done();       // empty marks of this pass
        if (T > 1) {
          u64* r = record_of(pass + 1, gu);
          word_store(r, bits_of(x));
          word_store(r + 1, bits_of(y));
          word_store(r + 2, bits_of(l.A[tid] * cs));
          word_store(r + 3, bits_of(l.A[tid] * sn));
        }
      }
      l.x[tid] = x;
      l.y[tid] = y;
      l.nx[tid] = l.A[tid] * cs;
      l.ny[tid] = l.A[tid] * sn;
      l.phi[tid] = phi;
      const double dx = fabs(min_image(x - l.xb[tid], Lx)), dy = fabs(min_image(y - l.yb[tid], Ly));
      const bool late = kHeun && T > 1;  // the answer comes one pass late
      if (fmax(dx, dy) >= (late ? 0.6 * hs : hs)) need |= kFlagRebuild;
      if (late && fmax(dx, dy) >= hs) need |= kFlagFast;
      if (need) atomicOr(&s_need, need);
    }
    if (moved && wave < nuw && (!kHeun || wide)) {
      if (kHeun) stores_done();  // empty marks of this pass
      publish(pass + 1);
    }
    ++xch;
    __syncthreads();  // new coordinates, s_need, s_next and s_fail visible
    if (!kHeun) {
      if (s_fail) {  // (in the first pass too: others may have the sums, and finish)
        if (tid == 0) give_up(kTeamStalled);
        return;
      }
      const int next = s_next;
      if (next == kAgain) {  // the same positions with new rows
        build = true;
        continue;
      }
      ++steps;
      if (next == kDone) break;  // finished at the state just evaluated
    }
    was_built = built;
    ++pass;
    limit = kStall;  // (everyone has come up)
    missed = kTeamStalled;
    if (steps == a.max_steps && !predicted) break;
    if (kHeun && T > 1 && tid == 0) put_flag(pass & 3, (unsigned)pass + 1, s_need);
  }
  if (kHeun && T > 1 && !outran && steps == a.max_steps) {
    // did the last evaluated pass have valid rows on every member?
    gather_flags((pass - 1) & 3, (unsigned)pass, kStall);
    __syncthreads();
    if (s_fail) {
      if (tid == 0) give_up(kTeamStalled);
      return;
    }
    outran = (s_bits & kFlagFast) && !was_built;
  }
  __syncthreads();
  if (kHeun && outran && tid == 0) {
    atomicOr(a.err + 1, kTeamFast);
    if (!predicted) {  // the step was counted
      s_S.gamma = s_gamma0;
      s_S.gamma_total = s_total0;
      s_S.step = s_S.step - 1;
    }
  }
  if (upd) {
    const bool back = kHeun && (predicted || outran);  // to the start of the step
    const double x = back ? l.ox[tid] : l.x[tid], y = back ? l.oy[tid] : l.y[tid];
    const double phi = back ? l.op[tid] : l.phi[tid];
    double sn, cs;
    rod_sincos(phi, &sn, &cs);
    b.x[gu] = x;
    b.y[gu] = y;
    b.phi[gu] = phi;
    b.nx[gu] = l.A[tid] * cs;
    b.ny[gu] = l.A[tid] * sn;
    if (kFire) {
      b.vx[gu] = l.vx[tid];
      b.vy[gu] = l.vy[tid];
      b.vpsi[gu] = l.vp[tid];
    }
    b.fx[gu] = l.fx[tid];
    b.fy[gu] = l.fy[tid];
    b.tau[gu] = l.tq[tid];
  }
  if (me == 0 && tid == 0) {
    if (!kHeun) {
      // (a stop counted the iteration that it did not take)
      const MinState& m = s_m[(steps - (s_end < 0 ? 1 : 0)) & 1];
      s_S.step = m.step;
      s_S.fire_dt = m.dt;
      s_S.fire_alpha = m.alpha;
      s_S.fire_npos = m.npos;
      s_S.prec = m.prec;
      if (s_end > 0) {
        s_S.converged = s_end;
        s_S.iters = m.step;
        s_S.frms = s_frms;
      }
    }
    a.scal[pk] = s_S;
  }
}

#define SC_TEAM_INST(M, H)                                      \
  template __global__ void k_team<M, false, false, H>(TeamArgs); \
  template __global__ void k_team<M, true, false, H>(TeamArgs);  \
  template __global__ void k_team<M, false, true, H>(TeamArgs);  \
  template __global__ void k_team<M, true, true, H>(TeamArgs);
#define SC_TEAM_INST_SHAPE(H)                                              \
  SC_TEAM_INST(kTeamFire, H)                                               \
  SC_TEAM_INST(kTeamGd, H)                                                 \
  SC_TEAM_INST(kTeamHeun, H)                                               \
  template __global__ void k_team<kTeamHeunSe, false, false, H>(TeamArgs); \
  template __global__ void k_team<kTeamHeunSe, true, false, H>(TeamArgs);
SC_TEAM_INST_SHAPE(0)
SC_TEAM_INST_SHAPE(1)
SC_TEAM_INST(kTeamFire, 2)
#undef SC_TEAM_INST_SHAPE
#undef SC_TEAM_INST

}  // namespace sc
