// The last generations of a run as walks (k_tail).
//
// Sweeps advance a batch one generation at a time, so a run takes as many
// sweeps as its deepest chain of generations, and every sweep costs a fixed
// latency however few particles it holds: a transport launch whose slowest
// particle takes its substeps one after another, a draw launch whose slowest
// request takes its candidate rounds, an emission launch.  A 400 GeV muon's
// ~2,000 MuonE vertices are 2,000 generations.  Once few particles remain,
// each wave instead walks particles and their subtrees by itself, one particle
// per lane: substeps to the next hard interaction (propagate_particle,
// shower.py:509-601) and the process choice (665-698); when two thirds of the
// live lanes have got there, their accept/reject draws (draw_sample, 401-465),
// the wave's 64 lanes shared among them, process by process (the lowest
// accepted index is the sequential loop's candidate); and the children
// (sample_scattering, 467-507), appended to the store.  A lane goes on with its
// higher-energy child, so the chain that sets the run's length never waits; the
// lower-energy one goes on the wave's stack, from which free lanes take.  A
// full stack passes children to a spill list, and after its share of
// iterations a wave starts nothing more and leaves its stack there, so the
// next launch spreads the particles over all waves again.  (Particles past a
// list's end are marked in the store, and k_tail_gather lists them as lists
// empty.)  Every random number
// comes from the particle's own Philox stream, as in the sweeps, so the records
// are the sweeps' records, bit for bit.
//
// A muon's vertices follow one another, 13 substeps and a draw phase each, and
// the longest muon sets the run's length.  A wave with muons therefore keeps to
// them: their other children go straight to the spill list, muons of a list go
// to its back, and an empty wave takes from there first: an even share of
// every second wave of the launch, so that the other half of them take the
// list's front; alone in its wave while there are fewer muons than that.
//
// What bounds it: for small batches the latency of a substep (~600 dependent
// instructions) and of a draw phase (two waves per SIMD at most; VALU issue 30 %
// for 1,000 electrons of 10 GeV in graphite, 5.2 ms a run); for large ones VALU
// issue (74 % of the peak at 100,000 mixed primaries in lead, 148 ms, 40,000 in
// 71 ms, both at three waves per SIMD at most); with muons the longest of them
// (32,000 substeps and 2,400 phases, 70 ms alone).  A 400 GeV beam
// of 2,000 in lead, half of them muons: 85 ms; 137 ms with each muon among the
// particles of its own subtree; 264 ms (170 ms of that in the walk) with one
// particle per wave, every lane computing the same transport, and two atomics
// per draw on one line of per-process counters.
#pragma once

constexpr int kTailMaxDepth = 128;  // stack entries per wave
constexpr int kTailGroup = 4;       // walk launches queued per host check after the first
constexpr int kTailStepsPerParticle = 8;  // iterations of a wave per particle of its lanes' budget
constexpr int kTailPhaseSteps = 4;        // iterations a draw phase counts for
// Iterations after which a wave that holds muons starts no more particles, and,
// in a launch with muons on its list, a quarter of that for the others, whose
// iterations (64 lanes instead of a few) take about three times as long: caps
// on the budget's limit, but for a budget that never stops a wave.
constexpr int kMuonIters = 2048;

// Entries of a spill list: kListFront from its front, kListMuons muons from its
// end (a store with less room needs no more than that).  Lists as large as any
// store took 8 bytes a place beside it, gigabytes for large batches; these take
// 72 MB (with 3 * 2^20 at the front, 100,000 mixed primaries in lead took 5 %
// longer).
constexpr int64_t kListFront = 8 << 20, kListMuons = 1 << 20;
constexpr int32_t kMarked = (int32_t)0x80000000;  // bit of a particle's meta: waits, but is on no list

// A spill list: its entries, muons from `end` down.
struct WalkList {
  int32_t *list, *end;
  int64_t front, muons;  // room
};
struct TailParams {
  WalkList in, out;
  int32_t par;      // list `in` (counted at C_SPILL + par, C_MUSPILL + par)
  int32_t depth;    // stack entries per wave (1..kTailMaxDepth)
  int32_t limit;    // iterations after which a wave starts no more particles
};

// A wave's buffers in LDS.
struct WalkLds {
  int32_t stack[kTailMaxDepth];
  double x0[64];     // a lane's accepted point: the 1-D variable in float64,
  float4 xs[64];     //   the 4-D point as the draw kernels store it,
  int32_t tr[64];    //   the candidate count (negative: none in max_trials)
};
__device__ inline bool is_muon(int pid) { return pid == 13 || pid == -13; }

// Where walk_hand_on writes, in LDS: held in scalar registers throughout the
// walk its arguments cost 1 % of it.  The counter's address stays an argument,
// so that the atomic goes out at once (read from LDS first, 1 % of a muon beam).
struct WalkOut {
  WalkList to;
  int32_t* meta;
};
typedef __attribute__((address_space(3))) const WalkOut LdsWalkOut;

// The slots v (>= 0) of the calling lanes at the end of the next launch's list,
// muons from its back; those there is no room for are marked in the store (1).
__device__ __noinline__ int walk_hand_on(LdsWalkOut* out, unsigned long long* count, int32_t v, bool muon) {
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  int marked = 0;
  for (int m = 0; m < 2; ++m) {
    const bool mine = v >= 0 && muon == (m == 1);
    const unsigned long long om = __ballot(mine);
    if (!om) continue;
    unsigned long long o = 0;
    if (lane == 0) o = atomicAdd(count + (m ? C_MUSPILL - C_SPILL : 0), (unsigned long long)__popcll(om));
    int32_t* const at = m ? out->to.end : out->to.list;
    const int64_t room = m ? out->to.muons : out->to.front;
    o = shfl_u64(o, 0) + (unsigned long long)__popcll(om & below);
    if (mine) {
      if ((int64_t)o < room) {
        at[m ? -(int64_t)o : (int64_t)o] = v;
      } else {
        atomicOr(out->meta + v, kMarked);
        marked = 1;
      }
    }
  }
  return marked;
}

// Per-process draw statistics of a block.
struct WalkStats {
  unsigned long long trials[8], draws[8], viol[8];
};

// The draws of process P that the lanes in `mine` ask for (at least one), by
// the whole wave: results in W, indexed by the asking lane.  ie, mf: the asking
// lane's map energy and max_F.
template <int P>
__device__ inline void walk_draws(const DevTables& T, uint64_t seed, bool mine, double E_own, uint64_t sid_own,
                                  int ie, double mf, WalkLds& W, WalkStats& B) {
  constexpr int ND = proc_ndim<P>();
  const int lane = threadIdx.x & 63;
  const PetiteGridDesc& gd = T.d->grid[P];
  const int32_t ninc[4] = {gd.ninc[0], gd.ninc[1], gd.ninc[2], gd.ninc[3]};
  const uint32_t max_trials = T.max_trials;
  unsigned long long om = __ballot(mine);
  int lg = 0, n_open = __popcll(om);
  while ((n_open << (lg + 1)) <= 64) ++lg;
  int G = 1 << lg, gl = lane & (G - 1), g0 = lane - gl;
  int owner = nth_lane(om, lane >> lg);
  bool have = (lane >> lg) < n_open;
  double E = shfl_f64(E_own, owner);
  mf = shfl_f64(mf, owner);
  uint64_t sid = shfl_u64(sid_own, owner);
  ie = __shfl(ie, owner);
  const float* base = T.f32 + gd.node_off + (int64_t)ie * gd.stride;
  uint32_t j = draw_possible<P>(T) ? 0u : max_trials;
  while (true) {
    double x[4] = {0.0, 0.0, 0.0, 0.0};
    double w = 0.0, ua = 1.0, J = 0.0;
    const uint32_t jc = j + (uint32_t)gl;
    if (have) {
      w = candidate_w<P, ND>(T, E, base, ninc, seed, sid, jc, x, ua, J);
      if (ND == 4 && fabs(mf * ua - w) <= kRefBand * w) w = J * integrand_ref<P>(T, E, x);
    }
    const bool acc = have && (jc < max_trials) && (mf * ua < w);
    const unsigned long long gmask = (G == 64) ? ~0ull : (((1ull << G) - 1ull) << g0);
    const unsigned long long am = __ballot(acc) & gmask;
    if (have) {
      const bool over = !am && j + (uint32_t)G >= max_trials;
      if (am ? lane == __ffsll((long long)am) - 1 : (over && gl == 0)) {
        const uint32_t n = am ? jc + 1u : max_trials;
        W.tr[owner] = am ? (int32_t)n : -(int32_t)n;
        W.x0[owner] = x[0];
        W.xs[owner] = make_float4((float)x[0], (float)x[1], (float)x[2], (float)x[3]);
        atomicAdd(&B.trials[P], (unsigned long long)n);
        atomicAdd(&B.draws[P], 1ull);
        if (am && w > mf) atomicAdd(&B.viol[P], 1ull);
      }
      if (am || over) have = false;
      j += (uint32_t)G;
    }
    const unsigned long long lead = __ballot(have && gl == 0);
    if (lead == 0ull) break;
    n_open = __popcll(lead);
    int lg2 = lg;
    while ((n_open << (lg2 + 1)) <= 64) ++lg2;
    if (lg2 > lg) {
      // the lanes of the draws that are through join the open ones (draw_loop)
      const int src = nth_lane(lead, lane >> lg2);
      have = (lane >> lg2) < n_open;
      E = shfl_f64(E, src);
      mf = shfl_f64(mf, src);
      sid = shfl_u64(sid, src);
      base = (const float*)shfl_u64((unsigned long long)base, src);
      owner = __shfl(owner, src);
      j = __shfl(j, src);
      lg = lg2;
      G = 1 << lg;
      gl = lane & (G - 1);
      g0 = lane - gl;
    }
  }
}

// Walks the items [0, nres + n + n_spill_in): the particles the previous
// sweep handed on (live state in its resume records), the store slots
// [first, first + n), then the previous launch's spills.  range: the tail
// setup's {first, n, end, nres}.
// EU: waves per SIMD the registers are held to (168 of them and 23 spills for
// three; the run chooses).
constexpr int kWalkWaves = 4;  // waves per block
template <int EU>
__global__ __launch_bounds__(64 * kWalkWaves) __attribute__((amdgpu_waves_per_eu(EU))) void k_tail(
    DevTables T, DevStore S, uint64_t seed, double* shower_energy, unsigned long long* counters,
    const double* sig_lds_src, const int64_t* range, ResumeBuf RB, TailParams TPm) {
  const int64_t first = range[0], n = range[1];
  const int64_t nres = RB.rec ? range[3] : 0;
  const ResumeRec* rin = RB.rec ? RB.rec + (int64_t)(counters[C_RPARITY] & 1ull) * RB.cap : nullptr;
  // a count past the list is cut to the list (the others are marked)
  const int32_t* const spill_in = TPm.in.list;
  const int64_t total = nres + n + min((int64_t)counters[C_SPILL + TPm.par], TPm.in.front);
  const int64_t n_mu = min((int64_t)counters[C_MUSPILL + TPm.par], TPm.in.muons);
  // items per claim: an even share of every wave of the launch (of half of them
  // for muons), at most a lane's each
  const int64_t waves = (int64_t)gridDim.x * kWalkWaves;
  const int share = (int)min((int64_t)64, max((int64_t)1, (total + waves - 1) / waves));
  const int share_mu = (int)min((int64_t)64, max((int64_t)1, (2 * n_mu + waves - 1) / waves));
  if ((int64_t)blockIdx.x * kWalkWaves >= (total + share - 1) / share + (n_mu + share_mu - 1) / share_mu) return;
  // INT32_MAX: no wave stops (tail_limit), one with muons as little as the others
  const bool capped = TPm.limit != INT32_MAX;
  const int limit_mu = capped ? min(TPm.limit, kMuonIters) : TPm.limit;
  const int limit = capped && n_mu > 0 ? min(TPm.limit, kMuonIters / 4) : TPm.limit;
  HIP_DYNAMIC_SHARED(double, s_sig)
  __shared__ WalkLds s_walk[kWalkWaves];
  __shared__ WalkStats s_stat;
  __shared__ WalkOut s_out;
  for (int i = threadIdx.x; i < T.lds_doubles; i += blockDim.x) s_sig[i] = sig_lds_src[i];
  if (threadIdx.x == 0) s_out = WalkOut{TPm.out, S.meta};
  if (threadIdx.x < 8) s_stat.trials[threadIdx.x] = s_stat.draws[threadIdx.x] = s_stat.viol[threadIdx.x] = 0ull;
  __syncthreads();
  const LdsSigma L{s_sig};
  LdsWalkOut* const to_out = (LdsWalkOut*)&s_out;
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  WalkLds& W = s_walk[threadIdx.x >> 6];
  const int depth = TPm.depth < 1 ? 1 : (TPm.depth > kTailMaxDepth ? kTailMaxDepth : TPm.depth);
  // lane states: empty, stepping, at its end (parked), given a particle that
  // has not started
  enum { EMPTY = 0, STEP = 1, PARKED = 2, GIVEN = 3 };
  int mode = EMPTY;
  int sp = 0;              // stack entries (wave-uniform, as the next four)
  int iters = 0;
  bool exhausted = total <= 0, mu_exhausted = n_mu <= 0, fresh = true;
  bool muons = false;      // the wave holds muons, and keeps to them (see the head of the file)
  int32_t slot = 0;
  int pid = 0, shower = 0, gen = 0;
  uint32_t ch = 0xFFFu;
  uint64_t sid = 0;
  double m = 0.0, pme = 0.0, E = 0.0, dep = 0.0;
  double dz = 0.0;  // substep length; |p| of a particle that does not move
  float nx = 0.0f, ny = 0.0f, nz = 0.0f, rx = 0.0f, ry = 0.0f, rz = 0.0f, wgt = 0.0f;
  uint32_t k = 0;
  bool closing = false;
  unsigned int steps = 0, n_fail = 0, n_drop = 0, n_ovf = 0, n_marked = 0;  // of this lane in this launch
  while (true) {
    // past its share the wave starts no more: the next launch spreads what it leaves
    if (muons) muons = __ballot(mode != EMPTY && is_muon(pid)) != 0ull;
    const bool stop = iters >= (muons ? limit_mu : limit);
    // ---- free lanes take from the stack, then claim items (after a draw
    // phase, or when no lane is stepping)
    const unsigned long long im = __ballot(mode == EMPTY);
    int64_t rr = -1;
    if (im && !stop && !muons && (fresh || __ballot(mode == STEP) == 0ull)) {
      const int rank = __popcll(im & below);
      const int take = min(__popcll(im), sp);
      bool got = false, got_mu = false;
      if (!mu_exhausted && sp == 0 && im == ~0ull) {
        unsigned long long c = 0;
        if (lane == 0) c = atomicAdd(counters + C_MUCLAIM, (unsigned long long)share_mu);
        c = shfl_u64(c, 0);
        got = lane < share_mu && (int64_t)c + lane < n_mu;
        if (got) slot = TPm.in.end[-((int64_t)c + lane)];
        got_mu = (int64_t)c < n_mu;
        mu_exhausted = (int64_t)c + share_mu >= n_mu;
      }
      if (mode == EMPTY && rank < take) {
        slot = W.stack[sp - 1 - rank];
        got = true;
      }
      sp -= take;
      const int need = min(__popcll(im) - take, share);
      if (need > 0 && !exhausted && !got_mu) {
        unsigned long long c = 0;
        if (lane == 0) c = atomicAdd(counters + C_TRANSPORT, (unsigned long long)need);
        c = shfl_u64(c, 0);
        if (mode == EMPTY && !got && rank - take < need) {
          rr = (int64_t)c + (rank - take);
          got = rr < total;
          if (got) slot = rr < nres ? rin[rr].slot
                                    : (rr < nres + n ? (int32_t)(first + (rr - nres)) : spill_in[rr - nres - n]);
        }
        exhausted = (int64_t)c + need >= total;
      }
      if (got) {
        const float4 p0 = S.p0[slot], r0 = S.r0[slot];
        pid = S.pid[slot];
        sid = S.sid[slot];
        shower = S.shower[slot];
        gen = S.meta[slot] & 0xFFFF;
        E = (double)p0.x;
        nx = p0.y;
        ny = p0.z;
        nz = p0.w;
        rx = r0.x;
        ry = r0.y;
        rz = r0.z;
        wgt = r0.w;
        mode = GIVEN;
      }
      muons = __ballot(mode == GIVEN && is_muon(pid)) != 0ull;
    }
    // ---- the given particles' starts (k_transport's refill)
    if (mode == GIVEN) {
      ch = sum_channels(pid);
      m = pid_mass(pid);
      pme = fmax(fmax(min_calc(T, pid), T.min_energy), m);
      const float pn2 = norm2(nx, ny, nz);
      if (pn2 > 0.0f) {
        const float inv = rsqrtf(pn2);
        nx *= inv;
        ny *= inv;
        nz *= inv;
      }
      const bool still = ch == 0xFFFu && pid != 22;
      if (still) dz = sqrt((double)pn2);  // the others' |p| is formed when they finish
      dep = 0.0;
      k = 0;
      closing = false;
      mode = STEP;
      if (rr >= 0 && rr < nres) {
        // handed on by the last sweep: its live state
        const ResumeRec& R0 = rin[rr];
        E = R0.E;
        dep = R0.dep;
        dz = R0.dz;
        nx = R0.nx;
        ny = R0.ny;
        nz = R0.nz;
        rx = R0.rx;
        ry = R0.ry;
        rz = R0.rz;
        k = R0.k;
      } else if (E < pme || still) {
        mode = PARKED;  // ends where it starts (shower.py:532-536, 640-653)
      } else if (pid == 22) {
        // one exponential flight, no MCS (shower.py:538-553)
        const double mfp = L.mfp(22, E);
        const double dist = -mfp * (double)log1p_f32(-u01f(draw_block(seed, sid, 0, PURPOSE_STEP).x));
        rx += (float)(nx * dist);
        ry += (float)(ny * dist);
        rz += (float)(nz * dist);
        k = 1;
        mode = PARKED;
      }
    }
    fresh = false;
    unsigned long long am = __ballot(mode == STEP), wm = __ballot(mode == PARKED);
    if (am == 0ull && wm == 0ull) break;
    // a draw phase costs several substeps (loads, a round of candidates per
    // process, the kinematics): run at two thirds of the live lanes parked it
    // measures 15 % faster than at a third over the showers of 1 to 100,000
    // primaries, and a half or four fifths are in between
    if (am != 0ull && __popcll(wm) < 2 * __popcll(am)) {
      // ---- advances of the stepping lanes (k_transport's) until a phase is due
      const LdsSigma::Channel c0 = L.channel(ch & 0xFu), c1 = L.channel((ch >> 4) & 0xFu),
                              c2 = L.channel((ch >> 8) & 0xFu);
      do {
        ++iters;
        if (mode == STEP) {
          const bool in_close = closing;
          // the channels' records are on their way while the Philox block is formed
          LdsSigma::Pair r0{}, r1{}, r2{};
          if (T.sig_indexed) {
            const float l2 = __log2f((float)E);
            r0 = L.fetch(c0, l2);
            r1 = L.fetch(c1, l2);
            r2 = L.fetch(c2, l2);
            __builtin_amdgcn_sched_barrier(0);
          }
          const U4 u = draw_block(seed, sid, in_close ? 0u : k, in_close ? PURPOSE_CLOSE : PURPOSE_STEP);
          double Ssum;
          if (T.sig_indexed) {
            const double s01 = L.value(c0, r0, E) + L.value(c1, r1, E);
            const double s2 = L.value(c2, r2, E);
            Ssum = (ch >> 8) == 0xFu ? s01 : s01 + s2;
          } else {
            Ssum = L.nsigma_sum_ch(ch, E);
          }
          const double mfp = Ssum > 0.0 ? kCmToM / Ssum : 1.0e12;
          bool adv = true;
          double dist;
          uint32_t w_r, w_a;
          double m_lep = m;
          if (!in_close) {
            const double div = 6.0 + 14.0 * u01d(u.y);
            dz = mfp / div;
            dist = dz;
            w_r = u.z;
            w_a = u.w;
            const double ux = u01d(u.x);
            double thr = (double)__expf(-__builtin_amdgcn_rcpf((float)div));
            if (fabs(ux - thr) < 1.0e-5) thr = exp(-(dz / mfp));
            if (ux > thr) {
              adv = false;
              closing = true;
            }
          } else {
            const double distC = u01d(u.x);
            if (E < pme) {
              dist = distC * dz;
            } else {
              const float r2 = Ssum > 0.0 ? (float)(dz * Ssum * (1.0 / kCmToM)) : (float)(dz * 1.0e-12);
              dist = -mfp * (double)log1p_f32(expm1f(-r2) * (float)distC);
            }
            w_r = u.y;
            w_a = u.z;
            m_lep = kMe;
          }
          if (adv) charged_advance(T, dist, m, m_lep, w_r, w_a, E, nx, ny, nz, rx, ry, rz, dep);
          ++k;
          if (in_close) mode = PARKED;
          else if (E < pme) closing = true;
        }
        am = __ballot(mode == STEP);
        wm = __ballot(mode == PARKED);
      } while (am != 0ull && __popcll(wm) < 2 * __popcll(am));
      if (wm == 0ull) continue;
    }
    // ---- the parked lanes' final states and process choices (k_transport's finish)
    iters += kTailPhaseSteps;
    fresh = true;
    int want = -1;
    float4 pf = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (mode == PARKED) {
      steps += k;
      const double p = ch == 0xFFFu && pid != 22 ? dz : momentum(E, m);
      pf = make_float4((float)E, (float)(p * nx), (float)(p * ny), (float)(p * nz));
      S.pf[slot] = pf;
      S.rf[slot] = make_float4(rx, ry, rz, (float)k);
      if (E > pme) {
        int c0 = -1, c1 = -1, c2 = -1;
        switch (pid) {
          case 11: c0 = BREM; c1 = MOLLER; break;
          case -11: c0 = BREM; c1 = ANN; c2 = BHABHA; break;
          case 22: c0 = PAIRPROD; c1 = COMP; break;
          case 13: case -13: c0 = MUONE; c1 = MUONBREM; break;
          default: break;
        }
        if (c0 >= 0) {
          const float lf = __log2f((float)E);
          const double w0 = L.nsigma(c0, E, lf), w1 = L.nsigma(c1, E, lf);
          const double w2 = c2 >= 0 ? L.nsigma(c2, E, lf) : 0.0;
          const double SC = c2 >= 0 ? w0 + w1 + w2 : w0 + w1;
          if (SC > 0.0 && !isnan(SC)) {
            const double uu = u01d(draw_block(seed, sid, 0, PURPOSE_INTERACT).x) * SC;
            if (uu < w0) want = c0;
            else if (c2 < 0 || uu < w0 + w1) want = c1;
            else want = c2;
          }
        }
      }
      if (shower_energy) {
        unsafeAtomicAdd(shower_energy + 4 * shower + 0, dep);
        if (want < 0) unsafeAtomicAdd(shower_energy + 4 * shower + 1, E);
      }
      mode = EMPTY;
    }
    // ---- the draws, process by process (the map energies and max_F of all
    // of them first: one round of dependent loads)
    int ie = 0;
    double mf = 0.0;
    if (want >= 0) {
      ie = lu_key(T, want, E);
      mf = T.maxf[want * T.maxE + ie] * T.maxF_fudge;
    }
    for (unsigned long long todo = __ballot(want >= 0); todo;) {
      const int q = __shfl(want, __ffsll((long long)todo) - 1);
      const bool mine = want == q;
      switch (q) {
        case 0: walk_draws<0>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 1: walk_draws<1>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 2: walk_draws<2>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 3: walk_draws<3>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 4: walk_draws<4>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 5: walk_draws<5>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        case 6: walk_draws<6>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
        default: walk_draws<7>(T, seed, mine, E, sid, ie, mf, W, s_stat); break;
      }
      todo &= ~__ballot(mine);
    }
    // results written by other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // ---- the children (k_emit)
    V4 lab[2];
    int cpid[2] = {0, 0};
    bool keep[2] = {false, false};
    if (want >= 0) {
      if (W.tr[lane] <= 0) {
        ++n_fail;
        if (shower_energy) unsafeAtomicAdd(shower_energy + 4 * shower + 1, E);
      } else {
        const double az = u01d(draw_block(seed, sid, 0, PURPOSE_INTERACT).y);
        const float4 xv = W.xs[lane];
        const float xs[4] = {xv.x, xv.y, xv.z, xv.w};
        vertex_children(want, pid, E, xs, W.x0[lane], az, pf.y, pf.z, pf.w, lab, cpid);
        for (int c = 0; c < 2; ++c) {
          keep[c] = lab[c].e > T.min_energy;
          if (!keep[c]) {
            ++n_drop;
            if (shower_energy) unsafeAtomicAdd(shower_energy + 4 * shower + 2, lab[c].e);
          }
        }
        if (shower_energy && (want == COMP || want == ANN || want == MOLLER || want == BHABHA || want == MUONE))
          unsafeAtomicAdd(shower_energy + 4 * shower + 3, 1.0);
      }
    }
    // store slots: one atomic per wave and phase
    const unsigned long long k0 = __ballot(keep[0]), k1 = __ballot(keep[1]);
    if ((k0 | k1) == 0ull) continue;
    unsigned long long cb = 0;
    if (lane == 0) cb = atomicAdd(counters + C_STORE, (unsigned long long)(__popcll(k0) + __popcll(k1)));
    cb = shfl_u64(cb, 0) + (unsigned long long)(__popcll(k0 & below) + __popcll(k1 & below));
    int32_t cslot[2] = {-1, -1};
    uint64_t csid[2] = {0, 0};
    float4 cp[2];
    for (int c = 0; c < 2; ++c) {
      if (!keep[c]) continue;
      if ((int64_t)cb < S.capacity) {
        cslot[c] = (int32_t)cb;
        cp[c] = make_float4((float)lab[c].e, (float)lab[c].x, (float)lab[c].y, (float)lab[c].z);
        csid[c] = derive_sid(seed, sid, (uint32_t)c, PURPOSE_CHILD);
        S.p0[cb] = cp[c];
        S.r0[cb] = make_float4(rx, ry, rz, wgt);
        S.pid[cb] = cpid[c];
        S.parent[cb] = slot;
        S.meta[cb] = ((gen + 1) & 0xFFFF) | ((want + 1) << 16) | (c << 24);
        S.shower[cb] = shower;
        S.sid[cb] = csid[c];
      } else {
        ++n_ovf;
      }
      ++cb;
    }
    // the stores above are read by other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // the lane goes on with its higher-energy child, unless the wave stops; in
    // a wave with muons with its muon, and the others are handed on
    int higher = cslot[0] >= 0 && (cslot[1] < 0 || lab[1].e < lab[0].e) ? 0 : 1;
    bool hmu = false, lmu = false;
    if (muons) {
      hmu = is_muon(cpid[higher]);
      lmu = cslot[1 - higher] >= 0 && is_muon(cpid[1 - higher]);
      if (lmu && !hmu) {
        higher = 1 - higher;
        hmu = true;
        lmu = false;
      }
    }
    const int32_t hs = higher ? cslot[1] : cslot[0], ls = higher ? cslot[0] : cslot[1];
    const bool go_on = hs >= 0 && !stop && (hmu || !muons);
    for (int t = 0; t < 2; ++t) {
      const int32_t v = t == 0 ? (go_on ? -1 : hs) : ls;
      const unsigned long long pm = __ballot(v >= 0);
      if (!pm) continue;
      const int at = muons ? depth : sp + __popcll(pm & below);
      if (v >= 0 && at < depth) W.stack[at] = v;
      const int32_t out = at >= depth ? v : -1;
      if (__ballot(out >= 0))
        n_marked += walk_hand_on(to_out, counters + C_SPILL + (TPm.par ^ 1), out, t == 0 ? hmu : lmu);
      if (!muons) sp = min(depth, sp + __popcll(pm));
    }
    if (go_on) {
      const float4 c = higher ? cp[1] : cp[0];
      slot = hs;
      pid = higher ? cpid[1] : cpid[0];
      sid = higher ? csid[1] : csid[0];
      gen = (gen + 1) & 0xFFFF;
      E = (double)c.x;
      nx = c.y;
      ny = c.z;
      nz = c.w;
      mode = GIVEN;
    }
  }
  // ---- what the wave did not start goes to the next launch, and so do the
  // items no wave claimed (a handed-on one starts over there: its random
  // numbers are indexed by its substeps, so it ends the same)
  while (!exhausted) {
    unsigned long long c = 0;
    if (lane == 0) c = atomicAdd(counters + C_TRANSPORT, 64ull);
    c = shfl_u64(c, 0);
    exhausted = (int64_t)c + 64 >= total;
    const int64_t rr = (int64_t)c + lane;
    int32_t v = -1;
    if (rr < total)
      v = rr < nres ? rin[rr].slot
                    : (rr < nres + n ? (int32_t)(first + (rr - nres)) : spill_in[rr - nres - n]);
    n_marked += walk_hand_on(to_out, counters + C_SPILL + (TPm.par ^ 1), v, v >= 0 && is_muon(S.pid[v]));
  }
  while (!mu_exhausted) {
    unsigned long long c = 0;
    if (lane == 0) c = atomicAdd(counters + C_MUCLAIM, 64ull);
    c = shfl_u64(c, 0);
    mu_exhausted = (int64_t)c + 64 >= n_mu;
    const int64_t rr = (int64_t)c + lane;
    n_marked += walk_hand_on(to_out, counters + C_SPILL + (TPm.par ^ 1), rr < n_mu ? TPm.in.end[-rr] : -1, true);
  }
  for (int e0 = 0; e0 < sp; e0 += 64)
    n_marked += walk_hand_on(to_out, counters + C_SPILL + (TPm.par ^ 1), e0 + lane < sp ? W.stack[e0 + lane] : -1, false);
  {
    unsigned long long* const st = counters + C_STATS;
    const unsigned long long v[7] = {steps, steps, n_fail, n_drop, n_ovf, n_marked, 0ull};
    unsigned long long* const dst[7] = {st + ST_STEPS, counters + C_TAIL_STEPS, st + ST_NOSAMPLE, st + ST_DROPPED,
                                        st + ST_OVERFLOW, counters + C_MARKED, st};
    block_stat_add<7>(v, dst);
  }
  if (threadIdx.x < 8) {
    const int q = threadIdx.x;
    if (s_stat.draws[q]) {
      atomicAdd(counters + C_PTRIALS + q, s_stat.trials[q]);
      atomicAdd(counters + C_PDRAWS + q, s_stat.draws[q]);
      if (s_stat.viol[q]) atomicAdd(counters + C_PVIOL + q, s_stat.viol[q]);
    }
  }
}

// Iterations of a wave in walk launch number i (from 0): `budget` particles per
// lane in the first, twice as many in each later one, so that particles are
// spread often while their number grows and seldom once a few long chains
// remain (a spread costs a launch, and leaves a chain among other particles);
// budgets above 2^30 never stop a wave.  (kMuonIters caps the others' limits in
// launches with muons.)
static int32_t tail_limit(int32_t budget, int64_t i) {
  if (budget > (1 << 30)) return INT32_MAX;
  return (int32_t)std::min<int64_t>((int64_t)std::max(budget, 1) * kTailStepsPerParticle << std::min<int64_t>(i, 20),
                                    INT32_MAX);
}

// Start of a tail launch: the items are the particles handed on by the last
// sweep, every store entry appended since the last sweep or tail launch (no
// bound: the walk files no draw requests), and the previous launch's spills
// (in the list of parity `par`, whose counts are cut to it; the other list is
// cleared for this launch's).  Everything a tail launch appended was walked or
// spilled, so the launches after the first start past it.
__global__ void k_tail_setup(unsigned long long* ctr, int64_t* range, int64_t capacity, int64_t resume_cap,
                             TailParams P, bool first) {
  if (threadIdx.x == 0) {
    const int64_t big = (int64_t)1 << 62;
    const int64_t now = min((int64_t)ctr[C_STORE], capacity);
    const SweepRange sr = sweep_range(first ? range[2] : now, now, capacity, big, (int64_t)ctr[C_YIELD_OUT],
                                      resume_cap);
    range[0] = sr.first;
    range[1] = sr.n;
    range[2] = sr.first + sr.n;
    range[3] = sr.nres;
    ctr[C_YIELD_OUT] = 0ull;
    ctr[C_RPARITY] ^= 1ull;
    ctr[C_TRANSPORT] = 0ull;
    ctr[C_SPILL + P.par] = min(ctr[C_SPILL + P.par], (unsigned long long)P.in.front);
    ctr[C_MUSPILL + P.par] = min(ctr[C_MUSPILL + P.par], (unsigned long long)P.in.muons);
    ctr[C_SPILL + (P.par ^ 1)] = 0ull;
    ctr[C_MUSPILL + (P.par ^ 1)] = 0ull;
    ctr[C_MUCLAIM] = 0ull;
    ctr[C_GATHER] = ctr[C_MARKED];
    if (sr.n > 0 || sr.nres > 0 || (ctr[C_SPILL + P.par] | ctr[C_MUSPILL + P.par] | ctr[C_MARKED]) != 0ull)
      ctr[C_SWEEPS] += 1ull;
  }
}

// The marked particles onto the coming launch's list, as many as it has room
// for: one atomic per block, list and 4,096 store entries.  A launch that finds
// none marked ends at once.
constexpr int kGatherRun = 16;
__global__ __launch_bounds__(256) void k_tail_gather(DevStore S, unsigned long long* ctr, TailParams P) {
  if (ctr[C_GATHER] == 0ull) return;
  __shared__ unsigned int s_n[2][4];
  __shared__ unsigned long long s_base[2];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  const int64_t n = min((int64_t)ctr[C_STORE], S.capacity);
  constexpr int64_t kWaveRun = 64 * kGatherRun, kBlockRun = 4 * kWaveRun;
  unsigned long long listed = 0ull;
  for (int64_t b0 = (int64_t)blockIdx.x * kBlockRun; b0 < n; b0 += (int64_t)gridDim.x * kBlockRun) {
    const int64_t w0 = b0 + wid * kWaveRun;
    unsigned int c[2] = {0u, 0u};
    for (int j = 0; j < kGatherRun; ++j) {
      const int64_t i = w0 + j * 64 + lane;
      const bool marked = i < n && S.meta[i] < 0;
      const unsigned long long m = __ballot(marked);
      if (!m) continue;
      const unsigned int mu = (unsigned int)__popcll(__ballot(marked && is_muon(S.pid[i])));
      c[0] += (unsigned int)__popcll(m) - mu;
      c[1] += mu;
    }
    if (lane == 0) {
      s_n[0][wid] = c[0];
      s_n[1][wid] = c[1];
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      const unsigned int t = s_n[threadIdx.x][0] + s_n[threadIdx.x][1] + s_n[threadIdx.x][2] + s_n[threadIdx.x][3];
      s_base[threadIdx.x] =
          t ? atomicAdd(ctr + (threadIdx.x ? C_MUSPILL : C_SPILL) + P.par, (unsigned long long)t) : 0ull;
    }
    __syncthreads();
    unsigned long long o[2] = {s_base[0], s_base[1]};
    for (int w = 0; w < wid; ++w) {
      o[0] += s_n[0][w];
      o[1] += s_n[1][w];
    }
    for (int j = 0; j < kGatherRun; ++j) {
      const int64_t i = w0 + j * 64 + lane;
      const bool marked = i < n && S.meta[i] < 0;
      if (!__ballot(marked)) continue;
      const bool muon = marked && is_muon(S.pid[i]);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool mine = marked && muon == (q == 1);
        const unsigned long long m = __ballot(mine);
        const int64_t at = (int64_t)(o[q] + __popcll(m & below));
        if (mine && at < (q ? P.in.muons : P.in.front)) {
          *(q ? P.in.end - at : P.in.list + at) = (int32_t)i;
          S.meta[i] &= ~kMarked;
          ++listed;
        }
        o[q] += (unsigned long long)__popcll(m);
      }
    }
    __syncthreads();  // s_n and s_base are read before the next run writes them
  }
  const unsigned long long v[1] = {0ull - listed};
  unsigned long long* const dst[1] = {ctr + C_MARKED};
  block_stat_add<1>(v, dst);
}
