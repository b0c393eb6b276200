// Dark-vector production over a shower record (DarkShower.generate_dark_shower,
// src/PETITE/dark_shower.py:806-849).
//
// k_dark_select reads each SM record once and, for every active process with
// a positive weight (GetBSMWeights, 595-647), writes an entry: the weight, the
// pair's dark stream, and the state produce_bsm_particle (721-804) reaches
// before its draw: interaction energy from the drate table, multiple
// scattering over the distance travelled and the energy lost.  Entries that
// need draw_dark_sample go to the per-process draw regions; k_dark_emit turns
// every entry into its vector (threshold shortcuts, bound-electron Compton,
// radiative return, dark bremsstrahlung) and rotates it into the lab frame.
//
// Random numbers of one pair come from dsid = derive_sid(seed, sid, code,
// PURPOSE_DARK): INTERACT block 0 (x drate bin, y MCS radius, z MCS azimuth
// with its sign in bit 0, w kinematic azimuth), INTERACT block 1 (x the bound
// electron's cos(theta), y the azimuth of its frame), BOUND_E blocks (pairs of
// bound-electron momentum accept/reject uniforms) and the VEGAS candidates.
#pragma once

namespace dark {

enum Family { F_BREM_E = 0, F_BREM_P = 1, F_MUBREM = 2, F_ANN = 3 };
enum State { S_NONE = 0, S_DRAW = 1, S_DIRECT = 2 };
constexpr int kPePairs = 1 << 16;

struct Entries {
  int32_t* parent;   // SM store slot
  int32_t* flag;     // code | state << 8
  double* weight;    // wg * parent weight
  double* E;         // energy after the drate step (pf[0] of produce_bsm_particle)
  float4* dir;       // unit direction of pf
  uint64_t* dsid;    // dark stream
  int64_t cap;
};

// Interval lo with x[lo] <= v < x[lo+1] (v inside [x0, x_{n-1})): an O(1)
// guess g0 + (v' - v0) * inv on uniform grids (in v' = ln v or v itself),
// corrected against the stored nodes; bisection when inv = 0.
__device__ inline int find_interval(const double* x, int n, double v, float guess_arg, double v0, double inv) {
  int lo;
  if (inv > 0.0) {
    lo = (int)((guess_arg - (float)v0) * (float)inv);
    lo = lo < 0 ? 0 : (lo > n - 2 ? n - 2 : lo);
    while (lo > 0 && x[lo] > v) --lo;
    while (lo < n - 2 && x[lo + 1] <= v) ++lo;
  } else {
    lo = 0;
    int hi = n - 1;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (x[mid] <= v) lo = mid; else hi = mid;
    }
  }
  return lo;
}

// numpy.interp on an ascending grid (slope form), 0 outside [x0, x_{n-1}]
// (scipy interp1d with fill_value=0, dark_shower.py:447-452).
__device__ inline double interp_fill0(const double* x, const double* y, int n, double E, double lnE0 = 0.0,
                                      double inv_dlog = 0.0) {
  if (n <= 0 || !(E >= x[0]) || E > x[n - 1]) return 0.0;
  if (E == x[n - 1]) return y[n - 1];
  const int lo = find_interval(x, n, E, __logf((float)E), lnE0, inv_dlog);
  const double slope = (y[lo + 1] - y[lo]) / (x[lo + 1] - x[lo]);
  return slope * (E - x[lo]) + y[lo];
}

// interpolate1d in log10-log10 with fill -20 (dark_shower.py:31-46, 294-309);
// l = log10(E).
__device__ inline double loglog(const double* lx, const double* ly, int n, double l, double l0 = 0.0,
                                double inv_dl = 0.0) {
  if (n <= 0 || l < lx[0] || l > lx[n - 1]) return 1.0e-20;
  if (l == lx[n - 1]) return pow(10.0, ly[n - 1]);
  const int lo = find_interval(lx, n, l, (float)l, l0, inv_dl);
  const double slope = (ly[lo + 1] - ly[lo]) / (lx[lo + 1] - lx[lo]);
  return pow(10.0, slope * (l - lx[lo]) + ly[lo]);
}

__device__ inline int family_of(int code, int pid) {
  if (code == DARKBREM) return pid == 11 ? F_BREM_E : (pid == -11 ? F_BREM_P : -1);
  if (code == DARKANN) return pid == -11 ? F_ANN : -1;
  if (code == DARKMUONBREM) return (pid == 13 || pid == -13) ? F_MUBREM : -1;
  return -1;
}

// Quantities of one SM particle shared by the weights of every mass.
struct WeightArgs {
  double E0;
  float lf;    // logf(E0): guess of the geometric-grid interval
  double l10;  // log10(E0) for the log-log DarkComp table
  double den;  // n*sigma_PairProd + n*sigma_Comp at E0 (photons)
};

__device__ inline WeightArgs weight_args(const DevTables& T, int pid, double E0) {
  WeightArgs a;
  a.E0 = E0;
  a.lf = __logf((float)E0);
  a.l10 = pid == 22 ? log10(E0) : 0.0;
  a.den = pid == 22 ? nsigma(T, PAIRPROD, E0) + nsigma(T, COMP, E0) : 0.0;
  return a;
}

// GetBSMWeights (dark_shower.py:595-647), eps^2 included.
__device__ inline double bsm_weight(const DevTables& T, const PetiteDarkDesc& D, const double* b, int pid, int code,
                                    const WeightArgs& a) {
  const double E0 = a.E0;
  if (code == DARKCOMP) {
    if (pid != 22 || E0 < D.min_comp || E0 < T.min_calc[2]) return 0.0;
    const double* lx = b + D.comp_off;
    const double num = loglog(lx, lx + D.comp_n, D.comp_n, a.l10, D.comp_l0, D.comp_inv_dl);
    return D.eps2 * (num / a.den);
  }
  const int f = family_of(code, pid);
  if (f < 0) return 0.0;
  const double thr = (code == DARKBREM) ? D.min_brem : (code == DARKANN ? D.min_ann : D.min_muon_brem);
  if (E0 < thr) return 0.0;
  const double* x = b + D.w_off[f];
  const int n = D.w_n[f];
  if (n <= 0 || !(E0 >= x[0]) || E0 > x[n - 1]) return 0.0;
  const double* y = x + n;
  if (E0 == x[n - 1]) return D.eps2 * y[n - 1];
  const int lo = find_interval(x, n, E0, a.lf, D.w_lnE0[f], D.w_inv_dlog[f]);
  const double slope = (y[lo + 1] - y[lo]) / (x[lo + 1] - x[lo]);
  return D.eps2 * (slope * (E0 - x[lo]) + y[lo]);
}

// numpy's sum of a short row: sequential below 8 terms, else eight partial
// sums combined pairwise and the remainder added in order.
__device__ inline double np_sum(const double* r, int n, int stride) {
  if (n < 8) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) s += r[i * stride];
    return s;
  }
  double s = ((r[0] + r[stride]) + (r[2 * stride] + r[3 * stride])) +
             ((r[4 * stride] + r[5 * stride]) + (r[6 * stride] + r[7 * stride]));
  for (int i = 8; i < n; ++i) s += r[i * stride];
  return s;
}

// Interaction energy of produce_bsm_particle (dark_shower.py:741-756): the
// saved energy Ei (the largest <= E0, clamped to the table), a bin drawn with
// probability proportional to its rate, shifted by E0 - Ei.  Returns false
// when the row's rates sum to zero (the reference returns None).
__device__ inline bool drate_energy(const PetiteDarkDesc& D, const double* b, int f, double E0, double u,
                                    double& E_int) {
  const int n = D.d_n[f];
  if (n <= 0) return false;
  const double* Es = b + D.d_off[f];
  const double* cnt = Es + n;
  const double* rows = cnt + n;
  int i;
  if (E0 < Es[0]) {
    i = 0;
  } else if (E0 > Es[n - 1]) {
    i = n - 1;
  } else {
    int lo = 0, hi = n;  // largest i with Es[i] <= E0
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (Es[mid] <= E0) lo = mid; else hi = mid;
    }
    i = lo;
  }
  const int c = (int)cnt[i];
  const double* row = rows + (int64_t)i * 2 * PETITE_DARK_DRATE_BINS;
  const double tot = np_sum(row + 1, c, 2);
  if (!(tot != 0.0) || c <= 0) return false;
  double cdf[PETITE_DARK_DRATE_BINS];
  double acc = 0.0;
  for (int k = 0; k < c; ++k) {
    acc += row[2 * k + 1] / tot;
    cdf[k] = acc;
  }
  int k = c - 1;
  for (int j = 0; j < c; ++j) {
    if (cdf[j] / acc > u) {
      k = j;
      break;
    }
  }
  E_int = row[2 * k] + (E0 - Es[i]);
  return true;
}

// A block's share of a counter: thread-wise `want`, the thread's slot returned
// (meaningless where !want), one atomic per block.  Per wave, the two counters'
// atomics of 1.4e6 records x 3 processes, served one after another, held the
// selection at 0.80 ms (0.33 ms with one per block; blocks of 1,024 threads
// spill and gain nothing).  Every thread of a block of 256 calls it; two calls
// in a row use different LDS.
template <typename C>
__device__ inline C block_slot(bool want, C* counter) {
  __shared__ unsigned int s_n[4];
  __shared__ C s_base;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned long long m = __ballot(want);
  if (lane == 0) s_n[wid] = (unsigned int)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned int t = s_n[0] + s_n[1] + s_n[2] + s_n[3];
    s_base = t ? atomicAdd(counter, (C)t) : (C)0;
  }
  __syncthreads();
  C o = s_base + (C)__popcll(m & ((1ull << lane) - 1ull));
  for (int w = 0; w < wid; ++w) o += (C)s_n[w];
  __syncthreads();  // read before the next call writes
  return o;
}

__global__ __launch_bounds__(256) void k_dark_select(DevTables T, PetiteDarkDesc D, const double* b, DevStore S,
                                                     int64_t first, int64_t n, uint64_t seed, Entries Q,
                                                     Requests R, unsigned long long* n_entries,
                                                     unsigned long long* stats) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = t < n;
  const int64_t i = first + t;
  int pid = 0;
  float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f), pf = p0;
  double wpar = 0.0;
  uint64_t sid = 0;
  if (live) {
    pid = S.pid[i];
    p0 = S.p0[i];
    pf = S.pf[i];
    wpar = (double)S.r0[i].w;
    sid = S.sid[i];
  }
  const double E0 = (double)p0.x;
  const WeightArgs wa = weight_args(T, pid, E0);
  unsigned long long n_zero = 0;
  for (int a = 0; a < D.n_active; ++a) {
    const int code = D.active[a];  // wave-uniform
    const double wg = live ? bsm_weight(T, D, b, pid, code, wa) : 0.0;
    const bool want = wg > 0.0;
    const unsigned long long slot = block_slot(want, n_entries);
    int state = S_NONE;
    int64_t e = -1;
    double E = 0.0;
    float nx = 0.f, ny = 0.f, nz = 0.f;
    if (want) {
      e = (int64_t)slot;
      const uint64_t dsid = derive_sid(seed, sid, (uint32_t)code, PURPOSE_DARK);
      const int f = (code == DARKCOMP) ? -1 : family_of(code, pid);
      const double m_part = pid_mass(pid);
      state = S_DIRECT;
      if (f >= 0) {
        const U4 w0 = draw_block(seed, dsid, 0, PURPOSE_INTERACT);
        double E_int = 0.0;
        if (!drate_energy(D, b, f, E0, u01d(w0.x), E_int)) {
          state = S_NONE;
          ++n_zero;
        } else {
          // scatter the initial momentum over the distance (m_lepton = m_e,
          // dark_shower.py:753-755), then lose E0 - E_int.  beta comes from the
          // on-shell |p| = sqrt(E0^2 - m^2): a float32 record's |p| can round to E0.
          const double dist = (E0 - E_int) / T.dEdx;
          const double px = p0.y, py = p0.z, pz = p0.w;
          const double pn = sqrt(px * px + py * py + pz * pz);
          const double pon = sqrt(fmax(E0 * E0 - m_part * m_part, 0.0));
          if (pn > 0.0 && pon > 0.0) {
            nx = (float)(px / pn);
            ny = (float)(py / pn);
            nz = (float)(pz / pn);
            mcs_rotate(T, nx, ny, nz, E0, pon, m_part, kMe, dist, w0.y, w0.z);
          }
          double Eu = E0 - (E0 - E_int);
          if (Eu <= m_part) Eu = m_part;
          if (!(sqrt(Eu * Eu - m_part * m_part) > 0.0)) nx = ny = nz = 0.0f;
          E = Eu;
        }
      } else {
        E = (double)pf.x;
        const double pn = sqrt((double)pf.y * pf.y + (double)pf.z * pf.z + (double)pf.w * pf.w);
        if (pn > 0.0) {
          nx = (float)(pf.y / pn);
          ny = (float)(pf.z / pn);
          nz = (float)(pf.w / pn);
        }
      }
      if (state == S_DIRECT) {
        const bool shortcut = (code == DARKANN && E <= D.E_res) || (code == DARKCOMP && E <= D.E_C);
        if (!shortcut) state = S_DRAW;
      }
      if (e < Q.cap) {
        Q.parent[e] = (int32_t)i;
        Q.flag[e] = code | (state << 8);
        Q.weight[e] = wg * wpar;
        Q.E[e] = E;
        Q.dir[e] = make_float4(nx, ny, nz, 0.0f);
        Q.dsid[e] = dsid;
      }
    }
    const bool drq = want && state == S_DRAW && e < Q.cap;
    const unsigned int rb = block_slot(drq, R.count + code);
    if (drq) {
      const int64_t k = (int64_t)code * R.cap + rb;
      R.slot[k] = (int32_t)e;
      R.E[k] = E;
    }
  }
  wave_stat(stats, 0, n_zero);
}

// draw_pe_sample (dark_shower.py:706-719): pe uniform in [0, 1 MeV) accepted
// against the 1s momentum density normalised at its maximum.
__device__ inline double electron_wf(double pe, double lam) {
  const double d = pe * pe + lam * lam;
  return 32.0 / kPi * (lam * lam * lam * lam * lam) * pe * pe / (d * d * d * d);
}
__device__ inline bool draw_pe(uint64_t seed, uint64_t dsid, double Zeff, double& pe) {
  const double lam = kAlpha * Zeff * kMe;
  const double c = electron_wf(lam / sqrt(3.0), lam);
  for (int k = 0; k < kPePairs / 2; ++k) {
    const U4 w = draw_block(seed, dsid, (uint32_t)k, PURPOSE_BOUND_E);
    double x = 1.0e-3 * u01d(w.x);
    if (u01d(w.y) < electron_wf(x, lam) / c) {
      pe = x;
      return true;
    }
    x = 1.0e-3 * u01d(w.z);
    if (u01d(w.w) < electron_wf(x, lam) / c) {
      pe = x;
      return true;
    }
  }
  return false;
}

// compton_fourvecs_boundelectron (kinematics.py:134-183): the vector.
__device__ inline V4 kin_compton_bound(double Eg, double mV, double ct, double Pe, double cte, double u_ph,
                                       double u_phie) {
  const double m = kMe;
  const double s = m * m + 2.0 * Eg * (sqrt(m * m + Pe * Pe) - cte * Pe);
  const double rs = sqrt(s);
  const double Ee = (s - mV * mV + m * m) / (2.0 * rs);
  const double EV = (s + mV * mV - m * m) / (2.0 * rs);
  const double pF = sqrt(Ee * Ee - m * m);
  const double bnum = sqrt(Eg * Eg + 2.0 * cte * Eg * Pe + Pe * Pe);
  const double b0 = bnum / (Eg + sqrt(m * m + Pe * Pe));
  const double g0 = 1.0 / sqrt(1.0 - b0 * b0);
  double sph, cph;
  sincos(2.0 * kPi * u_ph, &sph, &cph);
  const double st = sqrt(1.0 - ct * ct);
  const double vx = pF * st * sph, vy = pF * st * cph, vz = b0 * g0 * EV - g0 * pF * ct;
  const double ctz = (Eg + cte * Pe) / bnum;
  const double stz = sqrt(1.0 - ctz * ctz);
  double spe, cpe;
  sincos(2.0 * kPi * u_phie, &spe, &cpe);
  return V4{g0 * EV - b0 * g0 * pF * ct, ctz * cpe * vx - spe * vy + stz * cpe * vz,
            ctz * spe * vx + cpe * vy + stz * spe * vz, -stz * vx + ctz * vz};
}

// radiative_return_fourvecs (kinematics.py:267-299) with the boost of
// radiative_return.py:18-24 into the frame of the electron at rest.
__device__ inline V4 kin_radiative_return(double E, double u, double mV) {
  const double m = kMe;
  const double s = 2.0 * m * (m + E);
  const double beta = (2.0 * kAlpha / kPi) * (log(s / (m * m)) - 1.0);
  const double umax = pow(1.0 - mV * mV / s, beta / 2.0);
  const double x1 = 1.0 - pow(u * umax, 2.0 / beta);
  const double x2 = mV * mV / (x1 * s);
  const double rs = sqrt(s);
  const double E1 = x1 * rs / 2.0, E2 = x2 * rs / 2.0;
  const double v0 = E1 + E2, v3 = E1 - E2;
  // p = (rs/2, 0, 0, -sqrt(s/4 - m^2))
  const double p0 = rs / 2.0, p3 = -sqrt(s / 4.0 - m * m);
  const double rsq = sqrt(p0 * p0 - p3 * p3);
  const double w0 = (p0 * v0 - p3 * v3) / rsq;
  const double c1 = (v0 + w0) / (rsq + p0);
  return V4{w0, 0.0, 0.0, v3 - c1 * p3};
}

struct EmitOut {
  float4* p;
  float4* r;
  int32_t* parent;
  int32_t* meta;
};

__global__ __launch_bounds__(256) void k_dark_emit(DevTables T, PetiteDarkDesc D, DevStore S, Entries Q, int64_t n_e,
                                                   const float* x_res, const int32_t* trials_res, EmitOut O,
                                                   int64_t out_base, uint64_t seed, double* yield,
                                                   unsigned long long* stats) {
  double wsum[4] = {0.0, 0.0, 0.0, 0.0};
  unsigned long long n_vec = 0, n_pe_fail = 0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n_e; e += stride) {
    const int flag = Q.flag[e];
    const int code = flag & 0xFF;
    const int state = flag >> 8;
    const int32_t slot = Q.parent[e];
    double w = Q.weight[e];
    const double E = Q.E[e];
    const double mV = T.mV;
    bool ok = state != S_NONE;
    V4 v{0.0, 0.0, 0.0, 0.0};
    if (ok && state == S_DIRECT) {
      if (code == DARKANN) {
        v = V4{sqrt(E * E - kMe * kMe + mV * mV), 0.0, 0.0, sqrt(E * E - kMe * kMe)};
      } else {
        v = V4{sqrt(E * E + mV * mV), 0.0, 0.0, E};
      }
    } else if (ok) {
      ok = trials_res[e] > 0;
      if (ok) {
        const float* xs = x_res + 4 * e;
        const uint64_t dsid = Q.dsid[e];
        const U4 w0 = draw_block(seed, dsid, 0, PURPOSE_INTERACT);
        if (code == DARKCOMP) {
          const U4 w1 = draw_block(seed, dsid, 1, PURPOSE_INTERACT);
          double pe = 0.0;
          if (!draw_pe(seed, dsid, T.Zeff, pe)) {
            ok = false;
            ++n_pe_fail;
          } else {
            const double c0 = -1.0 + 2.0 * u01d(w1.x);
            const double s = kMe * kMe + 2.0 * E * (sqrt(kMe * kMe + pe * pe) - c0 * pe);
            const double Ee = (s - mV * mV + kMe * kMe) / (2.0 * sqrt(s));
            if (Ee < kMe) {
              v = V4{mV, 0.0, 0.0, 0.0};
              w = 0.0;
            } else {
              v = kin_compton_bound(E, mV, (double)xs[0], pe, c0, u01d(w0.w), u01d(w1.y));
            }
          }
        } else if (code == DARKANN) {
          v = kin_radiative_return(E, (double)xs[0], mV);
        } else {
          // l_to_lV_fourvecs (kinematics.py:43-68): the vector
          const double wv = (double)xs[0] * E;
          const double ct = 1.0 - pow(10.0, (double)xs[1]);
          const double k = sqrt(wv * wv - mV * mV);
          double sa, ca;
          sincos(2.0 * kPi * u01d(w0.w), &sa, &ca);
          const double st = sqrt(1.0 - ct * ct);
          v = V4{wv, k * ca * st, k * sa * st, k * ct};
        }
      }
    }
    float4 pv = make_float4(0.f, 0.f, 0.f, 0.f), rv = pv;
    if (ok) {
      const float4 d = Q.dir[e];
      double ox, oy, oz;
      frame_apply_d((double)d.x, (double)d.y, (double)d.z, v, ox, oy, oz);
      pv = make_float4((float)v.e, (float)ox, (float)oy, (float)oz);
      const float4 rf = S.rf[slot];
      rv = make_float4(rf.x, rf.y, rf.z, (float)w);
      ++n_vec;
#pragma unroll
      for (int k = 0; k < 4; ++k) wsum[k] += code - DARKBREM == k ? w : 0.0;
    }
    const int64_t o = out_base + e;
    O.p[o] = pv;
    O.r[o] = rv;
    O.parent[o] = slot;
    O.meta[o] = code | (ok ? 0x100 : 0);
  }
  // the yields and counts: one atomic per block and process (per wave they took
  // five sixths of the kernel: 0.42 ms, now 0.06, for 1.1e6 entries)
  __shared__ double s_y[4][4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int k = 0; k < 4; ++k) {
    double s = wsum[k];
    for (int off = 32; off > 0; off >>= 1) s += shfl_f64(s, lane ^ off);
    if (lane == 0) s_y[k][wid] = s;
  }
  const unsigned long long v[2] = {n_vec, n_pe_fail};
  unsigned long long* const dst[2] = {stats + 1, stats + 2};
  block_stat_add<2>(v, dst);  // (synchronises the block)
  if (threadIdx.x < 4) {
    const double t = (s_y[threadIdx.x][0] + s_y[threadIdx.x][1]) + (s_y[threadIdx.x][2] + s_y[threadIdx.x][3]);
    if (t != 0.0) unsafeAtomicAdd(yield + threadIdx.x, t);
  }
}

// ------------------------------------------------------ meson decays ------
constexpr int TWO_BODY = 12;  // TwoBody_BSMDecay: dark process code of the output entries

// TwoBody_BSMDecay of pi0 / eta / eta' records (dark_shower.py:633-640,
// 836-844): weight meson_w (1 - r^2)^3 with r = m_V / m_M, and the vector of
// the decay M -> gamma V, isotropic in the meson's rest frame (cos theta and
// phi uniform; particle.py:209-254 with V second) and boosted along the
// meson's final momentum with the boost_matrix of particle.py:187-207; the
// vector sits at the meson's end point.  Meson masses are the PDG values of
// mass_dict.  Entries are appended after out_base through *count; an entry
// beyond capacity is counted but not written.
// Slots, the yield sum and the vector count are aggregated per block (one
// atomic of each per 1024 records): per-wave atomics on the three shared
// addresses serialised the kernel (845 us for 4e6 records).
constexpr int kMesonBlock = 1024;
__global__ __launch_bounds__(kMesonBlock) void k_meson_decay(DevTables T, PetiteDarkDesc D, DevStore S, int64_t first,
                                                             int64_t n, uint64_t seed, EmitOut O, int64_t out_base,
                                                             int64_t capacity, unsigned long long* count,
                                                             double* yield, unsigned long long* stats) {
  __shared__ unsigned int wave_off[kMesonBlock / 64];
  __shared__ double wave_w[kMesonBlock / 64];
  __shared__ unsigned long long block_base;
  const int64_t i = first + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  bool have = false;
  double w = 0.0;
  float4 pv = make_float4(0.f, 0.f, 0.f, 0.f), rv = pv;
  if (i < first + n) {
    const int pid = S.pid[i];
    const int k = pid == 111 ? 0 : (pid == 221 ? 1 : (pid == 331 ? 2 : -1));
    const double mM = k == 0 ? 0.1349768 : (k == 1 ? 0.547862 : 0.95778);
    const double mV = T.mV;
    if (k >= 0 && D.meson_w[k] > 0.0 && mV / mM < 1.0) {
      const double r = mV / mM;
      const double q = 1.0 - r * r;
      const double wg = D.meson_w[k] * q * q * q;
      w = wg * (double)S.r0[i].w;
      const uint64_t dsid = derive_sid(seed, S.sid[i], (uint32_t)TWO_BODY, PURPOSE_DARK);
      const U4 u = draw_block(seed, dsid, 0, PURPOSE_INTERACT);
      const double ct = -1.0 + 2.0 * u01d(u.x);
      const double phi = 2.0 * kPi * u01d(u.y);
      const double st = sqrt(1.0 - ct * ct);
      const double E2 = (mM * mM + mV * mV) / (2.0 * mM);
      const double pF = (mM * mM - mV * mV) / (2.0 * mM);  // the photon's energy = |p| (m_gamma = 0)
      double sp, cp;
      sincos(phi, &sp, &cp);
      const double v[4] = {E2, pF * st * sp, pF * st * cp, pF * ct};
      const float4 pf = S.pf[i];
      const double E0 = pf.x, px = pf.y, py = pf.z, pz = pf.w;
      const double gam = E0 / mM;
      const double beta = gam == 1.0 ? 1.0 : sqrt(1.0 - 1.0 / (gam * gam));
      const double pm = sqrt(px * px + py * py + pz * pz);
      double o[4] = {v[0], v[1], v[2], v[3]};
      if (pm != 0.0) {
        const double b[3] = {beta * px / pm, beta * py / pm, beta * pz / pm};
        const double g1 = (gam - 1.0) / (beta * beta);
        const double bv = b[0] * v[1] + b[1] * v[2] + b[2] * v[3];
        o[0] = gam * v[0] + gam * bv;
        for (int a = 0; a < 3; ++a) o[a + 1] = gam * b[a] * v[0] + v[a + 1] + g1 * b[a] * bv;
      }
      pv = make_float4((float)o[0], (float)o[1], (float)o[2], (float)o[3]);
      const float4 rf = S.rf[i];
      rv = make_float4(rf.x, rf.y, rf.z, (float)w);
      have = true;
    }
  }
  const unsigned long long m = __ballot(have);
  double s = have ? w : 0.0;
  for (int off = 32; off > 0; off >>= 1) s += shfl_f64(s, lane ^ off);
  if (lane == 0) {
    wave_off[wave] = (unsigned int)__popcll(m);
    wave_w[wave] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int tot = 0;
    double sw = 0.0;
    for (int k = 0; k < kMesonBlock / 64; ++k) {
      const unsigned int c = wave_off[k];
      wave_off[k] = tot;  // exclusive prefix: the wave's first slot in the block
      tot += c;
      sw += wave_w[k];
    }
    block_base = tot ? atomicAdd(count, (unsigned long long)tot) : 0ull;
    if (tot) {
      unsafeAtomicAdd(yield + 4, sw);
      atomicAdd(stats + 1, (unsigned long long)tot);
    }
  }
  __syncthreads();
  if (have) {
    const int64_t o = out_base + (int64_t)(block_base + wave_off[wave]) + __popcll(m & ((1ull << lane) - 1ull));
    if (o < capacity) {
      O.p[o] = pv;
      O.r[o] = rv;
      O.parent[o] = (int32_t)i;
      O.meta[o] = TWO_BODY | 0x100;
    }
  }
}

// ------------------------------------------------------ m_V-continuous yield --
// Each mass point's sum over the record is a table lookup and (but for
// DarkAnn) an exponential per particle, in float64.  The record's energies and
// weights go to a list per species once, so that a wave works on one process;
// a block holds several points' sums in registers, and the grid's y dimension
// covers the rest, so that a particle's logarithms serve kYieldGroup points
// and a short record still fills the chip.  The blocks' sums go to rows of
// their own and one kernel adds those (atomics of every wave on the points'
// sums, all in four cache lines, were served one after another).  19e6 records
// x 32 points with gradients: 3.0 ms (interpolation 1.96, bound 0.75, lists
// 0.31); two scans of mixed species with unpacked tables took 10.6 ms.
constexpr int kYieldBatch = 32;   // points of a pass
constexpr int kYieldGroup = 8;     // points of a block of k_dark_yield
constexpr int kBoundGroup = 4;    // points of a block of k_bound_yield
constexpr int kYieldComp = 4;     // table of DarkComp beside the four weight families
constexpr int kYieldSpecies = 4;  // e-, e+, photons, mu-+
constexpr double kLn10 = 2.302585092994045684;

// One grid interval: x .. xn, the value at x and the slope.  The last node has
// xn = inf and slope 0.
struct alignas(32) YieldRow {
  double x, xn, y, slope;
};

// One process' table at one trained mass: a weight in E (the linear families)
// or log10 n sigma in log10 E (DarkComp).
struct YieldTable {
  double thr;       // lowest energy with a weight
  double x0, x1;    // grid ends
  double g0, inv;   // guess of the interval from ln E (log10 E for DarkComp); inv = 0: bisection
  double eps2, ln_eps2;
  int32_t n, off;   // rows
};

struct YieldTables {
  YieldTable t[PETITE_MAX_MASSES][kYieldComp + 1];
  const YieldRow* rows;
  int32_t n_mass;
};

// Mass points of one pass (ascending m_V): segment j[k] (trained masses j[k]
// and the next), t and dt/dm_V, and eps^2 for the bound-electron tables.
struct YieldPoints {
  int32_t n;
  int32_t j[kYieldBatch];
  double t[kYieldBatch];
  double dtdm[kYieldBatch];
  double eps2[kYieldBatch];
};

// The particles of one species: entry i at Ew[i] or, for the list that fills
// its array from the end, Ew[-i]; photons with log10 E and ln(n sigma_PP +
// n sigma_Comp) beside.
struct YieldList {
  const float2* Ew;
  const double2* ph;
  int32_t dir;
  const unsigned long long* count;  // on the device
};

// find_interval over rows.
template <typename Row>
__device__ inline int find_row(const Row* r, int n, double v, float guess_arg, double g0, double inv) {
  int lo;
  if (inv > 0.0) {
    lo = (int)((guess_arg - (float)g0) * (float)inv);
    lo = lo < 0 ? 0 : (lo > n - 1 ? n - 1 : lo);
    while (lo > 0 && r[lo].x > v) --lo;
    while (lo < n - 1 && r[lo].xn <= v) ++lo;
  } else {
    lo = 0;
    int hi = n;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (r[mid].x <= v) lo = mid; else hi = mid;
    }
  }
  return lo;
}

struct YieldArgs {
  double E0, l10, ln_den;  // (the last two of photons)
  float lf;
};

// Weight of one trained mass, as (w, ln w): GetBSMWeights with that mass's
// tables (dark_shower.py:595-647).  DarkComp's log-log table (fill -20) gives
// ln w = ln eps^2 - ln(n sigma_PP + n sigma_Comp) + ln 10 * L directly (w
// itself is formed only where the linear branch needs it; w = 1 marks it
// positive); the other families take the log of the interpolated weight.
template <bool COMP>
__device__ inline void yield_weight(const YieldTable& t, const YieldRow* rows, const YieldArgs& a, double& wv,
                                    double& lam) {
  wv = lam = 0.0;
  if (a.E0 < t.thr) return;
  const YieldRow* r = rows + t.off;
  if (COMP) {
    double L = -20.0;
    if (t.n > 0 && !(a.l10 < t.x0 || a.l10 > t.x1)) {
      const YieldRow R = r[find_row(r, t.n, a.l10, (float)a.l10, t.g0, t.inv)];
      L = R.slope * (a.l10 - R.x) + R.y;
    }
    wv = 1.0;
    lam = t.ln_eps2 - a.ln_den + kLn10 * L;
    return;
  }
  if (t.n <= 0 || !(a.E0 >= t.x0) || a.E0 > t.x1) return;
  const YieldRow R = r[find_row(r, t.n, a.E0, a.lf, t.g0, t.inv)];
  wv = t.eps2 * (R.slope * (a.E0 - R.x) + R.y);
  lam = wv > 0.0 ? log(wv) : 0.0;
}

// Bound-electron tables at one point's m_V: the interval weights and, in the
// derivative's terms, with u = x - x_lo and dots for d/dm_V of the nodes,
//   d/dm [y_lo + u (y_hi - y_lo) / (x_hi - x_lo)] = c0 + c1 u.
struct alignas(16) BoundRow {
  double x, xn, y, slope, c0, c1;
};

// Species list (0 e-, 1 e+, 2 photon, 3 mu-+; -1 other) of a record's pid.
__device__ inline int species_of(int pid) {
  switch (pid) {
    case 11: return 0;
    case -11: return 1;
    case 22: return 2;
    case 13:
    case -13: return 3;
    default: return -1;
  }
}

// The lists of the species in `mask`: e- from the front of Ew[0], e+ from its
// end, photons from the front of Ew[1], muons from its end (cap entries each).
// Each wave lists a run of kListRun x 64 consecutive records: a first look
// counts its entries, one atomic per block and list reserves the block's
// share, a second look writes them.
constexpr int kListRun = 16;
__global__ __launch_bounds__(256) void k_yield_lists(DevStore S, int64_t first, int64_t n, uint32_t mask, float2* Ew,
                                                     int64_t cap, unsigned long long* counts) {
  __shared__ unsigned int s_cnt[kYieldSpecies][4];
  __shared__ unsigned long long s_base[kYieldSpecies];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  constexpr int64_t kWaveRun = 64 * kListRun, kBlockRun = 4 * kWaveRun;
  for (int64_t b0 = (int64_t)blockIdx.x * kBlockRun; b0 < n; b0 += (int64_t)gridDim.x * kBlockRun) {
    const int64_t w0 = b0 + wid * kWaveRun;
    unsigned int c[kYieldSpecies] = {0u, 0u, 0u, 0u};
    for (int j = 0; j < kListRun; ++j) {
      const int64_t i = w0 + j * 64 + lane;
      const int sp = i < n ? species_of(S.pid[first + i]) : -1;
#pragma unroll
      for (int q = 0; q < kYieldSpecies; ++q) c[q] += (unsigned int)__popcll(__ballot(sp == q && ((mask >> q) & 1u)));
    }
    if (lane == 0)
      for (int q = 0; q < kYieldSpecies; ++q) s_cnt[q][wid] = c[q];
    __syncthreads();
    if (threadIdx.x < kYieldSpecies) {
      const int q = threadIdx.x;
      const unsigned int tot = s_cnt[q][0] + s_cnt[q][1] + s_cnt[q][2] + s_cnt[q][3];
      s_base[q] = tot ? atomicAdd(counts + q, (unsigned long long)tot) : 0ull;
    }
    __syncthreads();
    unsigned long long o[kYieldSpecies];
#pragma unroll
    for (int q = 0; q < kYieldSpecies; ++q) {
      o[q] = s_base[q];
      for (int w = 0; w < wid; ++w) o[q] += s_cnt[q][w];
    }
    for (int j = 0; j < kListRun; ++j) {
      const int64_t i = w0 + j * 64 + lane;
      const int sp = i < n ? species_of(S.pid[first + i]) : -1;
#pragma unroll
      for (int q = 0; q < kYieldSpecies; ++q) {
        const bool in = sp == q && ((mask >> q) & 1u);
        const unsigned long long m = __ballot(in);
        if (in) {
          const int64_t at = (int64_t)(o[q] + __popcll(m & below));
          float2* const A = Ew + (q >> 1) * cap;
          A[(q & 1) ? cap - 1 - at : at] = make_float2(S.p0[first + i].x, S.r0[first + i].w);
        }
        o[q] += (unsigned long long)__popcll(m);
      }
    }
    __syncthreads();  // s_cnt and s_base are read before the next run writes them
  }
}

// log10 E and the log of the total rate of the listed photons.
__global__ __launch_bounds__(256) void k_yield_photons(DevTables T, YieldList L, double2* out) {
  const int64_t n = (int64_t)*L.count, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const double E0 = (double)L.Ew[i].x;
    out[i] = make_double2(log10(E0), log(nsigma(T, PAIRPROD, E0) + nsigma(T, COMP, E0)));
  }
}

// The block's sums of its points k0 .. k0 + G - 1 into the block's row.
template <bool GRAD, int G>
__device__ inline void yield_row(const double* y, const double* dy, int k0, int n_pts, double* part) {
  __shared__ double s_sum[4][2 * G];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < G; ++k) {
    double a = y[k], b = GRAD ? dy[k] : 0.0;
    for (int off = 32; off > 0; off >>= 1) {
      a += shfl_f64(a, lane ^ off);
      if (GRAD) b += shfl_f64(b, lane ^ off);
    }
    if (lane == 0) {
      s_sum[wid][2 * k] = a;
      s_sum[wid][2 * k + 1] = b;
    }
  }
  __syncthreads();
  const int q = threadIdx.x;
  if (q < 2 * G && k0 + (q >> 1) < n_pts)
    part[(int64_t)blockIdx.x * (2 * kYieldBatch) + 2 * k0 + q] =
        (s_sum[0][q] + s_sum[1][q]) + (s_sum[2][q] + s_sum[3][q]);
}

// Sums over the rows of every kernel of a pass, added to the points' totals.
__global__ __launch_bounds__(256) void k_yield_sum(const double* part, int64_t rows, double* acc) {
  __shared__ double s_sum[256];
  const int q = blockIdx.x;  // 2 k: yield, 2 k + 1: derivative
  double s = 0.0;
  for (int64_t r = threadIdx.x; r < rows; r += 256) s += part[r * (2 * kYieldBatch) + q];
  s_sum[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s_sum[threadIdx.x] += s_sum[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) acc[q] += s_sum[0];
}

// A process' sums over one species: w W(m_k) and w dW/dm(m_k) (GRAD = false:
// the yield alone).  Between trained masses j and j+1 a particle's weight is
// interpolated geometrically, W = exp(ln w_j + t ln(w_j+1 / w_j)), where both
// are positive, linearly otherwise.  Points of one segment, and of the next,
// share the trained masses' weights.
template <bool GRAD, bool COMP>
__global__ __launch_bounds__(256) void k_dark_yield(const YieldTables* __restrict__ Yp, int fam, YieldList L,
                                                    YieldPoints P, double* __restrict__ part) {
  constexpr int G = kYieldGroup;
  const YieldTables& Y = *Yp;
  const YieldRow* const rows = Y.rows;
  const int k0 = blockIdx.y * G;
  double y[G], dy[G];
#pragma unroll
  for (int k = 0; k < G; ++k) y[k] = dy[k] = 0.0;
  const int64_t n = (int64_t)*L.count, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float2 Ew = L.Ew[L.dir * i];
    const double w = (double)Ew.y;
    YieldArgs a{};
    a.E0 = (double)Ew.x;
    if (COMP) {
      const double2 ph = L.ph[i];
      a.l10 = ph.x;
      a.ln_den = ph.y;
    } else {
      a.lf = __logf(Ew.x);
    }
    double lo = 0.0, hi = 0.0, llo = 0.0, lhi = 0.0;
    int jc = -2;
#pragma unroll
    for (int k = 0; k < G; ++k) {
      if (k0 + k >= P.n) break;
      const int j = P.j[k0 + k];
      if (j != jc) {
        if (j == jc + 1) {
          lo = hi;
          llo = lhi;
        } else {
          yield_weight<COMP>(Y.t[j][fam], rows, a, lo, llo);
        }
        hi = lo;
        lhi = llo;
        if (j + 1 < Y.n_mass) yield_weight<COMP>(Y.t[j + 1][fam], rows, a, hi, lhi);
        jc = j;
      }
      const double t = P.t[k0 + k];
      double W, dW;
      if (lo > 0.0 && hi > 0.0) {
        const double r = lhi - llo;
        W = exp(llo + t * r);
        dW = GRAD ? W * r * P.dtdm[k0 + k] : 0.0;
      } else {
        const double l = COMP ? (lo > 0.0 ? exp(llo) : 0.0) : lo;
        const double h = COMP ? (hi > 0.0 ? exp(lhi) : 0.0) : hi;
        W = l + t * (h - l);
        dW = GRAD ? (h - l) * P.dtdm[k0 + k] : 0.0;
      }
      y[k] += w * W;
      if (GRAD) dy[k] += w * dW;
    }
  }
  yield_row<GRAD, G>(y, dy, k0, P.n, part);
}

// Rows of the bound-electron tables of point k from slot k * nv (m_k) and the
// node derivatives in slot k * nv + 1 (quad::k_bound_deriv; nv = 1: none):
// DarkAnn's W in E, then DarkComp's log10 n sigma in log10 E.
__global__ __launch_bounds__(256) void k_bound_rows(const double* tab, int32_t stride, int32_t nv, BoundRow* rows) {
  constexpr int n = quad::kBoundGrid;
  const int i = threadIdx.x, comp = blockIdx.y;
  if (i >= n) return;
  const double* x = tab + (int64_t)blockIdx.x * nv * stride + (comp ? 4 * n : 0);
  const double* y = x + (comp ? n : 3 * n);
  const double* dx = x + stride;
  const double* dy = y + stride;
  const bool last = i == n - 1;
  BoundRow R{x[i], last ? (double)INFINITY : x[i + 1], y[i], 0.0, nv == 3 ? dy[i] : 0.0, 0.0};
  if (!last) {
    const double inv = 1.0 / (R.xn - R.x), dv = y[i + 1] - R.y;
    R.slope = dv / (R.xn - R.x);
    if (nv == 3) {
      R.c0 = dy[i] - dv * dx[i] * inv;
      R.c1 = inv * ((dy[i + 1] - dy[i]) - dv * (dx[i + 1] - dx[i]) * inv);
    }
  }
  rows[((int64_t)blockIdx.x * 2 + comp) * n + i] = R;
}

// The bound-electron processes' part of the yield (DarkAnn of positrons,
// DarkComp of photons) from the tables at the points' masses, held in LDS:
// W and dW/dm_V are the rows' interpolants, in log10 space for DarkComp (W =
// eps^2 10^L / den, dW = W ln 10 dL).  Below the thresholds, and for DarkAnn
// outside the grid, W = dW = 0; outside DarkComp's grid L = -20.
template <bool GRAD, bool COMP>
__global__ __launch_bounds__(256) void k_bound_yield(const quad::BoundSlot* __restrict__ slot,
                                                     const BoundRow* __restrict__ rows, int32_t nv, double min_photon,
                                                     YieldList L, YieldPoints P, double* __restrict__ part) {
  constexpr int G = kBoundGroup, N = quad::kBoundGrid;
  __shared__ BoundRow s_row[G][N];
  const int k0 = blockIdx.y * G;
  double thr[G], g0[G], inv[G], y[G], dy[G];
#pragma unroll
  for (int k = 0; k < G; ++k) {
    y[k] = dy[k] = thr[k] = g0[k] = inv[k] = 0.0;
    if (k0 + k >= P.n) continue;
    const quad::BoundSlot& S = slot[(k0 + k) * nv];
    thr[k] = COMP ? fmax(S.min_comp, min_photon) : S.min_ann;
    g0[k] = COMP ? S.l0c : S.lnEa0;
    inv[k] = COMP ? S.inv_dlc : S.inv_dln_a;
    for (int i = threadIdx.x; i < N; i += 256) s_row[k][i] = rows[((int64_t)(k0 + k) * 2 + (COMP ? 1 : 0)) * N + i];
  }
  __syncthreads();
  const int64_t n = (int64_t)*L.count, stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float2 Ew = L.Ew[L.dir * i];
    const double E0 = (double)Ew.x, w = (double)Ew.y;
    double v = E0, ln_den = 0.0;
    if (COMP) {
      const double2 ph = L.ph[i];
      v = ph.x;
      ln_den = ph.y;
    }
    const float g = COMP ? (float)v : __logf(Ew.x);
#pragma unroll
    for (int k = 0; k < G; ++k) {
      if (k0 + k >= P.n) break;
      const BoundRow* const r = s_row[k];
      if (E0 < thr[k]) continue;
      const bool out = COMP ? (v < r[0].x || v > r[N - 1].x) : !(v >= r[0].x && v <= r[N - 1].x);
      if (!COMP && out) continue;
      double val = -20.0, d = 0.0;
      if (!out) {
        const int lo = find_row(r, N, v, g, g0[k], inv[k]);
        const double u = v - r[lo].x;
        val = r[lo].slope * u + r[lo].y;
        if (GRAD) d = r[lo].c0 + r[lo].c1 * u;
      }
      if (COMP) {
        val = exp(kLn10 * val - ln_den);
        d = val * kLn10 * d;
      }
      y[k] += w * val;
      if (GRAD) dy[k] += w * d;
    }
  }
#pragma unroll
  for (int k = 0; k < G; ++k) {
    const double e2 = k0 + k < P.n ? P.eps2[k0 + k] : 0.0;
    y[k] *= e2;
    dy[k] *= e2;
  }
  yield_row<GRAD, G>(y, dy, k0, P.n, part);
}

}  // namespace dark
