// spectrum.hip -- gfx950 kernels and C ABI for the spectral radiation integral.
//
// What is computed (per spectral point g and particle p, reference semantics):
//   far : F_p(g) = sum_s A_s(n) exp(i omega (t_s - n.x_s))             kernel_farfield.cl:59-97
//         A_s(n) = c1 (n - bbar_s) - c2 a_s,  c2 = 1/(1 - n.bbar_s),
//         c1 = (n.a_s) c2^2,  bbar_s = (b_s + b_{s+1})/2,  a_s = (b_{s+1} - b_s)/dt
//   near: F_p(g) = sum_s [n/R^2 + i omega (b_s - n)/R] exp(i omega (t_s + R_s))
//                                                                      kernel_nearfield.cl:58-92
//   a step contributes only if |phase_s - phase_{s-1}| < pi (phase_{-1} = 0),
//   kernel_farfield.cl:69-72; snapshots add w dt^2 |F|^2 (or sqrt(w) dt F for
//   the coherent outputs) when it_start + it + 2 hits itSnaps[iSnap],
//   kernel_farfield.cl:100-106.
//
// How it is laid out on gfx950:
//   * A block owns one direction (far) or screen point (near) and a run of
//     T*M omegas: each of the T = 64*waves threads holds M omegas (the k-th
//     omega of thread t is chunk*T*M + k*T + t', t' = t with the 64-omega runs
//     dealt to the waves in an order rotated by the tile index, so every
//     output access of a wave covers 64 consecutive doubles).  A tile index
//     also carries a particle slice q; the slices of one tile are summed in
//     slice order by a second kernel.
//   * A pre-pass (k_step_prep) computes the direction-independent data of
//     every sample once per call: far a and the mean velocity of the interval,
//     near the velocity.
//   * The block walks its particles (CSR) and their steps in tiles of T steps.
//     Stage: thread t computes, in FP64, everything of step t0+t that does not
//     depend on omega -- tau = t - n.x (far) or t + |P - x| (near) and the
//     amplitude words -- and stores it in LDS.  Sweep: every thread reads
//     the tile back with broadcast LDS reads and accumulates its omegas.  The
//     omega-independent work is paid once per (point, step) and shared by the
//     block's T*M omegas.
//   * Amplitude words: far A.e_theta, A.e_phi (A is perpendicular to n; the
//     record rebuilds x, y, z); near v1 = (b - n)/R and v2 = n/R^2.
//   * Sweeps:
//       F64 direct    FP64 phase omega*tau, |dphase| < pi filter exactly as the
//                     reference forms it, FP64 sin/cos (pi/128 reduction, an
//                     LDS table of sin/cos(i pi/128), short polynomials), FP64
//                     sums; 1 or 2 omegas per thread.
//       split direct  (grids without a constant step) FP64 phase in
//                     revolutions -> v_fract_f64 -> v_sin_f32/v_cos_f32, the
//                     filter in its threshold form |omega|/2pi < 1/(2|dtau|),
//                     FP32 sums with a Kahan fold per swept segment.
//     Split spectra on linear grids run another kernel, factored.h: there the
//     sums over the steps are matrix products of a few sines per step.
//   * Records: with one snapshot and one output each thread sums its points
//     over the block's particles in LDS and writes once; otherwise outputs are
//     read-modify-written per particle record by the one thread that owns
//     them.  No atomics anywhere, so results do not depend on scheduling.
//   * An internal output kind writes each particle's complex field separately
//     (the adjoint's forward pass).
//
// All code here is compiled with -ffp-contract=off: the FP64 stage reproduces
// the reference's expression order term by term, and fused multiply-adds are
// written out explicitly where they are wanted (the sweep accumulations).
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <math.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "synchrad_amd.h"
#include "common.h"
#include "tile_params.h"
#include "factored.h"

namespace sr {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

const char *last_error() { return g_err; }

}  // namespace sr

namespace {

using namespace sr;

enum { SWEEP_DIRECT = 0, SWEEP_REC = 1 };

template <int V>
using IC = std::integral_constant<int, V>;

// ---------------------------------------------------------------------------
// the tile kernel
// ---------------------------------------------------------------------------
// Dynamic LDS of the split sweeps: the Kahan sum S and compensation C of every
// thread's NC*M accumulators, [2][NC*M][T] floats; a thread only ever touches
// its own column, so no barrier guards them.
template <int MODE, int M>
constexpr size_t kahan_lds_bytes(int T) {
  return (size_t)2 * (MODE == SR_MODE_FAR ? 4 : 6) * M * T * sizeof(float);
}

__device__ __forceinline__ float fmx(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmx(double a, double b, double c) { return fma(a, b, c); }

// One step's contribution to one frequency's sums acc[NC], from the step's
// amplitude words a[NA] and e^{i phase} = cn + i sn.  Far: [A cos | A sin]
// with NA words each (split: A.e_theta, A.e_phi; FP64: A_x, A_y, A_z).
// Near: the field itself, F_c += (v2_c + i omega v1_c) e^{i phase} with
// a = [v1 (3) | v2 (3)] and w = omega (kernel_nearfield.cl:87-91: c1 =
// omega v1, c2 = v2), as [Re F (3) | Im F (3)].
template <int MODE, int NA, typename X>
__device__ __forceinline__ void accumulate(X *acc, const X *a, X cn, X sn, X w) {
  if constexpr (MODE == SR_MODE_FAR) {
#pragma unroll
    for (int c = 0; c < NA; c++) {
      acc[c] = fmx(a[c], cn, acc[c]);
      acc[NA + c] = fmx(a[c], sn, acc[NA + c]);
    }
  } else {
    const X wc = w * cn, ws = w * sn;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      acc[c] = fmx(a[3 + c], cn, fmx(-a[c], ws, acc[c]));
      acc[3 + c] = fmx(a[3 + c], sn, fmx(a[c], wc, acc[3 + c]));
    }
  }
}
// The split sweeps' register partials of one frequency.  Far: as accumulate.
// Near: the two amplitude parts kept apart, [v2 cos | v2 sin | v1 sin | v1 cos]
// (12 sums, 12 FMAs per step and no multiplication by omega); the Kahan fold
// forms the field's [Re F | Im F] = [v2 cos - omega v1 sin | v2 sin + omega
// v1 cos] from them once per tile.
template <int MODE, int NA>
__device__ __forceinline__ void split_acc(float *acc, const float *a, float cn, float sn) {
  if constexpr (MODE == SR_MODE_FAR) {
#pragma unroll
    for (int c = 0; c < NA; c++) {
      acc[c] = fmx(a[c], cn, acc[c]);
      acc[NA + c] = fmx(a[c], sn, acc[NA + c]);
    }
  } else {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      acc[c] = fmx(a[3 + c], cn, acc[c]);
      acc[3 + c] = fmx(a[3 + c], sn, acc[3 + c]);
      acc[6 + c] = fmx(a[c], sn, acc[6 + c]);
      acc[9 + c] = fmx(a[c], cn, acc[9 + c]);
    }
  }
}

// Dynamic LDS after the Kahan state: the per-thread particle sums of the
// single output when KParams::acc_lds is set, [M][T] doubles.
template <int M>
constexpr size_t acc_lds_bytes(int T) {
  return (size_t)M * T * sizeof(double);
}

// amplitude words per staged step: far A.e_theta, A.e_phi; near v1 and v2
// (three components each)
template <int MODE, int PREC>
constexpr int amp_words() {
  return MODE == SR_MODE_FAR ? 2 : 6;
}

// Dynamic LDS before the Kahan state: one tile of T staged steps -- tau
// (double), the split threshold (double) and the amplitude words -- sized by the
// launched block, so that one-wave blocks do not hold a 256-step tile's LDS.
template <int MODE, int PREC>
constexpr size_t stage_lds_bytes(int T) {
  constexpr bool split = PREC == SR_PREC_SPLIT;
  return (size_t)T * (sizeof(double) + (split ? sizeof(double) : 0) +
                      amp_words<MODE, PREC>() * (split ? sizeof(float) : sizeof(double)));
}

// rows of a [n][T] LDS array: rows[c][j]
template <typename X>
struct LdsRows {
  X *base;
  int T;
  __device__ X *operator[](int c) const { return base + c * T; }
};

// Register budget per variant, as the minimum number of waves each SIMD must
// be able to hold: the split sweep keeps its Kahan state in LDS, so its
// registers hold the partial sums of M omegas plus one staged step group.
#ifndef SR_WAVE_ROTATE
#define SR_WAVE_ROTATE 1
#endif
#ifndef SR_DIRECT_WAVES
#define SR_DIRECT_WAVES 3
#endif
// split direct sweep in 4-step groups
#ifndef SR_DIRECT_GROUP
#define SR_DIRECT_GROUP 1
#endif
#ifndef SR_F64_WAVES
#define SR_F64_WAVES 4
#endif
// steps per iteration of the direct sweep's step loop (FP64 and the split tail)
#ifndef SR_F64_UNROLL
#define SR_F64_UNROLL 4
#endif
#ifndef SR_F64_WAVES2
#define SR_F64_WAVES2 4
#endif
#ifndef SR_F64_NEAR_WAVES2
#define SR_F64_NEAR_WAVES2 SR_F64_WAVES2
#endif
template <int MODE, int PREC, int M>
struct WavesPerEU {
  static constexpr int value =
      (PREC == SR_PREC_F64) ? (M == 2 ? (MODE == SR_MODE_NEAR ? SR_F64_NEAR_WAVES2 : SR_F64_WAVES2)
                                      : SR_F64_WAVES)
                            : (M >= 4 ? 2 : SR_DIRECT_WAVES);
};

// PRE: the step data come from the pre-pass records (batch calls); without
// them (the per-particle and no-allocation calls) the stage forms them from u.
// RECORDS: the sweep of a staged tile is split at the snapshot records in it, for launches
// with several and one group of threads; else the steps up to a record are staged by
// themselves, in the groups' parts (with one record the shorter code: 120 tracks of up to
// 20000 steps on a 256 x 32 x 32 log grid 36.7 ms against 37.1, FP64 24 x 4000 17.0 against
// 17.4)
template <int MODE, int PREC, int M, bool PRE, bool RECORDS>
__global__ void __launch_bounds__(PREC == SR_PREC_F64 && !RECORDS ? kWave * kMaxParts : kMaxT)
__attribute__((amdgpu_waves_per_eu(WavesPerEU<MODE, PREC, M>::value)))
k_spectrum(const KParams p) {
  static_assert(PREC == SR_PREC_SPLIT || M <= 2, "the FP64 sweep holds one or two omegas per thread");
  using Amp = typename std::conditional<PREC == SR_PREC_SPLIT, float, double>::type;
  constexpr bool kSplit = (PREC == SR_PREC_SPLIT);
  // amplitude words per step.  Far: A is perpendicular to n
  // (n.A = c1 (1 - n.bbar) - c2 n.a = 0 with c1 = (n.a) c2^2), so it is kept
  // as its two components on e_theta, e_phi (the reference sums A_x, A_y, A_z;
  // the two agree to rounding).  Near: v1 = (b - n)/R and v2 = n/R^2.
  constexpr int NA = amp_words<MODE, PREC>();
  constexpr int NC = (MODE == SR_MODE_FAR) ? 2 * NA : 6;   // real accumulators per omega
  constexpr int NP = (MODE == SR_MODE_FAR) ? NC : 12;      // split register partials per omega
  constexpr bool kParts = !kSplit && !RECORDS;             // several groups of threads
  constexpr int kMaxW = kParts ? kMaxParts : kMaxT / kWave;   // waves per block

  extern __shared__ __align__(16) char s_dyn_raw[];
  // FP64 sin/cos table (sincos_table) and the largest |omega| of the grid
  constexpr bool kTab = !kSplit && (SR_F64_TABLE != 0);
  __shared__ double2 s_sct[kTab ? kSinCosTab : 1];
  __shared__ double s_wmax[kTab ? kMaxW : 1];
  __shared__ int s_vote[kMaxW];   // per-wave votes of a block-wide any/all

  // the block's groups of T threads each hold the tile's omegas and sweep a part of
  // every track; their sums meet at the records
  const int P = kParts ? p.parts : 1;
  const int T = kParts ? (int)blockDim.x / P : (int)blockDim.x;
  const int grp = kParts ? uni((int)threadIdx.x / T) : 0;
  const int tid = (int)threadIdx.x - grp * T;
  const int W = T / kWave;
  const int wv = uni(tid / kWave);   // wave-uniform: its derived indices stay scalar
  const int lane = tid % kWave;
  // FP64: a tile whose |tau| * om_abs_max reaches kTabMaxPhase / 2 takes the
  // sin/cos table's wide-phase form
  double om_abs_max = 0.0;
  if (kTab) {
    for (int i = threadIdx.x; i < kSinCosTab; i += blockDim.x) {
      double sv, cv;
      sincospi((double)i / (kSinCosTab / 2), &sv, &cv);
      s_sct[i] = make_double2(sv, cv);
    }
    double m = 0.0;
    for (int64_t i = threadIdx.x; i < (int64_t)p.n_omega; i += blockDim.x) m = fmax(m, fabs(p.omega[i]));
    for (int o = kWave / 2; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if (lane == 0) s_wmax[grp * W + wv] = m;
    __syncthreads();
    for (int w = 0; w < P * W; w++) om_abs_max = fmax(om_abs_max, s_wmax[w]);
  }
  // dynamic LDS: the groups' staged tiles (s_tau[T], s_thr[T] (split), s_amp[NA][T]),
  // then the Kahan state (split), the particle sums, and the groups' sums of one
  // amplitude word on their way to the first group
  double *const s_tau = (double *)(s_dyn_raw + grp * stage_lds_bytes<MODE, PREC>(T));
  double *const s_thr = s_tau + T;
  const LdsRows<Amp> s_amp{(Amp *)(s_tau + (kSplit ? 2 : 1) * T), T};
  float *const s_dyn = (float *)(s_dyn_raw + P * stage_lds_bytes<MODE, PREC>(T));
  float *const s_ks = s_dyn + tid;                       // S[c*M+k] at s_ks[(c*M+k)*T]
  float *const s_kc = s_dyn + (size_t)NC * M * T + tid;  // C likewise
  // particle sums of the single output, k-th omega at s_acc[k*T]
  double *const s_acc = (double *)((char *)s_dyn + (kSplit ? kahan_lds_bytes<MODE, M>(T) : 0)) + tid;
  double *const s_sum = s_acc + (p.acc_lds ? M * T : 0);   // [P - 1][M][T]
  const double dt = p.dt;
  const double dtInv = 1.0 / dt;
  const bool spheric = (p.comp == SR_COMP_SPHERIC || p.comp == SR_COMP_SPHERIC_COMPLEX);

  for (int64_t ti = blockIdx.x; ti < p.n_tiles; ti += gridDim.x) {
    const uint32_t tile = p.tile_order ? (uint32_t)p.tile_order[ti] : (uint32_t)ti;
    const uint32_t rest = udiv(tile, p.div_chunks);
    const uint32_t chunk = tile - rest * p.n_chunks;
    const uint32_t qs = udiv(rest, p.div_dir);
    const uint32_t dir = rest - qs * p.n_dir;
    const int q = (int)qs;
    const uint32_t iPhi = udiv(dir, p.div_theta);
    const uint32_t iTh = dir - iPhi * p.n_theta;

    // geometry of the block's point (kernel_farfield.cl:40-42, 384-387;
    // kernel_nearfield.cl:40-42): far n, e_theta, e_phi; near the screen point
    // P.  Formed where it is used (from the block's uniform axis values, scalar
    // loads) rather than held in registers through the sweep.
    // (near: the screen point is held, which measured fewer spilled registers
    // in the FP64 near-field sweeps)
    struct Geom {
      double gx, gy, gz, thx, thy, thz, phx, phy;
    };
    double ngx = 0.0, ngy = 0.0, ngz = 0.0;
    if (MODE == SR_MODE_NEAR) {
      // the block's screen point is wave-uniform: kept in scalar registers
      const double r = p.radius[iTh];
      if (p.screen_y) {
        ngx = unid(r);
        ngy = unid(p.screen_y[iPhi]);
      } else {
        ngx = unid(r * p.cos_p[iPhi]);
        ngy = unid(r * p.sin_p[iPhi]);
      }
      ngz = p.l_screen;
    }
    auto geom = [&]() {
      Geom q;
      if (MODE == SR_MODE_FAR) {
        const double st = p.sin_t[iTh], ct = p.cos_t[iTh];
        const double sp = p.sin_p[iPhi], cp = p.cos_p[iPhi];
        q.gx = st * cp; q.gy = st * sp; q.gz = ct;
        q.thx = ct * cp; q.thy = ct * sp; q.thz = -st;
        q.phx = -sp; q.phy = cp;
      } else {
        q.gx = ngx; q.gy = ngy; q.gz = ngz;
        q.thx = q.thy = q.thz = q.phx = q.phy = 0.0;
      }
      return q;
    };

    // the block's omegas are dealt to its waves in 64-omega runs; the low runs
    // keep the most steps, so the run -> wave assignment is rotated by the tile
    // index to spread the heavy waves of co-resident blocks over the SIMDs
    const int vw = SR_WAVE_ROTATE ? (int)((wv + tile) & (uint32_t)(W - 1)) : wv;   // W is 1, 2 or 4
    // the omega index of the thread's k-th omega: lane of run k*W + vw
    auto omega_slot = [&](int k) { return (int)(chunk * T * M + (k * W + vw) * kWave + lane); };
    int wi[M];
    bool valid[M];
    double om[M];
#pragma unroll
    for (int k = 0; k < M; k++) {
      wi[k] = omega_slot(k);
      valid[k] = wi[k] < (int)p.n_omega;
      om[k] = valid[k] ? p.omega[wi[k]] : 0.0;
    }
    double om_rev[M];
    float omf[M];   // omega of the near field's v1 term (far: unused)
#pragma unroll
    for (int k = 0; k < M; k++) {
      om_rev[k] = om[k] * kInv2Pi;
      omf[k] = (float)om[k];
    }
    bool tile_wide = false;   // FP64: the tile's phases may reach kTabMaxPhase / 2
    // output c of this tile (slices: the slice's partial spectra), formed where it is written
    auto dst = [&](int c) -> double * {
      return (p.slices > 1 && p.part_stride == 0)
                 ? p.scratch + ((int64_t)q * p.n_out + c) * p.n_grid * p.n_snaps
                 : p.out[c];
    };

    if (late_s(p.acc_lds) && grp == 0) {
#pragma unroll
      for (int k = 0; k < M; k++) s_acc[k * T] = 0.0;
    }
    const int64_t p_lo = p.slice_lo[q], p_hi = p.slice_lo[q + 1];
    for (int64_t ip = p_lo; ip < p_hi; ip++) {
      const Particle pt = load_particle(p, ip);
      if (pt.n <= 0) continue;
      const int64_t n_act = min(pt.n - 1, (int64_t)pt.ite - 1);
      const double wpdt2 = pt.w * dt * dt;
      const double wpdt = sqrt(pt.w) * dt;

      SnapCursor cur;
      cur.init(pt, p.n_snaps);

      // F64: running sums fs; split: segment partials ps (registers), Kahan
      // sum and compensation in LDS
      double prev[M];
      double fs[M][NC];
      float ps[M][NP];
#pragma unroll
      for (int k = 0; k < M; k++) {
        prev[k] = 0.0;
#pragma unroll
        for (int c = 0; c < NC; c++) fs[k][c] = 0.0;
#pragma unroll
        for (int c = 0; c < NP; c++) ps[k][c] = 0.f;
      }
      if (kSplit) {
#pragma unroll
        for (int i = 0; i < NC * M; i++) {
          s_ks[i * T] = 0.f;
          s_kc[i * T] = 0.f;
        }
      }

      // adds this particle's snapshot value into the outputs the thread owns.
      // Records are rare; the split sweeps walk their omegas one at a time
      // (not unrolled, everything re-derived from k) so that the record code
      // does not set the kernel's register budget.
      // one omega's record: F are its sums (FP64), omk its 2 pi omega
      auto emit_k = [&](uint32_t slot, int k, int wk, const double *F, double omk) {
        double re[3], im[3];
        if constexpr (MODE == SR_MODE_FAR) {
          // F = F_theta e_theta + F_phi e_phi (spheric, kernel_farfield.cl:442-445:
          // the radial part n.F is 0, as n.A is)
          if (spheric) {
            re[0] = 0.0; re[1] = F[0]; re[2] = F[1];
            im[0] = 0.0; im[1] = F[2]; im[2] = F[3];
          } else {
            const Geom q = geom();
            re[0] = F[0] * q.thx + F[1] * q.phx; re[1] = F[0] * q.thy + F[1] * q.phy; re[2] = F[0] * q.thz;
            im[0] = F[2] * q.thx + F[3] * q.phx; im[1] = F[2] * q.thy + F[3] * q.phy; im[2] = F[2] * q.thz;
          }
        } else {
          // near: the sums are the field, [Re F (3) | Im F (3)]
          (void)omk;
#pragma unroll
          for (int c = 0; c < 3; c++) {
            re[c] = F[c];
            im[c] = F[3 + c];
          }
        }
        double v[kMaxOut];
        switch (p.comp) {
          case kCompField:
#pragma unroll
            for (int c = 0; c < 3; c++) {
              v[2 * c] = re[c];
              v[2 * c + 1] = im[c];
            }
            break;
          case SR_COMP_TOTAL:
            v[0] = wpdt2 * ((re[0] * re[0] + re[1] * re[1] + re[2] * re[2]) +
                            (im[0] * im[0] + im[1] * im[1] + im[2] * im[2]));
            break;
          case SR_COMP_CARTESIAN:
          case SR_COMP_SPHERIC:
#pragma unroll
            for (int c = 0; c < 3; c++) v[c] = wpdt2 * (re[c] * re[c] + im[c] * im[c]);
            break;
          default: {
            const double ff = (MODE == SR_MODE_FAR && p.comp == SR_COMP_CARTESIAN_COMPLEX)
                                  ? p.form_factor[wk] : 1.0;
#pragma unroll
            for (int c = 0; c < 3; c++) {
              v[2 * c] = wpdt * (ff * re[c]);
              v[2 * c + 1] = wpdt * (ff * im[c]);
            }
          }
        }
        if (late_s(p.acc_lds)) {
          s_acc[k * T] += v[0];
        } else {
          const int64_t g = (int64_t)slot * p.n_grid + (int64_t)dir * p.n_omega + late(wk) +
                            (ip - p.part_base) * p.part_stride;
#pragma unroll
          for (int c = 0; c < kMaxOut; c++)
            if (c < p.n_out) dst(c)[g] += v[c];
        }
      };
      auto emit = [&](uint32_t slot) {
        if constexpr (kSplit) {
#pragma unroll 1
          for (int k = 0; k < M; k++) {
            const int wk = omega_slot(k);
            if (wk >= (int)p.n_omega) continue;
            double F[NC];
#pragma unroll
            for (int c = 0; c < NC; c++)
              F[c] = (double)s_ks[(c * M + k) * T] - (double)s_kc[(c * M + k) * T];
            emit_k(slot, k, wk, F, p.omega[wk]);
          }
        } else {
          // FP64: the sums live in registers, so the loop is unrolled
#pragma unroll
          for (int k = 0; k < M; k++)
            if (valid[k]) emit_k(slot, k, wi[k], fs[k], om[k]);
        }
      };

      // one staged step of the direct sweeps; WIDE (FP64): the tile's phases
      // may reach the sin/cos table's limit
      auto direct_step = [&](int j, auto Wc) {
        const double tau = s_tau[j];
        const double thr = kSplit ? s_thr[j] : 0.0;
        Amp a[NA];
#pragma unroll
        for (int c = 0; c < NA; c++) a[c] = s_amp[c][j];
#pragma unroll
        for (int k = 0; k < M; k++) {
          // FP64: phase in radians and the reference's exact test
          // |phase_s - phase_{s-1}| < pi.  Split: phase in revolutions
          // (omega/2pi precomputed) and the same inequality in its
          // threshold form |omega|/2pi < thr_s, staged per step; the two
          // can disagree only within rounding of the boundary.
          const double ph = (kSplit ? om_rev[k] : om[k]) * tau;
          bool act;
          if (kSplit) {
            act = valid[k] && (fabs(om_rev[k]) < thr);
          } else {
            const double d = ph - prev[k];
            prev[k] = ph;
            act = valid[k] && (fabs(d) < kPi);
          }
          if (act) {
            if (kSplit) {
              float sn, cn;
              sincos_rev(ph, &sn, &cn);
              float af[NA];
#pragma unroll
              for (int c = 0; c < NA; c++) af[c] = (float)a[c];
              split_acc<MODE, NA>(ps[k], af, cn, sn);
            } else {
              double sn, cn;
              if (kTab)
                sincos_table(ph, s_sct, decltype(Wc)::value != 0, &sn, &cn);
              else
                sincos_reduced(ph, &sn, &cn);
              double ad[NA];
#pragma unroll
              for (int c = 0; c < NA; c++) ad[c] = (double)a[c];
              accumulate<MODE, NA>(fs[k], ad, cn, sn, om[k]);
            }
          }
        }
      };
      // steps [j, jend) of the direct sweep.  Split: single steps up to a
      // multiple of 4, then groups of 4 read with 16-byte LDS reads (each
      // frequency still skipped where the filter rejects it), then the tail
      auto direct_sweep = [&](int &j, int jend) {
        if constexpr (kSplit && SR_DIRECT_GROUP) {
          const int jg = min(jend, (j + 3) & ~3);
          for (; j < jg; j++) direct_step(j, IC<0>());
          for (; j + 4 <= jend; j += 4) {
            const double2 t01 = *(const double2 *)&s_tau[j];
            const double2 t23 = *(const double2 *)&s_tau[j + 2];
            const double2 h01 = *(const double2 *)&s_thr[j];
            const double2 h23 = *(const double2 *)&s_thr[j + 2];
            float4 av[NA];
#pragma unroll
            for (int c = 0; c < NA; c++) av[c] = *(const float4 *)&s_amp[c][j];
            const double tq[4] = {t01.x, t01.y, t23.x, t23.y};
            const double hq[4] = {h01.x, h01.y, h23.x, h23.y};
#pragma unroll
            for (int q = 0; q < 4; q++) {
              float a[NA];
#pragma unroll
              for (int c = 0; c < NA; c++) a[c] = lane4(av[c], q);
#pragma unroll
              for (int k = 0; k < M; k++) {
                if (valid[k] && fabs(om_rev[k]) < hq[q]) {
                  float sn, cn;
                  sincos_rev(om_rev[k] * tq[q], &sn, &cn);
                  split_acc<MODE, NA>(ps[k], a, cn, sn);
                }
              }
            }
          }
        }
        if (kTab && tile_wide) {
          for (; j < jend; j++) direct_step(j, IC<1>());
          return;
        }
#pragma unroll SR_F64_UNROLL
        for (; j < jend; j++) direct_step(j, IC<0>());
      };
      // split: Kahan fold of the segment's partial sums into the LDS S, C
      auto kahan_fold = [&]() {
        if (!kSplit) return;
#pragma unroll
        for (int k = 0; k < M; k++) {
          float part[NC];
#pragma unroll
          for (int c = 0; c < NC; c++) part[c] = ps[k][c];
          if constexpr (MODE != SR_MODE_FAR) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
              part[c] = fmx(-omf[k], ps[k][6 + c], part[c]);
              part[3 + c] = fmx(omf[k], ps[k][9 + c], part[3 + c]);
            }
          }
#pragma unroll
          for (int c = 0; c < NC; c++) {
            float &S = s_ks[(c * M + k) * T];
            float &C = s_kc[(c * M + k) * T];
            const float yv = part[c] - C;
            const float tv = S + yv;
            C = (tv - S) - yv;
            S = tv;
          }
#pragma unroll
          for (int c = 0; c < NP; c++) ps[k][c] = 0.f;
        }
      };

      // FP64: tau of one step, as the stage forms it
      auto tau_at = [&](int64_t s) {
        const int64_t gs = pt.off + s;
        const double time = (double)(uint32_t)(pt.its + (uint32_t)s) * dt;
        const Geom q = geom();
        if (MODE == SR_MODE_FAR) return time - (p.x[gs] * q.gx + p.y[gs] * q.gy + p.z[gs] * q.gz);
        const double rx = q.gx - p.x[gs], ry = q.gy - p.y[gs], rz = q.gz - p.z[gs];
        return time + sqrt(rx * rx + ry * ry + rz * rz);
      };

      // stages the group's steps [t0, t0 + cnt), cnt <= T
      auto stage_tile = [&](int64_t t0, int cnt) {
        __syncthreads();  // previous tile fully consumed
        int st_wide = 0;
        if (tid < cnt) {
          // ---- stage: omega-independent part of step s = t0 + tid, in FP64 ----
          const int64_t s = t0 + tid;
          const int64_t gs = pt.off + s;
          const double time = (double)(uint32_t)(pt.its + (uint32_t)s) * dt;
          const double xs = p.x[gs], ys = p.y[gs], zs = p.z[gs];
          const Geom q = geom();
          const double gx = q.gx, gy = q.gy, gz = q.gz;
          const double thx = q.thx, thy = q.thy, thz = q.thz, phx = q.phx, phy = q.phy;
          double tau;
          Amp st_amp[NA];
          // split: tau_{s-1} (phase_{-1} = 0 at the first step)
          double st_prev = 0.0;
          const bool own_prev = kSplit && s > 0;
          if (MODE == SR_MODE_FAR) {
            // kernel_farfield.cl:65-94
            tau = time - (xs * gx + ys * gy + zs * gz);
            if (own_prev) {
              const double tp = (double)(uint32_t)(pt.its + (uint32_t)(s - 1)) * dt;
              st_prev = tp - (p.x[gs - 1] * gx + p.y[gs - 1] * gy + p.z[gs - 1] * gz);
            }
            double ax, ay, az, mx, my, mz;
            if constexpr (PRE) {
              const double2 *r = (const double2 *)(p.pre + 6 * gs);
              const double2 r0 = r[0], r1 = r[1], r2 = r[2];
              ax = r0.x; ay = r0.y; az = r1.x;
              mx = r1.y; my = r2.x; mz = r2.y;
            } else {
              step_am(p.ux, p.uy, p.uz, gs, dtInv, &ax, &ay, &az, &mx, &my, &mz);
            }
            double c1 = ax * gx + ay * gy + az * gz;
            double c2 = 1.0 - (mx * gx + my * gy + mz * gz);
            // split: the amplitude ends in FP32, so the hardware reciprocal
            // (relative error <= 4.6e-8 measured on gfx950) with one Newton
            // step (~1e-15) replaces the IEEE division
            if (kSplit) {
              const double r = __builtin_amdgcn_rcp(c2);
              c2 = fma(r, fma(-c2, r, 1.0), r);
            } else {
              c2 = 1.0 / c2;
            }
            c1 = c1 * c2 * c2;
            const double Ax = c1 * (gx - mx) - c2 * ax;
            const double Ay = c1 * (gy - my) - c2 * ay;
            const double Az = c1 * (gz - mz) - c2 * az;
            // the two transverse components; the record rebuilds x, y, z
            st_amp[0] = (Amp)(thx * Ax + thy * Ay + thz * Az);
            st_amp[1] = (Amp)(phx * Ax + phy * Ay);
          } else {
            // kernel_nearfield.cl:67-88; omega of c1 = omega v1 is applied in the sums
            double b0x, b0y, b0z;
            if constexpr (PRE) {
              const double *r = p.pre + 3 * gs;
              b0x = r[0]; b0y = r[1]; b0z = r[2];
            } else {
              const double g0 = gamma_inv(p.ux[gs], p.uy[gs], p.uz[gs]);
              b0x = p.ux[gs] * g0; b0y = p.uy[gs] * g0; b0z = p.uz[gs] * g0;
            }
            const double rx = gx - xs, ry = gy - ys, rz = gz - zs;
            const double R = sqrt(rx * rx + ry * ry + rz * rz);
            tau = time + R;
            if (own_prev) {
              const double tp = (double)(uint32_t)(pt.its + (uint32_t)(s - 1)) * dt;
              const double qx = gx - p.x[gs - 1], qy = gy - p.y[gs - 1], qz = gz - p.z[gs - 1];
              st_prev = tp + sqrt(qx * qx + qy * qy + qz * qz);
            }
            const double rInv = 1.0 / R;
            const double nx = rInv * rx, ny = rInv * ry, nz = rInv * rz;
            const double r2 = rInv * rInv;
            st_amp[0] = (Amp)(rInv * (b0x - nx));
            st_amp[1] = (Amp)(rInv * (b0y - ny));
            st_amp[2] = (Amp)(rInv * (b0z - nz));
            st_amp[3] = (Amp)(r2 * nx);
            st_amp[4] = (Amp)(r2 * ny);
            st_amp[5] = (Amp)(r2 * nz);
          }
          const int pos = late(tid);   // the staged slots' LDS addresses formed here
          if (kTab) st_wide = fabs(tau) * om_abs_max >= 0.5 * kTabMaxPhase;
          if constexpr (kSplit) {
            // |omega tau_s - omega tau_{s-1}| < pi  <=>  |omega|/2pi < (1/2)/|tau_s - tau_{s-1}|
            // (the hardware reciprocal with one Newton step, as for c2; the raw
            // one, 4.6e-8, moved enough boundary decisions to raise the largest
            // element error of the betatron spectrum from 1e-7 to 6e-7)
            // (d = 0: +inf, always active, as the division gives; the Newton
            // step alone would make it fma(-0, inf, 1) = NaN)
            const double d = fabs(tau - st_prev);
            const double r = __builtin_amdgcn_rcp(d);
            s_thr[pos] = (d == 0.0) ? INFINITY : 0.5 * fma(r, fma(-d, r, 1.0), r);
          }
          s_tau[pos] = tau;
#pragma unroll
          for (int c = 0; c < NA; c++) s_amp[c][pos] = st_amp[c];
        }
        // FP64: a vote through one ballot per wave and an LDS word per wave (the
        // block is one-dimensional: unlike the library's work-group reductions
        // this keeps no y/z work-item ids alive, which cost the near-field
        // variant two spilled registers)
        if constexpr (kTab) {
          const uint64_t b = __ballot(st_wide != 0);
          if (lane == 0) s_vote[grp * W + wv] = (b != 0) ? 1 : 0;
          __syncthreads();
          int any = 0;
          for (int w = 0; w < W; w++) any |= s_vote[grp * W + w];
          tile_wide = uni(any) != 0;
        } else {
          __syncthreads();
        }
      };
      auto emit_next = [&]() {
        if (grp == 0) emit(cur.slot);
        const int64_t last = cur.next;
        cur.slot++;
        cur.advance(pt, p.n_snaps, last);
      };

      if constexpr (!RECORDS) {
        // the steps up to each snapshot record, [done, seg_hi), cut into the groups'
        // parts of `per` steps (P is a power of two); the records after the last active
        // step (global it_range mode) see the final sums
        int64_t done = 0;
        while (cur.next >= 0) {
          const int64_t seg_hi = max(done, min(cur.next + 1, n_act));
          const int64_t per = (seg_hi - done + P - 1) >> __builtin_ctz(P);
          const int64_t lo = min(done + grp * per, seg_hi), hi = min(lo + per, seg_hi);
          if (!kSplit) {
            // FP64: the phase before the part's first step (phase_{-1} = 0)
            const double before = lo > 0 ? tau_at(lo - 1) : 0.0;
#pragma unroll
            for (int k = 0; k < M; k++) prev[k] = om[k] * before;
          }
          for (int64_t it = 0; it < per; it += T) {
            const int cnt = uni((int)max((int64_t)0, min((int64_t)T, hi - lo - it)));
            stage_tile(lo + it, cnt);
            int j = 0;
            direct_sweep(j, cnt);
            kahan_fold();
          }
          done = seg_hi;
          if (kParts && P > 1) {
            // the other groups' sums so far go to the first group, one word at a time
#pragma unroll
            for (int c = 0; c < NC; c++) {
              __syncthreads();
              if (grp > 0) {
#pragma unroll
                for (int k = 0; k < M; k++) {
                  s_sum[((grp - 1) * M + k) * T] = fs[k][c];
                  fs[k][c] = 0.0;
                }
              }
              __syncthreads();
              if (grp == 0) {
                for (int q1 = 0; q1 < P - 1; q1++)
#pragma unroll
                  for (int k = 0; k < M; k++) fs[k][c] += s_sum[(q1 * M + k) * T];
              }
            }
          }
          emit_next();
        }
      } else {
        // tiles of T steps, their sweep split at the records (one electron's 1600 steps on
        // 256 x 32 x 32, 100 and 400 records: log grid 377 and 1178 us, FP64 534 and 1123;
        // with a tile staged anew after each record 411 and 1309, 754 and 2359)
        for (int64_t t0 = 0; t0 < n_act && cur.next >= 0; t0 += T) {
          const int cnt = uni((int)min((int64_t)T, n_act - t0));
          stage_tile(t0, cnt);
          int j = 0;
          while (j < cnt && cur.next >= 0) {
            const bool here = cur.next < t0 + cnt;
            direct_sweep(j, uni(here ? (int)(cur.next - t0) + 1 : cnt));
            kahan_fold();
            if (here) emit_next();
          }
        }
        // records after the last active step (global it_range mode) see the final sums
        while (cur.next >= 0) emit_next();
      }
    }
    if (late_s(p.acc_lds) && grp == 0) {
#pragma unroll 1
      for (int k = 0; k < M; k++) {
        const int wk = omega_slot(k);
        if (wk < (int)p.n_omega) dst(0)[(int64_t)dir * p.n_omega + wk] += s_acc[k * T];
      }
    }
  }
}


// ---------------------------------------------------------------------------
// heaviest tiles first
// ---------------------------------------------------------------------------
// A far-field tile's time grows with the share of its (omega, step) pairs that
// the filter keeps, which varies several-fold over the directions (near the
// beam axis most pairs are kept).  Launched in index order, the last blocks
// keep a few CUs busy while the rest of the GPU idles; so each tile's time is
// estimated from a sample of steps and the tiles are launched heaviest first.
// Every tile writes only its own outputs, so the order changes no result.
#ifndef SR_ORDER_SAMPLES
#define SR_ORDER_SAMPLES 256
#endif
#ifndef SR_ORDER_STEP_COST
#define SR_ORDER_STEP_COST 0.1f
#endif
constexpr int kOrderSamples = SR_ORDER_SAMPLES;
constexpr int64_t kOrderMinTiles = 2048;
constexpr int64_t kOrderMaxTiles = 65536;
constexpr double kOrderMinEvals = 1e10;
// the ranking compares every pair of tiles (2.3 ms for 32768 tiles); it is
// used when the launch has at least kOrderEvalsPerTile2 * tiles^2 evaluations
// (about 100 times the ranking's time at 5e12 evaluations/s)
constexpr double kOrderEvalsPerTile2 = 1.2e3;
// launches from this size on are planned with more particle slices (finer tiles)
constexpr double kOrderSliceEvals = 1e12;
constexpr float kOrderStepCost = SR_ORDER_STEP_COST;   // a step's fixed work, in units of a fully kept step's sweep

// cost[tile] for every (direction, omega chunk), the same for each particle
// slice: sum over sampled intervals of kOrderStepCost + the share of the
// chunk's |omega|/2pi range below the interval's threshold 1/(2|dtau|)
__global__ void k_tile_cost(const KParams p, int64_t run_len, float *cost) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)p.n_dir * p.n_chunks) return;
  const uint32_t chunk = (uint32_t)(i % p.n_chunks);
  const uint32_t dir = (uint32_t)(i / p.n_chunks);
  const uint32_t iPhi = dir / p.n_theta;
  const uint32_t iTh = dir - iPhi * p.n_theta;
  const double st = p.sin_t[iTh], ct = p.cos_t[iTh];
  const double nx = st * p.cos_p[iPhi], ny = st * p.sin_p[iPhi], nz = ct;
  const int64_t first = (int64_t)chunk * run_len;
  const int64_t last = min(first + run_len, (int64_t)p.n_omega);
  double wlo = 1e300, whi = 0.0;
  for (int64_t w = first; w < last; w++) {
    const double a = fabs(p.omega[w]) * kInv2Pi;
    wlo = fmin(wlo, a);
    whi = fmax(whi, a);
  }
  float c = 0.f;
  const int64_t n = p.n_points;
  for (int k = 0; k < kOrderSamples; k++) {
    const int64_t g = 1 + (int64_t)k * (n - 1) / kOrderSamples;   // intervals (g-1, g); rarely across particles
    const double dtau = p.dt - (nx * (p.x[g] - p.x[g - 1]) + ny * (p.y[g] - p.y[g - 1]) + nz * (p.z[g] - p.z[g - 1]));
    const double thr = 0.5 / fabs(dtau);
    double f = (whi > wlo) ? (thr - wlo) / (whi - wlo) : (thr > wlo ? 1.0 : 0.0);
    f = fmin(fmax(f, 0.0), 1.0);
    c += kOrderStepCost + (float)f;
  }
  if (!(c >= 0.f && c <= 1e30f)) c = 0.f;   // a strict order below needs no NaN
  for (int q = 0; q < p.slices; q++) cost[chunk + (int64_t)p.n_chunks * (dir + (int64_t)p.n_dir * q)] = c;
}

// order[rank] = tile, rank = tiles that cost more, or as much with a smaller
// index: a permutation (the key (-cost, index) is a strict total order).
// (Keeping the particle slices in launch order and sorting only within each,
// for cache locality, measured 10 % slower on the 20000-particle batch.)
__global__ void __launch_bounds__(256) k_tile_rank(const float *cost, int64_t n, int32_t *order) {
  __shared__ float s_c[256];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const float ci = i < n ? cost[i] : 0.f;
  int64_t rank = 0;
  for (int64_t j0 = 0; j0 < n; j0 += 256) {
    __syncthreads();
    // past n: -1, below every cost, so never counted
    s_c[threadIdx.x] = (j0 + threadIdx.x < n) ? cost[j0 + threadIdx.x] : -1.f;
    __syncthreads();
    int cnt = 0;
#pragma unroll 16
    for (int jj = 0; jj < 256; jj++) {
      const float cj = s_c[jj];
      cnt += (cj > ci || (cj == ci && j0 + jj < i)) ? 1 : 0;
    }
    rank += cnt;
  }
  if (i < n) order[rank] = (int32_t)i;
}

// Direction-independent data of every sample (the stage's inputs that do not
// depend on the spectral point), computed once per launch: far a, bbar of the
// interval (i, i+1) (kernel_farfield.cl:74-83); near b_i (kernel_nearfield.cl:
// 79-82).  The expressions are the stage's own, so the results are identical.
template <int MODE>
__global__ void k_step_prep(const double *ux, const double *uy, const double *uz, int64_t n, double dt,
                            double *pre) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (MODE == SR_MODE_FAR) {
    double ax = 0.0, ay = 0.0, az = 0.0, mx = 0.0, my = 0.0, mz = 0.0;
    if (i + 1 < n) step_am(ux, uy, uz, i, 1.0 / dt, &ax, &ay, &az, &mx, &my, &mz);
    double2 *r = (double2 *)(pre + 6 * i);
    r[0] = make_double2(ax, ay);
    r[1] = make_double2(az, mx);
    r[2] = make_double2(my, mz);
  } else {
    const double g0 = gamma_inv(ux[i], uy[i], uz[i]);
    double *r = pre + 3 * i;
    r[0] = ux[i] * g0; r[1] = uy[i] * g0; r[2] = uz[i] * g0;
  }
}

// out[c][i] += sum_q scratch[q][c][i], q in order
__global__ void k_reduce_slices(const KParams p) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)p.n_out * p.n_grid * p.n_snaps;
  if (i >= total) return;
  const int64_t per = (int64_t)p.n_grid * p.n_snaps;
  const int c = (int)(i / per);
  const int64_t g = i - (int64_t)c * per;
  double s = 0.0;
  for (int q = 0; q < p.slices; q++) s += p.scratch[((int64_t)q * p.n_out + c) * per + g];
  p.out[c][g] += s;
}

__global__ void k_fill_zero(double *buf, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) buf[i] = 0.0;
}

}  // namespace

// ---------------------------------------------------------------------------
// scratch of the no-allocation entry point
// ---------------------------------------------------------------------------
// sr_spectrum_batch_noalloc keeps its workspace (the particle slices' partial
// spectra and the tile launch order) in this array instead of a caller's
// buffer.  Each GPU holds its own copy from the library's load to the end of
// the process.  On the host the name is only a stand-in: its device address
// on the current GPU comes from hipGetSymbolAddress, once per GPU.
constexpr size_t kNoAllocScratchBytes = SR_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// device address of `scratch` on the current GPU, looked up on the first call
// made with that GPU current
int noalloc_scratch(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(SR_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(SR_ERR_UNSUPPORTED, "device %d: at most %d devices", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(SR_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return SR_OK;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
int outputs_for(int32_t mode, int32_t comp) {
  if (mode == SR_MODE_FAR) {
    switch (comp) {
      case SR_COMP_TOTAL: return 1;
      case SR_COMP_CARTESIAN: case SR_COMP_SPHERIC: return 3;
      case SR_COMP_CARTESIAN_COMPLEX: case SR_COMP_SPHERIC_COMPLEX: return 6;
    }
  } else if (mode == SR_MODE_NEAR) {
    switch (comp) {
      case SR_COMP_TOTAL: return 1;
      case SR_COMP_CARTESIAN: return 3;
      case SR_COMP_CARTESIAN_COMPLEX: return 6;
    }
  }
  return -1;
}

struct Plan {
  int sweep;     // SWEEP_*
  int waves;     // waves per block
  int M;         // omegas per thread
  int groups;    // recurrence: groups of 32 omegas per tile (factored.h)
  int parts;     // FP64: groups of threads that share a tile's steps
  int slices;
  int64_t blocks;
};

// omegas per thread each direct variant is built for
int allowed_m(int mode, int prec, int m) {
  if (prec == SR_PREC_F64) return m == 1 || m == 2;
  return m == 1 || m == 2 || (mode == SR_MODE_FAR && m == 4);
}

// vector instructions per step of a factored tile: the stage and the factors
double factored_cost(bool far, int groups) {
  if (far) return 2.5 + (groups == 4 ? 4.75 : groups == 8 ? 5.5 : 7.5);
  return 9.75;
}

// FP64: steps up to a record that each group of threads has at least.  The groups meet at
// every record: one electron's 1600 steps on 32 x 4 x 4 with a record every 80, 32 and 16
// steps 110, 216, 308 us at 16 (4, 2, 1 groups), 108, 192, 330 at 8, 152, 276, 308 at 32;
// 8 electrons on 100 x 12 x 12 297, 385, 459, at 8 352, 385, 546
constexpr int64_t kPartSteps = 16;

// omegas of one tile
int64_t tile_run(const Plan &pl) {
  return pl.sweep == SWEEP_REC ? 32 * (int64_t)pl.groups : (int64_t)kWave * pl.waves * pl.M;
}

int64_t mean_steps(const sr_tracks &t) { return t.n_particles > 0 ? t.n_points / t.n_particles : 0; }

// Tile shape: prefer the largest omega run per block (T*M) that is mostly
// used, then enough particle slices to put ~8 waves on each of the 1024 SIMDs.
// n_points: samples of the batch (0: unknown), for the size of the launch;
// mean_steps: per particle, for the groups that share a tile's steps
Plan make_plan(const sr_grid &g, const sr_opts &o, int64_t n_particles, uint32_t n_snaps, int64_t n_points,
               int64_t mean_steps) {
  Plan pl;
  const int64_t n_om = g.n_omega;
  const int64_t n_dir = (int64_t)g.n_theta * g.n_phi;
  const bool far = g.mode == SR_MODE_FAR;
  const int64_t spread = n_dir * std::min<int64_t>(std::max<int64_t>(n_particles, 1), kMaxSlices);
  // steps up to a record
  const int64_t record_steps = mean_steps / std::max<int64_t>(1, n_snaps);
  // AUTO: the factored tiles for split spectra on linear grids of more than one 64-omega
  // wave, from the record length on at which the rest of their queues, the fold and the
  // waves' meeting at each record are paid for (direct against factored: 1000 betatron
  // tracks of 32, 64 and 128 steps, 12 x 12 directions: 128 omegas 0.81, 1.02, 1.08 times, 512
  // 0.99, 1.34, 1.66, complex 256 omegas 0.80, 0.98, 1.20; 24 tracks of 1600 steps with a
  // record every 64 and 133: 512 omegas 1.05, 1.37, complex 0.65, 0.80, with every
  // 266 1.21).  On fewer omegas a far-field sine for each costs no more than forming the
  // factors (32 betatron electrons on 64 x 32 x 32: 3.38 ms against 3.62; on 72 omegas 6.8
  // against 3.6), but long tracks on too few directions to fill the GPU take the factored
  // tiles there too: the direct sweep has no more waves than tiles, a factored tile's steps
  // are shared by four (one electron x 6000 steps on 24 x 20 x 4 495 us against 86; 32 x
  // 1100 and 4000 on 2 to 64 omegas at a spread of 1920, 1.16 and 1.39 times).  Near field:
  // the same, and from 256 steps on where the GPU is full (40 tracks on 64 x 16 x 16: 0.78
  // times at 128 steps, 1.00 at 256, 1.19 at 512)
  const bool six = o.comp == kCompField || outputs_for(g.mode, o.comp) == 6;
  const bool full = n_om / ((n_om + 511) / 512) >= 384;   // tiles of 512 omegas, three quarters used
  bool pays = record_steps >= (six ? 96 : n_snaps > 1 ? 80 : far && full ? 32 : 64);
  if (n_om <= kWave)
    pays = pays && (far ? mean_steps >= 1008 && spread < 2048 : record_steps >= 256 || spread < 2048);
  pl.sweep = SWEEP_DIRECT;
  if (o.precision == SR_PREC_SPLIT && g.omega_step != 0.0 &&
      (o.sweep == SR_SWEEP_RECURRENCE || (o.sweep == SR_SWEEP_AUTO && pays)))
    pl.sweep = SWEEP_REC;
  // FP64: groups of threads that may share a tile's steps: blocks of at most
  // kMaxParts waves, two staged tiles of steps for each, and of the steps up to a
  // record kPartSteps
  auto part_limit = [&](int w) -> int64_t {
    if (o.precision != SR_PREC_F64) return 1;
    return std::max<int64_t>(1, std::min<int64_t>({kMaxParts / w, mean_steps / (2 * kWave * w), record_steps / kPartSteps}));
  };
  int64_t chunks;
  if (pl.sweep == SWEEP_REC) {
    // groups of 32 omegas per tile (factored.h): the number whose tiles cost least
    // (factored_cost)
    pl.M = (far && o.omega_per_lane != 2 && o.omega_per_lane != 1) ? 4 : 2;
    const int max_groups = pl.M == 4 ? 16 : far ? 8 : 4;
    double best = INFINITY;
    pl.groups = 4;
    for (int ng = 4; ng <= max_groups; ng *= 2) {
      const int64_t c = (n_om + 32 * ng - 1) / (32 * ng);
      const double cost = (double)c * factored_cost(far, ng);
      if (cost < best) {
        best = cost;
        pl.groups = ng;
      }
    }
    chunks = (n_om + 32 * pl.groups - 1) / (32 * pl.groups);
    // waves of a block share a tile's steps.  One each, but two for 16 groups
    // (betatron beam, 24 x 8000 steps on 512 x 32 x 32: 8.1 ms against 9.1; the
    // near-field screen with 4 groups the other way, 6.9 against 7.6), and more
    // where the tiles and particle slices leave the GPU short of waves (one
    // undulator electron on 256 x 32 x 32: 71 us with two, 94 with one), as long as a
    // wave has four stages' steps of each track: each fills queues of its own (30 x 200
    // steps on 600 x 40 x 20, three words: 0.71 ms with one, 1.08 with two; 100 x 400 on
    // 512 x 16 x 16 0.68 against 0.82); one stage each where even the tiles of two waves
    // leave half of the CUs without one.  Of a record's steps a wave has half a stage's
    // or more, a second wave for 16 groups' sake four stages' (24 x 1600 steps on 512 x 12
    // x 12, a record every 133: two waves 1.15 times one)
    auto shared = [&](int w, int stages) {
      return mean_steps >= (int64_t)w * stages * (kWave - 1) && record_steps >= w * (kWave / 2);
    };
    pl.waves = pl.groups == 16 && record_steps >= 2 * 4 * (kWave - 1) ? 2 : 1;
    while (pl.waves < 4 && ((shared(2 * pl.waves, 4) && chunks * pl.waves * spread < 2048) ||
                            (shared(2 * pl.waves, 1) && chunks * pl.waves * spread < 512)))
      pl.waves *= 2;
    if (o.waves_per_block > 0) pl.waves = o.waves_per_block;
  } else {
    pl.groups = 0;
    int best_w = 1, best_m = 1;
    double best_score = -1;
    const int m_opts[3] = {1, 2, 4};
    for (int w = 1; w <= 4; w *= 2) {
      for (int mi = 0; mi < 3; mi++) {
        const int m = m_opts[mi];
        if (!allowed_m(g.mode, o.precision, m)) continue;
        const int64_t run = (int64_t)kWave * w * m;
        const int64_t c = (n_om + run - 1) / run;
        const double eff = (double)n_om / (double)(c * run);
        if (eff < 0.75) continue;
        // M = 2 measured fastest, with groups of threads also against twice the waves
        // (256 omegas FP64: one undulator electron 0.38 ms at 2 x 2 waves, 0.42 at 1 x 4;
        // without them 100 omegas on 12 x 12, 200 records: 0.41 ms at 1 x 2, 0.74 at 2 x 1)
        const double mpref = (m == 2) ? (part_limit(w) > 1 ? 0.03 : 0.02) : 0.0;
        // launches too small to fill the GPU (one particle: no slices to add
        // waves) prefer the plan with the most waves: 256 CUs hold ~8K waves
        const double fill = std::min(1.0, (double)(c * n_dir * w * part_limit(w) *
                                                   std::min<int64_t>(std::max<int64_t>(n_particles, 1), kMaxSlices)) /
                                              8192.0);
        const double score = eff * fill + 0.01 * w + mpref;
        if (score > best_score) { best_score = score; best_w = w; best_m = m; }
      }
    }
    pl.waves = o.waves_per_block > 0 ? o.waves_per_block : best_w;
    pl.M = o.omega_per_lane > 0 ? o.omega_per_lane : best_m;
    if (!allowed_m(g.mode, o.precision, pl.M)) pl.M = 1;
    const int64_t run = (int64_t)kWave * pl.waves * pl.M;
    chunks = (n_om + run - 1) / run;
  }
  const int64_t base_waves = chunks * n_dir * pl.waves;
  int s = 1;
  if (o.slices > 0) {
    s = o.slices;
  } else {
    // particle slices until the launch has ~8K waves; large launches until
    // ~64K: smaller tiles leave a shorter tail (betatron beam +3 %, the uneven
    // 20000-particle batch +20 % at 16 slices, the near-field screen +6 % at
    // 12 of equal-cost tiles).  Far-field tiles run heaviest first, and only
    // as far as they stay orderable: more slices without the order would
    // lengthen the tail instead.
    const double evals = (double)n_points * (double)(n_om * n_dir);
    const bool far_ordered = g.mode == SR_MODE_FAR && o.tile_order == 0;
    const bool big = evals >= kOrderSliceEvals && (g.mode != SR_MODE_FAR || far_ordered);
    // factored tiles: ~32K waves from 1e10 evaluations on (24 x 4000 steps and
    // more), where the finer tiles' shorter tail outweighs summing the slices:
    // 48 electrons on the near-field screen 19.5 ms against 20.4 at 8K, 256 on
    // 128 x 32 x 32 24.2 against 29.0
    const bool fine = pl.sweep == SWEEP_REC && evals >= kOrderMinEvals;
    const int64_t target = big ? 64 * 1024 : fine ? 32 * 1024 : 8 * 1024;
    auto orderable = [&](int64_t tiles) {
      return tiles <= kOrderMaxTiles && evals >= kOrderEvalsPerTile2 * (double)tiles * (double)tiles;
    };
    while (s < kMaxSlices && base_waves * s < target && (int64_t)(s * 2) <= n_particles &&
           (!(big && far_ordered) || orderable(chunks * n_dir * s * 2)))
      s *= 2;
  }
  if (s > n_particles) s = (int)std::max<int64_t>(1, n_particles);
  pl.slices = s;
  // FP64: launches short of waves (a few particles on a few directions) let several
  // groups of threads share each tile's steps, up to the 4K waves that run at once
  // (powers of two, so that blocks of 2 to 16 waves fill a CU's 16).  One undulator
  // electron, 1600 steps: on 32 x 4 x 4 46 us with the groups, 228 without; on
  // 256 x 32 x 32 (2 groups) 646 us through the calculator against 679; the adjoint of
  // 8 electrons on 100 x 12 x 12 674 us against 772.  From 4K waves on the launch is the
  // same as without.
  pl.parts = 1;
  while (2 * pl.parts <= part_limit(pl.waves) && base_waves * s * pl.parts < 4096) pl.parts *= 2;
  pl.blocks = chunks * n_dir * s;
  return pl;
}

template <int MODE, int PREC, int M>
hipError_t launch_t(const KParams &kp, int64_t grid, int threads, hipStream_t st) {
  const int T = threads / kp.parts;
  const size_t lds = kp.parts * stage_lds_bytes<MODE, PREC>(T) +
                     ((PREC == SR_PREC_SPLIT) ? kahan_lds_bytes<MODE, M>(T) : 0) +
                     (kp.acc_lds ? acc_lds_bytes<M>(T) : 0) + (kp.parts - 1) * acc_lds_bytes<M>(T);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(threads), lds, st, kp); };
  if (kp.n_snaps > 1 && kp.parts == 1) {
    if (kp.pre) launch(k_spectrum<MODE, PREC, M, true, true>);
    else launch(k_spectrum<MODE, PREC, M, false, true>);
  } else {
    if (kp.pre) launch(k_spectrum<MODE, PREC, M, true, false>);
    else launch(k_spectrum<MODE, PREC, M, false, false>);
  }
  return hipGetLastError();
}

template <int MODE, int NG>
hipError_t launch_factored(const KParams &kp, int64_t grid, int threads, hipStream_t st) {
  const size_t lds = factored_lds<MODE, NG>(threads / kWave, kp.acc_lds != 0);
  if (kp.pre)
    hipLaunchKernelGGL((k_factored<MODE, NG, true>), dim3((unsigned)grid), dim3(threads), lds, st, kp);
  else
    hipLaunchKernelGGL((k_factored<MODE, NG, false>), dim3((unsigned)grid), dim3(threads), lds, st, kp);
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_mode(const Plan &pl, int prec, const KParams &kp, int64_t grid, int threads,
                       hipStream_t st) {
  if (prec == SR_PREC_F64) {
    if (pl.M == 2) return launch_t<MODE, SR_PREC_F64, 2>(kp, grid, threads, st);
    return launch_t<MODE, SR_PREC_F64, 1>(kp, grid, threads, st);
  }
  if (pl.sweep == SWEEP_REC) {
    if (pl.groups == 4) return launch_factored<MODE, 4>(kp, grid, threads, st);
    if (MODE == SR_MODE_FAR && pl.groups == 16)
      return launch_factored<MODE, (MODE == SR_MODE_FAR ? 16 : 4)>(kp, grid, threads, st);
    return launch_factored<MODE, (MODE == SR_MODE_FAR ? 8 : 4)>(kp, grid, threads, st);
  }
  if (MODE == SR_MODE_FAR && pl.M == 4)
    return launch_t<MODE, SR_PREC_SPLIT, (MODE == SR_MODE_FAR ? 4 : 2)>(kp, grid, threads, st);
  if (pl.M == 2) return launch_t<MODE, SR_PREC_SPLIT, 2>(kp, grid, threads, st);
  return launch_t<MODE, SR_PREC_SPLIT, 1>(kp, grid, threads, st);
}

int check_grid(const sr_grid *g) {
  if (!g) return fail(SR_ERR_INVALID, "grid is NULL");
  if (g->mode != SR_MODE_FAR && g->mode != SR_MODE_NEAR)
    return fail(SR_ERR_INVALID, "grid.mode %d is not far (0) or near (1)", g->mode);
  if (g->n_omega == 0 || g->n_theta == 0 || g->n_phi == 0)
    return fail(SR_ERR_INVALID, "grid sizes must be >= 1 (got %u, %u, %u)", g->n_omega, g->n_theta,
                g->n_phi);
  if (!g->omega) return fail(SR_ERR_INVALID, "grid axis pointer is NULL");
  if (g->screen_y && g->mode != SR_MODE_NEAR)
    return fail(SR_ERR_INVALID, "screen_y (a Cartesian screen) is a near-field grid");
  if (!g->screen_y && (!g->sin_phi || !g->cos_phi)) return fail(SR_ERR_INVALID, "grid axis pointer is NULL");
  if (g->mode == SR_MODE_FAR && (!g->sin_theta || !g->cos_theta))
    return fail(SR_ERR_INVALID, "far grid needs sin_theta and cos_theta");
  if (g->mode == SR_MODE_NEAR && !g->radius) return fail(SR_ERR_INVALID, "near grid needs radius");
  if (!isfinite(g->omega_step)) return fail(SR_ERR_INVALID, "omega_step must be finite");
  const double npts = (double)g->n_omega * g->n_theta * g->n_phi;
  if (npts > 4.0e9) return fail(SR_ERR_INVALID, "grid has more than 4e9 points");
  return SR_OK;
}

int check_opts(const sr_grid *g, const sr_opts *o) {
  if (!o) return fail(SR_ERR_INVALID, "opts is NULL");
  if (outputs_for(g->mode, o->comp) < 0)
    return fail(SR_ERR_INVALID, "comp %d is not available in mode %d", o->comp, g->mode);
  if (o->precision != SR_PREC_F64 && o->precision != SR_PREC_SPLIT)
    return fail(SR_ERR_INVALID, "precision %d is not F64 (0) or SPLIT (1)", o->precision);
  if (!(o->omega_per_lane == 0 || o->omega_per_lane == 1 || o->omega_per_lane == 2 ||
        o->omega_per_lane == 4))
    return fail(SR_ERR_INVALID, "omega_per_lane must be 0, 1, 2 or 4");
  if (!(o->waves_per_block == 0 || o->waves_per_block == 1 || o->waves_per_block == 2 ||
        o->waves_per_block == 4))
    return fail(SR_ERR_INVALID, "waves_per_block must be 0, 1, 2 or 4");
  if (o->slices < 0 || o->slices > kMaxSlices)
    return fail(SR_ERR_INVALID, "slices must be in [0, %d]", kMaxSlices);
  if (o->persistent < 0) return fail(SR_ERR_INVALID, "persistent must be >= 0");
  if (o->tile_order != 0 && o->tile_order != 1) return fail(SR_ERR_INVALID, "tile_order must be 0 or 1");
  if (o->sweep < SR_SWEEP_AUTO || o->sweep > SR_SWEEP_RECURRENCE)
    return fail(SR_ERR_INVALID, "sweep must be SR_SWEEP_AUTO, _DIRECT or _RECURRENCE");
  if (o->sweep == SR_SWEEP_RECURRENCE && (o->precision != SR_PREC_SPLIT || g->omega_step == 0.0))
    return fail(SR_ERR_INVALID, "the recurrence sweep needs SR_PREC_SPLIT and a constant omega_step");
  if (g->mode == SR_MODE_FAR && o->comp == SR_COMP_CARTESIAN_COMPLEX && !o->form_factor)
    return fail(SR_ERR_INVALID, "far cartesian_complex needs form_factor");
  return SR_OK;
}

void fill_grid(KParams &kp, const sr_grid &g, const sr_opts &o, int n_out, double *const *outs) {
  kp.comp = o.comp;
  kp.n_omega = g.n_omega;
  kp.n_theta = g.n_theta;
  kp.n_phi = g.n_phi;
  kp.omega = g.omega;
  kp.sin_t = g.sin_theta;
  kp.cos_t = g.cos_theta;
  kp.radius = g.radius;
  kp.sin_p = g.sin_phi;
  kp.cos_p = g.cos_phi;
  kp.l_screen = g.l_screen;
  kp.screen_y = g.screen_y;
  kp.omega_step = g.omega_step;
  kp.form_factor = o.form_factor;
  kp.n_grid = (int64_t)g.n_omega * g.n_theta * g.n_phi;
  kp.n_out = n_out;
  for (int c = 0; c < kMaxOut; c++) kp.out[c] = c < n_out ? outs[c] : nullptr;
  kp.n_dir = g.n_theta * g.n_phi;
}

// balanced contiguous particle slices by step count
void slice_particles(KParams &kp, int slices, int64_t n_particles, const int64_t *offsets_host) {
  kp.slice_lo[0] = 0;
  if (offsets_host && slices > 1) {
    const int64_t total = offsets_host[n_particles] - offsets_host[0];
    int64_t i = 0;
    for (int q = 1; q < slices; q++) {
      const double target = (double)total * q / slices + (double)offsets_host[0];
      while (i < n_particles && (double)offsets_host[i] < target) i++;
      kp.slice_lo[q] = std::max(kp.slice_lo[q - 1], i);
    }
  } else {
    for (int q = 1; q < slices; q++) kp.slice_lo[q] = n_particles * q / slices;
  }
  kp.slice_lo[slices] = n_particles;
}

// workspace of a batch call: the slices' partial spectra, then the
// direction-independent step data
size_t scratch_bytes(const Plan &pl, int n_out, int64_t n_grid, uint32_t n_snaps) {
  // rounded to 256 bytes: the step records after it are read with 16-byte loads
  return pl.slices > 1 ? ((size_t)pl.slices * n_out * (size_t)n_grid * n_snaps * sizeof(double) + 255) / 256 * 256
                       : 0;
}
size_t pre_bytes(int mode, int64_t n_points) {
  return (size_t)(mode == SR_MODE_FAR ? 6 : 3) * (size_t)n_points * sizeof(double);
}
// the tile costs and launch order (batch calls in the far field with enough
// tiles and work to have a tail worth ordering), 0 otherwise
size_t order_bytes(const Plan &pl, const sr_grid &g, const sr_opts &o, int64_t n_points) {
  const double evals = (double)n_points * g.n_omega * g.n_theta * g.n_phi;
  if (g.mode != SR_MODE_FAR || o.tile_order != 0 || n_points < 2 || pl.blocks < kOrderMinTiles ||
      pl.blocks > kOrderMaxTiles || evals < kOrderMinEvals ||
      evals < kOrderEvalsPerTile2 * (double)pl.blocks * (double)pl.blocks)
    return 0;
  return ((size_t)pl.blocks * (sizeof(float) + sizeof(int32_t)) + 255) / 256 * 256;
}

// want_pre: compute the step data into the workspace (batch calls); the
// single-particle entry points and the no-allocation batch call compute it in
// the stage instead.  need_order: bytes of the tile launch order (0: index
// order), order_bytes() for batch calls.  Workspace layout: the slices'
// partial spectra, the step data, the tile costs and order.
int run(KParams &kp, const Plan &pl, const sr_grid &g, const sr_opts &o, void *ws, size_t ws_bytes,
        hipStream_t st, bool want_pre = false, size_t need_order = 0) {
  const int threads = kWave * pl.waves * pl.parts;
  kp.parts = pl.parts;
  const int64_t run = tile_run(pl);
  kp.n_chunks = (uint32_t)((g.n_omega + run - 1) / run);
  kp.slices = pl.slices;
  kp.n_tiles = pl.blocks;
  if (pl.blocks >= ((int64_t)1 << 31))
    return fail(SR_ERR_UNSUPPORTED, "%lld tiles in one launch: at most 2^31 - 1", (long long)pl.blocks);
  kp.div_chunks = make_udiv(kp.n_chunks);
  kp.div_dir = make_udiv(kp.n_dir);
  kp.div_theta = make_udiv(kp.n_theta);
  kp.acc_lds = (kp.n_out == 1 && kp.n_snaps == 1) ? 1 : 0;
  // per-particle outputs are disjoint: slices write them in place
  const size_t need = kp.part_stride ? 0 : scratch_bytes(pl, kp.n_out, kp.n_grid, kp.n_snaps);
  const size_t need_pre = want_pre ? pre_bytes(g.mode, kp.n_points) : 0;
  hipError_t e;
  if (need + need_pre + need_order && (!ws || ws_bytes < need + need_pre + need_order))
    return fail(SR_ERR_WORKSPACE, "workspace of %zu bytes needed, %zu given", need + need_pre + need_order,
                ws_bytes);
  kp.tile_order = nullptr;
  if (need_order) {
    float *cost = (float *)((char *)ws + need + need_pre);
    int32_t *order = (int32_t *)(cost + pl.blocks);
    const int64_t pairs = (int64_t)kp.n_dir * kp.n_chunks;
    hipLaunchKernelGGL(k_tile_cost, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, st, kp, run, cost);
    hipLaunchKernelGGL(k_tile_rank, dim3((unsigned)((pl.blocks + 255) / 256)), dim3(256), 0, st,
                       (const float *)cost, (int64_t)pl.blocks, order);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(SR_ERR_HIP, "tile order launch: %s", hipGetErrorString(e));
    kp.tile_order = order;
  }
  if (need_pre) {
    kp.pre = (const double *)((char *)ws + need);
    const int64_t n = kp.n_points;
    if (g.mode == SR_MODE_FAR)
      hipLaunchKernelGGL(k_step_prep<SR_MODE_FAR>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, kp.ux,
                         kp.uy, kp.uz, n, kp.dt, (double *)kp.pre);
    else
      hipLaunchKernelGGL(k_step_prep<SR_MODE_NEAR>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, kp.ux,
                         kp.uy, kp.uz, n, kp.dt, (double *)kp.pre);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(SR_ERR_HIP, "step data launch: %s", hipGetErrorString(e));
  }
  if (need) {
    kp.scratch = (double *)ws;
    const int64_t n = (int64_t)(need / sizeof(double));
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, kp.scratch, n);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(SR_ERR_HIP, "workspace clear: %s", hipGetErrorString(e));
  } else {
    kp.scratch = nullptr;
  }
  int64_t grid = pl.blocks;
  if (o.persistent > 0) grid = std::min<int64_t>(grid, o.persistent);
  if (grid <= 0) return SR_OK;
  e = (g.mode == SR_MODE_FAR) ? launch_mode<SR_MODE_FAR>(pl, o.precision, kp, grid, threads, st)
                              : launch_mode<SR_MODE_NEAR>(pl, o.precision, kp, grid, threads, st);
  if (e != hipSuccess) return fail(SR_ERR_HIP, "tile kernel launch: %s", hipGetErrorString(e));
  if (need) {
    const int64_t total = (int64_t)kp.n_out * kp.n_grid * kp.n_snaps;
    hipLaunchKernelGGL(k_reduce_slices, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, kp);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(SR_ERR_HIP, "slice reduction launch: %s", hipGetErrorString(e));
  }
  return SR_OK;
}

int check_tracks(const sr_tracks *t) {
  if (!t) return fail(SR_ERR_INVALID, "tracks is NULL");
  if (t->n_particles < 0 || t->n_points < 0) return fail(SR_ERR_INVALID, "negative track sizes");
  if (t->n_particles == 0) return SR_OK;
  if (!t->offsets || !t->x || !t->y || !t->z || !t->ux || !t->uy || !t->uz || !t->weight ||
      !t->it_start || !t->it_end || !t->it_snaps)
    return fail(SR_ERR_INVALID, "a track pointer is NULL");
  if (t->n_snaps == 0) return fail(SR_ERR_INVALID, "n_snaps must be >= 1");
  if (t->snaps_stride != 0 && t->snaps_stride != t->n_snaps)
    return fail(SR_ERR_INVALID, "snaps_stride must be 0 or n_snaps");
  if (!(t->dt != 0.0) || !isfinite(t->dt)) return fail(SR_ERR_INVALID, "dt must be finite and non-zero");
  return SR_OK;
}

int single_particle(int32_t mode, int32_t comp, double *const *outs, const double *x, const double *y,
                    const double *z, const double *ux, const double *uy, const double *uz, double wp,
                    uint32_t itStart, uint32_t itEnd, uint32_t nSteps, const sr_grid &g, double dt,
                    uint32_t nSnaps, const uint32_t *itSnaps, int32_t precision, void *stream) {
  int rc = check_grid(&g);
  if (rc) return rc;
  sr_opts o;
  memset(&o, 0, sizeof(o));
  o.comp = comp;
  o.precision = precision;
  if ((rc = check_opts(&g, &o))) return rc;
  // the reference would loop 2^32 times (itEnd == 0) or read out of bounds (nSteps == 0)
  if (itEnd == 0) return fail(SR_ERR_INVALID, "itEnd must be >= 1");
  if (nSteps == 0) return fail(SR_ERR_INVALID, "nSteps must be >= 1");
  if (nSnaps == 0 || !itSnaps) return fail(SR_ERR_INVALID, "nSnaps must be >= 1 with itSnaps");
  if (!x || !y || !z || !ux || !uy || !uz) return fail(SR_ERR_INVALID, "a track pointer is NULL");
  if (!(dt != 0.0) || !isfinite(dt)) return fail(SR_ERR_INVALID, "dt must be finite and non-zero");
  const int n_out = outputs_for(mode, comp);
  for (int c = 0; c < n_out; c++)
    if (!outs[c]) return fail(SR_ERR_INVALID, "output %d is NULL", c);
  KParams kp;
  memset(&kp, 0, sizeof(kp));
  kp.offsets = nullptr;
  kp.x = x; kp.y = y; kp.z = z; kp.ux = ux; kp.uy = uy; kp.uz = uz;
  kp.it_snaps = itSnaps;
  kp.n_snaps = nSnaps;
  kp.snaps_stride = 0;
  kp.dt = dt;
  kp.single_n = nSteps;
  kp.single_w = wp;
  kp.single_its = itStart;
  kp.single_ite = itEnd;
  fill_grid(kp, g, o, n_out, outs);
  Plan pl = make_plan(g, o, 1, nSnaps, nSteps, std::min(nSteps, itEnd));
  pl.slices = 1;  // one particle: no slices, no workspace
  slice_particles(kp, 1, 1, nullptr);
  return run(kp, pl, g, o, nullptr, 0, (hipStream_t)stream);
}

}  // namespace

namespace sr {

int step_prep(const sr_tracks &t, int32_t mode, double *pre, hipStream_t st) {
  const int64_t n = t.n_points;
  if (mode == SR_MODE_FAR)
    hipLaunchKernelGGL(k_step_prep<SR_MODE_FAR>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, t.ux, t.uy,
                       t.uz, n, t.dt, pre);
  else
    hipLaunchKernelGGL(k_step_prep<SR_MODE_NEAR>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, t.ux, t.uy,
                       t.uz, n, t.dt, pre);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SR_OK : fail(SR_ERR_HIP, "step data launch: %s", hipGetErrorString(e));
}

namespace {
// samples of particles [p_begin, p_end): exact with the host offsets, else
// the batch's mean
int64_t chunk_points(const sr_tracks &t, int64_t p_begin, int64_t p_end) {
  if (t.offsets_host) return t.offsets_host[p_end] - t.offsets_host[p_begin];
  return t.n_particles ? t.n_points * (p_end - p_begin) / t.n_particles : 0;
}
sr_opts fields_opts(const sr_opts &request) {
  sr_opts o;
  memset(&o, 0, sizeof(o));
  o.comp = kCompField;
  o.precision = request.precision;
  if (request.sweep == SR_SWEEP_DIRECT) o.sweep = SR_SWEEP_DIRECT;
  // every particle's field has its own output, so particle slices cost no
  // reduction: split fields take the finest tiles (the adjoint workload's
  // 256 x 4000 steps on 128 x 32 x 32: 41.4 ms at 32 slices against 42.7 at
  // the library plan's 8, heaviest first); FP64 keeps the plan (90.6 ms
  // against 93.1 at 32)
  if (o.precision == SR_PREC_SPLIT) o.slices = kMaxSlices;
  return o;
}
}  // namespace

size_t fields_order_space(const sr_tracks &t, const sr_grid &g, const sr_opts &request, int64_t n_particles) {
  const Plan pl = make_plan(g, fields_opts(request), std::max<int64_t>(n_particles, 1), 1, 0, mean_steps(t));
  if (pl.blocks > kOrderMaxTiles) return 0;
  return ((size_t)pl.blocks * (sizeof(float) + sizeof(int32_t)) + 255) / 256 * 256;
}

int spectrum_fields(const sr_tracks &t, const sr_grid &g, const sr_opts &request, int64_t p_begin, int64_t p_end,
                    const double *pre, double *F, hipStream_t st, void *order_ws, size_t order_ws_bytes) {
  KParams kp;
  memset(&kp, 0, sizeof(kp));
  kp.offsets = t.offsets;
  kp.x = t.x; kp.y = t.y; kp.z = t.z; kp.ux = t.ux; kp.uy = t.uy; kp.uz = t.uz;
  kp.weight = t.weight;
  kp.it_start = t.it_start;
  kp.it_end = t.it_end;
  kp.it_snaps = t.it_snaps;
  kp.n_snaps = 1;
  kp.snaps_stride = t.snaps_stride;
  kp.dt = t.dt;
  kp.n_points = t.n_points;
  kp.pre = pre;
  const sr_opts o = fields_opts(request);
  const int64_t np = p_end - p_begin;
  const int64_t n_grid = (int64_t)g.n_omega * g.n_theta * g.n_phi;
  double *outs[kMaxOut];
  for (int c = 0; c < 6; c++) outs[c] = F + (int64_t)c * np * n_grid;
  fill_grid(kp, g, o, 6, outs);
  const Plan pl = make_plan(g, o, np, 1, 0, mean_steps(t));
  for (int q = 0; q <= pl.slices; q++) kp.slice_lo[q] = p_begin + np * q / pl.slices;
  kp.part_base = p_begin;
  kp.part_stride = n_grid;
  // heaviest tiles first where the launch is large enough and the caller
  // gave room for the order
  size_t ob = order_ws ? order_bytes(pl, g, o, chunk_points(t, p_begin, p_end)) : 0;
  if (ob > order_ws_bytes) ob = 0;
  return run(kp, pl, g, o, order_ws, order_ws_bytes, st, false, ob);
}

}  // namespace sr

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int sr_abi_version(void) { return SR_ABI_VERSION; }

const char *sr_last_error(void) { return sr::last_error(); }

int sr_num_outputs(int32_t mode, int32_t comp) {
  const int n = outputs_for(mode, comp);
  return n < 0 ? fail(SR_ERR_INVALID, "comp %d is not available in mode %d", comp, mode) : n;
}

int sr_workspace_bytes(const sr_tracks *tracks, const sr_grid *grid, const sr_opts *opts,
                       size_t *bytes) {
  int rc;
  if (!bytes) return fail(SR_ERR_INVALID, "bytes is NULL");
  *bytes = 0;
  if ((rc = check_tracks(tracks)) || (rc = check_grid(grid)) || (rc = check_opts(grid, opts))) return rc;
  if (tracks->n_particles == 0) return SR_OK;
  const Plan pl = make_plan(*grid, *opts, tracks->n_particles, tracks->n_snaps, tracks->n_points, mean_steps(*tracks));
  *bytes = scratch_bytes(pl, outputs_for(grid->mode, opts->comp),
                         (int64_t)grid->n_omega * grid->n_theta * grid->n_phi, tracks->n_snaps) +
           pre_bytes(grid->mode, tracks->n_points) + order_bytes(pl, *grid, *opts, tracks->n_points);
  return SR_OK;
}

int sr_spectrum_batch(const sr_tracks *t, const sr_grid *g, const sr_opts *o, double *const *outs,
                      void *workspace, size_t workspace_bytes, void *stream) {
  int rc;
  if ((rc = check_tracks(t)) || (rc = check_grid(g)) || (rc = check_opts(g, o))) return rc;
  if (t->n_particles == 0) return SR_OK;
  const int n_out = outputs_for(g->mode, o->comp);
  if (!outs) return fail(SR_ERR_INVALID, "outs is NULL");
  for (int c = 0; c < n_out; c++)
    if (!outs[c]) return fail(SR_ERR_INVALID, "output %d is NULL", c);
  KParams kp;
  memset(&kp, 0, sizeof(kp));
  kp.offsets = t->offsets;
  kp.x = t->x; kp.y = t->y; kp.z = t->z; kp.ux = t->ux; kp.uy = t->uy; kp.uz = t->uz;
  kp.weight = t->weight;
  kp.it_start = t->it_start;
  kp.it_end = t->it_end;
  kp.it_snaps = t->it_snaps;
  kp.n_snaps = t->n_snaps;
  kp.snaps_stride = t->snaps_stride;
  kp.dt = t->dt;
  kp.n_points = t->n_points;
  fill_grid(kp, *g, *o, n_out, outs);
  const Plan pl = make_plan(*g, *o, t->n_particles, t->n_snaps, t->n_points, mean_steps(*t));
  slice_particles(kp, pl.slices, t->n_particles, t->offsets_host);
  return run(kp, pl, *g, *o, workspace, workspace_bytes, (hipStream_t)stream, true,
             order_bytes(pl, *g, *o, t->n_points));
}

int sr_plan(const sr_tracks *t, const sr_grid *g, const sr_opts *o, sr_plan_info *info) {
  int rc;
  if (!info) return fail(SR_ERR_INVALID, "info is NULL");
  memset(info, 0, sizeof(*info));
  if ((rc = check_tracks(t)) || (rc = check_grid(g)) || (rc = check_opts(g, o))) return rc;
  const Plan pl = make_plan(*g, *o, std::max<int64_t>(t->n_particles, 1), t->n_snaps, t->n_points, mean_steps(*t));
  info->sweep = pl.sweep == SWEEP_REC ? SR_SWEEP_RECURRENCE : SR_SWEEP_DIRECT;
  info->omega_per_lane = pl.M;
  info->waves_per_block = pl.waves;
  info->slices = pl.slices;
  info->tiles = pl.blocks;
  info->ordered = order_bytes(pl, *g, *o, t->n_points) > 0 ? 1 : 0;
  return SR_OK;
}

namespace {
// the candidate's plan fields over the base request's output and precision
sr_opts candidate_opts(const sr_opts &base, const sr_opts &cand) {
  sr_opts o = cand;
  o.comp = base.comp;
  o.precision = base.precision;
  o.form_factor = base.form_factor;
  return o;
}
}  // namespace

int sr_autotune_workspace_bytes(const sr_tracks *t, const sr_grid *g, const sr_opts *base,
                                const sr_opts *candidates, int n_candidates, size_t *bytes) {
  if (!bytes) return fail(SR_ERR_INVALID, "bytes is NULL");
  *bytes = 0;
  if (!base || !candidates || n_candidates <= 0) return fail(SR_ERR_INVALID, "no candidates");
  for (int i = 0; i < n_candidates; i++) {
    const sr_opts o = candidate_opts(*base, candidates[i]);
    size_t b = 0;
    if (sr_workspace_bytes(t, g, &o, &b) == SR_OK) *bytes = std::max(*bytes, b);
  }
  return SR_OK;
}

int sr_autotune(const sr_tracks *t, const sr_grid *g, const sr_opts *base, const sr_opts *candidates,
                int n_candidates, double *const *outs, void *workspace, size_t workspace_bytes, int warmup,
                int reps, void *stream, float *ms, int *best) {
  int rc;
  if (!base || !candidates || n_candidates <= 0 || !ms || !best)
    return fail(SR_ERR_INVALID, "sr_autotune needs a base request, candidates, ms[] and best");
  if ((rc = check_tracks(t)) || (rc = check_grid(g)) || (rc = check_opts(g, base))) return rc;
  if (reps < 1 || warmup < 0) return fail(SR_ERR_INVALID, "reps must be >= 1 and warmup >= 0");
  hipStream_t st = (hipStream_t)stream;
  hipEvent_t e0, e1;
  hipError_t e = hipEventCreate(&e0);
  if (e != hipSuccess) return fail(SR_ERR_HIP, "hipEventCreate: %s", hipGetErrorString(e));
  e = hipEventCreate(&e1);
  if (e != hipSuccess) {
    (void)hipEventDestroy(e0);
    return fail(SR_ERR_HIP, "hipEventCreate: %s", hipGetErrorString(e));
  }
  *best = -1;
  float best_ms = INFINITY;
  rc = SR_OK;
  for (int i = 0; i < n_candidates && rc == SR_OK; i++) {
    ms[i] = INFINITY;
    const sr_opts o = candidate_opts(*base, candidates[i]);
    size_t need = 0;
    if (check_opts(g, &o) != SR_OK || sr_workspace_bytes(t, g, &o, &need) != SR_OK || need > workspace_bytes)
      continue;   // a plan this request cannot run (or cannot fit) is not a candidate
    // untimed runs (code objects, caches), then reps timed ones
    for (int r = 0; r < warmup && rc == SR_OK; r++)
      rc = sr_spectrum_batch(t, g, &o, outs, workspace, workspace_bytes, stream);
    if (rc != SR_OK) break;
    e = hipEventRecord(e0, st);
    for (int r = 0; r < reps && rc == SR_OK && e == hipSuccess; r++)
      rc = sr_spectrum_batch(t, g, &o, outs, workspace, workspace_bytes, stream);
    if (e == hipSuccess) e = hipEventRecord(e1, st);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float elapsed = 0.f;
    if (e == hipSuccess && rc == SR_OK) e = hipEventElapsedTime(&elapsed, e0, e1);
    if (e != hipSuccess) {
      rc = fail(SR_ERR_HIP, "timing candidate %d: %s", i, hipGetErrorString(e));
      break;
    }
    if (rc != SR_OK) break;
    ms[i] = elapsed / (float)reps;
    if (ms[i] < best_ms) {
      best_ms = ms[i];
      *best = i;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc == SR_OK && *best < 0) rc = fail(SR_ERR_INVALID, "no candidate plan can run this request");
  return rc;
}

int sr_spectrum_batch_noalloc(const sr_tracks *t, const sr_grid *g, const sr_opts *o, double *const *outs,
                              void *stream) {
  int rc;
  if ((rc = check_tracks(t)) || (rc = check_grid(g)) || (rc = check_opts(g, o))) return rc;
  if (t->n_particles == 0) return SR_OK;
  const int n_out = outputs_for(g->mode, o->comp);
  if (!outs) return fail(SR_ERR_INVALID, "outs is NULL");
  for (int c = 0; c < n_out; c++)
    if (!outs[c]) return fail(SR_ERR_INVALID, "output %d is NULL", c);
  void *scr = nullptr;
  if ((rc = noalloc_scratch(&scr))) return rc;
  KParams kp;
  memset(&kp, 0, sizeof(kp));
  kp.offsets = t->offsets;
  kp.x = t->x; kp.y = t->y; kp.z = t->z; kp.ux = t->ux; kp.uy = t->uy; kp.uz = t->uz;
  kp.weight = t->weight;
  kp.it_start = t->it_start;
  kp.it_end = t->it_end;
  kp.it_snaps = t->it_snaps;
  kp.n_snaps = t->n_snaps;
  kp.snaps_stride = t->snaps_stride;
  kp.dt = t->dt;
  kp.n_points = t->n_points;
  fill_grid(kp, *g, *o, n_out, outs);
  Plan pl = make_plan(*g, *o, t->n_particles, t->n_snaps, t->n_points, mean_steps(*t));
  // the same plan as sr_spectrum_batch; a tuned slice count is halved until
  // the slices' partial spectra and the tile order fit the scratch array
  auto need = [&](const Plan &p) {
    return scratch_bytes(p, n_out, kp.n_grid, t->n_snaps) + order_bytes(p, *g, *o, t->n_points);
  };
  while (o->slices == 0 && pl.slices > 1 && need(pl) > kNoAllocScratchBytes) {
    pl.blocks /= pl.slices;
    pl.slices /= 2;
    pl.blocks *= pl.slices;
  }
  if (need(pl) > kNoAllocScratchBytes)
    return fail(SR_ERR_WORKSPACE,
                "this request needs %zu bytes of scratch (%d particle slices); the no-allocation entry "
                "point holds %zu: ask for fewer slices (opts.slices) or use sr_spectrum_batch",
                need(pl), pl.slices, kNoAllocScratchBytes);
  slice_particles(kp, pl.slices, t->n_particles, t->offsets_host);
  return run(kp, pl, *g, *o, scr, kNoAllocScratchBytes, (hipStream_t)stream, false,
             order_bytes(pl, *g, *o, t->n_points));
}

int sr_far_total(double *spectrum, const double *x, const double *y, const double *z,
                 const double *ux, const double *uy, const double *uz, double wp, uint32_t itStart,
                 uint32_t itEnd, uint32_t nSteps, const double *omega, const double *sinTheta,
                 const double *cosTheta, const double *sinPhi, const double *cosPhi, uint32_t nOmega,
                 uint32_t nTheta, uint32_t nPhi, double dt, uint32_t nSnaps, const uint32_t *itSnaps,
                 int32_t precision, void *stream) {
  sr_grid g;
  memset(&g, 0, sizeof(g));
  g.mode = SR_MODE_FAR;
  g.n_omega = nOmega; g.n_theta = nTheta; g.n_phi = nPhi;
  g.omega = omega; g.sin_theta = sinTheta; g.cos_theta = cosTheta; g.sin_phi = sinPhi; g.cos_phi = cosPhi;
  double *outs[1] = {spectrum};
  return single_particle(SR_MODE_FAR, SR_COMP_TOTAL, outs, x, y, z, ux, uy, uz, wp, itStart, itEnd,
                         nSteps, g, dt, nSnaps, itSnaps, precision, stream);
}

int sr_far_cartesian(double *spectrum1, double *spectrum2, double *spectrum3, const double *x,
                     const double *y, const double *z, const double *ux, const double *uy,
                     const double *uz, double wp, uint32_t itStart, uint32_t itEnd, uint32_t nSteps,
                     const double *omega, const double *sinTheta, const double *cosTheta,
                     const double *sinPhi, const double *cosPhi, uint32_t nOmega, uint32_t nTheta,
                     uint32_t nPhi, double dt, uint32_t nSnaps, const uint32_t *itSnaps,
                     int32_t precision, void *stream) {
  sr_grid g;
  memset(&g, 0, sizeof(g));
  g.mode = SR_MODE_FAR;
  g.n_omega = nOmega; g.n_theta = nTheta; g.n_phi = nPhi;
  g.omega = omega; g.sin_theta = sinTheta; g.cos_theta = cosTheta; g.sin_phi = sinPhi; g.cos_phi = cosPhi;
  double *outs[3] = {spectrum1, spectrum2, spectrum3};
  return single_particle(SR_MODE_FAR, SR_COMP_CARTESIAN, outs, x, y, z, ux, uy, uz, wp, itStart, itEnd,
                         nSteps, g, dt, nSnaps, itSnaps, precision, stream);
}

int sr_near_total(double *spectrum, const double *x, const double *y, const double *z,
                  const double *ux, const double *uy, const double *uz, double wp, uint32_t itStart,
                  uint32_t itEnd, uint32_t nSteps, const double *omega, const double *radius,
                  const double *sinPhi, const double *cosPhi, double distanceToScreen, uint32_t nOmega,
                  uint32_t nRadius, uint32_t nPhi, double dt, uint32_t nSnaps, const uint32_t *itSnaps,
                  int32_t precision, void *stream) {
  sr_grid g;
  memset(&g, 0, sizeof(g));
  g.mode = SR_MODE_NEAR;
  g.n_omega = nOmega; g.n_theta = nRadius; g.n_phi = nPhi;
  g.omega = omega; g.radius = radius; g.sin_phi = sinPhi; g.cos_phi = cosPhi;
  g.l_screen = distanceToScreen;
  double *outs[1] = {spectrum};
  return single_particle(SR_MODE_NEAR, SR_COMP_TOTAL, outs, x, y, z, ux, uy, uz, wp, itStart, itEnd,
                         nSteps, g, dt, nSnaps, itSnaps, precision, stream);
}

int sr_near_cartesian(double *spectrum1, double *spectrum2, double *spectrum3, const double *x,
                      const double *y, const double *z, const double *ux, const double *uy,
                      const double *uz, double wp, uint32_t itStart, uint32_t itEnd, uint32_t nSteps,
                      const double *omega, const double *radius, const double *sinPhi,
                      const double *cosPhi, double distanceToScreen, uint32_t nOmega, uint32_t nRadius,
                      uint32_t nPhi, double dt, uint32_t nSnaps, const uint32_t *itSnaps,
                      int32_t precision, void *stream) {
  sr_grid g;
  memset(&g, 0, sizeof(g));
  g.mode = SR_MODE_NEAR;
  g.n_omega = nOmega; g.n_theta = nRadius; g.n_phi = nPhi;
  g.omega = omega; g.radius = radius; g.sin_phi = sinPhi; g.cos_phi = cosPhi;
  g.l_screen = distanceToScreen;
  double *outs[3] = {spectrum1, spectrum2, spectrum3};
  return single_particle(SR_MODE_NEAR, SR_COMP_CARTESIAN, outs, x, y, z, ux, uy, uz, wp, itStart, itEnd,
                         nSteps, g, dt, nSnaps, itSnaps, precision, stream);
}

}  // extern "C"
