// adjoint_factored.h -- the transpose sweep of the split-precision adjoint on a
// linear omega grid as matrix products (gfx950 MFMA).  Included by adjoint.hip,
// after AParams.
//
// A step needs, for each coefficient word, P = sum_omega Re(conj(C) e^{i omega tau})
// and R = sum_omega omega Im(conj(C) e^{i omega tau}), C = H F.  The frequencies
// are taken in groups of 32 around centres alpha_a at offsets +-beta_b, beta_b = (b +
// 1/2) domega, as in the forward (factored.h):
//   P = sum_a cos(alpha_a tau) U_a + sin(alpha_a tau) V_a,
//   U_a, V_a = sum_b (cos(beta_b tau), sin(beta_b tau)) . (coefficients of a, b)
// U and V of all groups are one real matrix product per direction, coefficient
// table (8 rows a group with two words) x basis (32: cos and sin of 16 offsets, the
// same for every group) over the steps, in fp16 word pairs with FP32 sums (hi hi + hi
// lo + lo hi, the dropped lo lo below 2^-22); the combination over the groups is two
// FMAs per word and group.  A step thus costs the sines of 7 + NG phases and 64 NG
// multiply-adds on the matrix cores where the rotation loop took 14 instructions for
// each of 32 NG frequencies.
//
// The |dphase| < pi filter: a step keeps the frequencies with |omega|/2pi below its
// threshold.  Tiles that no step of the wave keeps a whole group of are skipped, groups
// that a step does not keep whole are left out of its combination, and a group that steps
// cut (on betatron tracks four waves in five have one, rarely two) is a second product
// with the basis masked step by step: of the table's two sides +-beta_b apart, eight rows
// each, only the side that the step cuts, added to nothing or taken off the whole group.
// (Both sides in a product of their own, 24 matrix instructions a group instead of 12: the
// backward of 256 electrons x 4000 steps on 128 x 32 x 32 33.3 ms against 30.0.)
//
// Work split: a first kernel forms each (particle, direction)'s coefficient table in the
// matrix operand's order, a wave a table; then a block owns (particle, direction group,
// run of T steps).  A thread holds its step's data and nine gradient sums in registers
// over all directions of the group, so the slab is written once a launch.  The matrix
// product wants the steps in columns and the tables in rows: lane (c, q) of a wave holds
// the basis of step c at offsets 4 q .. 4 q + 3, and receives word q of step c for two
// groups at a time.  Each wave reads the tables by itself, a tile ahead of its use: with
// tables staged in LDS for the block, whose waves then meet every five directions, the
// waves that cut groups hold up the others (9.9 ms against 8.0, before the masked
// product).
//
// Bound: vector instructions (FP64 step geometry and gradient chain about a third, the
// basis' word pairs about a third) with the matrix products beneath.  64 betatron
// electrons x 4000 steps on 128 x 32 x 32: 5.9 ms and 0.17 ms for the tables, against
// 8.6 ms of the rotation loop; summing the cut groups frequency by frequency in FP32
// instead of the masked product 7.5 ms.
#pragma once

#include "factored.h"

namespace {

constexpr int kAdjRow = 68;   // float2 per factor row: a wave's steps and a bank shift
// LDS of a wave: factors, masks, the geometry of 64 directions
constexpr int kAdjWaveBytes = 7 * kAdjRow * 8 + kWave * 4 + 32 + kWave * 64;
constexpr int kAdjMaxT = 256;

// steps of a particle that enter its record (none: no record)
__device__ __forceinline__ int64_t adj_steps(const AParams &p, const Particle &pt) {
  if (pt.n <= 0) return 0;
  SnapCursor cur;
  cur.init(pt, 1);
  const int64_t n_act = min(pt.n - 1, (int64_t)pt.ite - 1);
  return cur.next >= 0 ? max((int64_t)0, min(n_act, cur.next + 1)) : 0;
}

// groups per omega tile, sets of four result words
template <bool TWO>
constexpr int adj_tile_groups() {
  return TWO ? 16 : 8;
}
template <bool TWO>
constexpr int adj_sets() {
  return TWO ? 1 : 2;
}
// one table of ng groups (a direction and omega tile of one particle): matrix fragments
// [t][set][hi, lo][lane], FP32 coefficients [omega][re.., im..], scales
// [group][set][word], the groups with coefficients that are not finite (a bit each)
template <bool TWO>
struct AdjRecord {
  static constexpr int NCW = TWO ? 2 : 3, NSET = adj_sets<TWO>();
  int ng;
  __host__ __device__ constexpr size_t raw_at() const { return (size_t)(ng / 2) * NSET * 2048; }
  __host__ __device__ constexpr size_t scl_at() const { return raw_at() + (size_t)ng * kGroup * 8 * NCW; }
  __host__ __device__ constexpr size_t flag_at() const { return scl_at() + (size_t)ng * NSET * 16; }
  __host__ __device__ constexpr size_t bytes() const { return flag_at() + 16; }
};
// LDS of a sweep block: the waves' own, the frequencies, the group bounds
constexpr size_t adj_lds_bytes(int waves, int ng) {
  return (size_t)waves * kAdjWaveBytes + (size_t)ng * (kGroup + 3) * 8 + 16;
}
// A group's table as two, of the offsets -beta_b and +beta_b apart.  A lane holds a row's 4
// cos and 4 sin columns, its neighbour (lane ^ 1) the group's other row; with the row of
// cos(alpha tau) (a+ + a-, b+ - b-) and that of sin(alpha tau) (b+ + b-, a- - a+), the
// lower parts are (a-, -b-) and (b-, a-), the upper ones the rest.  Lanes with bit 1 clear
// form the lower part of their row, the others the upper
__device__ __forceinline__ void two_sides(uint4v th, uint4v tl, float one, uint4v *oh, uint4v *ol) {
  float v[8];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const half2v h = __builtin_bit_cast(half2v, (uint32_t)th[k]), l = __builtin_bit_cast(half2v, (uint32_t)tl[k]);
    v[2 * k] = ((float)h.x + (float)l.x) * 0.5f;
    v[2 * k + 1] = ((float)h.y + (float)l.y) * 0.5f;
  }
  const int ln = (int)threadIdx.x;
  const float sg = ((ln ^ (ln >> 1)) & 1) ? -1.f : 1.f;
  float u[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    // (quad_perm 1, 0, 3, 2)
    const float o = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v[k ^ 4]), 0xb1, 0xf, 0xf, true));
    u[k] = k < 4 ? __builtin_fmaf(sg, o, v[k]) : __builtin_fmaf(-sg, o, v[k]);
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint2 w = split_values(u[2 * k], u[2 * k + 1], one);
    (*oh)[k] = w.x;
    (*ol)[k] = w.y;
  }
}
// waves of a table block
constexpr int kTabWaves = 4;

// ---- coefficient tables of directions [dir_lo, dir_lo + dir_n) from the particles'
// fields and dL/dS, and the weights' gradient.  A wave takes the directions of (particle,
// weight group) in turn: a lane the two frequencies alpha_a -+ beta_b, 16 lanes a group.
// Formed in LDS, so that the table's 2-byte scatter stays there and it leaves in 16-byte
// stores ----
template <bool TWO>
__global__ void __launch_bounds__(kTabWaves * kWave) k_adjoint_tables(const AParams p) {
  constexpr int NCW = TWO ? 2 : 3;
  constexpr int NSET = adj_sets<TWO>();
  extern __shared__ __align__(16) char s_dyn_raw[];
  const int ng = p.tile_groups;
  const AdjRecord<TWO> rec{ng};
  const int wv = uni(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  char *const s_rec = s_dyn_raw + wv * rec.bytes();
  float *const s_raw = (float *)(s_rec + rec.raw_at());
  float *const s_scl = (float *)(s_rec + rec.scl_at());
  uint32_t *const s_flag = (uint32_t *)(s_rec + rec.flag_at());
  // the first launch clears the slabs (and starts the weights' sums)
  const bool first_launch = p.dir_lo == 0 && p.chunk_base == 0;
  if (first_launch) {
    const int64_t n = (int64_t)p.n_groups * kSlabWords * p.n_points;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
      p.slab[i] = 0.0;
  }
  const int64_t unit = (int64_t)blockIdx.x * kTabWaves + wv;
  if (unit >= p.chunk_n * p.n_wgroups) return;   // (no block-wide barrier below)
  const int64_t lp = unit % p.chunk_n;
  const int qw = (int)(unit / p.chunk_n);
  const int64_t ip = p.chunk_base + lp;
  const Particle pt = load_particle(p, ip);
  double *const sum_w = p.slab_w + (int64_t)qw * p.n_particles + ip;
  if (adj_steps(p, pt) == 0) {
    if (lane == 0 && p.dir_lo == 0) *sum_w = 0.0;
    return;
  }
  const double wdt2 = pt.w * p.dt * p.dt;
  const uint32_t d_lo = p.dir_lo + (uint32_t)((int64_t)p.dir_n * qw / p.n_wgroups);
  const uint32_t d_hi = p.dir_lo + (uint32_t)((int64_t)p.dir_n * (qw + 1) / p.n_wgroups);
  const int64_t fstride = p.chunk_n * p.n_grid;
  double gw_acc = 0.0;

  for (uint32_t dir = d_lo; dir < d_hi; dir++) {
    const uint32_t iPhi = dir / p.n_theta;
    const uint32_t iTh = dir - iPhi * p.n_theta;
    const double st = p.sin_t[iTh], ct = p.cos_t[iTh], sp = p.sin_p[iPhi], cp = p.cos_p[iPhi];
    for (int wt = 0; wt < p.n_wtiles; wt++) {
      const int w0 = wt * ng * kGroup;
      const int n_om = min(ng * kGroup, (int)p.n_omega - w0);
      sr::wave_sync();
      uint32_t odd = 0;
      for (int idx = lane; idx < ng * 16; idx += kWave) {
        const int g = idx >> 4, b = idx & 15;
        double pr[2][NCW], pi[2][NCW], om2[2];   // H F at alpha - beta, alpha + beta
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int wi = g * kGroup + (h ? 16 + b : 15 - b);
#pragma unroll
          for (int c = 0; c < NCW; c++) { pr[h][c] = 0.0; pi[h][c] = 0.0; }
          om2[h] = 0.0;
          if (wi < n_om) {
            om2[h] = p.omega[w0 + wi] * kInv2Pi;
            const int64_t gidx = (int64_t)dir * p.n_omega + w0 + wi;
            const int64_t fi = lp * p.n_grid + gidx;
            double Fr[3], Fi[3], G[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
              Fr[c] = p.F[(int64_t)(2 * c) * fstride + fi];
              Fi[c] = p.F[(int64_t)(2 * c + 1) * fstride + fi];
              G[c] = p.dS[TWO ? 0 : c][gidx];
            }
#pragma unroll
            for (int c = 0; c < 3; c++) gw_acc += p.dt * p.dt * G[c] * (Fr[c] * Fr[c] + Fi[c] * Fi[c]);
            if constexpr (TWO) {
              const double H = 2.0 * wdt2 * G[0];
              pr[h][0] = H * (Fr[0] * (ct * cp) + Fr[1] * (ct * sp) - Fr[2] * st);
              pr[h][1] = H * (Fr[1] * cp - Fr[0] * sp);
              pi[h][0] = H * (Fi[0] * (ct * cp) + Fi[1] * (ct * sp) - Fi[2] * st);
              pi[h][1] = H * (Fi[1] * cp - Fi[0] * sp);
            } else {
#pragma unroll
              for (int c = 0; c < 3; c++) {
                const double H = 2.0 * wdt2 * G[c];
                pr[h][c] = H * Fr[c];
                pi[h][c] = H * Fi[c];
              }
            }
          }
          float *rw = s_raw + wi * 2 * NCW;
#pragma unroll
          for (int c = 0; c < NCW; c++) { rw[c] = (float)pr[h][c]; rw[NCW + c] = (float)pi[h][c]; }
        }
#pragma unroll
        for (int wd = 0; wd < 2 * NCW; wd++) {
          // word wd: P_c, or R_c, whose coefficients are (-omega Im C, omega Re C)
          const int c = wd % NCW;
          const bool is_r = wd >= NCW;
          const double ar0 = is_r ? -om2[0] * pi[0][c] : pr[0][c], ai0 = is_r ? om2[0] * pr[0][c] : pi[0][c];
          const double ar1 = is_r ? -om2[1] * pi[1][c] : pr[1][c], ai1 = is_r ? om2[1] * pr[1][c] : pi[1][c];
          // row of cos(alpha tau): cos, sin beta columns; row of sin(alpha tau)
          const double v[4] = {ar1 + ar0, ai1 - ai0, ai1 + ai0, ar0 - ar1};
          // the group's word scaled by a power of two to values below 2^14
          int e = 0;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const int ek = (int)((uint64_t)__double_as_longlong(v[k]) >> 52) & 0x7ff;
            e = max(e, ek == 0x7ff ? 0 : ek);
            odd |= ek == 0x7ff ? 1u << g : 0u;
          }
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) e = max(e, __shfl_xor(e, o));
          const double scale = __longlong_as_double((int64_t)min(2046, 2059 - e) << 52);
          const int set = TWO ? 0 : wd / NCW, q = TWO ? wd : c;
          if (b == 0) s_scl[(g * NSET + set) * 4 + q] = ldexpf(1.0f, 1023 - min(2046, 2059 - e));
          _Float16 *const row = (_Float16 *)s_rec + (size_t)((g >> 1) * NSET + set) * 2 * kWave * 8;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const int r = 4 * q + 2 * (g & 1) + (k >> 1);
            const int at = ((b >> 2) * 16 + r) * 8 + (b & 3) + 4 * (k & 1);
            const float x = (float)(v[k] * scale);
            const _Float16 hi = (_Float16)x;
            row[at] = hi;
            row[kWave * 8 + at] = (_Float16)(x - (float)hi);
          }
        }
      }
      for (int o = 1; o < kWave; o <<= 1) odd |= (uint32_t)__shfl_xor((int)odd, o);
      if (lane == 0) *s_flag = odd;
      sr::wave_sync();
      uint4v *const dst = (uint4v *)(p.tab + (((size_t)lp * p.n_wtiles + wt) * p.dir_n + (dir - p.dir_lo)) * rec.bytes());
      for (int i = lane; i < (int)(rec.bytes() / 16); i += kWave) dst[i] = ((const uint4v *)s_rec)[i];
    }
  }
  // this launch's part of the weight's gradient, in a fixed order
  for (int off = kWave / 2; off > 0; off >>= 1) gw_acc += __shfl_down(gw_acc, off, kWave);
  if (lane == 0) *sum_w = p.dir_lo == 0 ? gw_acc : *sum_w + gw_acc;
}

template <bool TWO>
__global__ void __launch_bounds__(kAdjMaxT) __attribute__((amdgpu_waves_per_eu(TWO ? 3 : 2)))
k_adjoint_factored(const AParams p) {
  constexpr int NCW = TWO ? 2 : 3;
  constexpr int NSET = adj_sets<TWO>();
  extern __shared__ __align__(16) char s_dyn_raw[];

  const int T = blockDim.x, W = T / kWave;
  const int tid = threadIdx.x;
  const int wv = uni(tid / kWave), lane = tid % kWave;
  const int ng = p.tile_groups;
  const int nt = ng / 2;                        // matrix tiles of 16 rows (two groups) per set
  char *ptr = s_dyn_raw;
  auto carve = [&](size_t bytes) { char *r = ptr; ptr += bytes; return r; };
  const AdjRecord<TWO> rec{ng};
  double *const s_om = (double *)carve((size_t)ng * kGroup * 8);                      // omega / 2pi
  double *const s_alpha = (double *)carve((size_t)ng * 8);                            // group centres / 2pi
  double *const s_lo = (double *)carve((size_t)ng * 8);                               // bounds of |omega| / 2pi
  double *const s_hi = (double *)carve((size_t)ng * 8);
  uint32_t *const s_cross = (uint32_t *)carve(16);   // groups on both sides of zero, groups of ascending |omega|
  auto s_up = [&](int g) { return ((s_cross[1] >> g) & 1u) != 0; };
  char *const s_own = ptr + wv * kAdjWaveBytes;
  float2 *const s_fac = (float2 *)s_own;        // [7][kAdjRow]: e^{i (4 k1 + 1/2) d}, e^{i k0 d}
  float4 *const s_al = (float4 *)s_own;         // then, twice [64]: cos, sin of two group centres
  float *const s_out = (float *)s_own;          // then [set][word][64]
  uint32_t *const s_msk = (uint32_t *)(s_own + 7 * kAdjRow * 8 + 32);
  double *const s_geo = (double *)(s_msk + kWave);   // [64 directions][n, e_theta, e_phi x, y]

  const int n_ranges = p.n_ranges;
  const int rg = (int)(blockIdx.x % (uint32_t)n_ranges);
  const int64_t rest = blockIdx.x / (uint32_t)n_ranges;
  const int64_t lp = rest % p.chunk_n;
  const int q_dir = (int)(rest / p.chunk_n);
  const int64_t ip = p.chunk_base + lp;
  const double dt = p.dt;
  const float one = late_s(1.0f);
  const double step_inv = 1.0 / fabs(p.domega_rev);
  const int col = lane & 15, quad = lane >> 4;

  const Particle pt = load_particle(p, ip);
  const int64_t n_use = adj_steps(p, pt);
  const uint32_t d_lo = (uint32_t)((int64_t)p.dir_n * q_dir / p.n_groups);
  const uint32_t d_hi = (uint32_t)((int64_t)p.dir_n * (q_dir + 1) / p.n_groups);
  double *slab = p.slab + (int64_t)q_dir * kSlabWords * p.n_points;

  int n_om = 0;
  // how many of group g's frequencies a step of threshold thr keeps, those of smallest
  // |omega|; the group's |omega| ascend (up) or descend.  On a linear grid the count is
  // known to one, and the threshold's own comparison settles it
  auto kept_of = [&](int g, bool up, double thr) -> int {
    const double *w = s_om + g * kGroup;
    const int cnt = min(kGroup, n_om - g * kGroup);
    int r = min((int)fmin(fmax((thr - s_lo[g]) * step_inv, 0.0), 31.0) + 1, cnt - 1);
    const double in = fabs(w[up ? max(r - 1, 0) : cnt - max(r, 1)]), out = fabs(w[up ? r : cnt - 1 - r]);
    // (past the grid's end a descending group's frequencies count as kept: zeros)
    return r + ((out < thr && r < cnt - 1) ? 1 : (!(in < thr) && r > 0) ? -1 : 0) + (up ? 0 : kGroup - cnt);
  };

  for (int64_t base = (int64_t)rg * T; base < n_use; base += (int64_t)n_ranges * T) {
    const int64_t s = base + tid;
    const bool active = s < n_use;
    const bool wave_active = base + wv * kWave < n_use;
    // the step (idle lanes: a step at rest at the origin, whose sums go nowhere)
    double xs = 0.0, ys = 0.0, zs = 0.0;
    double a[3] = {0.0, 0.0, 0.0}, m[3] = {0.0, 0.0, 0.0};
    const int64_t gs = pt.off + s;
    if (active) {
      xs = p.x[gs]; ys = p.y[gs]; zs = p.z[gs];
      // direction-independent part of the step (kernel_farfield.cl:74-83)
      const double *am = p.pre + 6 * gs;
#pragma unroll
      for (int c = 0; c < 3; c++) { a[c] = am[c]; m[c] = am[3 + c]; }
    }
    // the step before the wave's first (the others' is the lane below)
    const int64_t s_w = base + wv * kWave;
    double xp = 0.0, yp = 0.0, zp = 0.0;
    if (wave_active && s_w > 0) {
      xp = unid(p.x[pt.off + s_w - 1]); yp = unid(p.y[pt.off + s_w - 1]); zp = unid(p.z[pt.off + s_w - 1]);
    }
    double acc9[kSlabWords];
#pragma unroll
    for (int k = 0; k < kSlabWords; k++) acc9[k] = 0.0;

    for (int wt = 0; wt < p.n_wtiles; wt++) {
    const int w0 = wt * ng * kGroup;
    n_om = min(ng * kGroup, (int)p.n_omega - w0);
    __syncthreads();   // the previous omega tile's bounds are read
    if (tid < 2) s_cross[tid] = 0;
    __syncthreads();
    for (int i = tid; i < ng * kGroup; i += T) s_om[i] = i < n_om ? p.omega[w0 + i] * kInv2Pi : 0.0;
    for (int i = tid; i < ng; i += T) {
      const int first = i * kGroup, last = min(first + kGroup, n_om) - 1;
      double al = 0.0, lo = 0.0, hi = 0.0;    // a group past the grid's end: all kept, all zero
      if (first <= last) {
        const double wa = p.omega[w0 + first] * kInv2Pi, wb = p.omega[w0 + last] * kInv2Pi;
        al = fma(15.5, p.domega_rev, wa);
        hi = fmax(fabs(wa), fabs(wb));
        lo = fmin(fabs(wa), fabs(wb));
        if (fabs(wb) >= fabs(wa)) atomicOr(&s_cross[1], 1u << i);
        if ((wa < 0.0) != (wb < 0.0)) {
          lo = 0.0;
          atomicOr(&s_cross[0], 1u << i);
        }
      }
      s_alpha[i] = al; s_lo[i] = lo; s_hi[i] = hi;
    }
    __syncthreads();
    if (wave_active) {
      double w_top = 0.0;
      for (int g = 0; g < ng; g++) w_top = fmax(w_top, s_hi[g]);
      const char *rec_at = p.tab + (((size_t)lp * p.n_wtiles + wt) * p.dir_n + d_lo) * rec.bytes();
      // ---- transpose sweep: lanes = steps, loop over the directions ----
      for (uint32_t d = d_lo; d < d_hi; d++, rec_at += rec.bytes()) {
        // the first tile's operands, used after the basis is formed
        const uint4v *tab = (const uint4v *)rec_at + lane;
        const float *scl = (const float *)(rec_at + rec.scl_at()) + quad;
        uint4v th[NSET], tl[NSET];
#pragma unroll
        for (int set = 0; set < NSET; set++) {
          th[set] = tab[set * 2 * kWave];
          tl[set] = tab[(set * 2 + 1) * kWave];
        }
        const uint32_t dl = (d - d_lo) & (kWave - 1);
        if (dl == 0) {
          sr::wave_sync();
          const uint32_t dir = p.dir_lo + min(d + lane, d_hi - 1);
          const uint32_t iPhi = dir / p.n_theta;
          const uint32_t iTh = dir - iPhi * p.n_theta;
          const double st = p.sin_t[iTh], ct = p.cos_t[iTh], sp = p.sin_p[iPhi], cp = p.cos_p[iPhi];
          double *q = s_geo + 8 * lane;
          q[0] = st * cp; q[1] = st * sp; q[2] = ct;
          q[3] = ct * cp; q[4] = ct * sp; q[5] = -st;
          q[6] = -sp; q[7] = cp;
          sr::wave_sync();
        }
        const double *const gq = s_geo + 8 * dl;
        double tau, dtau;
        {
          const double nx = gq[0], ny = gq[1], nz = gq[2];
          const double time = (double)(uint32_t)(pt.its + (uint32_t)s) * dt;
          const double tp = (double)(uint32_t)(pt.its + (uint32_t)(s_w - 1)) * dt;
          tau = time - (xs * nx + ys * ny + zs * nz);
          const double below = lane_below(tau);
          const double first = s_w > 0 ? tp - (xp * nx + yp * ny + zp * nz) : 0.0;
          dtau = active ? fabs(tau - (lane == 0 ? first : below)) : 0.0;
        }
        // basis factors of the lane's step
        const double dr = p.domega_rev * tau;
#pragma unroll
        for (int k = 0; k < 7; k++) {
          float sn, cs;
          sincos_rev(k < 4 ? dr * (4.0 * k + 0.5) : dr * (k - 3.0), &sn, &cs);
          s_fac[k * kAdjRow + lane] = make_float2(cs, sn);
        }
        // steps that keep every frequency need no threshold (the comparison below is
        // on the safe side of its rounding)
        const bool all_kept = w_top * dtau < 0.5 * (1.0 - 1e-12);
        const bool cuts = __ballot(!all_kept) != 0;
        double thr = 0.0;
        uint32_t whole = 0, part = 0;
        uint32_t slow = 0;           // cut groups that the masked product does not take
        int cut_at = 0, cut_r = 0;   // the lane's cut group and its kept count
        if (cuts) {
          thr = 0.5 / dtau;
          for (int g = 0; g < ng; g++) {
            const uint32_t w = s_hi[g] < thr, l = s_lo[g] < thr;
            whole |= w << g;
            part |= (l & ~w) << g;
          }
          // a step that keeps more than half of the group it cuts takes it whole, less the
          // offsets of one side that it drops; else it takes the kept offsets of one side.
          // Groups on both sides of zero and coefficients that are not finite go apart
          if (part != 0) {
            const uint32_t odd = *(const uint32_t *)(rec_at + rec.flag_at()) | *s_cross;
            slow = part & odd;
            part &= ~odd;
            slow |= part & (part - (part != 0));   // (a grid across zero can be cut on both sides)
            if (part != 0) {
              cut_at = __builtin_ctz(part);
              cut_r = kept_of(cut_at, s_up(cut_at), thr);
              part = 1u << cut_at;
              if (cut_r > 16) whole |= part;
            }
          }
          s_msk[lane] = whole;
        }
        sr::wave_sync();
        // the wave's matrix operand: basis of steps 16 blk + col
        uint4v bh[4], bl[4];
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
          const int at = 16 * blk + col;
          const float2 x1 = s_fac[quad * kAdjRow + at];
          float c[4], sn[4];
          c[0] = x1.x;
          sn[0] = x1.y;
#pragma unroll
          for (int k = 1; k < 4; k++) {
            const float2 x0 = s_fac[(3 + k) * kAdjRow + at];
            c[k] = __builtin_fmaf(x1.x, x0.x, -(x1.y * x0.y));
            sn[k] = __builtin_fmaf(x1.x, x0.y, x1.y * x0.x);
          }
#pragma unroll
          for (int k = 0; k < 2; k++) {
            const uint2 wc = split_values(c[2 * k], c[2 * k + 1], one), ws = split_values(sn[2 * k], sn[2 * k + 1], one);
            bh[blk][k] = wc.x; bl[blk][k] = wc.y;
            bh[blk][2 + k] = ws.x; bl[blk][2 + k] = ws.y;
          }
        }
        uint32_t mk[4] = {0, 0, 0, 0};
        if (cuts) {
#pragma unroll
          for (int blk = 0; blk < 4; blk++) mk[blk] = s_msk[16 * blk + col];
        }
        sr::wave_sync();   // the factors are read: their LDS holds the group centres' phasors now
        float out[NSET][4];
#pragma unroll
        for (int set = 0; set < NSET; set++)
#pragma unroll
          for (int blk = 0; blk < 4; blk++) out[set][blk] = 0.f;
        // the centres' phasors of the lane's step, a tile ahead
        auto centres = [&](int t, int buf) {
          float4 v;
          sincos_rev(s_alpha[2 * t] * tau, &v.y, &v.x);
          sincos_rev(s_alpha[2 * t + 1] * tau, &v.w, &v.z);
          s_al[buf * kWave + lane] = v;
        };
        auto operands = [&](int t) {
#pragma unroll
          for (int set = 0; set < NSET; set++) {
            th[set] = tab[(t * NSET + set) * 2 * kWave];
            tl[set] = tab[((t * NSET + set) * 2 + 1) * kWave];
          }
        };
        // the tiles with a group that a step of the wave keeps whole
        uint32_t need = (1u << nt) - 1;
        if (cuts) {
          need = 0;
          for (int t = 0; t < nt; t++) need |= __ballot((whole >> (2 * t)) & 3u) != 0 ? 1u << t : 0u;
        }
        int t = need != 0 ? __builtin_ctz(need) : 0;
        if (need != 0) {
          if (t != 0) operands(t);
          centres(t, 0);
        }
        sr::wave_sync();
#pragma unroll 1
        for (int buf = 0; need != 0; buf ^= 1) {
          need &= need - 1;
          const int next = need != 0 ? __builtin_ctz(need) : -1;
          float sc[NSET][2];
#pragma unroll
          for (int set = 0; set < NSET; set++) {
            sc[set][0] = scl[(2 * t * NSET + set) * 4];
            sc[set][1] = scl[((2 * t + 1) * NSET + set) * 4];
          }
          float4 av[4];
#pragma unroll
          for (int blk = 0; blk < 4; blk++) av[blk] = s_al[buf * kWave + 16 * blk + col];
          if (next >= 0) centres(next, buf ^ 1);
          sr::wave_sync();
#pragma unroll
          for (int set = 0; set < NSET; set++) {
            float4v U[4];
#pragma unroll
            for (int blk = 0; blk < 4; blk++) U[blk] = mfma16(tl[set], bh[blk], (float4v)(0.f));
#pragma unroll
            for (int blk = 0; blk < 4; blk++) U[blk] = mfma16(th[set], bl[blk], U[blk]);
#pragma unroll
            for (int blk = 0; blk < 4; blk++) U[blk] = mfma16(th[set], bh[blk], U[blk]);
            const float sc0 = sc[set][0], sc1 = sc[set][1];
            if (next >= 0) {
              th[set] = tab[(next * NSET + set) * 2 * kWave];
              tl[set] = tab[((next * NSET + set) * 2 + 1) * kWave];
            }
            float u0[4], u1[4];
#pragma unroll
            for (int blk = 0; blk < 4; blk++) {
              u0[blk] = __builtin_fmaf(av[blk].x, U[blk][0], av[blk].y * U[blk][1]);
              u1[blk] = __builtin_fmaf(av[blk].z, U[blk][2], av[blk].w * U[blk][3]);
            }
            if (cuts) {
              // (selected, not multiplied by zero: a coefficient that is not finite stays
              // with the steps that keep it)
#pragma unroll
              for (int blk = 0; blk < 4; blk++) {
                const uint32_t k = mk[blk] >> (2 * t);
                u0[blk] = (k & 1u) ? u0[blk] : 0.f;
                u1[blk] = (k & 2u) ? u1[blk] : 0.f;
              }
            }
#pragma unroll
            for (int blk = 0; blk < 4; blk++)
              out[set][blk] = __builtin_fmaf(sc1, u1[blk], __builtin_fmaf(sc0, u0[blk], out[set][blk]));
          }
          t = next;
        }
        // the groups that steps of the wave cut, mostly one: the table's two sides, eight rows
        // each, times the basis masked to the offsets from |16 - kept| on -- the side kept if
        // that is less than half of the group, the side dropped, to be subtracted, if more
        if (cuts) {
          for (int g = 0; g < ng; g++) {
            const bool mine = part != 0 && cut_at == g;
            if (__ballot(mine) == 0) continue;
            const bool up = s_up(g);
            float2 ph;
            sincos_rev(s_alpha[g] * tau, &ph.y, &ph.x);
            const bool more = cut_r > 16;
            const bool low = mine && more != up, high = mine && more == up;
            const float cs = more ? -ph.x : ph.x, sn = more ? -ph.y : ph.y;
            const uint32_t from = mine ? (uint32_t)(more ? cut_r - 16 : 16 - cut_r) : 16u;
            sr::wave_sync();
            s_msk[lane] = from | (from << 16);
            // (selected, not multiplied by zero: the phase of a step at a position that is
            // not finite stays out of its sums, as the step does)
            s_al[lane] = make_float4(low ? cs : 0.f, low ? sn : 0.f, high ? cs : 0.f, high ? sn : 0.f);
            sr::wave_sync();
#pragma unroll
            for (int set = 0; set < NSET; set++) {
              const uint4v *tb = (const uint4v *)rec_at + ((g >> 1) * NSET + set) * 2 * kWave + ((lane & ~2) | (2 * (g & 1)));
              uint4v gh, gl;
              two_sides(tb[0], tb[kWave], one, &gh, &gl);
              const float sc = scl[(g * NSET + set) * 4];
#pragma unroll
              for (int blk = 0; blk < 4; blk++) {
                const short2v fr = __builtin_bit_cast(short2v, s_msk[16 * blk + col]);
                const float4 al = s_al[16 * blk + col];
                uint4v mh, ml;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                  // offsets 4 quad + 2 k, + 1: all ones where from <= offset
                  const short b0 = (short)(4 * quad + 2 * k + 1);
                  const short2v off = {b0, (short)(b0 + 1)};
                  const uint32_t mm = __builtin_bit_cast(uint32_t, (short2v)((fr - off) >> 15));
#pragma unroll
                  for (int h = 0; h < 4; h += 2) {
                    mh[h + k] = bh[blk][h + k] & mm;
                    ml[h + k] = bl[blk][h + k] & mm;
                  }
                }
                float4v U = mfma16(gl, mh, (float4v)(0.f));
                U = mfma16(gh, ml, U);
                U = mfma16(gh, mh, U);
                const float u = __builtin_fmaf(al.x, U[0], al.y * U[1]) + __builtin_fmaf(al.z, U[2], al.w * U[3]);
                out[set][blk] = __builtin_fmaf(sc, u, out[set][blk]);
              }
            }
          }
        }
        // back to a step per lane
        sr::wave_sync();
#pragma unroll
        for (int set = 0; set < NSET; set++)
#pragma unroll
          for (int blk = 0; blk < 4; blk++) s_out[(set * 4 + quad) * kWave + 16 * blk + col] = out[set][blk];
        sr::wave_sync();
        float P[NCW], R[NCW];
#pragma unroll
        for (int c = 0; c < NCW; c++) {
          P[c] = s_out[c * kWave + lane];
          R[c] = s_out[(TWO ? NCW + c : 4 + c) * kWave + lane];
        }
        // the cut groups left: only the frequencies that are kept may be touched
        while (slow != 0) {
          const int g = __builtin_ctz(slow);
          slow &= slow - 1;
          for (int j = g * kGroup; j < min((g + 1) * kGroup, n_om); j++) {
            const double w = s_om[j];
            if (!(fabs(w) < thr)) continue;
            float sn, cs;
            sincos_rev(w * tau, &sn, &cs);
            const float *rw = (const float *)(rec_at + rec.raw_at()) + j * 2 * NCW;
#pragma unroll
            for (int c = 0; c < NCW; c++) {
              P[c] = __builtin_fmaf(rw[c], cs, __builtin_fmaf(rw[NCW + c], sn, P[c]));
              R[c] = __builtin_fmaf((float)w, __builtin_fmaf(rw[c], sn, -rw[NCW + c] * cs), R[c]);
            }
          }
        }
        sr::wave_sync();   // read before the next direction's factors
        const double nv[3] = {gq[0], gq[1], gq[2]};
        auto dot3 = [](const double *u, double x, double y, double z) { return fma(u[0], x, fma(u[1], y, u[2] * z)); };
        const double mn = dot3(m, nv[0], nv[1], nv[2]);
        const double c2 = 1.0 / (1.0 - mn);
        const double c1 = dot3(a, nv[0], nv[1], nv[2]) * c2 * c2;
        double Q[3], AR, nmg, ag;
        if constexpr (TWO) {
          // everything on e_theta, e_phi: A and dL/dA have no part along n
          const double et[3] = {gq[3], gq[4], gq[5]}, ep[2] = {gq[6], gq[7]};
          const double mt = dot3(m, et[0], et[1], et[2]), mp = fma(m[0], ep[0], m[1] * ep[1]);
          const double at = dot3(a, et[0], et[1], et[2]), ap = fma(a[0], ep[0], a[1] * ep[1]);
          const double p0 = (double)P[0], p1 = (double)P[1];
          AR = -fma(fma(c1, mt, c2 * at), (double)R[0], fma(c1, mp, c2 * ap) * (double)R[1]);
          nmg = -fma(mt, p0, mp * p1);
          ag = fma(at, p0, ap * p1);
          Q[0] = fma(p0, et[0], p1 * ep[0]);
          Q[1] = fma(p0, et[1], p1 * ep[1]);
          Q[2] = p0 * et[2];
        } else {
          AR = 0.0; nmg = 0.0; ag = 0.0;
#pragma unroll
          for (int c = 0; c < 3; c++) {
            Q[c] = (double)P[c];
            AR += (c1 * (nv[c] - m[c]) - c2 * a[c]) * (double)R[c];
            nmg += (nv[c] - m[c]) * Q[c];
            ag += a[c] * Q[c];
          }
        }
        AR *= 2.0 * kPi;   // revolutions -> radians
        const double ka = c2 * c2 * nmg, km = fma(2.0 * c1 * c2, nmg, -(c2 * c2 * ag));
#pragma unroll
        for (int c = 0; c < 3; c++) {
          acc9[c] = fma(nv[c], AR, acc9[c]);
          acc9[3 + c] = fma(nv[c], km, fma(-c1, Q[c], acc9[3 + c]));
          acc9[6 + c] = fma(nv[c], ka, fma(-c2, Q[c], acc9[6 + c]));
        }
      }
    }
    }
    if (active) {
#pragma unroll
      for (int k = 0; k < kSlabWords; k++) slab[(int64_t)k * p.n_points + gs] += acc9[k];
    }
  }
}

}  // namespace
