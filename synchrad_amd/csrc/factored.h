// factored.h -- the split-precision spectrum on a linear omega grid as matrix
// products (gfx950 MFMA).
//
// On a linear grid a direction's 32*NG frequencies are NG groups of 32 around
// group centres alpha_a, at offsets +-beta_b, beta_b = (b + 1/2) domega:
//   cos((alpha +- beta) tau) = cos a cos b -+ sin a sin b
//   sin((alpha +- beta) tau) = sin a cos b +- cos a sin b
// so the sums over the steps s of A_s e^{i omega tau_s} at all of them are the
// four real products P_uv[a][b] = sum_s (A_s u(alpha_a tau_s)) v(beta_b tau_s),
// u, v in {cos, sin}: matrices of 16 rows (a) x 16 columns (b) contracted over
// the steps.  A step then costs four phasors and NG + 16 products of them instead of
// a sine or a rotation for each of the 32*NG frequencies, and the multiply-adds run
// on the matrix cores.
//
// FP32 in fp16 matrix instructions: every factor x is two fp16 words, x = hi +
// lo with hi = fp16(x), lo = fp16(x - hi) (22 to 24 bits), and a product is
// hi hi + hi lo + lo hi (the dropped lo lo is below 2^-22 of the product), each
// exact in the FP32 accumulator's product.  Each amplitude word is scaled by a power
// of two per track stretch so that its values stay in fp16's range.  The
// FP32 accumulators hold a few blocks of steps, then go into FP64 sums.
//
// Phases: per step the stage takes tau * domega/2 and the first group's centre
// phase to revolutions in FP64 and removes whole turns.  A block of steps forms, per
// step and side (columns, rows), the phasors of the first phase p and of the spacing d
// by FP64 polynomials, and from them e^{i (p + 4 k1 d)} and e^{i k0 d}, k1, k0 = 0..3, by
// FP64 products, rounded to FP32 in LDS; column or row 4 k1 + k0 is the FP32 product of
// two of these.
//
// The |dphase| < pi filter keeps, at step s, the K_s frequencies of smallest
// |omega| (threshold form, as in the direct sweep; K_s by the same comparison
// with the grid's own values).  Steps that keep all of the tile's frequencies
// and steps that cut them go through separate queues: for the former no mask is
// needed; for the latter the groups below K_s enter as they are and the one
// group that K_s cuts (row a = K_s / 32) enters a second product with masked
// columns.  Steps that keep nothing are dropped.
//
// Work split: a block owns a tile (direction or screen point, run of 32*NG
// frequencies, particle slice); its W waves take the 63-step stretches of each
// track in turn (one lane of a stretch recomputes the step before it, whose tau
// the filter needs), each with its own queues and accumulators, and meet only at
// snapshot records.
#pragma once

#include "tile_params.h"

namespace sr {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef short short2v __attribute__((ext_vector_type(2)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kGroup = 32;        // frequencies per group
constexpr int kBlockSteps = 32;   // steps per matrix product (its contracted length)
constexpr int kQueue = 96;        // ring capacity: 31 left over + 64 new
// blocks of steps between two folds of the FP32 accumulators into FP64.  A fold
// costs about as much as a third of a block; fewer blocks round less.  Over 29
// far- and near-field cases of 1 to 290 tracks the error against FP64 was 0.2 to
// 0.95 times that of sines rotated in FP32 and summed by Kahan's rule at 3 far and 8
// near (far at
// 8: up to 1.5 times, betatron tracks of 4000 steps; 24 betatron electrons on 512 x
// 32 x 32 take 7.68 ms at 3 against 7.43 at 8)
template <int MODE>
constexpr int fold_blocks() {
  return MODE == SR_MODE_FAR ? 3 : 8;
}

template <int MODE>
constexpr int factored_words() {
  return MODE == SR_MODE_FAR ? 2 : 6;
}
// bytes of one step queue: half-step phase, centre phase, amplitude words, kept
// count
template <int MODE>
constexpr int queue_bytes() {
  return kQueue * (16 + 4 * factored_words<MODE>() + 2);
}
// factors of one block of steps: for the columns and for the rows, e^{i(p + 4 k1
// d)} and e^{i k0 d}, k1, k0 = 0..3, a row of 32 steps for each word.  The words of
// one kind (k = 0..3) are laid out so that a wave's 16 different 16-byte reads of
// them (4 k, 4 groups of 8 steps) fall on different LDS banks, and the two sides
// half the banks apart, so that the 64 lanes' writes do too.
enum { FAC_1RE, FAC_1IM, FAC_0RE, FAC_0IM, FAC_0NIM, FAC_KINDS };
constexpr int kFactorKind = 136;
constexpr int kFactorSide = 736;
__device__ __forceinline__ constexpr int factor_at(int kind, int k) { return kind * kFactorKind + 32 * k + 4 * (k >> 1); }
constexpr int kFactorBytes = 2 * kFactorSide * 4;
// the tile's constants, read where they are used instead of held in registers
enum { TC_GX, TC_GY, TC_GZ, TC_THX, TC_THY, TC_THZ, TC_PHX, TC_PHY, TC_DT, TC_HALF, TC_C0, TC_WLO, TC_WHI, TC_INV, TC_COUNT };
template <int MODE>
constexpr int wave_bytes() {
  return 3 * queue_bytes<MODE>() + kFactorBytes;
}
template <int MODE, int NG>
constexpr size_t factored_lds(int waves, bool acc) {
  return (size_t)(TC_COUNT + NG * kGroup) * 8 + (size_t)waves * wave_bytes<MODE>() + (acc ? (size_t)NG * kGroup * 8 : 0);
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// value of the previous lane (lane 0: unspecified)
__device__ __forceinline__ double lane_below(double v) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)((uint64_t)b >> 32), 0x138, 0xf, 0xf, true);
  return __longlong_as_double((int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// The value unchanged, in one register from here on (an empty asm statement): the
// halves of a pair are then read from the packed word instead of being formed twice
__device__ __forceinline__ half2v packed(half2v h) {
  uint32_t v = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(v));
  return __builtin_bit_cast(half2v, v);
}
// (as above for an FP32 value: the compiler would otherwise round a mixed FMA to
// fp16 in the instruction that does so, which runs at half the rate of the FP32
// mixed FMA and the packed conversion together: 8.5 against 4.4 cycles each)
__device__ __forceinline__ float keep(float v) {
  asm("" : "+v"(v));
  return v;
}
// two products t0 m0, t1 m1 as two packed fp16 words: high words rounded from the
// products, low words from the unrounded products minus the high words
__device__ __forceinline__ uint2 split_pair(float t0, float m0, float t1, float m1) {
  float2v x;
  x.x = t0 * m0;
  x.y = t1 * m1;
  const half2v h = packed(__builtin_convertvector(x, half2v));
  float2v r;
  r.x = keep(__builtin_fmaf(t0, m0, -(float)h.x));
  r.y = keep(__builtin_fmaf(t1, m1, -(float)h.y));
  const half2v l = __builtin_convertvector(r, half2v);
  return make_uint2(__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l));
}
// two values as two packed fp16 words (one: an opaque 1)
__device__ __forceinline__ uint2 split_values(float x0, float x1, float one) {
  float2v x;
  x.x = x0;
  x.y = x1;
  const half2v h = packed(__builtin_convertvector(x, half2v));
  float2v r;
  r.x = keep(__builtin_fmaf(x0, one, -(float)h.x));
  r.y = keep(__builtin_fmaf(x1, one, -(float)h.y));
  const half2v l = __builtin_convertvector(r, half2v);
  return make_uint2(__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, l));
}

__device__ __forceinline__ float4v mfma16(uint4v a, uint4v b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, a), __builtin_bit_cast(half8v, b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t below_mask(int bound, uint32_t k) {
  // per 16-bit half: all ones where bound < k (both below 2^15)
  const short2v v = (short2v)(short)bound - __builtin_bit_cast(short2v, k);
  return __builtin_bit_cast(uint32_t, v >> 15);
}

// e^{2 pi i rev} for |rev| <= 1/2, about 2e-10 absolute: polynomials of the
// quarter angle (least-maximum fits on |x| <= pi/4: sin to x^9, 2.3e-12; cos to
// x^8, 5.4e-11), squared twice
__device__ __forceinline__ void phasor(double rev, double *c, double *s) {
  const double x = rev * 1.5707963267948966;
  const double z = x * x;
  double ps = fma(z, 2.7160140045195716e-06, -0.00019839043768864802);
  ps = fma(ps, z, 0.008333328238709012);
  ps = fma(ps, z, -0.16666666627998977);
  double pc = fma(z, 2.4390450554142482e-05, -0.0013886763792706424);
  pc = fma(pc, z, 0.04166662332428502);
  pc = fma(pc, z, -0.4999999972510758);
  double sn = fma(x * z, ps, x), cn = fma(z, pc, 1.0);
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const double t = sn + sn;
    const double c2 = fma(-t, sn, 1.0);
    sn = t * cn;
    cn = c2;
  }
  *c = cn;
  *s = sn;
}

// waves per SIMD each variant is held to: the largest count at which nothing is
// spilled (16 groups without the pre-pass: two values; a spilled register costs more than the wave: with 0.3 KB of scratch per
// lane the far kernels ran 1.5 to 3 times slower)
template <int MODE, int NG>
constexpr int factored_waves() {
  return (MODE == SR_MODE_FAR && NG == 4) ? 3 : 2;
}
template <int MODE, int NG, bool PRE>
__global__ void __launch_bounds__(kMaxT) __attribute__((amdgpu_waves_per_eu(factored_waves<MODE, NG>())))
k_factored(const KParams p) {
  constexpr int NW = factored_words<MODE>();
  constexpr int NB = NG * 2 * NW / 16;     // 16-row blocks of the left factor
  constexpr int NAL = NG / 4;              // groups per lane of the result
  // the cut groups' sums: field sums (re, im of each word) where cos and sin rows
  // are separate blocks, else P_uv
  constexpr int ND = NG == 16 ? NB : 2 * NB;
  constexpr int kRun = NG * kGroup;

  extern __shared__ __align__(16) char s_raw[];
  const int W = blockDim.x / kWave;
  const int tid = threadIdx.x;
  const int wv = uni(tid / kWave);
  const int lane = tid % kWave;
  double *const s_tc = (double *)s_raw;
  double *const s_om = s_tc + TC_COUNT;                                   // |omega|/2pi of the tile, ascending
  char *const s_waves = (char *)(s_om + kRun);
  char *const s_own = s_waves + wv * wave_bytes<MODE>();
  double *const s_acc = (double *)(s_waves + W * wave_bytes<MODE>());
  auto q_xh = [&](int q) { return (double *)(s_own + q * queue_bytes<MODE>()); };
  auto q_c0 = [&](int q) { return q_xh(q) + kQueue; };
  auto q_amp = [&](int q) { return (float *)(q_c0(q) + kQueue); };        // [NW][kQueue]
  auto q_cnt = [&](int q) { return (uint16_t *)(q_amp(q) + NW * kQueue); };

  float *const s_fac = (float *)(s_own + 3 * queue_bytes<MODE>());         // columns, then rows
  // the lane's place in the matrix factors: row (group and trigonometric
  // function; both functions where a row is a group) of the left one, column of
  // the right one, and the factors it multiplies (rows that hold one function:
  // cos = re re + im (-im), sin = re im + im re)
  struct Lanes {
    int kg, rc, row_a, row_w;
    const float *col1, *col0, *row1, *row0p, *row0q;
  };
  auto lanes = [&]() {
    Lanes L;
    const int lb = late(lane);
    L.kg = lb >> 4;
    L.rc = lb & 15;
    L.row_a = NG == 16 ? L.rc : NG == 8 ? L.rc >> 1 : L.rc >> 2;
    const int row_u = NG == 16 ? 0 : L.rc & 1;
    L.row_w = NG == 4 ? (L.rc >> 1) & 1 : 0;
    const float *f = s_fac + 8 * L.kg;
    L.col1 = f + factor_at(FAC_1RE, L.rc >> 2);
    L.col0 = f + factor_at(FAC_0RE, L.rc & 3);
    L.row1 = f + kFactorSide + factor_at(FAC_1RE, L.row_a >> 2);
    L.row0p = f + kFactorSide + factor_at(row_u ? FAC_0IM : FAC_0RE, L.row_a & 3);
    L.row0q = f + kFactorSide + factor_at(row_u ? FAC_0RE : FAC_0NIM, L.row_a & 3);
    return L;
  };
  // held in registers where there is room, else formed once per block of steps
  constexpr bool kHoist = NG < 16;
  const Lanes held = lanes();
  const double dt = p.dt;
  const float one = late_s(1.0f);
  const bool spheric = (p.comp == SR_COMP_SPHERIC || p.comp == SR_COMP_SPHERIC_COMPLEX);

  for (int64_t ti = blockIdx.x; ti < p.n_tiles; ti += gridDim.x) {
    const uint32_t tile = p.tile_order ? (uint32_t)p.tile_order[ti] : (uint32_t)ti;
    const uint32_t rest = udiv(tile, p.div_chunks);
    const uint32_t chunk = tile - rest * p.n_chunks;
    const uint32_t qs = udiv(rest, p.div_dir);
    const uint32_t dir = rest - qs * p.n_dir;
    const int slice = (int)qs;
    const uint32_t iPhi = udiv(dir, p.div_theta);
    const uint32_t iTh = dir - iPhi * p.n_theta;

    // output c of this tile (slices: the slice's partial spectra)
    auto dst = [&](int c) -> double * {
      return (p.slices > 1 && p.part_stride == 0)
                 ? p.scratch + ((int64_t)slice * p.n_out + c) * p.n_grid * p.n_snaps
                 : p.out[c];
    };

    // The run's frequencies in the order of ascending |omega|: one part, or two
    // where the run crosses zero (swept one after the other)
    const int k0 = (int)chunk * kRun, k1 = min(k0 + kRun, (int)p.n_omega);
    const double w_a = unid(p.omega[k0]), w_b = unid(p.omega[k1 - 1]);
    int kz = k0;                                  // crossing: first frequency past zero
    const bool crossing = (w_a < 0.0 && w_b > 0.0) || (w_a > 0.0 && w_b < 0.0);
    if (crossing) {
      int lo = k0, hi = k1 - 1;                   // the sign of omega[lo] is w_a's, of omega[hi] not
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        const double w = unid(p.omega[mid]);
        if ((w_a < 0.0) ? (w < 0.0) : (w > 0.0)) lo = mid; else hi = mid;
      }
      kz = hi;
    }
    for (int part = 0; part < (crossing ? 2 : 1); part++) {
      int first, count, sgn;
      if (!crossing) {
        sgn = fabs(w_b) >= fabs(w_a) ? 1 : -1;
        first = sgn > 0 ? k0 : k1 - 1;
        count = k1 - k0;
      } else if (part == 0) {
        sgn = -1; first = kz - 1; count = kz - k0;
      } else {
        sgn = 1; first = kz; count = k1 - kz;
      }
      const double om_first = unid(p.omega[first]);
      const double step = (double)sgn * p.omega_step;                       // signed step along the order
      const double half_rev = 0.5 * step * kInv2Pi;                         // half a step, revolutions per length
      const double c0_rev = (om_first + 15.5 * step) * kInv2Pi;             // centre of the first group
      __syncthreads();   // an earlier part or tile of this block is done with s_om, s_acc
      const int td = late(tid);
      for (int j = td; j < kRun; j += blockDim.x)
        s_om[j] = j < count ? fabs(p.omega[first + sgn * j]) * kInv2Pi : INFINITY;
      if (p.acc_lds)
        for (int j = td; j < kRun; j += blockDim.x) s_acc[j] = 0.0;
      if (td == 0) {
        // geometry of the block's point (kernel_farfield.cl:40-42, 384-387;
        // kernel_nearfield.cl:40-42): far n, e_theta, e_phi; near the screen point
        if (MODE == SR_MODE_FAR) {
          const double st = p.sin_t[iTh], ct = p.cos_t[iTh];
          const double sp = p.sin_p[iPhi], cp = p.cos_p[iPhi];
          s_tc[TC_GX] = st * cp; s_tc[TC_GY] = st * sp; s_tc[TC_GZ] = ct;
          s_tc[TC_THX] = ct * cp; s_tc[TC_THY] = ct * sp; s_tc[TC_THZ] = -st;
          s_tc[TC_PHX] = -sp; s_tc[TC_PHY] = cp;
        } else {
          const double r = p.radius[iTh];
          s_tc[TC_GX] = p.screen_y ? r : r * p.cos_p[iPhi];
          s_tc[TC_GY] = p.screen_y ? p.screen_y[iPhi] : r * p.sin_p[iPhi];
          s_tc[TC_GZ] = p.l_screen;
        }
        s_tc[TC_DT] = dt;
        s_tc[TC_HALF] = half_rev;
        s_tc[TC_C0] = c0_rev;
        s_tc[TC_WLO] = fabs(om_first) * kInv2Pi;
        s_tc[TC_WHI] = fabs(p.omega[first + sgn * (count - 1)]) * kInv2Pi;
        s_tc[TC_INV] = 1.0 / fabs(step * kInv2Pi);
      }
      __syncthreads();

      const int64_t p_lo = p.slice_lo[slice], p_hi = p.slice_lo[slice + 1];
      for (int64_t ip = p_lo; ip < p_hi; ip++) {
        const Particle pt = load_particle(p, ip);
        if (pt.n <= 0) continue;
        const int64_t n_act = max((int64_t)0, min(pt.n - 1, (int64_t)pt.ite - 1));
        SnapCursor cur;
        cur.init(pt, p.n_snaps);
        if (cur.next < 0) continue;   // no record: the sums go nowhere

        // the queued amplitude words are scaled by 2^ex[word], following the track's
        // own amplitudes only, so that a particle's field does not depend on the
        // particles swept before it; each word by itself, so that a small component
        // keeps its relative accuracy
        constexpr int kUnset = -2000;   // scales every word to zero
        int ex[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) ex[w] = kUnset;
        // FP64 field sums, [group][word][Re+, Im+, Re-, Im-] (+-: the group's
        // upper and lower half)
        double acc[NAL][NW][4];
#pragma unroll
        for (int a = 0; a < NAL; a++)
#pragma unroll
          for (int w = 0; w < NW; w++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[a][w][i] = 0.0;
        int64_t done = 0;             // steps summed so far

        while (cur.next >= 0) {
          const int64_t seg_hi = min(cur.next + 1, n_act);
          // ---- steps [done, seg_hi) ----
          float4v C[NB][2];           // P_uv of whole groups (v: cos, sin columns)
          float4v D[2][ND];           // cut groups: kept lower part, dropped upper part
#pragma unroll
          for (int g = 0; g < NB; g++)
#pragma unroll
            for (int v = 0; v < 2; v++) C[g][v] = (float4v)(0.f);
#pragma unroll
          for (int g = 0; g < ND; g++) {
            D[0][g] = (float4v)(0.f);
            D[1][g] = (float4v)(0.f);
          }
          bool cut_low = false, cut_up = false;
          int head[3] = {0, 0, 0}, fill[3] = {0, 0, 0}, blocks = 0;
          int64_t t0 = done + (int64_t)(kWave - 1) * wv;
          const int64_t stride = (int64_t)(kWave - 1) * W;

          // one matrix-product block: 32 queued steps of queue q
          auto sweep_block = [&](auto type) {
            constexpr int q = decltype(type)::value;
            constexpr bool CUT = q != 0;
            wave_sync();   // the block before has read its factors
            const Lanes L = kHoist ? held : lanes();
            const int at = head[q] + 8 * L.kg;
            // ---- the block's factors: lanes 0..31 the columns' of step l, lanes
            // 32..63 the rows' of step l - 32, in FP64 (4 k1 + k0 = k: phase p + k d) ----
            {
              const int ln = late(lane), l = ln & 31;
              const double xh = q_xh(q)[head[q] + l], c0 = q_c0(q)[head[q] + l];
              const double ph = ln < 32 ? xh : c0;
              double d = xh * (ln < 32 ? 2.0 : 2.0 * kGroup);
              d = d - rint(d);
              double pr, pi, dr, di;
              phasor(ph, &pr, &pi);
              phasor(d, &dr, &di);
              float *f = s_fac + (ln < 32 ? 0 : kFactorSide) + l;
              auto put0 = [&](int k, double r, double i) {
                f[factor_at(FAC_0RE, k)] = (float)r;
                f[factor_at(FAC_0IM, k)] = (float)i;
                if (NG < 16) f[factor_at(FAC_0NIM, k)] = -(float)i;
              };
              put0(0, 1.0, 0.0);
              put0(1, dr, di);
              const double e2r = fma(-(di + di), di, 1.0), e2i = (dr + dr) * di;
              put0(2, e2r, e2i);
              put0(3, fma(e2r, dr, -(e2i * di)), fma(e2r, di, e2i * dr));
              const double e4r = fma(-(e2i + e2i), e2i, 1.0), e4i = (e2r + e2r) * e2i;
#pragma unroll
              for (int k = 0; k < 4; k++) {
                f[factor_at(FAC_1RE, k)] = (float)pr;
                f[factor_at(FAC_1IM, k)] = (float)pi;
                const double nr = fma(pr, e4r, -(pi * e4i));
                pi = fma(pr, e4i, pi * e4r);
                pr = nr;
              }
            }
            wave_sync();
            // right factor: cos, sin of the column's phase
            uint4v vh[2], vl[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
              const float4 r1 = *(const float4 *)(L.col1 + 4 * j), i1 = *(const float4 *)(L.col1 + kFactorKind + 4 * j);
              const float4 r0 = *(const float4 *)(L.col0 + 4 * j), i0 = *(const float4 *)(L.col0 + kFactorKind + 4 * j);
              float c[4], sn[4];
#pragma unroll
              for (int i = 0; i < 4; i++) {
                c[i] = __builtin_fmaf(lane4(r1, i), lane4(r0, i), -(lane4(i1, i) * lane4(i0, i)));
                sn[i] = __builtin_fmaf(lane4(r1, i), lane4(i0, i), lane4(i1, i) * lane4(r0, i));
              }
#pragma unroll
              for (int i = 0; i < 2; i++) {
                const uint2 wc = split_values(c[2 * i], c[2 * i + 1], one), ws = split_values(sn[2 * i], sn[2 * i + 1], one);
                vh[0][2 * j + i] = wc.x; vl[0][2 * j + i] = wc.y;
                vh[1][2 * j + i] = ws.x; vl[1][2 * j + i] = ws.y;
              }
            }
            // left factor's cos, sin of the row's phase
            float tc[8], ts[8];
#pragma unroll
            for (int j = 0; j < 2; j++) {
              const float4 r1 = *(const float4 *)(L.row1 + 4 * j), i1 = *(const float4 *)(L.row1 + kFactorKind + 4 * j);
              if constexpr (NG == 16) {
                const float4 r0 = *(const float4 *)(L.row0p + 4 * j), i0 = *(const float4 *)(L.row0p + kFactorKind + 4 * j);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                  tc[4 * j + i] = __builtin_fmaf(lane4(r1, i), lane4(r0, i), -(lane4(i1, i) * lane4(i0, i)));
                  ts[4 * j + i] = __builtin_fmaf(lane4(r1, i), lane4(i0, i), lane4(i1, i) * lane4(r0, i));
                }
              } else {
                const float4 a0 = *(const float4 *)(L.row0p + 4 * j), b0 = *(const float4 *)(L.row0q + 4 * j);
#pragma unroll
                for (int i = 0; i < 4; i++)
                  ts[4 * j + i] = __builtin_fmaf(lane4(r1, i), lane4(a0, i), lane4(i1, i) * lane4(b0, i));
              }
            }
            // masks of the cut: the rows that enter whole (lower cut: those below the
            // cut group; upper cut: with it), the cut row, and its kept columns of
            // the lower half (lower cut) or dropped ones of the upper half (upper cut)
            uint4v m_full, m_cut, m_col;
            if constexpr (CUT) {
              const uint4v kk = *(const uint4v *)(q_cnt(q) + at);
#pragma unroll
              for (int j = 0; j < 4; j++) {
                const uint32_t r = kk[j] & 0x001f001fu;
                const uint32_t below = below_mask(kGroup * L.row_a + kGroup - 1, kk[j]), upto = below_mask(kGroup * L.row_a, kk[j]);
                m_full[j] = q == 1 ? below : upto;
                m_cut[j] = upto & ~below;
                m_col[j] = q == 1 ? below_mask(15 - L.rc, r) : ~below_mask(16 + L.rc, r);
              }
            }
            // the cut row's right factors: cos, sin, and (field sums) -sin columns
            uint4v ch[3], cl[3];
            if constexpr (CUT) {
              ch[0] = vh[0] & m_col; cl[0] = vl[0] & m_col;
              ch[1] = vh[1] & m_col; cl[1] = vl[1] & m_col;
              if constexpr (NG == 16) {
                ch[2] = (vh[1] & m_col) ^ 0x80008000u;
                cl[2] = (vl[1] & m_col) ^ 0x80008000u;
              }
            }
            uint4v fh[NB], fl[NB];
            const float *as = q_amp(q) + at;
#pragma unroll
            for (int g = 0; g < NB; g++) {
              const int w = NG == 16 ? g >> 1 : NG == 8 ? g : 0;
              const float *ap = NG == 4 ? as + (2 * g + L.row_w) * kQueue : as + w * kQueue;
              const float4 a0 = *(const float4 *)ap, a1 = *(const float4 *)(ap + 4);
              const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
              uint4v uh, ul;
#pragma unroll
              for (int j = 0; j < 4; j++) {
                const float t0v = (NG == 16 && (g & 1) == 0) ? tc[2 * j] : ts[2 * j];
                const float t1v = (NG == 16 && (g & 1) == 0) ? tc[2 * j + 1] : ts[2 * j + 1];
                const uint2 u = split_pair(t0v, a[2 * j], t1v, a[2 * j + 1]);
                uh[j] = u.x;
                ul[j] = u.y;
              }
              if constexpr (CUT) {
                const uint4v kh = uh & m_cut, kl = ul & m_cut;
                uh &= m_full;
                ul &= m_full;
                // lower half, cos(alpha - beta) = cc + ss, sin(alpha - beta) = sc - cs;
                // upper half, cos(alpha + beta) = cc - ss, sin(alpha + beta) = sc + cs
                constexpr int plus = q == 1 ? 1 : 2, minus = q == 1 ? 2 : 1;
                const int d0 = NG == 16 ? 2 * (g >> 1) : 2 * g;
                const int b0 = NG == 16 ? ((g & 1) == 0 ? 0 : plus) : 0;
                const int b1 = NG == 16 ? ((g & 1) == 0 ? minus : 0) : 1;
                float4v &x = D[q - 1][d0], &y = D[q - 1][d0 + 1];
                x = mfma16(kh, ch[b0], x);
                y = mfma16(kh, ch[b1], y);
                C[g][0] = mfma16(uh, vh[0], C[g][0]);
                C[g][1] = mfma16(uh, vh[1], C[g][1]);
                x = mfma16(kl, ch[b0], x);
                y = mfma16(kl, ch[b1], y);
                C[g][0] = mfma16(ul, vh[0], C[g][0]);
                C[g][1] = mfma16(ul, vh[1], C[g][1]);
                x = mfma16(kh, cl[b0], x);
                y = mfma16(kh, cl[b1], y);
                C[g][0] = mfma16(uh, vl[0], C[g][0]);
                C[g][1] = mfma16(uh, vl[1], C[g][1]);
              } else {
                fh[g] = uh;
                fl[g] = ul;
              }
            }
            if constexpr (!CUT) {
#pragma unroll
              for (int g = 0; g < NB; g++)
#pragma unroll
                for (int v = 0; v < 2; v++) C[g][v] = mfma16(fh[g], vh[v], C[g][v]);
#pragma unroll
              for (int g = 0; g < NB; g++)
#pragma unroll
                for (int v = 0; v < 2; v++) C[g][v] = mfma16(fl[g], vh[v], C[g][v]);
#pragma unroll
              for (int g = 0; g < NB; g++)
#pragma unroll
                for (int v = 0; v < 2; v++) C[g][v] = mfma16(fh[g], vl[v], C[g][v]);
            }
          };

          for (;;) {
            // uniform per wave: every lane of a wave takes the same path
            bool flush = true, rescale = false;
            int want[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) want[w] = ex[w];
            const bool has = t0 < seg_hi;
            if (has) {
              // ---- stage: lane l (1..63) forms the omega-independent part of step
              // s = t0 - 1 + l in FP64; lane 0 the tau of the step before them ----
              const int ln = late(tid) % kWave;
              const int nrem = (int)min((int64_t)(kWave - 1), seg_hi - t0);
              const uint32_t lc = (uint32_t)min(max(ln, t0 == 0 ? 1 : 0), nrem);   // loads stay inside the segment
              const int64_t base = pt.off + t0 - 1;
              const double xs = (p.x + base)[lc], ys = (p.y + base)[lc], zs = (p.z + base)[lc];
              const double time = (double)(pt.its + (uint32_t)(t0 - 1) + (uint32_t)ln) * s_tc[TC_DT];
              double tau, am[NW];
              if constexpr (MODE == SR_MODE_FAR) {
                double ax, ay, az, mx, my, mz;
                if constexpr (PRE) {
                  const double2 *r = (const double2 *)(p.pre + 6 * base) + 3 * lc;
                  const double2 r0 = r[0], r1 = r[1], r2 = r[2];
                  ax = r0.x; ay = r0.y; az = r1.x;
                  mx = r1.y; my = r2.x; mz = r2.y;
                } else {
                  step_am(p.ux, p.uy, p.uz, base + lc, 1.0 / dt, &ax, &ay, &az, &mx, &my, &mz);
                }
                // kernel_farfield.cl:65-94.  tau in the reference's order (it decides
                // the filter); the amplitude, which ends in 24 bits, in FMAs, its
                // transverse parts from n.e = 0: A.e = -(c1 m.e + c2 a.e)
                const double gx = s_tc[TC_GX], gy = s_tc[TC_GY], gz = s_tc[TC_GZ];
                tau = time - (xs * gx + ys * gy + zs * gz);
                const double na = fma(az, gz, fma(ay, gy, ax * gx));
                double c2 = fma(-mz, gz, fma(-my, gy, fma(-mx, gx, 1.0)));
                // the hardware reciprocal (4.6e-8) with one Newton step (~1e-15)
                const double r = __builtin_amdgcn_rcp(c2);
                c2 = fma(r, fma(-c2, r, 1.0), r);
                const double c1 = na * c2 * c2;
                const double thx = s_tc[TC_THX], thy = s_tc[TC_THY], thz = s_tc[TC_THZ];
                const double phx = s_tc[TC_PHX], phy = s_tc[TC_PHY];
                am[0] = -fma(c1, fma(mz, thz, fma(my, thy, mx * thx)), c2 * fma(az, thz, fma(ay, thy, ax * thx)));
                am[1] = -fma(c1, fma(my, phy, mx * phx), c2 * fma(ay, phy, ax * phx));
              } else {
                double bx, by, bz;
                if constexpr (PRE) {
                  const double *r = (p.pre + 3 * base) + 3 * lc;
                  bx = r[0]; by = r[1]; bz = r[2];
                } else {
                  const double ux = (p.ux + base)[lc], uy = (p.uy + base)[lc], uz = (p.uz + base)[lc];
                  const double g0 = gamma_inv(ux, uy, uz);
                  bx = ux * g0; by = uy * g0; bz = uz * g0;
                }
                // kernel_nearfield.cl:67-88; tau in the reference's order
                const double rx = s_tc[TC_GX] - xs, ry = s_tc[TC_GY] - ys, rz = s_tc[TC_GZ] - zs;
                const double R = sqrt(rx * rx + ry * ry + rz * rz);
                tau = time + R;
                const double r = __builtin_amdgcn_rcp(R);
                const double rInv = fma(r, fma(-R, r, 1.0), r);
                const double nx = rInv * rx, ny = rInv * ry, nz = rInv * rz;
                const double r2 = rInv * rInv;
                am[0] = rInv * (bx - nx); am[1] = rInv * (by - ny); am[2] = rInv * (bz - nz);
                am[3] = r2 * nx; am[4] = r2 * ny; am[5] = r2 * nz;
              }
              // |omega tau_s - omega tau_{s-1}| < pi <=> |omega|/2pi < (1/2)/|dtau|
              // (phase_{-1} = 0; dtau = 0: always)
              const double below = lane_below(tau);
              const double d = fabs(tau - (ln == 1 && t0 == 0 ? 0.0 : below));
              const double dr = __builtin_amdgcn_rcp(d);
              const double thr = (d == 0.0) ? INFINITY : 0.5 * fma(dr, fma(-d, dr, 1.0), dr);
              // kept frequencies: the count of s_om[j] < thr (ascending; NaN: none),
              // by the grid's step and then the neighbouring values themselves
              const double est = fmin(fmax((thr - s_tc[TC_WLO]) * s_tc[TC_INV], 0.0), (double)max(count - 2, 0));
              const int e = (int)est + 1;
              int K = s_om[e] < thr ? e + 1 : (s_om[e - 1] < thr ? e : e - 1);
              if (ln == 0 || ln > nrem) K = 0;
              // the scaled words, the largest of each kind among the kept steps between 1
              // and 2^15 (fp16's high words below 2^16, its low words, of 2^-24 or more,
              // within 2^-24 of the largest); outside, the queues are emptied first
              float af[NW];
              bool out = false;
              const uint64_t kept = __ballot(K > 0);
#pragma unroll
              for (int w = 0; w < NW; w++) {
                af[w] = (float)ldexp(am[w], ex[w]);
                const uint64_t high = __ballot(!(fabsf(af[w]) < 32768.f)) & kept;
                if (high != 0 || (__ballot(fabsf(af[w]) >= 1.f) & kept) == 0)
                  out = out || high != 0 || (__ballot(am[w] != 0.0) & kept) != 0;
              }
              if (out) {
#pragma unroll
                for (int w = 0; w < NW; w++) {
                  double m = (K > 0 && fabs(am[w]) < INFINITY) ? fabs(am[w]) : 0.0;
                  for (int o = kWave / 2; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
                  m = unid(m);
                  const double ms = ldexp(m, ex[w]);
                  // amplitudes too small for any scale keep the last one they asked for
                  if (m > 0.0 && !(ms >= 2.0 && ms < 32768.0)) {
                    want[w] = uni(max(-1000, min(1000, 11 - ilogb(m))));
                    rescale = rescale || want[w] != ex[w];
                  }
                }
              }
              // (nothing swept or queued under the old scales, as at a track's start: they change
              // here, not by another pass)
              if (rescale && blocks + fill[0] + fill[1] + fill[2] == 0) {
#pragma unroll
                for (int w = 0; w < NW; w++) {
                  ex[w] = want[w];
                  af[w] = (float)ldexp(am[w], ex[w]);
                }
                rescale = false;
              }
              if (!rescale) {
                flush = false;
                const uint64_t bf = __ballot(K == count);
                const uint64_t bu = __ballot((K & (kGroup - 1)) > kGroup / 2) & ~bf, bl = kept & ~bf & ~bu;
                if (K > 0) {
                  const bool up = (K & (kGroup - 1)) > kGroup / 2;
                  const int q1 = K == count ? 0 : up ? 2 : 1;
                  const uint64_t b = q1 == 0 ? bf : q1 == 1 ? bl : bu;
                  const int at = q1 == 0 ? head[0] + fill[0] : q1 == 1 ? head[1] + fill[1] : head[2] + fill[2];
                  int pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, at));
                  if (pos >= kQueue) pos -= kQueue;
                  double xh = s_tc[TC_HALF] * tau, c0 = s_tc[TC_C0] * tau;
                  xh = xh - rint(xh);
                  c0 = c0 - rint(c0);
                  q_xh(q1)[pos] = xh;
                  q_c0(q1)[pos] = c0;
#pragma unroll
                  for (int c = 0; c < NW; c++) q_amp(q1)[c * kQueue + pos] = af[c];
                  q_cnt(q1)[pos] = (uint16_t)K;
                }
                fill[0] += __popcll(bf);
                fill[1] += __popcll(bl);
                fill[2] += __popcll(bu);
                t0 += stride;
              }
            }
            // ---- sweep the full blocks; before a record or a rescaling all ----
            if (flush) {
#pragma unroll
              for (int q1 = 0; q1 < 3; q1++) {
                const int ln = late(tid) % kWave;
                if (ln >= fill[q1] && ln < kBlockSteps && fill[q1] > 0) {
#pragma unroll
                  for (int c = 0; c < NW; c++) q_amp(q1)[c * kQueue + head[q1] + ln] = 0.f;
                  q_cnt(q1)[head[q1] + ln] = 0;
                  q_xh(q1)[head[q1] + ln] = 0.0;
                  q_c0(q1)[head[q1] + ln] = 0.0;
                }
                if (fill[q1] > 0) fill[q1] = max(fill[q1], kBlockSteps);
              }
            }
            wave_sync();
            auto drain = [&](auto type) {
              constexpr int q = decltype(type)::value;
              while (fill[q] >= kBlockSteps) {
                sweep_block(type);
                fill[q] -= kBlockSteps;
                head[q] = head[q] == kQueue - kBlockSteps ? 0 : head[q] + kBlockSteps;
                blocks++;
                cut_low = cut_low || q == 1;
                cut_up = cut_up || q == 2;
              }
            };
            drain(std::integral_constant<int, 0>());
            drain(std::integral_constant<int, 1>());
            drain(std::integral_constant<int, 2>());
            wave_sync();
            // ---- fold into the FP64 sums ----
            if (blocks >= fold_blocks<MODE>() || (flush && blocks > 0)) {
              double un[NW];   // 2^-ex
#pragma unroll
              for (int w = 0; w < NW; w++)
                un[w] = ex[w] == kUnset ? 0.0 : __longlong_as_double((int64_t)(1023 - ex[w]) << 52);
#pragma unroll
              for (int a = 0; a < NAL; a++)
#pragma unroll
                for (int w = 0; w < NW; w++) {
                  auto at_g = [&](int u) { return NG == 16 ? 2 * w + u : NG == 8 ? w : w >> 1; };
                  auto at_r = [&](int u) { return NG == 16 ? a : NG == 8 ? 2 * a + u : 2 * (w & 1) + u; };
                  auto P = [&](int u, int v) { return C[at_g(u)][v][at_r(u)]; };
                  float f[4] = {P(0, 0) - P(1, 1), P(1, 0) + P(0, 1), P(0, 0) + P(1, 1), P(1, 0) - P(0, 1)};
                  auto Q = [&](int h, int u, int v) { return D[h][NG == 16 ? 2 * w + v : 2 * at_g(u) + v][NG == 16 ? a : at_r(u)]; };
                  if (cut_low) {
                    f[2] += NG == 16 ? Q(0, 0, 0) : Q(0, 0, 0) + Q(0, 1, 1);
                    f[3] += NG == 16 ? Q(0, 0, 1) : Q(0, 1, 0) - Q(0, 0, 1);
                  }
                  if (cut_up) {
                    f[0] -= NG == 16 ? Q(1, 0, 0) : Q(1, 0, 0) - Q(1, 1, 1);
                    f[1] -= NG == 16 ? Q(1, 0, 1) : Q(1, 1, 0) + Q(1, 0, 1);
                  }
                  const double us = un[w];
#pragma unroll
                  for (int i = 0; i < 4; i++) acc[a][w][i] = fma((double)f[i], us, acc[a][w][i]);
                }
#pragma unroll
              for (int g = 0; g < NB; g++)
#pragma unroll
                for (int v = 0; v < 2; v++) C[g][v] = (float4v)(0.f);
#pragma unroll
              for (int g = 0; g < ND; g++) {
                if (cut_low) D[0][g] = (float4v)(0.f);
                if (cut_up) D[1][g] = (float4v)(0.f);
              }
              cut_low = cut_up = false;
              blocks = 0;
            }
            if (rescale) {
#pragma unroll
              for (int w = 0; w < NW; w++) ex[w] = want[w];
            }
            if (!has) break;
          }
          done = max(done, seg_hi);

          // ---- record (kernel_farfield.cl:100-106): the waves' sums meet in LDS,
          // one (group, half) slice at a time, and one wave writes it ----
          const double wpdt2 = pt.w * dt * dt;
          const double wpdt = sqrt(pt.w) * dt;
          // everything the record derives from the lane is formed here, not held
          // in registers through the sweeps
          const int ln = late(tid) % kWave, kgr = ln >> 4, rcr = ln & 15;
          double *const own = (double *)s_own;
#pragma unroll 1
          for (int sl = 0; sl < 2 * NAL; sl++) {
#pragma unroll
            for (int a = 0; a < NAL; a++)
#pragma unroll
              for (int h = 0; h < 2; h++)
                if (sl == 2 * a + h) {
#pragma unroll
                  for (int w = 0; w < NW; w++) {
                    own[(2 * w) * kWave + ln] = acc[a][w][2 * h];
                    own[(2 * w + 1) * kWave + ln] = acc[a][w][2 * h + 1];
                  }
                }
            if (W > 1) __syncthreads(); else wave_sync();
            if (wv == (sl & (W - 1))) {
              double F[NW][2];
#pragma unroll
              for (int w = 0; w < NW; w++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                  double sum = 0.0;
                  for (int v = 0; v < W; v++)
                    sum += ((const double *)(s_waves + v * wave_bytes<MODE>()))
                        [(2 * w + i) * kWave + ln];
                  F[w][i] = sum;
                }
              const int a = NG == 16 ? 4 * kgr + (sl >> 1) : NG == 8 ? 2 * kgr + (sl >> 1) : kgr;
              const int j = kGroup * a + ((sl & 1) ? 15 - rcr : 16 + rcr);
              if (j < count) {
                const int wk = first + sgn * j;
                double re[3], im[3];
                if constexpr (MODE == SR_MODE_FAR) {
                  // F = F_theta e_theta + F_phi e_phi (spheric, kernel_farfield.cl:442-445)
                  if (spheric) {
                    re[0] = 0.0; re[1] = F[0][0]; re[2] = F[1][0];
                    im[0] = 0.0; im[1] = F[0][1]; im[2] = F[1][1];
                  } else {
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                      const double th = s_tc[TC_THX + c], ph = c < 2 ? s_tc[TC_PHX + c] : 0.0;
                      re[c] = c < 2 ? F[0][0] * th + F[1][0] * ph : F[0][0] * th;
                      im[c] = c < 2 ? F[0][1] * th + F[1][1] * ph : F[0][1] * th;
                    }
                  }
                } else {
                  // sum (v2 + i omega v1) e^{i phase}
                  const double om = p.omega[wk];
#pragma unroll
                  for (int c = 0; c < 3; c++) {
                    re[c] = F[3 + c][0] - om * F[c][1];
                    im[c] = F[3 + c][1] + om * F[c][0];
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
                if (p.acc_lds) {
                  s_acc[sl * kWave + ln] += v[0];
                } else {
                  const int64_t g = (int64_t)cur.slot * p.n_grid + (int64_t)dir * p.n_omega + wk +
                                    (ip - p.part_base) * p.part_stride;
#pragma unroll
                  for (int c = 0; c < kMaxOut; c++)
                    if (c < p.n_out) dst(c)[g] += v[c];
                }
              }
            }
            if (W > 1) __syncthreads(); else wave_sync();
          }
          const int64_t last = cur.next;
          cur.slot++;
          cur.advance(pt, p.n_snaps, last);
        }
      }
      if (p.acc_lds) {
        __syncthreads();
        const int ln = late(tid) % kWave, kgr = ln >> 4, rcr = ln & 15;
        for (int sl = wv; sl < 2 * NAL; sl += W) {
          const int a = NG == 16 ? 4 * kgr + (sl >> 1) : NG == 8 ? 2 * kgr + (sl >> 1) : kgr;
          const int j = kGroup * a + ((sl & 1) ? 15 - rcr : 16 + rcr);
          if (j < count) dst(0)[(int64_t)dir * p.n_omega + first + sgn * j] += s_acc[sl * kWave + ln];
        }
      }
    }
  }
}

}  // namespace sr
