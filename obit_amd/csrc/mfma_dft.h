// mfma_dft.h -- the parts the matrix-core DFT kernels share (dft.hip,
// beam.hip): phasors from FP64 phases, exchange between half-waves, FP16
// operand parts.
#pragma once
#include <hip/hip_runtime.h>
#include "phasor.h"

namespace obit {

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// e(t) for a phase in turns formed in FP64: reduced to [-1/2, 1/2] first,
// then the hardware sin / cos (HW) or the Taylor polynomial
template <bool HW>
__device__ __forceinline__ float2 eturn(double t) {
  float sn, cs;
  if (HW) sincos_turns_hw((float)(t - rint(t)), &sn, &cs);
  else sincos_turns_poly((float)(t - rint(t)), &sn, &cs);
  return make_float2(cs, sn);
}

// a value of the first half-wave (lanes 0..31) and of the second
// (32..63) in every lane: lo[l] = x[l mod 32], hi[l] = x[32 + l mod 32]
// (v_permlane32_swap exchanges lanes 32..63 of its first operand with
// lanes 0..31 of its second)
__device__ __forceinline__ void swap_halves(float2 x, float2 &lo, float2 &hi) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x.x), __float_as_uint(x.x), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x.y), __float_as_uint(x.y), false, false);
  lo = make_float2(__uint_as_float(a[0]), __uint_as_float(b[0]));
  hi = make_float2(__uint_as_float(a[1]), __uint_as_float(b[1]));
}

// FP16 parts of (x, y), each pair packed in a 32-bit word (x in the low
// half): hi = fp16(x), fp16(y) rounded to nearest; lo = fp16(x - hi.x),
// fp16(y - hi.y), the differences formed in FP32 from the FP16 values.
// The differences are formed by v_fma_mix_f32 and packed by one conversion:
// v_fma_mixlo_f16 / v_fma_mixhi_f16, which would form and pack them in two
// instructions, issue at half rate (9 cycles measured against 5), so four
// full-rate instructions take fewer cycles than those three.
__device__ __forceinline__ void split_pair(float x, float y, unsigned &hi, unsigned &lo) {
  float dx, dy;
  asm("v_cvt_pk_f16_f32 %0, %4, %5\n\t"
      "v_fma_mix_f32 %2, -%0, 1.0, %4 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mix_f32 %3, -%0, 1.0, %5 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_cvt_pk_f16_f32 %1, %2, %3"
      : "=&v"(hi), "=&v"(lo), "=&v"(dx), "=&v"(dy)
      : "v"(x), "v"(y));
}

// (x, y) -> (y, -x) of an FP16 pair
__device__ __forceinline__ unsigned swap_neg(unsigned v) {
  unsigned r;
  asm("v_pk_add_f16 %0, %1, 0 op_sel:[1,0] op_sel_hi:[0,0] neg_hi:[1,0]" : "=v"(r) : "v"(v));
  return r;
}

// ---- sums over components by blocks of 16 channels ----
//
// M_e[t][b] = sum_k X_k[t] Y_ke[b] of one row by one wave (described at
// k_beam_mm): X_k[t] = G_k(t) e(psi df t), t = -8 .. 7, Y_ke[b] = C_keb e(psi f_b).
namespace mm {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int kTile = 32;          // components a tile
// slots of a 4-component block: 32 rows (A) or 16 columns (B) + 1 (k_dft_mfma's
// layout); 16-byte slots of one operand part
constexpr int kRA = 33, kRB = 17;
constexpr int kSlotsA = 8 * kRA, kSlotsB = 8 * kRB;
constexpr int kSlots = 2 * kSlotsA + 2 * kSlotsB;  // of a wave
constexpr int kT = 16;             // channels of a block
constexpr int kPass = 16;          // blocks of a pass
// Largest residual of the factored amplitudes, relative to the component's
// largest amplitude in the same block, that the matrix-core kernels take.  It is
// the worst channel's (a steep spectrum at both ends of a pass); the model's error
// stays below that of the channel walks, whose worst is 1.3e-6 of the peak.
constexpr float kFitTol = 1e-6f;

struct Blk {
  double fc;            // nu/nu0 of channel ch0 + 8
  int IF, ch0;          // first channel (t = -8)
  int vlo, vhi;         // channels the block writes
  int jc;               // beam channel
  float s;              // df (1 / fc - 1 / f0), f0 the pass's reference
};

// exponent that brings a largest value (float bits) to [2^13, 2^14)
__host__ __device__ __forceinline__ int shift_of(unsigned bits) {
  const int e = (int)((bits >> 23) & 255u) - 126;
  return bits == 0u ? 0 : 14 - e;
}

static __global__ void k_clear(unsigned *a, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) a[i] = 0u;
}

// The factors A_kb G_k(t) (1 + kappa_k tau(t) s_b) of the amplitude table
// (rows of ldk floats, ldif an IF, of which nchan are channels), one thread a
// component and pass; resid: the largest relative residual, amax (may be
// null): the largest |A| of every block (float bits, both cleared before).  G is
// the shape of the pass's reference block, its middle one where it can be; A and the slope of each block
// are taken at two channels 0.7 of the way to its ends, which halves the error
// of the linear term at them; kappa is the slopes' least-squares fit to s_b.
static __global__ __launch_bounds__(64) void k_fit(const float *__restrict__ tab, int nchan, int ldif, long long ldk,
                                                 const Blk *__restrict__ blk, int nblk, const float *__restrict__ r0,
                                                 int ncomp, int ncpad, float *__restrict__ Ab, float *__restrict__ G,
                                                 unsigned *__restrict__ kap, unsigned *__restrict__ resid,
                                                 unsigned *__restrict__ amax) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, ps = blockIdx.y;
  const int b0 = ps * kPass, nb = min(kPass, nblk - b0);
  float worst = 0.0f, top[kPass] = {};
  if (k < ncomp) {
    const float *row = tab + (long long)k * ldk;
    auto amp = [&](int b, int t) {
      const int ch = min(max(blk[b].ch0 + 8 + t, 0), nchan - 1);
      return (double)row[(long long)blk[b].IF * ldif + ch];
    };
    // the reference: a block whose 16 channels are of one run, if there is one
    auto fit_ref = [&](int b) { return amp(b, 0) != 0.0 && blk[b].vhi == blk[b].ch0 + kT - 1; };
    int ref = b0 + nb / 2;
    for (int i = 0; i < nb && !fit_ref(ref); ++i) ref = b0 + i;
    const double a0 = amp(ref, 0);
    double g[kT];
    for (int t = -8; t < 8; ++t) {
      g[t + 8] = a0 != 0.0 ? amp(ref, t) / a0 : 1.0;
      // (a shape that varies more would cost X's low FP16 part bits; the residual tells)
      if (!(fabs(g[t + 8]) > 0.25 && fabs(g[t + 8]) < 4.0)) g[t + 8] = 1.0;
      g[t + 8] = (double)(float)g[t + 8];
      G[((long long)ps * kT + t + 8) * ncpad + k] = (float)g[t + 8];
    }
    const double r = r0[ps];
    auto tau = [&](int t) { return (double)t - (double)t * (double)t * r; };
    auto ends = [&](int b, int &t1, int &t2) {
      const double lo = blk[b].vlo - blk[b].ch0 - 8, hi = blk[b].vhi - blk[b].ch0 - 8;
      const double m = 0.5 * (lo + hi), w = 0.35 * (hi - lo);
      t1 = (int)rint(m - w);
      t2 = (int)rint(m + w);
    };
    double num = 0.0, den = 0.0;
    for (int b = b0; b < b0 + nb; ++b) {
      int t1, t2;
      ends(b, t1, t2);
      const double p1 = amp(b, t1) / g[t1 + 8], p2 = amp(b, t2) / g[t2 + 8];
      const double d = p1 * tau(t2) - p2 * tau(t1), s = blk[b].s;
      if (t2 > t1 && d != 0.0 && s != 0.0) {
        num += (p2 - p1) / d * s;
        den += s * s;
      }
    }
    double ka = den > 0.0 ? num / den : 0.0;
    if (!(fabs(ka) < 1e3)) ka = 0.0;
    const _Float16 kh = (_Float16)(float)ka;
    ka = (double)(float)kh;
    kap[(long long)ps * ncpad + k] = (unsigned)__builtin_bit_cast(unsigned short, kh) * 0x10001u;
#pragma unroll
    for (int i = 0; i < kPass; ++i) {
      const int b = b0 + i;
      if (i >= nb) break;
      int t1, t2;
      ends(b, t1, t2);
      const double s = blk[b].s;
      double off = 0.0, big = 0.0;
      const double A = 0.5 * (amp(b, t1) / (g[t1 + 8] * (1.0 + ka * tau(t1) * s)) +
                              amp(b, t2) / (g[t2 + 8] * (1.0 + ka * tau(t2) * s)));
      Ab[(long long)b * ncpad + k] = (float)A;
      top[i] = fabsf((float)A);
      for (int ch = blk[b].vlo; ch <= blk[b].vhi; ++ch) {
        const int t = ch - blk[b].ch0 - 8;
        const double a = amp(b, t), e = fabs(a - (double)(float)A * g[t + 8] * (1.0 + ka * tau(t) * s));
        big = fmax(big, fabs(a));
        off = (e >= off) ? e : (e < off ? off : INFINITY);  // a NaN counts as infinite
      }
      const float res = big > 0.0 ? (float)(off / big) : (off > 0.0 ? INFINITY : 0.0f);
      worst = res >= 0.0f ? fmaxf(worst, res) : INFINITY;
    }
  } else if (k < ncpad) {
    for (int t = 0; t < kT; ++t) G[((long long)ps * kT + t) * ncpad + k] = 1.0f;
    kap[(long long)ps * ncpad + k] = 0u;
    for (int b = b0; b < b0 + nb; ++b) Ab[(long long)b * ncpad + k] = 0.0f;
  }
  for (int o = 32; o > 0; o >>= 1) worst = fmaxf(worst, __shfl_xor(worst, o));
  if ((threadIdx.x & 63) == 0 && worst > 0.0f) atomicMax(resid, __float_as_uint(worst));
  if (amax) {
#pragma unroll
    for (int i = 0; i < kPass; ++i) {
      float t = top[i];
      for (int o = 32; o > 0; o >>= 1) t = fmaxf(t, __shfl_xor(t, o));
      if ((threadIdx.x & 63) == 0 && i < nb && t > 0.0f) atomicMax(amax + b0 + i, __float_as_uint(t));
    }
  }
}

// The sums over components kBeg .. kEnd - 1 (kBeg a multiple of 32; so is kEnd,
// or it is ncomp) for the 8 blocks of this lane's half-wave at -f_b = fc[b].
// lds: the wave's operand area.  prod: a table of C by (block offset po, then
// component), REAL floats, or conj C as float2 in steps of pm (NE 1) or
// float4 (NE 2), zero from ncomp to the end of the last tile.  AMP: G points at
// the shape of slot 0 of the half (t = 0 or -1), gstep to the next slot's;
// kap: (kappa, kappa) pairs.  PREC: hardware sin / cos for P and the steps (0), for
// P (1), for neither (2).  o[T][e][r], d2: lanes 0..31 hold the real parts
// of slot c = 4 (lane / 16) + r of tile T (t = c, or -(c + 1) for T = 0), lanes 32
// on the imaginary, of column lane mod 16 (half-wave, block).
template <bool AMP, int NE, bool REAL, int PREC>
__device__ __forceinline__ void sum(uint4 *lds, const double *__restrict__ cx, const double *__restrict__ cy,
                                    const double *__restrict__ cz, int ncomp, int kBeg, int kEnd, double u, double v,
                                    double w, double df, const double (&fc)[8], const unsigned (&po)[8],
                                    const void *__restrict__ prod, unsigned pm, const float *__restrict__ G, int gstep,
                                    const unsigned *__restrict__ kap, double (&o)[2][NE][4], f4 (&d2)[2][NE]) {
  const int lane = threadIdx.x & 63;
  uint4 *sAh = lds, *sAl = sAh + kSlotsA, *sBh = sAl + kSlotsA, *sBl = sBh + kSlotsB;
  const int i = lane & 15, qd = lane >> 4;   // matrix-step roles
  const int kc = lane & 31, h = lane >> 5;   // set-up roles: component, half
  unsigned *wA = reinterpret_cast<unsigned *>(sAh + (kc >> 2) * kRA + 16 * h) + (kc & 3);
  unsigned *wB = reinterpret_cast<unsigned *>(sBh + (kc >> 2) * kRB + 8 * h) + (kc & 3);
  constexpr int kLoA = 4 * kSlotsA, kLoB = 4 * kSlotsB;  // words from the _h to the _l array
  const double wdf = h ? 6.0 * df : df;
#pragma unroll
  for (int T = 0; T < 2; ++T)
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      d2[T][e] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int r = 0; r < 4; ++r) o[T][e][r] = 0.0;
    }
  // the next tile's positions, read a tile ahead
  double nx, ny, nz;
  auto fetch = [&](int k0) {
    const int k = min(k0 + kc, ncomp - 1);
    nx = cx[k];
    ny = cy[k];
    nz = cz[k];
  };
  fetch(kBeg);
  for (int k4 = kBeg; k4 < kEnd; k4 += 2 * kTile) {
    f4 acc[2][NE];
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int e = 0; e < NE; ++e) acc[T][e] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int kt = 0; kt < 2; ++kt) {
      const int k0 = k4 + kt * kTile;
      if (k0 >= kEnd) break;
      // this tile's products and shape, used after the powers below
      const unsigned kp = (unsigned)(k0 + kc);
      float4 pr[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (REAL) {
          pr[b] = make_float4(static_cast<const float *>(prod)[po[b] + kp], 0.0f, 0.0f, 0.0f);
        } else if (NE == 1) {
          const float2 x = static_cast<const float2 *>(prod)[pm * (po[b] + kp)];
          pr[b] = make_float4(x.x, x.y, 0.0f, 0.0f);
        } else {
          pr[b] = static_cast<const float4 *>(prod)[po[b] + kp];
        }
      }
      float g[8];
      if (AMP) {
        // slot c of this half: t = c (second half) or -(c + 1)
#pragma unroll
        for (int c = 0; c < 8; ++c) g[c] = G[(int)kp + c * gstep];
      }
      const double psi = fma(w, nz, fma(v, ny, u * nx));
      fetch(k0 + kTile);
      {
        const float2 s1 = eturn<PREC == 0>(psi * wdf);
        float2 z[9];
        swap_halves(s1, z[1], z[6]);
        z[2] = cmul(z[1], z[1]);
        z[3] = cmul(z[2], z[1]);
        auto cjmul = [](float2 a, float2 b) {  // a conj(b)
          return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
        };
        z[4] = cjmul(z[6], z[2]);
        z[5] = cjmul(z[6], z[1]);
        z[7] = cmul(z[6], z[1]);
        z[8] = cmul(z[6], z[2]);
        z[0] = make_float2(1.0f, 0.0f);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          float xr = h ? z[c].x : z[c + 1].x, xi = h ? z[c].y : -z[c + 1].y;
          if (AMP) { xr *= g[c]; xi *= g[c]; }
          unsigned xh, xl;
          split_pair(xr, xi, xh, xl);
          wA[4 * c] = xh;
          wA[4 * c + kLoA] = xl;
          wA[4 * (c + 8)] = swap_neg(xh);
          wA[4 * (c + 8) + kLoA] = swap_neg(xl);
        }
      }
      // the first correlation's Y into the operand area, the second's kept
      // until the first's are read
      unsigned y1h[8], y1l[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const float2 pg = eturn<PREC != 2>(psi * fc[b]);  // conj P
        const float2 y0 = REAL ? make_float2(pr[b].x * pg.x, pr[b].x * pg.y)
                               : cmul(pg, make_float2(pr[b].x, pr[b].y));
        unsigned yh, yl;
        split_pair(y0.x, y0.y, yh, yl);
        wB[4 * b] = yh;
        wB[4 * b + kLoB] = yl;
        if (NE == 2) {
          const float2 y1 = cmul(pg, make_float2(pr[b].z, pr[b].w));
          split_pair(y1.x, y1.y, y1h[b], y1l[b]);
        }
      }
      // a wave's LDS accesses complete in order: writes, reads, writes, reads
      h8 ah[2][2], al[2][2];  // [step][tile]
      asm volatile("" ::: "memory");
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        h8 bh[2], bl[2];
        if (e) {
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            wB[4 * b] = y1h[b];
            wB[4 * b + kLoB] = y1l[b];
          }
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (!e) {
#pragma unroll
            for (int T = 0; T < 2; ++T) {
              const int at = (qd + 4 * s) * kRA + 16 * T + i;
              ah[s][T] = __builtin_bit_cast(h8, sAh[at]);
              al[s][T] = __builtin_bit_cast(h8, sAl[at]);
            }
          }
          bh[s] = __builtin_bit_cast(h8, sBh[(qd + 4 * s) * kRB + i]);
          bl[s] = __builtin_bit_cast(h8, sBl[(qd + 4 * s) * kRB + i]);
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
          for (int T = 0; T < 2; ++T)
            acc[T][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s][T], bh[s], acc[T][e], 0, 0, 0);
#pragma unroll
          for (int T = 0; T < 2; ++T)
            acc[T][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s][T], bl[s], acc[T][e], 0, 0, 0);
#pragma unroll
          for (int T = 0; T < 2; ++T)
            acc[T][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[s][T], bh[s], acc[T][e], 0, 0, 0);
          if (AMP) {
            const h8 ks = __builtin_bit_cast(h8, *reinterpret_cast<const uint4 *>(kap + k0 + 4 * (qd + 4 * s)));
#pragma unroll
            for (int T = 0; T < 2; ++T)
              d2[T][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s][T] * ks, bh[s], d2[T][e], 0, 0, 0);
          }
        }
      }
    }
#pragma unroll
    for (int T = 0; T < 2; ++T)
#pragma unroll
      for (int e = 0; e < NE; ++e)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[T][e][r] += (double)acc[T][e][r];
  }
}

}  // namespace mm

}  // namespace obit
