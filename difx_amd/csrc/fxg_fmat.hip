// Matrix F-engine: the F-engine of the FX hot path for 2-bit real data with its FFT on the FP16
// matrix cores, at FP32 accuracy.  What one FFT block computes is what fxg_fengine.hip's kernels
// compute (Mode::process, mode.cpp:634-1374) for fringe rotation orders 0 and 1.
//
// With n = s + 64 t and k = k2 + 32 k1 (L = 2048: t, k2 < 32, s, k1 < 64) and a rotator whose
// phase is linear in n,
//   X[k] = sum_s W_64^(s k1) * T[s][k2] * Y[s][k2],   Y[s][k2] = sum_t x[s + 64 t] M[t][k2]
//   M[t][k2] = W_32^(t k2) step[t],  T[s][k2] = W_2048^(s k2) sub[s]
// (step and sub the rotator at 64 t and at s).  Both sums are matrix products:
//   stage 1   Y = M x.  The samples are real and take four values +-1, +-H: x = xh + xl with xh
//             and xl FP16 numbers (H = 427/128 and a remainder), exact to FP32 rounding.  M is
//             built per FFT and freq in FP32 and split into two FP16 numbers, M = Mh + Ml, so
//             Y = Mh xh + Ml xh + Mh xl, products of 11-bit factors summed in FP32.
//   stage 2   Z = T Y and then, s and s + 32 together, E = Z_s + Z_(s+32) and D = Z_s - Z_(s+32)
//             in FP32; the even k1 are a product of a constant matrix with E and the odd ones of
//             another with D (half the work of one over 64 values of s), split the same way,
//             X = Wh Zh + Wl Zh + Wh Zl, only for the kept half of the channels.
// The dropped terms Ml xl and Wl Zl are below 2^-22 of the ones kept.  Powers of two keep every
// FP16 part out of the subnormal range and are taken out again in FP32.
//
// One wavefront does one FFT of one datastream, freq by freq, with no barrier: the transposition
// between the stages goes through its own 9 KB of LDS, E and then D.  Eight wavefronts (one
// workgroup per CU) share the constant tables in LDS and take consecutive FFTs, so that their
// stores fill whole lines of the 16-bit spectra.  M and T serve both bands of a freq.
//
// Measured at 16 stations x 16 bands x 15625 FFTs (16-bit spectra): 16.5 ms per subint with the
// vector FFT, 10.7 ms with this kernel; spectra of FP32 jobs come out with a smaller error against
// 64 bits than before (visibilities of 10 stations 1.1e-7 -> 7.4e-8).  The vector FFT issues 52.8
// vector instructions per sample, this one 24 and 96 matrix instructions per 4096 samples.  What
// bounds it now is power: the clock falls from 2.36 to 1.97 GHz under it, one matrix instruction
// costs as much as 16 vector ones, and both are busy 60 and 28 % of the cycles left.
#include "fxg_fe_common.h"
#include <algorithm>
#include <cmath>

namespace {

typedef _Float16 fm_h8 __attribute__((ext_vector_type(8)));
typedef float fm_f16 __attribute__((ext_vector_type(16)));
typedef unsigned fm_u4 __attribute__((ext_vector_type(4)));

constexpr int FM_L = 2048, FM_C = FM_L / 2; // FFT length and channels
constexpr int FM_NW = 8;                    // wavefronts per workgroup
constexpr int FM_HS = 36;                   // words per row of an exchange plane (conflict-free 16-byte reads)
constexpr int FM_PLANE = 32 * FM_HS;
constexpr int FM_TAB = 64 + 32;              // per wavefront: sub and step, then fsub and fstep phasors
constexpr int FM_WORDS = 16 * 64;           // per wavefront: sample words of bands 8-15
constexpr int FM_OWN = 2 * FM_PLANE + 2 * FM_TAB + FM_WORDS;
constexpr float FM_MSCALE = 4096.0f;        // of M and W
constexpr float FM_XSCALE = 16.0f;          // of the samples
constexpr float FM_ZSCALE = 256.0f;         // of E and D: at most 64 H, so below 65504 scaled

// The two FP16 parts of a pair of floats: hi rounded to nearest, lo the rest rounded.
__device__ __forceinline__ void fm_split(float a, float b, unsigned& hi, unsigned& lo) {
  float ra, rb;
  asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(ra) : "v"(hi), "v"(a));
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(rb) : "v"(hi), "v"(b));
  asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(lo) : "v"(ra), "v"(rb));
}

__device__ __forceinline__ fm_f16 fm_mfma(fm_u4 a, fm_u4 b, fm_f16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(fm_h8, a), __builtin_bit_cast(fm_h8, b), c, 0, 0, 0);
}

// exp(2 pi i ph) for a phase in turns: reduced in double, then FP32 sin/cos of half turns
__device__ __forceinline__ float2 fm_turn(double ph) {
  const float r = (float)(ph - rint(ph));
  float sn, cs;
  sincospif(2.0f * r, &sn, &cs);
  return make_float2(cs, sn);
}

// Orders the wavefront's own LDS writes before its following LDS reads: LDS instructions of one
// wavefront execute in order, so only the compiler has to keep them so.
__device__ __forceinline__ void fm_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace

size_t fxg_fmat_lds() {
  return sizeof(float) * (FMAT_TABLE_WORDS + FM_NW * FM_OWN);
}

// The constant tables, in the lane order in which they are read (words):
//   W    [odd k1 2][k-step 4][hi, lo][lane 64][4]: FP16 pairs of the stage 2 matrices, rows
//        2 j + (re, im) of k1 = 2 j + odd, columns 2 s + (re, im)
//   tc   [half of s 2][j / 2 8][lane 64][j % 2] (re, im) of W_2048^(s k2) / scales
//   mc   [row tile 2][k-step 2][pair of t 4][lane 64] (A, B, A', B'): M = step.re A + step.im B
void fxg_fmat_tables(uint32_t* out) {
  uint32_t* w = out;
  for (int odd = 0; odd < 2; ++odd)
    for (int ks = 0; ks < 4; ++ks)
      for (int lane = 0; lane < 64; ++lane)
        for (int e = 0; e < 8; e += 2) {
          const int row = lane & 31, k1 = 2 * (row >> 1) + odd, im = row & 1;
          const int s = 8 * ks + 4 * (lane >> 5) + (e >> 1);
          const double a = TWO_PI_D * ((s * k1) & 63) / 64.0;
          const double v[2] = {im ? -std::sin(a) : std::cos(a), im ? std::cos(a) : std::sin(a)};
          uint16_t h[2], l[2];
          for (int q = 0; q < 2; ++q) {
            const double x = v[q] * (double)FM_MSCALE;
            const _Float16 hh = (_Float16)x;
            const _Float16 ll = (_Float16)(x - (double)hh);
            h[q] = __builtin_bit_cast(uint16_t, hh);
            l[q] = __builtin_bit_cast(uint16_t, ll);
          }
          const int at = (((odd * 4 + ks) * 2) * 64 + lane) * 4 + (e >> 1);
          w[at] = h[0] | ((uint32_t)h[1] << 16);
          w[at + 64 * 4] = l[0] | ((uint32_t)l[1] << 16);
        }
  float* tc = reinterpret_cast<float*>(out + FMAT_W_WORDS);
  const double tsc = (double)FM_ZSCALE / ((double)FM_MSCALE * (double)FM_XSCALE);
  for (int st = 0; st < 2; ++st)
    for (int j = 0; j < 16; ++j)
      for (int lane = 0; lane < 64; ++lane) {
        const int s = 32 * st + (lane & 31), k2 = 16 * (j >> 3) + 4 * ((j >> 1) & 3) + 2 * (lane >> 5) + (j & 1);
        const double a = -TWO_PI_D * (double)(s * k2) / 2048.0;
        float* p = tc + (((st * 8 + (j >> 1)) * 64 + lane) * 2 + (j & 1)) * 2;
        p[0] = (float)(std::cos(a) * tsc);
        p[1] = (float)(std::sin(a) * tsc);
      }
  float* mc = tc + FMAT_T_WORDS;
  for (int rt = 0; rt < 2; ++rt)
    for (int ks = 0; ks < 2; ++ks)
      for (int p = 0; p < 4; ++p)
        for (int lane = 0; lane < 64; ++lane)
          for (int q = 0; q < 2; ++q) {
            const int row = 32 * rt + (lane & 31), k2 = row >> 1, im = row & 1;
            const int t = 16 * ks + 8 * (lane >> 5) + 2 * p + q;
            const double a = TWO_PI_D * ((t * k2) & 31) / 32.0;
            float* o = mc + (((rt * 2 + ks) * 4 + p) * 64 + lane) * 4 + 2 * q;
            o[0] = (float)(im ? -std::sin(a) : std::cos(a));
            o[1] = (float)(im ? std::cos(a) : std::sin(a));
          }
}

template <int ORDER>
__global__ void __launch_bounds__(64 * FM_NW, 2) k_fmat(FengineArgs args, const uint32_t* __restrict__ tables, int nds,
                                                       int nfs) {
  extern __shared__ fm_u4 fm_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hf = lane >> 5;
  const fm_u4* sW = fm_smem;
  const float4* sT = reinterpret_cast<const float4*>(reinterpret_cast<uint32_t*>(fm_smem) + FMAT_W_WORDS);
  const float4* sM = reinterpret_cast<const float4*>(reinterpret_cast<uint32_t*>(fm_smem) + FMAT_W_WORDS + FMAT_T_WORDS);
  uint32_t* own = reinterpret_cast<uint32_t*>(fm_smem) + FMAT_TABLE_WORDS + wave * FM_OWN;
  // exchange planes (hi, lo) [k2][s], FP16 (re, im) pairs: written by column s, read by row k2
  uint32_t* xw = own + 2 * hf * FM_HS + c;
  const uint32_t* xr = own + c * FM_HS + 4 * hf;
  float2* sub = reinterpret_cast<float2*>(own + 2 * FM_PLANE);
  float2* stp = sub + 64;
  float2* fsub = sub;                                // sub and stp are done with when these are made
  float2* fstp = fsub + 32;
  fm_u4* whi = reinterpret_cast<fm_u4*>(sub + FM_TAB) + lane;   // [4 groups][lane]
  for (int i = tid; i < FMAT_TABLE_WORDS / 4; i += 64 * FM_NW) fm_smem[i] = reinterpret_cast<const fm_u4*>(tables)[i];
  __syncthreads();                                   // the only barrier: from here each wavefront is on its own

  // work items: (freq part, datastream, eight consecutive FFTs, one per wavefront)
  const int nunit = args.nffts_pad / FM_NW;
  const int nitems = nunit * nds * nfs;
  const int cap = args.chunkcap;
  for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
    const int unit = item % nunit, rest = item / nunit;
    const int d = args.dslist[rest % nds], fpart = rest / nds;
    const CDevDs ds = (CDevDs)(args.ds + d);
    const int nrec = ds->nrecbands, spf = ds->spf;
    const GBytes data = (GBytes)args.run[d].data;
    const int nframes = args.run[d].nframes;
    const GBytes fv = (GBytes)(args.fvalid + ds->fvalid_off);
    const int2* __restrict__ fz = args.fzone + ds->fvalid_off;
    // levels of the four 2-bit codes as bytes of FP16 numbers: low bytes, high bytes (v_perm pools)
    uint32_t ph[2] = {0, 0}, pl[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v = lut2(ds->format, q) * FM_XSCALE;
      const _Float16 h = (_Float16)v;
      const _Float16 l = (_Float16)(v - (float)h);
      const uint32_t hb = __builtin_bit_cast(uint16_t, h), lb = __builtin_bit_cast(uint16_t, l);
      ph[0] |= (hb & 255u) << (8 * q); ph[1] |= (hb >> 8) << (8 * q);
      pl[0] |= (lb & 255u) << (8 * q); pl[1] |= (lb >> 8) << (8 * q);
    }
    {
      const int lt = unit * FM_NW + wave;
      const FXG_CONST FftDelay& fd = ((const FXG_CONST FftDelay*)args.params)[(long long)d * cap + lt];   // scalar loads
      const bool fok = fd.ok != 0;
      const bool whole = fok && fd.weight == 1.0f;   // every sample of the window decodes
      // output scale, in a scalar register; flagged FFTs: zero spectra (mode.cpp:656-669)
      const float fs = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(
          int, fok ? ds->xsc * (1.0f / (FM_MSCALE * FM_ZSCALE)) : 0.0f)));

      // Samples n = 32 st + c + 64 (16 ks + 8 hf + e): each word shifted so that band b's field is
      // at bit 2 b, then pairs (e, e + 1) merged as 16-bit halves: bands 0-7 in registers, 8-15 in LDS
      // (as registers they would spill).
      uint32_t wlo[16];
      uint32_t okm = 0xffffffffu;                    // bit per sample: decodes
      {
        const double inv = 1.0 / (double)spf;
#pragma unroll
        for (int g = 0; g < 4; ++g) {                // (st, ks)
          const unsigned g0 = (unsigned)fd.n0 + (unsigned)(32 * (g >> 1) + c + 64 * (16 * (g & 1) + 8 * hf));
          unsigned fr0 = (unsigned)((double)g0 * inv);
          unsigned w0 = g0 - fr0 * (unsigned)spf;
          if (w0 >= (unsigned)spf) { w0 -= spf; ++fr0; }
          uint32_t w[8];
          unsigned q[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            unsigned fr = fr0, wi = w0 + 64u * e;
            if (spf >= 512) {                        // uniform: at most one frame edge
              if (wi >= (unsigned)spf) { wi -= spf; ++fr; }
            } else {
              const unsigned gs = g0 + 64u * e;
              fr = (unsigned)((double)gs * inv);
              wi = gs - fr * (unsigned)spf;
              if (wi >= (unsigned)spf) { wi -= spf; ++fr; }
            }
            q[e] = wi * (unsigned)nrec;
            w[e] = 0;
            if (fok && nframes > 0) {
              const unsigned frc = min(fr, (unsigned)(nframes - 1));
              w[e] = *(GWords)(data + (size_t)frc * (unsigned)ds->framebytes + (unsigned)ds->headerbytes + ((q[e] >> 4) << 2));
            }
            if (!whole) {
              const bool ok = fok && fr < (unsigned)nframes && sample_ok(fv[min(fr, (unsigned)max(nframes - 1, 0))], fz, fr, wi);
              if (!ok) okm &= ~(1u << (8 * g + e));
            }
          }
          fm_u4 hi;
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const uint32_t a = w[e] >> (2 * (q[e] & 15u)), b = w[e + 1] >> (2 * (q[e + 1] & 15u));
            wlo[4 * g + e / 2] = __builtin_amdgcn_perm(b, a, 0x05040100u);
            hi[e / 2] = __builtin_amdgcn_perm(b, a, 0x07060302u);
          }
          if (nrec > 8) whi[64 * g] = hi;
        }
      }

      for (int f = fpart; f < ds->nrecfreqs; f += nfs) {
        const FreqConst rf = load_freq(ds->rf[f]);
        if (rf.nbands == 0) continue;
        // the lane number, opaque in each freq: what is computed from it would otherwise be kept
        // across the loop, in spilled registers (a reload waits for every store before it)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int lc = ln & 31, lh = ln >> 5;
        // ---- rotator phasors (mode.cpp:883-955) at s and at 64 t
        if (ORDER == 1) {
          const double sx = fd.a / FM_L;           // delay per sample across the FFT
          double b0 = fd.b * rf.lofreq;
          if (ds->fractionallo) b0 += (rf.lofreq - (double)(int)rf.lofreq) * (double)fd.intdelay;
          double slope = sx * rf.lofreq;
          if (rf.looff) {
            slope -= ds->sampletime_us / 1e6 * rf.lo_offset_hz;
            b0 -= rf.lo_offset_hz * fd.fracwall;
            if (rf.isfraclooffset) b0 -= rf.fraclooffset * fd.intwall;
          }
          float2 p = fm_turn(-(slope * (double)ln + b0));
          if (rf.lsb && (ln & 1)) p = make_float2(-p.x, -p.y);   // X[C + c]: (-1)^s
          sub[ln] = p;
          if (lh == 0) {
            p = fm_turn(-(slope * (double)(64 * lc)));
            stp[lc] = make_float2(p.x * FM_MSCALE, p.y * FM_MSCALE);
          }
        } else {
          sub[ln] = make_float2(rf.lsb && (ln & 1) ? -1.0f : 1.0f, 0.0f);
          if (lh == 0) stp[lc] = make_float2(FM_MSCALE, 0.0f);
        }
        fm_wave_sync();
        // ---- M in two FP16 parts, as stage 1's left operand
        fm_u4 mh[2][2], ml[2][2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            const float4 sv = *reinterpret_cast<const float4*>(&stp[16 * ks + 8 * lh + 2 * p]);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
              const float4 k = sM[((rt * 2 + ks) * 4 + p) * 64 + ln];
              unsigned hi, lo;
              fm_split(fmaf(sv.x, k.x, sv.y * k.y), fmaf(sv.z, k.z, sv.w * k.w), hi, lo);
              mh[rt][ks][p] = hi;
              ml[rt][ks][p] = lo;
            }
          }

        // the compiler does not know what an asm writes: keep M's parts two instructions away from
        // the matrix instructions that read them
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 1");
        __builtin_amdgcn_sched_barrier(0);

        const float2 sv[2] = {sub[lc], sub[32 + lc]};
        // NB bands from kb on, which share M and T; WHOLE: every sample decodes
        auto bands = [&](const int kb, auto nb_c, auto whole_c) {
          constexpr int NB = decltype(nb_c)::value;
          constexpr bool WHOLE = decltype(whole_c)::value != 0;
          fm_f16 y[NB][2][2];                        // [band][half of s, then E and D][row tile]
          // ---- stage 1
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            const int band = ds->rf[f].band[kb + b];
            const int sh = 2 * (band & 7);
#pragma unroll
            for (int st = 0; st < 2; ++st) {
              fm_u4 bh[2], bl[2];
              auto decode = [&](const uint32_t* w) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                  for (int p = 0; p < 4; ++p) {
                    const uint32_t code = (w[4 * ks + p] >> sh) & 0x00030003u;
                    const uint32_t sel = __umul24(code, 0x0101u) + 0x04000400u;
                    uint32_t h = __builtin_amdgcn_perm(ph[1], ph[0], sel), l = __builtin_amdgcn_perm(pl[1], pl[0], sel);
                    if (!WHOLE) {                    // invalid samples decode to zero
                      const uint32_t m2 = okm >> (8 * (2 * st + ks) + 2 * p);
                      const uint32_t m = ((m2 & 1u) ? 0xffffu : 0u) | ((m2 & 2u) ? 0xffff0000u : 0u);
                      h &= m;
                      l &= m;
                    }
                    bh[ks][p] = h;
                    bl[ks][p] = l;
                  }
              };
              if (band < 8) {                        // uniform; the empty asm keep it a branch
                asm volatile("; low bands");
                decode(wlo + 8 * st);
                asm volatile("; low bands decoded");
              } else {
                asm volatile("; high bands");
                const fm_u4 w0 = whi[64 * (2 * st)], w1 = whi[64 * (2 * st + 1)];
                const uint32_t w[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
                decode(w);
                asm volatile("; high bands decoded");
              }
#pragma unroll
              for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int r = 0; r < 16; ++r) y[b][st][rt][r] = 0.0f;
#pragma unroll
              for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) y[b][st][rt] = fm_mfma(ml[rt][ks], bh[ks], y[b][st][rt]);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) y[b][st][rt] = fm_mfma(mh[rt][ks], bl[ks], y[b][st][rt]);
              }
#pragma unroll
              for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) y[b][st][rt] = fm_mfma(mh[rt][ks], bh[ks], y[b][st][rt]);
            }
          }
          // ---- twiddles; E and D in place
#pragma unroll
          for (int jc = 0; jc < 2; ++jc) {
            __builtin_amdgcn_sched_barrier(0);       // no earlier: registers
            float4 tt[8];                            // W_2048^(s k2) of 8 k2, both halves of s
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
              for (int j = 0; j < 4; ++j) tt[4 * st + j] = sT[(st * 8 + 4 * jc + j) * 64 + lane];
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) {
              const float4 ta = tt[jj >> 1], tb = tt[4 + (jj >> 1)];
              const float2 T0 = cmul(jj & 1 ? make_float2(ta.z, ta.w) : make_float2(ta.x, ta.y), sv[0]);
              const float2 T1 = cmul(jj & 1 ? make_float2(tb.z, tb.w) : make_float2(tb.x, tb.y), sv[1]);
#pragma unroll
              for (int b = 0; b < NB; ++b) {
                const float2 z0 = cmul(make_float2(y[b][0][jc][2 * jj], y[b][0][jc][2 * jj + 1]), T0);
                const float2 z1 = cmul(make_float2(y[b][1][jc][2 * jj], y[b][1][jc][2 * jj + 1]), T1);
                y[b][0][jc][2 * jj] = z0.x + z1.x;
                y[b][0][jc][2 * jj + 1] = z0.y + z1.y;
                y[b][1][jc][2 * jj] = z0.x - z1.x;
                y[b][1][jc][2 * jj + 1] = z0.y - z1.y;
              }
            }
          }
          // ---- exchange and stage 2: even k1 from E, odd k1 from D.  While the matrix
          // instructions of one k-step run, a quarter of the next exchange's values is split (in
          // place: two floats become the words of their hi and lo parts).
          fm_f16 acc[NB][2];
          auto split4 = [&](int i, int q) {          // values 4 q .. 4 q + 3 of exchange i
            fm_f16(&v)[2] = y[i % NB][i / NB];
#pragma unroll
            for (int j = 4 * q; j < 4 * q + 4; ++j) {
              unsigned hi, lo;
              fm_split(v[j >> 3][2 * (j & 7)], v[j >> 3][2 * (j & 7) + 1], hi, lo);
              v[j >> 3][2 * (j & 7)] = __builtin_bit_cast(float, hi);
              v[j >> 3][2 * (j & 7) + 1] = __builtin_bit_cast(float, lo);
            }
          };
#pragma unroll
          for (int q = 0; q < 4; ++q) split4(0, q);
#pragma unroll
          for (int i = 0; i < 2 * NB; ++i) {
            const int b = i % NB, o = i / NB;
            fm_wave_sync();                          // the previous reads of the planes are issued
#pragma unroll
            for (int j = 0; j < 16; ++j) {
              const int k2 = 16 * (j >> 3) + 4 * ((j >> 1) & 3) + (j & 1);      // + 2 hf
              xw[k2 * FM_HS] = __builtin_bit_cast(unsigned, (float)y[b][o][j >> 3][2 * (j & 7)]);
              xw[FM_PLANE + k2 * FM_HS] = __builtin_bit_cast(unsigned, (float)y[b][o][j >> 3][2 * (j & 7) + 1]);
            }
            fm_wave_sync();
            fm_u4 z[2][2], w[2][2];
            auto load = [&](int ks) {                // the loads of one k-step ahead of its products
              z[ks & 1][0] = *reinterpret_cast<const fm_u4*>(xr + 8 * ks);
              z[ks & 1][1] = *reinterpret_cast<const fm_u4*>(xr + FM_PLANE + 8 * ks);
#pragma unroll
              for (int q = 0; q < 2; ++q) w[ks & 1][q] = sW[((o * 4 + ks) * 2 + q) * 64 + lane];
            };
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][o][r] = 0.0f;
            load(0);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
              if (ks < 3) load(ks + 1);
              __builtin_amdgcn_sched_barrier(0);
              acc[b][o] = fm_mfma(w[ks & 1][1], z[ks & 1][0], acc[b][o]);
              acc[b][o] = fm_mfma(w[ks & 1][0], z[ks & 1][1], acc[b][o]);
              acc[b][o] = fm_mfma(w[ks & 1][0], z[ks & 1][0], acc[b][o]);
              if (i + 1 < 2 * NB) split4(i + 1, ks);
            }
          }
          // ---- fractional-sample phasors (mode.cpp:1030-1122), corrected channels, stores
          float2 frq[16];                            // of k1 = 8 (i / 4) + 4 hf + i % 4
          const int ch = lc + 128 * lh;               // channel of k1 = 4 hf; k1 + 1: 32 channels on
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            const int band = ds->rf[f].band[kb + b];
            if (b == 0 || ds->rf[f].newfrac[kb + b]) {
              if (kb + b == 0 || ds->rf[f].newfrac[kb + b]) {
                const float e = (float)((double)fd.fse - rf.clockoff + ds->rf[f].bhd[kb + b]);
                const double per = (double)e * ds->bw_mhz * (1.0 / FM_C);   // turns per channel
                double ph0 = 0.0;
                if (ORDER == 0) {                    // the post-F fringe phase (mode.cpp:1040-1049)
                  ph0 = fd.b * rf.lofreq;
                  if (ds->fractionallo) ph0 += fd.intdelay * (rf.lofreq - (int)rf.lofreq);
                  ph0 -= ((double)fd.intwall + fd.fracwall) * rf.lo_offset_hz;
                }
                // lanes 0-31: channel c (with the pol phase offset); 32-63: stride c of 32 channels
                float2 p = fm_turn(lh == 0 ? per * (double)lc - ph0 : per * (double)(32 * lc - (rf.lsb ? FM_C : 0)));
                if (lh == 0) {
                  const float2 pc = make_float2(ds->rf[f].pcre[kb + b], ds->rf[f].pcim[kb + b]);
                  if (!(pc.x == 1.0f && pc.y == 0.0f)) p = cmul(p, pc);
                  fsub[lc] = p;
                } else {
                  fstp[lc] = make_float2(p.x * fs, p.y * fs);
                }
                fm_wave_sync();
              }
              const float2 fc = fsub[lc];
#pragma unroll
              for (int i = 0; i < 16; i += 2) {
                const float4 fp = *reinterpret_cast<const float4*>(&fstp[8 * (i >> 2) + 4 * lh + (i & 3)]);
                frq[i] = cmul(fc, make_float2(fp.x, fp.y));
                frq[i + 1] = cmul(fc, make_float2(fp.z, fp.w));
              }
            }
            auto channels = [&](auto emit) {         // emit(k1 without its 4 hf, value)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const int r = 4 * (i >> 2) + 2 * ((i >> 1) & 1);
                emit(8 * (i >> 2) + (i & 3), cmul(make_float2(acc[b][i & 1][r], acc[b][i & 1][r + 1]), frq[i]));
              }
            };
            // (uniform bases plus a 32-bit byte offset per lane)
            if (args.out_mode == 0) {
              char* __restrict__ o = (char*)(args.spec32 + ds->spec_off + ((long long)band * cap + lt) * FM_C);
              const unsigned lo = 8u * (unsigned)ch;
              channels([&](int k1, float2 v) { *(float2*)(o + 256 * k1 + lo) = v; });
            } else {
              auto store16 = [&](auto mode_c) {
                constexpr int OM = decltype(mode_c)::value;
                const CDevXGroup xg = ((CDevXGroup)args.xgroups) + ds->band_xfreq[band];
                const int tw = xg->twlog;
                char* __restrict__ o = (char*)(args.spec16 + xg->spec_off + (long long)ds->band_xrow[band] * xg->rowstride +
                                               ((long long)lt << tw));
                const unsigned lo = 4u * ((((unsigned)(ch >> tw) * (unsigned)cap) << tw) + (unsigned)(ch & ((1 << tw) - 1)));
                const long long ks = 4LL * ((long long)(32 >> tw) * cap << tw);
                channels([&](int k1, float2 v) { *(uint32_t*)(o + k1 * ks + lo) = pack16m<OM>(v); });
                for (int z = 0; z < ds->nzout; ++z) {              // zoom windows of this band
                  if (ds->zout_band[z] != band) continue;
                  const int c0 = ds->zout_c0[z], nz = ds->zout_n[z];
                  const CDevXGroup zg = ((CDevXGroup)args.xgroups) + ds->zout_group[z];
                  const int zl = zg->twlog, zm = (1 << zl) - 1;
                  uint32_t* __restrict__ oz = args.spec16 + zg->spec_off + (long long)ds->zout_row[z] * zg->rowstride + ((long long)lt << zl);
                  channels([&](int k1, float2 v) {
                    const int cz = ch + 32 * k1 - c0;
                    if (cz >= 0 && cz < nz) oz[(((long long)(cz >> zl) * cap) << zl) + (cz & zm)] = pack16m<OM>(v);
                  });
                }
              };
              if (args.out_mode == 1) store16(IntC<1>());
              else store16(IntC<2>());
            }
          }
        };
        for (int kb = 0; kb < rf.nbands; kb += 2) {
          if (kb + 1 < rf.nbands) {
            if (whole) bands(kb, IntC<2>(), IntC<1>());
            else bands(kb, IntC<2>(), IntC<0>());
          } else {
            if (whole) bands(kb, IntC<1>(), IntC<1>());
            else bands(kb, IntC<1>(), IntC<0>());
          }
        }
      }
    }
  }
}

// Chunk FFTs of the nds datastreams of args.dslist (2-bit real, 2048-point FFTs).
int fxg_launch_fmat(const FengineArgs& a, int nds, int ncu, int nfreqs, const uint32_t* tables, hipStream_t st) {
  if (fxg_launch_fftparams(a, nds, st)) return -1;
  // where the FFTs do not fill the device, the freqs of an FFT go to different workgroups
  const int units = nds * (a.nffts_pad / FM_NW);
  const int nfs = std::max(1, std::min(nfreqs, 2 * ncu / std::max(1, units)));
  const int grid = std::min(ncu, units * nfs);
  const size_t lds = fxg_fmat_lds();
  static size_t raised[2] = {0, 0};
  if (a.rotorder == 1) {
    if (raise_lds(k_fmat<1>, lds, &raised[1])) return -1;
    hipLaunchKernelGGL(k_fmat<1>, dim3(grid), dim3(64 * FM_NW), lds, st, a, tables, nds, nfs);
  } else if (a.rotorder == 0) {
    if (raise_lds(k_fmat<0>, lds, &raised[0])) return -1;
    hipLaunchKernelGGL(k_fmat<0>, dim3(grid), dim3(64 * FM_NW), lds, st, a, tables, nds, nfs);
  } else {
    return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
