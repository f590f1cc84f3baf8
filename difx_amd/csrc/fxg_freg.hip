// F-engine for long FFTs (4096 to 32768 points) of real 2-bit and complex 8-bit samples with the
// whole FFT in the registers of one workgroup.  What one FFT computes is what the fused F-engine
// computes (Mode::process, mode.cpp:634-1374: decode, rotator, L-point FFT, channel selection,
// fractional-sample correction).
//
// L/32 threads hold 32 points each and run three Stockham passes of radix 32, 32 and L/1024; the
// two exchanges between them go through LDS as real parts and then imaginary parts, so that a
// 32768-point FFT takes 128 KB of it (a CU's 160 KB hold no complex one) and no spectrum passes
// through memory on its way.  Three passes instead of the five of the four-step kernel: fewer LDS
// trips, addresses and twiddles.  What bounds it is vector instructions: 76 per point at 32768
// points, 76 % of the cycles (the four-step kernel: 118, 65 %; it also wrote and read each
// spectrum once in L2 and MALL).  Measured, 16 stations, 1001 FFTs of 32768 points in 8 bands
// and 1001 of 16384 in 8: 22.1 -> 12.0 ms and 9.0 -> 4.5 ms; 8 stations, 1000 FFTs of 8192 points
// in 8 bands (k_fengine before): 1.61 -> 1.19 ms; 16 stations, 4096 points in 16 bands 3.5 -> 2.6 ms;
// 64 stations of complex 8-bit samples, 3906 FFTs of 4096 points: 6.3 -> 3.6 ms.
#include "fxg_fe_common.h"
#include <algorithm>
#include <cmath>
#include <vector>

namespace {

// Constant twiddles W32^M = exp(-2 pi i M / 32) = (-i)^q c (1 - i t) with |angle| <= pi/4: turn()
// gives (-i)^q (1 - i t) z, one fused multiply-add per component, and the factor c goes into the
// fused multiply-add of the butterfly that follows (Linzer and Feig's scheme): no separate
// multiplication, and one rounding per step.
constexpr double COSD[5] = {1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
                            0.70710678118654752440};     // cos(2 pi m / 32)
constexpr double TAND[5] = {0.0, 0.19891236737965800691, 0.41421356237309504880, 0.66817863791929891999, 1.0};
constexpr int tw_m(int M) { return (M & 31) - 8 * (((M & 31) + 4) / 8); }      // -4 .. 3
constexpr double tw_c(int M) { return COSD[tw_m(M) < 0 ? -tw_m(M) : tw_m(M)]; }
template <int M>
__device__ __forceinline__ float2 turn(float2 z) {
  constexpr int q = (((M & 31) + 4) / 8) & 3, m = tw_m(M);
  constexpr float t = (float)(m < 0 ? -TAND[-m] : TAND[m]);
  const float2 r = q == 0 ? z : q == 1 ? make_float2(z.y, -z.x) : q == 2 ? make_float2(-z.x, -z.y) : make_float2(-z.y, z.x);
  if (m == 0) return r;
  return make_float2(fmaf(t, r.y, r.x), fmaf(-t, r.x, r.y));
}
__device__ __forceinline__ float2 axpy(float c, float2 b, float2 a) { return make_float2(fmaf(c, b.x, a.x), fmaf(c, b.y, a.y)); }

// a + c b and a - c b
template <typename C>
__device__ __forceinline__ void bfly(float2& a, float2& b, C c) {
  constexpr float f = (float)C::v;
  const float2 s = f == 1.0f ? cadd(a, b) : axpy(f, b, a), d = f == 1.0f ? csub(a, b) : axpy(-f, b, a);
  a = s;
  b = d;
}
template <int A, int B>
struct RatioC { static constexpr double v = tw_c(A) / tw_c(B); };          // cos A / cos B
template <int A>
struct HalfC { static constexpr double v = COSD[4] * tw_c(A); };            // sqrt(1/2) cos A

// DFT4 and DFT8 of z[b] W32^(K b), natural order.
template <int K>
__device__ __forceinline__ void dft4k(float2* z) {
  float2 a0 = z[0], a1 = turn<K>(z[1]), a2 = turn<2 * K>(z[2]), a3 = turn<3 * K>(z[3]);
  bfly(a0, a2, RatioC<2 * K, 0>());
  bfly(a1, a3, RatioC<3 * K, K>());
  a3 = mul_negi(a3);
  bfly(a0, a1, RatioC<K, 0>());
  bfly(a2, a3, RatioC<K, 0>());
  z[0] = a0; z[1] = a2; z[2] = a1; z[3] = a3;
}
template <int K>
__device__ __forceinline__ void dft8k(float2* z) {
  float2 u0 = z[0], u1 = turn<K>(z[1]), u2 = turn<2 * K>(z[2]), u3 = turn<3 * K>(z[3]);
  float2 u4 = turn<4 * K>(z[4]), u5 = turn<5 * K>(z[5]), u6 = turn<6 * K>(z[6]), u7 = turn<7 * K>(z[7]);
  bfly(u0, u4, RatioC<4 * K, 0>());
  bfly(u2, u6, RatioC<6 * K, 2 * K>());
  bfly(u1, u5, RatioC<5 * K, K>());
  bfly(u3, u7, RatioC<7 * K, 3 * K>());
  bfly(u0, u2, RatioC<2 * K, 0>());
  bfly(u1, u3, RatioC<3 * K, K>());
  u3 = mul_negi(u3);
  bfly(u0, u1, RatioC<K, 0>());
  bfly(u2, u3, RatioC<K, 0>());
  u5 = make_float2(u5.x + u5.y, u5.y - u5.x);            // sqrt(2) W8^1
  u6 = mul_negi(u6);
  u7 = make_float2(u7.y - u7.x, -(u7.x + u7.y));         // sqrt(2) W8^3
  bfly(u4, u6, RatioC<2 * K, 0>());
  bfly(u5, u7, RatioC<3 * K, K>());
  u7 = mul_negi(u7);
  bfly(u4, u5, HalfC<K>());
  bfly(u6, u7, HalfC<K>());
  z[0] = u0; z[1] = u4; z[2] = u2; z[3] = u6; z[4] = u1; z[5] = u5; z[6] = u3; z[7] = u7;
}

// 32-point forward DFT as 4 x 8 in place: X[k1 + 4 k2] ends in x[8 k1 + k2].
__device__ __forceinline__ void dft32(float2* x) {
#pragma unroll
  for (int b = 0; b < 8; ++b) dft4(x[b], x[8 + b], x[16 + b], x[24 + b]);
  dft8k<0>(x);
  dft8k<1>(x + 8);
  dft8k<2>(x + 16);
  dft8k<3>(x + 24);
}
__host__ __device__ constexpr int reg32(int r) { return 8 * (r & 3) + (r >> 2); }   // register of X[r]

// 16-point forward DFT as 4 x 4 in place: X[k1 + 4 k2] ends in x[4 k1 + k2].
__device__ __forceinline__ void dft16p(float2* x) {
#pragma unroll
  for (int b = 0; b < 4; ++b) dft4(x[b], x[4 + b], x[8 + b], x[12 + b]);
  dft4k<0>(x);
  dft4k<2>(x + 4);
  dft4k<4>(x + 8);
  dft4k<6>(x + 12);
}

// The thread number, opaque to the compiler at each use: otherwise it computes the addresses of
// every phase of a band ahead of the band loop and, for want of registers, spills them.
__device__ __forceinline__ int opaque(int t) {
  asm volatile("" : "+v"(t));
  return t;
}
typedef const __attribute__((address_space(1))) uint16_t* GHalfs;
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// An FFT's parameters, uniform: read by scalar loads where they are used.
typedef const FXG_CONST FftDelay* CFftDelay;
__device__ __forceinline__ FftDelay load_delay(const FXG_CONST FftDelay& p) {
  FftDelay r;
  r.ok = p.ok; r.n0 = p.n0; r.fse = p.fse; r.intdelay = p.intdelay; r.a = p.a; r.b = p.b; r.c = p.c;
  r.weight = p.weight; r.intwall = p.intwall; r.fracwall = p.fracwall;
  return r;
}

template <int L>
struct RPlan {
  static constexpr int NT = L / 32;               // threads of an FFT
  static constexpr int R = L / 1024;              // radix of the last pass
  static constexpr int NB = 32 / R;               // its butterflies per thread
  static constexpr int G = L == 4096 ? 2 : 1;     // FFTs side by side in a workgroup
  static constexpr int TW1 = 31 * 32;             // twiddles of the second pass, [s - 1][k]
  static constexpr int TW2 = (R - 1) * 1024;      // and of the last, [s - 1][j]
  // register of X[t + q NT] after the last pass: butterfly q % NB, output q / NB
  static constexpr int reg(int q) {
    const int b = q % NB, r = q / NB;
    return R == 32 ? reg32(r) : R == 16 ? b * 16 + 4 * (r & 3) + (r >> 2) : b * R + r;
  }
};

template <int L>
size_t freg_lds_bytes(int cplx, int order, int phcap) {
  constexpr int G = RPlan<L>::G;
  return sizeof(float) * (size_t)L * G + sizeof(float2) * ((size_t)RPlan<L>::TW1 + 2 * (size_t)G * phcap) +
         sizeof(float) * ((order == 2 ? (size_t)G * phcap : 0) + (cplx ? 256 : 8)) + stage_lds_bytes(phcap);
}

}  // namespace

// Workgroup (x, y): FFTs [x * upw, ...) of datastream dslist[y], consecutive ones so that their
// 16-bit spectra complete each other's lines in one L2.  128 registers: at 32768
// points one workgroup of 16 waves per CU, at 16384 two of 8, below three of 4 (by LDS; 4096
// points two FFTs side by side), so that one works while the others wait.
template <int L, bool CPLX, int ORDER>
__global__ void __launch_bounds__(L / 32 * RPlan<L>::G, 4) k_freg(FengineArgs args, const float2* __restrict__ tw, int upw) {
  using P = RPlan<L>;
  constexpr int NT = P::NT, G = P::G, NTB = NT * G;
  extern __shared__ float2 fx_smem[];
  const int tid = threadIdx.x;
  const int g = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / NT), t0 = tid - g * NT;
  const int ph = args.phcap;
  float2* stw = fx_smem;                          // twiddles of the second pass
  float2* srot = stw + P::TW1 + g * ph;
  float2* sfrac = stw + P::TW1 + (G + g) * ph;
  float* xb = reinterpret_cast<float*>(stw + P::TW1 + 2 * G * ph) + g * L;    // exchange buffer
  float* squad = reinterpret_cast<float*>(stw + P::TW1 + 2 * G * ph) + G * L + g * ph;
  float* slev = reinterpret_cast<float*>(stw + P::TW1 + 2 * G * ph) + G * (ORDER == 2 ? L + ph : L);   // the sample levels
  float* scf = slev + (CPLX ? 256 : 8);                        // staged channel-frequency tables
  const int d = args.dslist[blockIdx.y];
  const CDevDs dsp = (CDevDs)(args.ds + d);
  for (int m = tid; m < P::TW1; m += NTB) stw[m] = tw[m];
  for (int m = tid; m < (CPLX ? 256 : 4); m += NTB) slev[m] = CPLX ? lut8(m) : lut2(dsp->format, m);
  stage_cf(args, dsp, scf, tid, NTB);
  const float2* __restrict__ tw2 = tw + P::TW1;
  DsConst k;
  k.C = dsp->C; k.S = dsp->S; k.NS = dsp->NS; k.NFS = dsp->NFS; k.nrec = dsp->nrecbands;
  k.nrecfreqs = dsp->nrecfreqs; k.fmt = dsp->format; k.spf = dsp->spf;
  k.framebytes = dsp->framebytes; k.headerbytes = dsp->headerbytes; k.nbits = dsp->nbits;
  k.fractionallo = dsp->fractionallo; k.sampletime_us = dsp->sampletime_us; k.dsb = dsp->dsb;
  const GBytes fv = (GBytes)(args.fvalid + dsp->fvalid_off);
  const int2* __restrict__ fz = args.fzone + dsp->fvalid_off;
  const GBytes data = (GBytes)args.run[d].data;
  const int nframes = args.run[d].nframes;
  const CFftDelay params = (CFftDelay)(args.params + (long long)d * args.chunkcap);
  const int S = k.S;
  const float xsc = dsp->xsc;
  const double inv_spf = 1.0 / (double)k.spf;
  const int nrl = 31 - __clz(k.nrec);              // the bands of 2-bit samples are a power of two
  const int cap = args.chunkcap;

  const int lt0 = blockIdx.x * upw, lt1 = min(lt0 + upw, args.nffts_pad);
  for (int lb = lt0; lb < lt1; lb += G) {          // (lt1 - lt0 is a multiple of G)
    const int lt = lb + g;
    const int n0 = params[lt].n0;
    const bool fok_all = params[lt].ok != 0;       // flagged FFTs: zero spectra (mode.cpp:656-669)
    const bool whole = fok_all && params[lt].weight == 1.0f;   // every sample of the window decodes
    const float fs = fok_all ? xsc : 0.0f;
    for (int f = 0; f < k.nrecfreqs; ++f) {
      const int nbands = dsp->rf[f].nbands;
      if (nbands == 0) continue;
      __syncthreads();                            // previous users of srot/sfrac are done
      {
      const FreqConst rf = load_freq(dsp->rf[f]);
      const FftDelay fd = load_delay(params[lt]);
      if (ORDER != 0) build_rotator<ORDER>(srot, squad, k, rf, fd, L, t0, NT);
      build_frac<ORDER>(sfrac, k, rf, CPLX, scf, fd, dsp->rf[f].bhd[0], make_float2(dsp->rf[f].pcre[0], dsp->rf[f].pcim[0]), t0, NT);
      }
      __syncthreads();
      uint32_t pk[2][2], okm = ~0u;
      for (int kb = 0; kb < nbands; ++kb) {
        const int band = dsp->rf[f].band[kb];
        if (kb > 0 && dsp->rf[f].newfrac[kb]) {    // another pol's phasor table (uniform branch)
          __syncthreads();                        // the previous band's phasor reads are done
          const FreqConst rf = load_freq(dsp->rf[f]);
          const FftDelay fd = load_delay(params[lt]);
          build_frac<ORDER>(sfrac, k, rf, CPLX, scf, fd, dsp->rf[f].bhd[kb], make_float2(dsp->rf[f].pcre[kb], dsp->rf[f].pcim[kb]), t0, NT);
        }
        // The 2-bit fields of this thread's samples n = t + s NT, for two bands at a time: a
        // sample word holds every band's field.
        if (!CPLX && (kb & 1) == 0) {
          const int t = opaque(t0);
          const int sh0 = 2 * band, sh1 = 2 * (kb + 1 < nbands ? dsp->rf[f].band[kb + 1] : band);
          pk[0][0] = pk[0][1] = pk[1][0] = pk[1][1] = 0u;
          // frame and sample within it: the quotient through the reciprocal of spf (exact after
          // the one correction: sample indices and spf stay below 2^31 and 2^20)
          const unsigned g0 = (unsigned)n0 + (unsigned)t;
          unsigned fr = (unsigned)((double)g0 * inv_spf);
          unsigned within = g0 - fr * (unsigned)k.spf;
          if (within >= (unsigned)k.spf) { within -= k.spf; ++fr; }
          unsigned pay = fr * (unsigned)k.framebytes + (unsigned)k.headerbytes;   // of the frame's payload
          auto next = [&](int s) {                // on to sample s: at most one frame on, or divide
            if (k.spf >= NT) {
              within += NT;
              const bool over = within >= (unsigned)k.spf;
              within -= over ? (unsigned)k.spf : 0u;
              pay += over ? (unsigned)k.framebytes : 0u;
              fr += over ? 1u : 0u;
            } else {
              const unsigned gs = g0 + (unsigned)(s * NT);
              fr = (unsigned)((double)gs * inv_spf);
              within = gs - fr * (unsigned)k.spf;
              if (within >= (unsigned)k.spf) { within -= k.spf; ++fr; }
              pay = fr * (unsigned)k.framebytes + (unsigned)k.headerbytes;
            }
          };
          if (whole) {
#pragma unroll
            for (int sb = 0; sb < 32; sb += 8) {
              uint32_t w[8], sh[8];
#pragma unroll
              for (int s = 0; s < 8; ++s) {
                const unsigned q = within << nrl;   // first field of the sample
                w[s] = *(GWords)(data + (pay + ((q >> 4) << 2)));
                sh[s] = 2u * (q & 15u);
                next(sb + s + 1);
              }
#pragma unroll
              for (int s = 0; s < 8; ++s) {
                const int at = 2 * ((sb + s) & 15), h = (sb + s) >> 4;
                const uint32_t x = w[s] >> sh[s];
                pk[0][h] |= ((x >> sh0) & 3u) << at;
                pk[1][h] |= ((x >> sh1) & 3u) << at;
              }
              fence();                            // eight loads in flight at a time
            }
          } else {
            okm = 0u;
#pragma unroll 1
            for (int s = 0; s < 32; ++s) {
              if (fok_all && fr < (unsigned)nframes && sample_ok(fv[fr], fz, fr, within)) {
                const unsigned q = within << nrl;
                const uint32_t w = *(GWords)(data + (pay + ((q >> 4) << 2)));
                const uint32_t x = w >> (2u * (q & 15u));
                const uint32_t a = ((x >> sh0) & 3u) << (2 * (s & 15)), b = ((x >> sh1) & 3u) << (2 * (s & 15));
                okm |= 1u << s;
                if (s < 16) { pk[0][0] |= a; pk[1][0] |= b; }
                else { pk[0][1] |= a; pk[1][1] |= b; }
              }
              next(s + 1);
            }
          }
        }
        float2 v[32];
        const bool lsb = dsp->rf[f].lsb != 0;
        const uint32_t p0 = kb & 1 ? pk[1][0] : pk[0][0], p1 = kb & 1 ? pk[1][1] : pk[0][1];
        fence();
        // order 2: the quadratic sub term^j, j = n/S (mode.cpp:1017-1024), of every eighth sample and
        // its step from one sample to the next (a chain of 32 factors was 1.9 times as far off)
        float2 qstart[4], qstep = make_float2(1.0f, 0.0f);
        if (ORDER == 2) {
          const int t = opaque(t0);
          const float th = squad[t & (S - 1)];
          float sn, cs;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sincosf((float)(t / S + 8 * i * (NT / S)) * th, &sn, &cs);
            qstart[i] = make_float2(cs, sn);
          }
          sincosf((float)(NT / S) * th, &sn, &cs);
          qstep = make_float2(cs, sn);
          fence();
        }
        if (CPLX) {
          // complex 8-bit samples: both bytes in one load, sixteen in flight; an invalid sample
          // reads the buffer's first bytes, if it has any
          const int t = opaque(t0);
          const unsigned g0 = (unsigned)n0 + (unsigned)t;
          const bool any = fok_all && nframes > 0;
          okm = whole ? ~0u : 0u;
#pragma unroll
          for (int sb = 0; sb < 32; sb += 16) {
            unsigned w[16];
#pragma unroll
            for (int s = 0; s < 16; ++s) {
              const unsigned gs = g0 + (unsigned)((sb + s) * NT);
              unsigned fr = (unsigned)((double)gs * inv_spf);
              unsigned within = gs - fr * (unsigned)k.spf;
              if (within >= (unsigned)k.spf) { within -= k.spf; ++fr; }
              bool ok = whole;
              if (!whole) {
                ok = any && fr < (unsigned)nframes && sample_ok(fv[fr], fz, fr, within);
                okm |= (ok ? 1u : 0u) << (sb + s);
              }
              const unsigned at = fr * (unsigned)k.framebytes + (unsigned)k.headerbytes + (within * (unsigned)k.nrec + band) * 2u;
              w[s] = any ? *(GHalfs)(data + (ok ? at : 0u)) : 0u;
            }
#pragma unroll
            for (int s = 0; s < 16; ++s) v[sb + s] = make_float2(slev[w[s] & 255u], slev[w[s] >> 8]);
            fence();
          }
        }
        {
          const int t = opaque(t0);
          const float2 sub = ORDER != 0 ? srot[t & (S - 1)] : make_float2(1.0f, 0.0f);
          float2 qpow = make_float2(1.0f, 0.0f);
          const float2* __restrict__ step = srot + S + t / S;    // NT is a multiple of S
#pragma unroll
          for (int s = 0; s < 32; ++s) {
            const float x = CPLX ? 0.0f : slev[((s < 16 ? p0 : p1) >> (2 * (s & 15))) & 3u];
            if (ORDER == 0) {
              v[s] = make_float2(x, 0.0f);
            } else {
              float2 rot = sub;
              if (ORDER == 2 && s % 8 == 0) qpow = qstart[s / 8];
              if (ORDER == 2) { rot = cmul(sub, qpow); qpow = cmul(qpow, qstep); }
              rot = cmul(rot, step[s * (NT / S)]);
              v[s] = CPLX ? cmul(rot, v[s]) : make_float2(x * rot.x, x * rot.y);
              // complex LSB: conj input gives the conjugate-flipped spectrum (mode.cpp:1186-1201)
              if (CPLX && lsb) v[s].y = -v[s].y;
            }
            if (s % 8 == 7) fence();
          }
          if (!whole) {
#pragma unroll
            for (int s = 0; s < 32; ++s)
              if (!((okm >> s) & 1u)) v[s] = make_float2(0.0f, 0.0f);
          }
        }
        // ---- pass 1, and its exchange: thread t writes entries 32 t + r, four at a time and
        // XORed with the row so that eight lanes fill the banks; a row is read as a permutation
        dft32(v);
        fence();
        {
          const int t = opaque(t0);
          const int rd = (t & ~31) + ((t & 31) ^ (4 * ((t >> 5) & 7)));
          float4* xw = reinterpret_cast<float4*>(xb) + 8 * t;
          __syncthreads();                        // the previous band's reads are done
#pragma unroll
          for (int i = 0; i < 8; ++i) xw[i ^ (t & 7)] = make_float4(v[i].x, v[8 + i].x, v[16 + i].x, v[24 + i].x);
          __syncthreads();
#pragma unroll
          for (int s = 0; s < 32; ++s) v[s].x = xb[(NT == 128 && (s & 1) ? rd ^ 16 : rd) + s * NT];
          __syncthreads();
#pragma unroll
          for (int i = 0; i < 8; ++i) xw[i ^ (t & 7)] = make_float4(v[i].y, v[8 + i].y, v[16 + i].y, v[24 + i].y);
          __syncthreads();
#pragma unroll
          for (int s = 0; s < 32; ++s) v[s].y = xb[(NT == 128 && (s & 1) ? rd ^ 16 : rd) + s * NT];
        }
        // ---- pass 2
        {
          const float2* twp = stw + (opaque(t0) & 31);
#pragma unroll
          for (int s = 1; s < 32; ++s) {
            v[s] = cmul(v[s], twp[(s - 1) * 32]);
            if (s % 8 == 7) fence();
          }
        }
        dft32(v);
        fence();
        {
          const int t = opaque(t0);
          float* xw = xb + (t >> 5) * 1024 + (t & 31);
          __syncthreads();
#pragma unroll
          for (int r = 0; r < 32; ++r) xw[r * 32] = v[reg32(r)].x;
          __syncthreads();
#pragma unroll
          for (int s = 0; s < 32; ++s) v[s].x = xb[t + s * NT];
          __syncthreads();
#pragma unroll
          for (int r = 0; r < 32; ++r) xw[r * 32] = v[reg32(r)].y;
          __syncthreads();
#pragma unroll
          for (int s = 0; s < 32; ++s) v[s].y = xb[t + s * NT];
        }
        // ---- pass 3: NB butterflies of R points, element s of butterfly b in register b + s NB;
        // its twiddles from L2 (one table entry per point and length), eight in flight
        float2 z[32];
        const int t = opaque(t0);
        const float2* __restrict__ twb = tw2;
        asm volatile("" : "+s"(twb));
#pragma unroll
        for (int b = 0; b < P::NB; ++b) {
          z[b * P::R] = v[b];
#pragma unroll
          for (int s0 = 1; s0 < P::R; s0 += 8) {
            float2 w[8];
#pragma unroll
            for (int s = 0; s < 8; ++s)
              if (s0 + s < P::R) w[s] = (twb + ((s0 + s - 1) * 1024 + b * NT))[(unsigned)t];
#pragma unroll
            for (int s = 0; s < 8; ++s)
              if (s0 + s < P::R) z[b * P::R + s0 + s] = cmul(v[b + (s0 + s) * P::NB], w[s]);
            if (P::R > 4 || (b & 1)) fence();
          }
          if (P::R == 32) dft32(z);
          else if (P::R == 16) dft16p(z + b * P::R);
          else if (P::R == 8) dft8k<0>(z + b * P::R);
          else dft4k<0>(z + b * P::R);
        }
        // ---- the kept channels c = t + m NT, times the fractional-sample phasor and the output
        // scale: real USB X[c], LSB X[C + c] (mode.cpp:1205); complex all, halves swapped for double
        // sideband (mode.cpp:1191-1192, 1211-1213)
        constexpr int KEEP = CPLX ? 32 : 16;
        if (CPLX && lsb && !k.dsb && t == 0) z[P::reg(0)].y = -z[P::reg(0)].y;   // DC is not flipped (mode.cpp:1199-1200)
        const float2 fsub0 = sfrac[t & (S - 1)];
        const float2 fsub = make_float2(fsub0.x * fs, fsub0.y * fs);
        const float2* __restrict__ fstep = sfrac + S + t / S;
        auto emit = [&](auto half_c) {
          constexpr int H = decltype(half_c)::value;
          if (args.out_mode == 0) {
            float2* __restrict__ o32 = args.spec32 + dsp->spec_off + ((long long)band * cap + lt) * k.C;
#pragma unroll
            for (int m = 0; m < KEEP; ++m) (o32 + m * NT)[(unsigned)t] = cmul(z[P::reg((H + m) & 31)], cmul(fsub, fstep[m * (NT / S)]));
            return;
          }
          auto store16 = [&](auto mode_c) {
            constexpr int OM = decltype(mode_c)::value;
            // channel c of FFT lt sits at (c / TW) cap TW + lt TW + c % TW of the row; NT is a
            // multiple of TW, so a uniform base per m and an offset per thread (below 2^32 bytes:
            // a chunk's FFTs hold fewer than 2^31 samples)
            const CDevXGroup xgr = ((CDevXGroup)args.xgroups) + dsp->band_xfreq[band];
            const int twl = xgr->twlog, twm = (1 << twl) - 1;
            uint32_t* __restrict__ o16 = args.spec16 + xgr->spec_off + (long long)dsp->band_xrow[band] * xgr->rowstride +
                                         ((long long)lt << twl);
            const unsigned ot = (((unsigned)(t >> twl) * (unsigned)cap) << twl) + (unsigned)(t & twm);
            const long long cs16 = ((long long)(NT >> twl) * cap) << twl;
            const bool zoom = dsp->nzout > 0;
#pragma unroll
            for (int m = 0; m < KEEP; ++m) {
              const uint32_t o = pack16m<OM>(cmul(z[P::reg((H + m) & 31)], cmul(fsub, fstep[m * (NT / S)])));
              (o16 + m * cs16)[ot] = o;
              if (zoom) z[P::reg((H + m) & 31)].x = __uint_as_float(o);   // kept for the windows
            }
            // zoom windows of this band: the same channels again, as rows of the zoom freq's group
            for (int zz = 0; zz < dsp->nzout; ++zz) {
              if (dsp->zout_band[zz] != band) continue;
              const int c0 = dsp->zout_c0[zz], nz = dsp->zout_n[zz];
              const CDevXGroup zg = ((CDevXGroup)args.xgroups) + dsp->zout_group[zz];
              const int zl = zg->twlog, zm = (1 << zl) - 1;
              uint32_t* __restrict__ oz = args.spec16 + zg->spec_off + (long long)dsp->zout_row[zz] * zg->rowstride +
                                          ((long long)lt << zl);
#pragma unroll
              for (int m = 0; m < KEEP; ++m) {
                const int cz = t + m * NT - c0;
                if (cz >= 0 && cz < nz) oz[(((long long)(cz >> zl) * cap) << zl) + (cz & zm)] = __float_as_uint(z[P::reg((H + m) & 31)].x);
              }
            }
          };
          if (args.out_mode == 1) store16(IntC<1>());
          else store16(IntC<2>());
        };
        if (CPLX ? k.dsb != 0 : lsb) emit(IntC<16>());
        else emit(IntC<0>());
      }
    }
  }
}

namespace {

template <int L, bool CPLX, int ORDER>
int launch(const FengineArgs& a, int nds, int ncu, const float2* tw, hipStream_t st) {
  static size_t raised = 0;
  constexpr int G = RPlan<L>::G;
  const size_t lds = freg_lds_bytes<L>(CPLX, ORDER, a.phcap);
  if (raise_lds(k_freg<L, CPLX, ORDER>, lds, &raised)) return -1;
  // four rounds of workgroups or more where there are that many FFTs, up to eight FFTs each per
  // group of threads
  const long long total = (long long)a.nffts_pad / G * nds, wgs = 4LL * ncu * (32768 / (L * G));
  const int upw = G * (int)std::max(1LL, std::min(8LL, total / wgs));
  hipLaunchKernelGGL((k_freg<L, CPLX, ORDER>), dim3((a.nffts_pad + upw - 1) / upw, nds), dim3(L / 32 * G), lds, st, a, tw, upw);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int L>
int launch_o(const FengineArgs& a, int cplx, int nds, int ncu, const float2* tw, hipStream_t st) {
  switch (a.rotorder) {
    case 0: return cplx || L <= 8192 ? -2 : launch<(L <= 8192 ? 16384 : L), false, 0>(a, nds, ncu, tw, st);
    case 1: return cplx ? launch<L, true, 1>(a, nds, ncu, tw, st) : launch<L, false, 1>(a, nds, ncu, tw, st);
    case 2: return cplx ? launch<L, true, 2>(a, nds, ncu, tw, st) : launch<L, false, 2>(a, nds, ncu, tw, st);
  }
  return -2;
}

}  // namespace

// Whether it takes FFTs of L points: phasor tables (phcap entries, sub-phasors of S) that leave room
// in LDS for one, two or three workgroups per CU (fewer would not cover each other's barriers), and S
// dividing the stride of a thread's samples.  Up to 8192 points of post-F rotation (order 0) stay
// with k_fengine, which puts two bands through one FFT there.
bool fxg_freg_takes(int L, int cplx, int nbits, int order, int S, int phcap) {
  if (nbits != (cplx ? 8 : 2) || (order == 0 && (cplx || L <= 8192))) return false;
  const size_t lds = L == 32768   ? freg_lds_bytes<32768>(cplx, order, phcap)
                     : L == 16384 ? freg_lds_bytes<16384>(cplx, order, phcap)
                     : L == 8192  ? freg_lds_bytes<8192>(cplx, order, phcap)
                     : L == 4096  ? freg_lds_bytes<4096>(cplx, order, phcap)
                                  : ~(size_t)0;
  return (L / 32) % S == 0 && (S & (S - 1)) == 0 && lds <= (L == 32768 ? 160u : L == 16384 ? 80u : 53u) * 1024u;
}

// Twiddles exp(-2 pi i k s / (Ns R)) of the second and the last pass, [s - 1][k] each: the same for
// every context, computed in FP64 once per length.
template <int L>
static const std::vector<float2>& tables() {
  static const std::vector<float2> t = [] {
    std::vector<float2> w(L), v;
    for (int j = 0; j < L; ++j) {
      const double a = -TWO_PI_D * (double)j / (double)L;
      w[j] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    for (int s = 1; s < 32; ++s)
      for (int k = 0; k < 32; ++k) v.push_back(w[k * s * (L / 1024)]);
    for (int s = 1; s < L / 1024; ++s)
      for (int j = 0; j < 1024; ++j) v.push_back(w[j * s]);
    return v;
  }();
  return t;
}
const std::vector<float2>& fxg_freg_tables(int L) {
  return L == 32768 ? tables<32768>() : L == 16384 ? tables<16384>() : L == 8192 ? tables<8192>() : tables<4096>();
}

int fxg_launch_freg(const FengineArgs& a, int L, int cplx, int nds, int ncu, const float2* tw, hipStream_t st) {
  if (fxg_launch_fftparams(a, nds, st)) return -1;
  switch (L) {
    case 4096: return launch_o<4096>(a, cplx, nds, ncu, tw, st);
    case 8192: return launch_o<8192>(a, cplx, nds, ncu, tw, st);
    case 16384: return launch_o<16384>(a, cplx, nds, ncu, tw, st);
    case 32768: return launch_o<32768>(a, cplx, nds, ncu, tw, st);
  }
  return -2;
}
