// X-engines and accumulation of the FX hot path on CDNA4.
//
// Plain FP32 path: every product accumulates
//   acc += F1[t][c] * conj(F2[t][c])
// over the FFTs of the subint in FP32, the vectorAddProduct_cf32 of Core::processdata
// (mpifxcorr/src/core.cpp:884-979, :963) for the cross products and of Mode::process for the
// autocorrelations (mode.cpp:1272, 1333-1339).  The matrix kernel takes the input x input
// matrix of the products' inputs per channel on FP32 matrix instructions; the per-product
// kernel (one thread per product and channel, FFT order) takes the products it leaves.
//
// MFMA path: per channel the visibilities of all inputs (station bands of one frequency)
// form the Hermitian matrix V = sum_t x_t x_t^H.  With x stored as interleaved (re, im)
// 16-bit pairs along time, the row of input n is A_n = (re_0, im_0, re_1, im_1, ...), so
//   Re V = A A^T            and   Im V = B A^T,  B_n = (im_0, -re_0, im_1, -re_1, ...)
// and both are 32x32x16 MFMA contractions whose A and B operands come from the same
// 16-byte load per lane.  FP32 accumulators live in registers for a whole chunk.
#include "fxg_internal.h"
#include <hip/hip_fp16.h>

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));


// Thread per (product, channel).  Parallel-hand autocorrelations keep a zero imaginary part,
// as F * conj(F) has in the reference's arithmetic.
__global__ void __launch_bounds__(256) k_xmac_f32(XPlainArgs a) {
  const DevProd p = a.prods[blockIdx.y];
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= p.nchan) return;
  const DevDs& d1 = a.ds[p.ds1];
  const DevDs& d2 = a.ds[p.ds2];
  const int C1 = d1.C, C2 = d2.C;
  const float2* s1 = a.spec32 + d1.spec_off + (long long)p.band1 * a.chunkcap * C1 + p.choff1 + c;
  const float2* s2 = a.spec32 + d2.spec_off + (long long)p.band2 * a.chunkcap * C2 + p.choff2 + c;
  const bool isauto = (p.ds1 == p.ds2) && (p.band1 == p.band2) && (p.choff1 == p.choff2);
  float2 acc = a.acc[p.acc_off + c];
  int t = 0;
  for (; t + 4 <= a.nffts; t += 4) {
    float2 x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) { x[u] = s1[(long long)(t + u) * C1]; y[u] = s2[(long long)(t + u) * C2]; }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      acc.x += x[u].x * y[u].x + x[u].y * y[u].y;
      acc.y += x[u].y * y[u].x - x[u].x * y[u].y;
    }
  }
  for (; t < a.nffts; ++t) {
    const float2 x = s1[(long long)t * C1], y = s2[(long long)t * C2];
    acc.x += x.x * y.x + x.y * y.y;
    acc.y += x.y * y.x - x.x * y.y;
  }
  if (isauto) acc.y = 0.0f;
  a.acc[p.acc_off + c] = acc;
}


// Matrix form of the plain FP32 X-engine.  Per channel and FFT the rows' spectra x give
//   S = re(x) (re(x) - im(x))^T + im(x) (re(x) + im(x))^T,
// one FP32 matrix product over k = (re, im), and V = x x^H follows from it:
//   re V = (S + S^T) / 2,  im V = (S - S^T) / 2
// (re V is symmetric and im V antisymmetric), so one FP32 matrix instruction per FFT does the
// work of a real and an imaginary one.  Inputs, products and sums stay FP32.
// A workgroup takes 16 channels (8 for R = 64) of one group, a line per row and FFT, and a range
// of the chunk's FFTs; TB FFTs at a time are staged in LDS as [FFT][row][channel] (one pad entry
// per row: a wave's reads, one row per lane, then hit distinct banks), double buffered, the next
// stage's loads in flight while the current one is multiplied.  Rows past the group stay zero.
// Runs of 64 FFTs are summed apart and then added to the total: one chain over 7800 FFTs of 10
// stations was 1.3e-6 off the 64-bit result, runs of 256 1.1e-7.  Sums of up to 256 FFTs take runs
// of 8 and those of up to 64 runs of 4 (FINE: half a stage of the 16-row tiles, in a kernel of its
// own, since in the long sums' the branch alone cost 1.4 %): there the run's own rounding is what is
// left.  With the lane-per-channel sums in four parts, runs of 16 and these the results are off by
// 9.6e-8, 1.09e-7 and 9.6e-8 for 24 FFTs of one baseline, by 1.10e-7, 9.4e-8 and 8.9e-8 for 200 of
// 4 stations dual pol and by 1.41e-7, 1.41e-7 and 1.35e-7 for 63 of 20; 8 freqs of 1024 channels of
// 10 stations and 63 FFTs take 143, now 146 us.  One matrix instruction at a time is worse again
// (the total's own rounding) and spills at 64 rows.
// R is the row count rounded up to 16, 32 or 64 (16x16x4 tiles, else 32x32x2).
template <int R>
struct XPTile {
  static constexpr int CT = R == 64 ? 8 : 16;             // channels
  static constexpr int NTH = R == 16 ? 256 : 512;
  static constexpr int NW = NTH / 64;
  static constexpr int CPW = CT / NW;                     // channels per wave: its sums and totals
                                                          // are 32 (R = 16), 64 or 128 registers
  static constexpr int TB = R == 64 ? 4 : 128 / R;        // FFTs per stage
  static constexpr int RS = CT + 1;                       // LDS entries per row
  static constexpr int STAGE = TB * R * RS;
  static constexpr int QN = TB * R * (CT / 2) / NTH;      // 16-byte loads per thread and stage
  static constexpr int NT = R == 64 ? 2 : 1;              // row tiles
};
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float float4_a8 __attribute__((ext_vector_type(4), aligned(8)));

template <int R, bool FINE>
__global__ void __launch_bounds__(XPTile<R>::NTH) k_xmac_f32_mat(XPMatArgs a) {
  using T = XPTile<R>;
  constexpr int NT = T::NT, CPW = T::CPW, TB = T::TB, RS = T::RS, QN = T::QN;
  constexpr int NREG = R == 16 ? 4 : 16;
  __shared__ float2 lds[2][T::STAGE];
  const XPItem it = a.items[blockIdx.x];
  const XPGroup g = a.groups[it.group];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = (int)((long long)it.split * a.nffts / g.nsplit);
  const int t1 = (int)((long long)(it.split + 1) * a.nffts / g.nsplit);
  const int nrun = max(1, (t1 - t0 <= 64 ? 4 : t1 - t0 <= 256 ? 8 : 64) / TB);   // stages summed before they join the total
  const int nc = g.C - it.c0;                             // channels left (the last item may be short)

  for (int i = tid; i < 2 * T::STAGE; i += T::NTH) (&lds[0][0])[i] = make_float2(0.0f, 0.0f);

  // load q of a stage, channel pair fastest, then row, then FFT
  const float2* src[QN];
  bool on[QN];
  int tq[QN], dst[QN];
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    const int q = tid + T::NTH * i;
    const int cp = 2 * (q % (T::CT / 2)), row = q / (T::CT / 2) % R;
    tq[i] = q / (T::CT / 2) / R;
    on[i] = row < g.nrows && cp < nc;
    dst[i] = (tq[i] * R + row) * RS + cp;
    src[i] = a.spec32 + a.rows[g.row0 + min(row, g.nrows - 1)] + (long long)(t0 + tq[i]) * g.stride + it.c0 + cp;
  }
  float4_a8 buf[QN];
  auto load = [&](int t) {
#pragma unroll
    for (int i = 0; i < QN; ++i) {
      buf[i] = float4_a8{0.0f, 0.0f, 0.0f, 0.0f};
      if (on[i] && t + tq[i] < t1) {
        if ((tid + T::NTH * i) % (T::CT / 2) * 2 + 1 < nc) {
          buf[i] = *reinterpret_cast<const float4_a8*>(src[i]);
        } else {                                          // the window's last channel, alone
          const float2 v = *src[i];
          buf[i].x = v.x;
          buf[i].y = v.y;
        }
      }
      src[i] += (long long)TB * g.stride;
    }
  };
  auto store = [&](float2* d) {
#pragma unroll
    for (int i = 0; i < QN; ++i)
      if (on[i]) {
        d[dst[i]] = make_float2(buf[i].x, buf[i].y);
        d[dst[i] + 1] = make_float2(buf[i].z, buf[i].w);
      }
  };

  // accumulators, [channel of the wave][row tile][column tile][register]
  typedef float accv __attribute__((ext_vector_type(NREG)));
  accv acc[CPW][NT][NT];
  const int cs = xp_floats(g.nrows);                      // floats per channel
  float* part = a.part + g.off + it.split * g.split_stride + (long long)(it.c0 + wave * CPW) * cs;
#pragma unroll
  for (int c = 0; c < CPW; ++c)
#pragma unroll
    for (int ti = 0; ti < NT; ++ti)
#pragma unroll
      for (int tj = 0; tj < NT; ++tj)
#pragma unroll
        for (int r = 0; r < NREG; ++r)
          acc[c][ti][tj][r] = 0.0f;
  accv tot[CPW][NT][NT];
#pragma unroll
  for (int c = 0; c < CPW; ++c)
#pragma unroll
    for (int ti = 0; ti < NT; ++ti)
#pragma unroll
      for (int tj = 0; tj < NT; ++tj) tot[c][ti][tj] = acc[c][ti][tj];

  // lane: row l % 32 (l % 16), k = l / 32: (re, im) of one FFT, or l / 16: (re, im) of two
  const int row = R == 16 ? lane & 15 : lane & 31;
  const bool im = R == 16 ? (lane >> 4) & 1 : lane >> 5;
  const int tk = R == 16 ? lane >> 5 : 0;
  const float sgn = im ? 1.0f : -1.0f;
  auto fold = [&] {
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
      for (int ti = 0; ti < NT; ++ti)
#pragma unroll
        for (int tj = 0; tj < NT; ++tj)
#pragma unroll
          for (int r = 0; r < NREG; ++r) {
            tot[c][ti][tj][r] += acc[c][ti][tj][r];
            acc[c][ti][tj][r] = 0.0f;
          }
  };
  auto step = [&](const float2* s) {
#pragma unroll
    for (int t = 0; t < TB; t += R == 16 ? 2 : 1) {
      if (FINE && t == TB / 2) fold();
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        float av[NT], bv[NT];
#pragma unroll
        for (int ti = 0; ti < NT; ++ti) {
          const float2 x = s[((t + tk) * R + row + 32 * ti) * RS + wave * CPW + c];
          av[ti] = im ? x.y : x.x;
          bv[ti] = fmaf(sgn, x.y, x.x);                   // re - im, re + im
        }
#pragma unroll
        for (int ti = 0; ti < NT; ++ti)
#pragma unroll
          for (int tj = 0; tj < NT; ++tj) {
            accv& v = acc[c][ti][tj];
            if constexpr (R == 16) v = __builtin_amdgcn_mfma_f32_16x16x4f32(av[ti], bv[tj], v, 0, 0, 0);
            else v = __builtin_amdgcn_mfma_f32_32x32x2f32(av[ti], bv[tj], v, 0, 0, 0);
          }
      }
    }
  };

  load(t0);
  __syncthreads();
  store(lds[0]);
  __syncthreads();
  int cur = 0, run = 0;
  for (int t = t0; t < t1; t += TB, cur ^= 1) {
    load(t + TB);                                         // past the end: zeros, not used
    step(lds[cur]);
    if (++run == nrun || t + TB >= t1) {
      run = 0;
      fold();
    }
    if (t + TB < t1) store(lds[cur ^ 1]);
    __syncthreads();
  }
  // the group's rows only, tile by tile in row order
#pragma unroll
  for (int ti = 0; ti < NT; ++ti)
#pragma unroll
    for (int tj = 0; tj < NT; ++tj) {
      const int h = xp_rows(g.nrows, ti), w = xp_rows(g.nrows, tj);
      float* pt = part + xp_tile(g.nrows, ti, tj);
#pragma unroll
      for (int r = 0; r < NREG; ++r) {
        const int i = R == 16 ? 4 * (lane >> 4) + r : 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (i >= h || row >= w) continue;
#pragma unroll
        for (int c = 0; c < CPW; ++c) {
          if (wave * CPW + c >= nc) continue;
          float* p = pt + c * cs + i * w + row;
          *p = a.first ? tot[c][ti][tj][r] : *p + tot[c][ti][tj][r];
        }
      }
    }
}

template <typename V8>
__device__ __forceinline__ floatx16 mfma32(V8 a, V8 b, floatx16 c);
template <>
__device__ __forceinline__ floatx16 mfma32<half8_t>(half8_t a, half8_t b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
template <>
__device__ __forceinline__ floatx16 mfma32<bf16x8_t>(bf16x8_t a, bf16x8_t b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// (re, im) pairs -> (im, -re) pairs: flip the sign bit of the 16-bit value moved to the
// high half.  Same bit manipulation for FP16 and BF16 (sign is bit 15).
__device__ __forceinline__ uint4 rot_negi(uint4 u) {
  uint4 r;
  r.x = ((u.x >> 16) | (u.x << 16)) ^ 0x80000000u;
  r.y = ((u.y >> 16) | (u.y << 16)) ^ 0x80000000u;
  r.z = ((u.z >> 16) | (u.z << 16)) ^ 0x80000000u;
  r.w = ((u.w >> 16) | (u.w << 16)) ^ 0x80000000u;
  return r;
}

// One workgroup = one tile of CT channels (8 or 16, the tile width of the group's spectra
// layout) of one group; each wavefront owns CPW channels (2 for one 32-row tile, 1 for two).
// The F-engine writes the 16-bit spectra channel-tile-blocked ([row][C/CT][t][CT]), so per
// k-step (8 FFTs) every input row contributes one contiguous run of 32 CT bytes.  The workgroup
// streams those runs into LDS as [channel][row][8 FFTs], double buffered, so each lane reads its
// MFMA operand (one row, 4 consecutive FFTs = 8 halves) with one 16-byte LDS load.  Rows beyond
// the group's inputs stay zero in LDS and are never fetched.
template <int NTILE, int CT_>
struct XTile {
  static constexpr int CPW = (NTILE == 1) ? 2 : 1;      // channels per wavefront
  static constexpr int CT = CT_;                         // channels per workgroup
  static constexpr int NW = CT / CPW;                    // wavefronts per workgroup
  static constexpr int NTH = 64 * NW;
  static constexpr int R = 32 * NTILE;                   // operand rows
  static constexpr int CSTR = R * 8 + 8;                 // 32-bit words per channel in LDS (padded:
                                                         // conflict-free chunk stores)
  static constexpr int QPR = 2 * CT;                     // 16-byte chunks per row per k-step
  static constexpr int QMAX = (R * QPR + NTH - 1) / NTH; // chunks per thread per k-step
  static_assert(NTH <= 1024, "workgroup size");
};

template <typename V8, int NTILE, int CT_>
__global__ void __launch_bounds__((XTile<NTILE, CT_>::NTH)) k_xmac_mfma(XMfmaArgs a) {
  using T = XTile<NTILE, CT_>;
  constexpr int NPAIR = NTILE * (NTILE + 1) / 2;
  constexpr int CPW = T::CPW, CT = T::CT, CSTR = T::CSTR, QPR = T::QPR, QMAX = T::QMAX, NTH = T::NTH;
  __shared__ uint4 lds_raw[2][(CT * CSTR) / 4];
  uint32_t* lds0 = reinterpret_cast<uint32_t*>(lds_raw[0]);
  uint32_t* lds1 = reinterpret_cast<uint32_t*>(lds_raw[1]);
  const DevXGroup g = a.groups[blockIdx.y];
  const int ct = blockIdx.x;
  const int c0 = ct * CT;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int row = lane & 31, half = lane >> 5;
  const int nq = g.nin * QPR;
  const uint32_t* gbase = a.spec16 + g.spec_off + (long long)ct * a.chunkcap * CT;

  for (int i = tid; i < 2 * (CT * CSTR) / 4; i += NTH)
    (&lds_raw[0][0])[i] = make_uint4(0u, 0u, 0u, 0u);

  floatx16 accr[CPW][NPAIR], acci[CPW][NPAIR];
  // the sums of channel c, tile pair p: the group's rows only; register r of a lane is element
  // (8 (r / 4) + 4 half + r % 4, row) of the tile
  const int cs = xh_floats(g.nin);
  float* acc0 = a.acc + g.acc_off + blockIdx.z * g.split_stride + (long long)(c0 + wave * CPW) * cs;
  auto sums = [&](auto&& f) {
    int p = 0;
#pragma unroll
    for (int ti = 0; ti < NTILE; ++ti)
#pragma unroll
      for (int tj = 0; tj <= ti; ++tj, ++p) {
        const int h = xp_rows(g.nin, ti), w = xp_rows(g.nin, tj);
        float* pt = acc0 + xh_tile(g.nin, p) + row;
        const int im = xh_len(g.nin, ti, tj);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = 8 * (r >> 2) + 4 * half + (r & 3);
          if (i >= h || row >= w) continue;
#pragma unroll
          for (int cw = 0; cw < CPW; ++cw) f(pt + cw * cs + i * w, im, cw, p, r);
        }
      }
  };
#pragma unroll
  for (int cw = 0; cw < CPW; ++cw)
#pragma unroll
    for (int p = 0; p < NPAIR; ++p)
#pragma unroll
      for (int r = 0; r < 16; ++r) accr[cw][p][r] = acci[cw][p][r] = 0.0f;
  if (!a.first)
    sums([&](const float* v, int im, int cw, int p, int r) {
      accr[cw][p][r] = v[0];
      acci[cw][p][r] = v[im];
    });

  // chunk q of a k-step: row r = q / QPR, FFT t = (q % QPR) / (CT/4), channel quad
  // h = q % (CT/4).  The loads are unconditional (a chunk past the group's inputs re-reads
  // row 0 and is not stored), so the compiler can count them exactly in its waits.
  constexpr int QPC = CT / 4;                    // channel quads per FFT
  auto gload = [&](int k, uint4* b) {
#pragma unroll
    for (int i = 0; i < QMAX; ++i) {
      const int q0 = tid + NTH * i;
      const int q = q0 < nq ? q0 : (q0 % QPR);
      const int r = q / QPR, rem = q % QPR;
      b[i] = *reinterpret_cast<const uint4*>(gbase + (long long)r * g.rowstride + (long long)(8 * k) * CT + rem * 4);
    }
  };
  auto lstore = [&](uint32_t* L, const uint4* b) {
#pragma unroll
    for (int i = 0; i < QMAX; ++i) {
      const int q = tid + NTH * i;
      if (q < nq) {
        const int r = q / QPR, rem = q % QPR;
        const int t = rem / QPC, h = rem % QPC;
        uint32_t* d = L + (4 * h) * CSTR + r * 8 + t;
        d[0] = b[i].x; d[CSTR] = b[i].y; d[2 * CSTR] = b[i].z; d[3 * CSTR] = b[i].w;
      }
    }
  };
  auto mfma_step = [&](const uint32_t* L) {
#pragma unroll
      for (int cw = 0; cw < CPW; ++cw) {
        const uint32_t* cb = L + (wave * CPW + cw) * CSTR + 4 * half;
        uint4 x[NTILE];
  #pragma unroll
        for (int ti = 0; ti < NTILE; ++ti) x[ti] = *reinterpret_cast<const uint4*>(cb + (row + 32 * ti) * 8);
        int pi = 0;
  #pragma unroll
        for (int ti = 0; ti < NTILE; ++ti) {
          const uint4 xr = rot_negi(x[ti]);
  #pragma unroll
          for (int tj = 0; tj <= ti; ++tj) {
            const V8 av = __builtin_bit_cast(V8, x[ti]);
            const V8 bv = __builtin_bit_cast(V8, x[tj]);
            const V8 arv = __builtin_bit_cast(V8, xr);
            accr[cw][pi] = mfma32<V8>(av, bv, accr[cw][pi]);
            acci[cw][pi] = mfma32<V8>(arv, bv, acci[cw][pi]);
            ++pi;
          }
        }
      }
  };

  // this workgroup's range of k-steps
  const int nka = a.nffts_pad / 8;
  const int k0 = (int)((long long)blockIdx.z * nka / g.nsplit), k1 = (int)((long long)(blockIdx.z + 1) * nka / g.nsplit);
  // one k-step of global loads in flight over a double-buffered LDS stage (two k-steps ahead
  // in registers measured slower)
  uint4 buf[QMAX];
  __syncthreads();
  if (k0 < k1) {                                  // uniform: a short chunk may leave a split empty
    gload(k0, buf);
    lstore(lds0, buf);
  }
  __syncthreads();
  for (int k = k0; k < k1; ++k) {
    uint32_t* cur = ((k - k0) & 1) ? lds1 : lds0;
    uint32_t* nxt = ((k - k0) & 1) ? lds0 : lds1;
    gload(min(k + 1, k1 - 1), buf);               // past the end: re-read, unused
    mfma_step(cur);
    if (k + 1 < k1) lstore(nxt, buf);
    __syncthreads();
  }

  sums([&](float* v, int im, int cw, int p, int r) {
    v[0] = accr[cw][p][r];
    v[im] = acci[cw][p][r];
  });
}

// The raw accumulator tiles to the products: a workgroup reads a block of tiles of a few
// channels of one group into LDS, whole lines at a time, summing the splits in order, and then
// writes one value per thread with the channel fastest, so each product gets 64- or 128-byte
// runs (read in place, the 4-byte values of one product are a channel's sums, up to 24 KB, apart).  A product whose
// channels go to the results as they are is written there, the others to their accumulators.
template <int NPL, int CH>
__device__ __forceinline__ void xr_gather(float* s, const float* p0, const float* p1, long long chf, int nch, int len,
                                          int cs, int nsplit, long long stride) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  const int q4 = len / 4;                                  // len: floats per channel and plane
#pragma unroll 2
  for (int e = threadIdx.x; e < CH * NPL * q4; e += 256) {
    const int ch = e / (NPL * q4), rem = e % (NPL * q4), pl = rem / q4, k = rem % q4;
    if (ch >= nch) break;                                  // channels ascend with e
    const v4* p = reinterpret_cast<const v4*>((NPL == 2 && pl ? p1 : p0) + ch * chf) + k;
    v4 v = *p;
    const long long st = stride / 4;
    int q = 1;
    for (; q + 4 <= nsplit; q += 4) {                      // four splits in flight
      const v4 a = p[q * st], b = p[(q + 1) * st], c = p[(q + 2) * st], d = p[(q + 3) * st];
      v += a; v += b; v += c; v += d;
    }
    for (; q < nsplit; ++q) v += p[q * st];
    *reinterpret_cast<v4*>(s + ch * cs + pl * len + 4 * k) = v;
  }
}

__device__ __forceinline__ void xr_put(const XReduceArgs& a, long long p, int c, float2 v) {
  if (p >= 0) a.acc[p + c] = v;
  else if (p < -1) a.res[-2 - p + c] = v;
}

// 16-bit X-engine: 16 channels, one pair of row tiles, eight rows (up to 256 floats of each part).
constexpr int XRH_CH = 16, XRH_CS = 512 + 4;
__global__ void __launch_bounds__(256) k_xreduce_h(XReduceArgs a) {
  __shared__ float s[XRH_CH * XRH_CS];
  const XRGroup g = a.groups[blockIdx.y];
  const int c0 = blockIdx.x * XRH_CH, ntp = g.ntile * (g.ntile + 1) / 2;
  int ti = 0, tj = blockIdx.z >> 2;
  const int i0 = 8 * (blockIdx.z & 3), tp = tj;
  while (tj > ti) { ++ti; tj -= ti; }
  if (c0 >= g.C || tp >= ntp || ti * 32 + i0 >= g.n) return;
  const int nch = min(XRH_CH, g.C - c0);
  const long long chf = xh_floats(g.n);
  const int w = xp_rows(g.n, tj), len = (min(8, xp_rows(g.n, ti) - i0) * w + 3) & ~3;
  const float* p = a.part + g.off + c0 * chf + xh_tile(g.n, tp) + i0 * w;
  // the places and the rows' scales are on their way while the parts are added: a small call's
  // reduction is a chain of such loads (5.5 us with them in the loop below)
  __shared__ float rs[8 + 32];
  const long long* pairs = a.pairs + g.pair0;
  constexpr int NE = 256 / (256 / XRH_CH);
  long long pp[NE], pq[NE];
#pragma unroll
  for (int k = 0; k < NE; ++k) {
    const int e = threadIdx.x / XRH_CH + k * (256 / XRH_CH), ri = ti * 32 + i0 + (e >> 5), rj = tj * 32 + (e & 31);
    const bool in = ri < g.n && rj < g.n;
    pp[k] = in ? pairs[ri * g.n + rj] : -1;
    pq[k] = in && ti != tj ? pairs[rj * g.n + ri] : -1;
  }
  if (threadIdx.x < 40) {
    const int r = threadIdx.x < 8 ? ti * 32 + i0 + (int)threadIdx.x : tj * 32 + (int)threadIdx.x - 8;
    rs[threadIdx.x] = r < g.n ? a.xscale[g.scale_off + r] : 1.0f;
  }
  xr_gather<2, XRH_CH>(s, p, p + xh_len(g.n, ti, tj), chf, nch, len, XRH_CS, g.nsplit, g.split_stride);
  __syncthreads();
  const int ch = threadIdx.x % XRH_CH;
  if (ch >= nch) return;
  const float* sc = s + ch * XRH_CS;
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    if (pp[n] == -1 && pq[n] == -1) continue;
    const int e = threadIdx.x / XRH_CH + n * (256 / XRH_CH), i = e >> 5, j = e & 31;
    const float inv = 1.0f / (rs[i] * rs[8 + j]);
    const int k = i * w + j;
    float2 v = make_float2(sc[k] * inv, sc[len + k] * inv);
    if (ti == tj && i0 + i == j) v.y = 0.0f;               // x conj(x) is real
    xr_put(a, pp[n], c0 + ch, v);
    xr_put(a, pq[n], c0 + ch, make_float2(v.x, -v.y));
  }
}

// FP32 X-engine: 8 channels, one pair of row tiles: S(ti, tj) and S(tj, ti).
constexpr int XRS_CH = 8, XRS_CS = 2048 + 8;
__global__ void __launch_bounds__(256) k_xreduce_s(XReduceArgs a) {
  __shared__ float s[XRS_CH * XRS_CS];
  const XRGroup g = a.groups[blockIdx.y];
  const int c0 = blockIdx.x * XRS_CH;
  int ti = 0, tj = blockIdx.z;
  while (tj > ti) { ++ti; tj -= ti; }
  if (c0 >= g.C || ti >= g.ntile) return;
  const int h = xp_rows(g.n, ti), w = xp_rows(g.n, tj), len = (h * w + 3) & ~3;
  const int nch = min(XRS_CH, g.C - c0);
  const long long chf = xp_floats(g.n);
  const float* p = a.part + g.off + c0 * chf;
  if (ti == tj)
    xr_gather<1, XRS_CH>(s, p + xp_tile(g.n, ti, tj), nullptr, chf, nch, len, XRS_CS, g.nsplit, g.split_stride);
  else
    xr_gather<2, XRS_CH>(s, p + xp_tile(g.n, ti, tj), p + xp_tile(g.n, tj, ti), chf, nch, len, XRS_CS, g.nsplit, g.split_stride);
  __syncthreads();
  const int ch = threadIdx.x % XRS_CH;
  if (ch >= nch) return;
  const long long* pairs = a.pairs + g.pair0;
  const float* sc = s + ch * XRS_CS;
  const float* st = sc + (ti == tj ? 0 : len);
  const int wl = w <= 16 ? 4 : 5;
#pragma unroll 4
  for (int e = threadIdx.x / XRS_CH; e < h << wl; e += 256 / XRS_CH) {
    const int i = e >> wl, j = e & ((1 << wl) - 1), ri = ti * 32 + i, rj = tj * 32 + j;
    if (j >= w) continue;
    const long long p = pairs[ri * g.n + rj], q = ti == tj ? -1 : pairs[rj * g.n + ri];
    if (p == -1 && q == -1) continue;
    const float x = sc[i * w + j], y = st[j * h + i];
    const float2 v = make_float2(0.5f * (x + y), 0.5f * (x - y));   // i = j: imaginary part 0
    xr_put(a, p, c0 + ch, v);
    xr_put(a, q, c0 + ch, make_float2(v.x, -v.y));
  }
}

// ---- accumulation into the slot results (core.cpp:1819-1853, 1258-1376) ----------------

// The uv-shift rotation of channel ch of a freq to a phase centre at applied delay dd (us),
// in the reference's steps (core.cpp:1699-1766, 1789-1808): FP64 turns of the sub phasor
// (channel within its rotate stride, plus the band edge) and of the step phasor (the stride),
// wrapped, as FP32 arguments of FP32 sin/cos; the value times the sub phasor, then the step.
constexpr double UV_TWO_PI = 6.283185307179586476925286766559;   // architecture.h.in:430

__device__ __forceinline__ float2 uv_rotate(float2 v, double dd, const UvFreq& q, int ch) {
  const int c = ch % q.rs, j = ch / q.rs;
  double edge = dd * q.lofreq;
  edge -= floor(edge);
  const double subf = q.lsb ? -(double)(q.rs - (c + 1)) * q.chbw : (double)c * q.chbw;
  const double stepf = q.lsb ? -(double)(q.nsteps - (j + 1)) * q.stepbw : (double)j * q.stepbw;
  const double t1 = dd * subf + edge;
  const double t2 = dd * stepf;
  const float a1 = (float)((t1 - floor(t1)) * UV_TWO_PI);
  const float a2 = (float)((t2 - floor(t2)) * UV_TWO_PI);
  float s1, c1, s2, c2;
  sincosf(a1, &s1, &c1);
  sincosf(a2, &s2, &c2);
  const float2 r = make_float2(c1 * v.x - s1 * v.y, c1 * v.y + s1 * v.x);
  return make_float2(r.x * c2 - r.y * s2, r.x * s2 + r.y * c2);
}

// One workgroup row per product.  SUMS: without the reduction's pass over LDS and memory, straight
// from the 16-bit X-engine's sums (a row of them per channel): a launch less, which is
// what counts in short uv-shift intervals of small arrays (see sums_read_directly).
template <bool SUMS>
__global__ void k_fin(const FinProd* e, const float2* acc, const float* part, float2* res, UvArgs uv) {
  const FinProd f = e[blockIdx.y];
  auto value = [&](int ch) {
    if (!SUMS) return acc[f.src + ch];
    const float* p = part + f.tile + (long long)ch * f.tstep;
    return make_float2(p[0] * f.sre, p[f.im] * f.sim);
  };
  const int co = blockIdx.x * blockDim.x + threadIdx.x;
  if (co >= f.nout) return;
  if (uv.P > 1 && f.bl >= 0) {                    // rotated into every phase centre's block
    const UvFreq q = uv.fq[f.fq];
    for (int p = 0; p < uv.P; ++p) {
      const double dd = uv.dd[f.bl * uv.P + p];
      const bool turn = fabs(dd) > 1.0e-20;
      float2 s = make_float2(0.f, 0.f);
      for (int k = 0; k < f.avg; ++k) {
        const int ch = co * f.avg + k;
        float2 v = value(ch);
        if (turn) v = uv_rotate(v, dd, q, ch);
        s.x += v.x; s.y += v.y;
      }
      if (f.avg > 1) { s.x /= (float)f.avg; s.y /= (float)f.avg; }
      float2* o = res + f.dst + (long long)p * f.pcstride + co;
      o->x += s.x; o->y += s.y;
    }
    return;
  }
  float2 s = make_float2(0.f, 0.f);
  for (int k = 0; k < f.avg; ++k) {
    const float2 v = value(co * f.avg + k);
    s.x += v.x; s.y += v.y;
  }
  if (f.avg > 1) { s.x /= (float)f.avg; s.y /= (float)f.avg; }
  float2 o = res[f.dst + co];
  o.x += s.x; o.y += s.y;
  res[f.dst + co] = o;
}


// Baseline weights (core.cpp:1005-1052, 1066-1112) and autocorrelation weights
// (core.cpp:1306-1370): sequential FP32 sums over the FFTs of the subint.

// One workgroup per entry: a strided partial sum per thread, then a tree over the block.  The time
// is the latency of the loads (125000 weights took 186 us with 256 threads and one load in flight
// each), so a thread has eight in flight, and long subints take 1024 threads.
template <int NTH>
__global__ void __launch_bounds__(NTH) k_fin_weights(const FinWeight* e, const float* w, int B, float* resf) {
  __shared__ float part[NTH];
  const FinWeight f = e[blockIdx.x];
  const float* w1 = w + (long long)f.ds1 * B;
  const float* w2 = f.ds2 >= 0 ? w + (long long)f.ds2 * B : nullptr;
  float s = 0.0f;
  for (int i = threadIdx.x; i < B; i += 8 * NTH) {
    float a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int at = i + k * NTH;
      a[k] = at < B ? w1[at] : 0.0f;
      b[k] = w2 && at < B ? w2[at] : 1.0f;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) s += a[k] * b[k];
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int h = NTH / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) resf[f.dstf] += part[0];
}

__global__ void k_zero(float* p, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = 0.0f;
}

// Visibility::addData (visibility.cpp:192-205): one subint's results into an integration.
__global__ void k_add(float* dst, const float* src, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    dst[i] += src[i];
}

// The shift decorrelation sums of a subint into their result words (core.cpp:1089-1104).
__global__ void k_add_at(const int* idx, const float* val, int n, float* resf) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) resf[idx[i]] += val[i];
}

__global__ void k_fill(float* p, long long n, float v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---- host-side launchers -------------------------------------------------------------
int fxg_launch_xplain_mat(const XPMatArgs& a, int R, int nsplit, int nitems, hipStream_t st) {
  const dim3 grid(nitems);
  const bool fine = (a.nffts + nsplit - 1) / nsplit <= 64;
  if (R == 16 && fine) hipLaunchKernelGGL((k_xmac_f32_mat<16, true>), grid, dim3(XPTile<16>::NTH), 0, st, a);
  else if (R == 16) hipLaunchKernelGGL((k_xmac_f32_mat<16, false>), grid, dim3(XPTile<16>::NTH), 0, st, a);
  else if (R == 32) hipLaunchKernelGGL((k_xmac_f32_mat<32, false>), grid, dim3(XPTile<32>::NTH), 0, st, a);
  else hipLaunchKernelGGL((k_xmac_f32_mat<64, false>), grid, dim3(XPTile<64>::NTH), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_xreduce(const XReduceArgs& a, int mfma, int ngroups, int maxC, int maxtp, hipStream_t st) {
  if (ngroups == 0) return 0;
  if (mfma)
    hipLaunchKernelGGL(k_xreduce_h, dim3((maxC + XRH_CH - 1) / XRH_CH, ngroups, 4 * maxtp), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(k_xreduce_s, dim3((maxC + XRS_CH - 1) / XRS_CH, ngroups, maxtp), dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_xplain(const XPlainArgs& a, int nprod, int maxchan, hipStream_t st) {
  dim3 grid((maxchan + 255) / 256, nprod);
  hipLaunchKernelGGL(k_xmac_f32, grid, dim3(256), 0, st, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename V8, int NTILE, int CT>
static void launch_x(const XMfmaArgs& b, int C, int ngroups, int nsplit, hipStream_t st) {
  hipLaunchKernelGGL((k_xmac_mfma<V8, NTILE, CT>), dim3(C / CT, ngroups, nsplit), dim3(XTile<NTILE, CT>::NTH), 0, st, b);
}

// groups [group0, group0 + ngroup_launch) share the tile count, channel count, tile width and
// splits of g
int fxg_launch_xmfma(const XMfmaArgs& a, int ngroup_launch, int group0, const DevXGroup& g, hipStream_t st) {
  XMfmaArgs b = a;
  const int ntile = g.ntile, C = g.C, twlog = g.twlog, ns = g.nsplit;
  b.groups = a.groups + group0;
  const int ct = 1 << twlog;
  if (C % ct || (ct != 8 && ct != 16) || (ntile != 1 && ntile != 2) || (ntile == 2 && ct != 8)) return -2;
  const int form = (a.mode == 1 ? 0 : 4) + (ntile == 1 ? 0 : 2) + (ct == 8 ? 0 : 1);
  switch (form) {
    case 0: launch_x<half8_t, 1, 8>(b, C, ngroup_launch, ns, st); break;
    case 1: launch_x<half8_t, 1, 16>(b, C, ngroup_launch, ns, st); break;
    case 2: launch_x<half8_t, 2, 8>(b, C, ngroup_launch, ns, st); break;
    case 4: launch_x<bf16x8_t, 1, 8>(b, C, ngroup_launch, ns, st); break;
    case 5: launch_x<bf16x8_t, 1, 16>(b, C, ngroup_launch, ns, st); break;
    case 6: launch_x<bf16x8_t, 2, 8>(b, C, ngroup_launch, ns, st); break;
    default: return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_fin(const FinProd* e, int n, int maxout, const float2* acc, const float* part, float2* res, const UvArgs& uv,
                   hipStream_t st) {
  if (n == 0) return 0;
  const dim3 grid((maxout + 255) / 256, n);
  if (part) hipLaunchKernelGGL(k_fin<true>, grid, dim3(256), 0, st, e, acc, part, res, uv);
  else hipLaunchKernelGGL(k_fin<false>, grid, dim3(256), 0, st, e, acc, part, res, uv);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_add_at(const int* idx, const float* val, int n, float* resf, hipStream_t st) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_add_at, dim3((n + 255) / 256), dim3(256), 0, st, idx, val, n, resf);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_fin_weights(const FinWeight* e, int n, const float* w, int B, float* resf, hipStream_t st) {
  if (n == 0) return 0;
  if (B > 8192) hipLaunchKernelGGL(k_fin_weights<1024>, dim3(n), dim3(1024), 0, st, e, w, B, resf);
  else hipLaunchKernelGGL(k_fin_weights<256>, dim3(n), dim3(256), 0, st, e, w, B, resf);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_zero(void* p, long long bytes, hipStream_t st) {
  if (bytes <= 0) return 0;
  const long long n = bytes / 4;
  long long blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, st, (float*)p, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_add(float* dst, const float* src, long long n, hipStream_t st) {
  if (n <= 0) return 0;
  long long blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_add, dim3((unsigned)blocks), dim3(256), 0, st, dst, src, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int fxg_launch_fill(float* p, long long n, float v, hipStream_t st) {
  if (n <= 0) return 0;
  long long blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, st, p, n, v);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}
