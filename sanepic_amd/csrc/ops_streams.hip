// ops_streams.hip -- the filter passes of detectors that share lines of sight.
//
// The passes over SkyStreams (kernels.h): 16 detectors behind one line of
// sight are 3 streams instead of 16, and pixels, angles and run records are
// read and written once for all of them.  Measured at 16 detectors x 2^24
// samples, NSIDE 512, segments of 2^20, against one stream per detector:
// gather + column pass 1264 -> 221 us, row pass 1140 -> 286 us, inverse pass
// 1585 -> 223 us, P^T 474 -> 101 us in FP64; FP32 at half the samples 450 ->
// 69, 284 -> 75, 436 -> 64 and 169 -> 51 us.

#include "ops_dev.h"

namespace {

// Block lb of a column pass: the three streams of a set take consecutive
// blocks, so they share the pixel, angle and map lines in their XCD's L2.
template <typename T>
__device__ __forceinline__ void stream_block(const OpArgs<T> &a, int64_t lb, int64_t ncb, int &v, int64_t &j,
                                             int64_t &cb) {
  const int64_t per = a.g.ppd * ncb, mixed = 3 * (int64_t)a.nset * per;
  int64_t r;
  if (lb < mixed) {
    const int64_t q = lb / 3;
    v = 3 * (int)(q / per) + (int)(lb - 3 * q);
    r = q % per;
  } else {
    v = 3 * a.nset + (int)((lb - mixed) / per);
    r = (lb - mixed) % per;
  }
  j = r / ncb;
  cb = r % ncb;
}

// (cos, sin) of a stored angle plus the stream's constant
__device__ __forceinline__ float2 stream_cs(uint64_t turn, uint32_t u) { return cs_of_turn(u, (uint32_t)(turn >> 32)); }
__device__ __forceinline__ double2 stream_cs(uint64_t turn, uint64_t u) {
  return cs_of_turn64_tab(u, s_turn_tab, turn);
}
__device__ __forceinline__ uint32_t stream_turn(const OpArgs<float> &a, int64_t g) { return a.ang[g]; }
__device__ __forceinline__ uint64_t stream_turn(const OpArgs<double> &a, int64_t g) { return a.ang64[g]; }

template <typename T, int PARTS>
__device__ __forceinline__ T stream_value(const OpArgs<T> &a, uint64_t turn, int64_t g) {
  const T *m = a.map + 3 * (int64_t)a.pix[g];
  if constexpr (PARTS == 1) {
    return m[0];
  } else {
    const VT<T> c = stream_cs(turn, stream_turn(a, g));
    const T p = fma(m[1], c.x, m[2] * c.y);
    return PARTS == 2 ? p : m[0] + p;
  }
}

template <typename T, int PARTS, int TS>
__device__ __forceinline__ void stream_load(const OpArgs<T> &a, uint64_t turn, int64_t ga, int64_t gb, bool hb,
                                            int64_t step, VT<T> (&v)[16]) {
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const T xa = stream_value<T, PARTS>(a, turn, ga + step * i);
    const T xb = stream_value<T, PARTS>(a, turn, gb + step * i);
    v[i] = mk<VT<T>>(xa, hb ? xb : (T)0);
  }
}

// Gather of a stream + column FFT (col_fwd_body over streams).  Bound by the
// latency of the pixel -> map loads like k_col_fwd; the I stream reads no
// angle, the others no I.
template <typename T, int LOG2N2>
__global__ __launch_bounds__(256) void k_col_fwd_st(OpArgs<T> a) {
  using V = VT<T>;
  constexpr int N2 = 1 << LOG2N2, TS = N2 / 16, B = 256 / TS;
  static_assert(LdsSize<LOG2N2, B>::value <= kLds, "LDS");
  __shared__ LdsE<V> lds[kLds];
  if constexpr (sizeof(T) == 8) {
    fill_turn_tab();
    __syncthreads();
  }
  const int tid = threadIdx.x, b = tid % B, t = tid / B;
  const int64_t N1 = a.g.N1, N = a.g.N;
  int vi;
  int64_t j, cb;
  stream_block(a, logical_block(a.xcd), N1 / B, vi, j, cb);
  const SkyStream st = a.vs[vi];
  const int64_t n1 = cb * B + b;
  const bool hb = 2 * j + 1 < a.g.nseg;  // the last pair of an odd segment count reads segment a twice
  const int64_t ga = ((int64_t)st.det * a.g.nseg + 2 * j) * N + n1 + N1 * (int64_t)t, gb = hb ? ga + N : ga;
  const int64_t step = N1 * (int64_t)TS;
  V v[16];
  if (st.parts == 1) stream_load<T, 1, TS>(a, st.turn, ga, gb, hb, step, v);
  else if (st.parts == 2) stream_load<T, 2, TS>(a, st.turn, ga, gb, hb, step, v);
  else stream_load<T, 3, TS>(a, st.turn, ga, gb, hb, step, v);
  fft_reg<V, -1, LOG2N2, B>(v, t, lds + b, a.tw4096);
  V *out = a.buf + ((int64_t)vi * a.g.ppd + j) * N;
  TwRun tr = tw_run<-1>(a.twlo64, a.twhi64, n1 * t, n1 * TS);
#pragma unroll
  for (int s = 0; s < 16; s++) out[(int64_t)(t + TS * s) * N1 + n1] = cmul(v[s], tw_next<V>(tr));
}

// Threads of a stream in the row pass: 16 values each of a row, one wave at
// least.  A CU's vector and LDS pipes serve the three streams of a block in
// turn, so a block holds no more rows than it must: at 4 detectors x 1 segment
// of 2^13 samples eight rows of 512 in 3 x 256 threads took 39 us on two CUs,
// two rows in 3 x 64 threads take 10.7 us on eight (a row pass of the four
// detectors 15 us).
template <int LOG2N1>
constexpr int row_group() {
  return LOG2N1 <= 10 ? 64 : 1 << (LOG2N1 - 4);
}

// What thread group k of row block lb works on: first the sets' blocks, whose
// groups hold the same rows of a set's three streams, then the detectors on
// their own (OWN), three rows' blocks of them in turn (live: false past the last).
// Blocks take the same rows of all of a stream's pairs back to back, so the
// rows of H or W come from L2 for all but the first.
struct RowAt {
  int64_t row;   // of the stream's buffer: stream, pair and N1-point row
  int64_t k2;
  int64_t j;     // pair
  int64_t wrow;  // first entry of the weights' row (H_00 of a set)
  int32_t set;   // set, or -1 and
  int32_t det;   // the detector
  bool live;
};
template <bool OWN, typename T>
__device__ __forceinline__ RowAt row_at(const OpArgs<T> &a, int64_t lb, int k, int b, int B) {
  const int64_t N1 = a.g.N1, N = a.g.N, ppd = a.g.ppd, per = ppd * (a.g.N2 / B), nmix = a.nset * per;
  RowAt w;
  const bool mixed = !OWN || lb < nmix;
  const int64_t nown = (a.nvs - 3 * (int64_t)a.nset) * per;
  int64_t o = mixed ? lb : 3 * (lb - nmix) + k;
  w.live = mixed || o < nown;
  if (!w.live) o = nown - 1;  // a group without rows of its own still joins the barriers
  const int64_t u = o / per, r = o % per;
  const int64_t v = mixed ? 3 * u + k : 3 * (int64_t)a.nset + u;
  w.j = r % ppd;
  w.k2 = r / ppd * B + b;
  w.row = (v * ppd + w.j) * N + w.k2 * N1;
  w.set = mixed ? (int32_t)u : -1;
  w.det = mixed ? 0 : a.vs[v].det;
  w.wrow = (mixed ? 6 * u : (int64_t)w.det) * N + w.k2 * N1;
  return w;
}

// Row pass of the sets: after the forward FFTs the spectra X_k of a set pass through the
// LDS (in halves of 8 values a thread in FP64, whose 3 x 34 KB hold no more at
// 4096) and thread group k forms U_k = sum_j H_kj X_j in place of the product
// with W.  Three streams in one block, since a pass of its own for the mixing
// would read and write them once more (16 of then 32 bytes a sample and
// stream).  OWN: the detectors on their own in the same launch (row_merged).
template <typename T, int LOG2N1, bool OWN>
__global__ __launch_bounds__(3 * row_group<LOG2N1>()) void k_row_mix(OpArgs<T> a) {
  using V = VT<T>;
  constexpr int G = row_group<LOG2N1>(), N1 = 1 << LOG2N1, TS = N1 / 16, B = G / TS;
  constexpr int HB = sizeof(T) == 8 ? 8 : 16;  // values exchanged at a time
  constexpr int R = LdsSize<LOG2N1, B>::value;  // a stream's region
  static_assert(HB * G * sizeof(V) <= R * sizeof(LdsE<V>), "exchange");
  __shared__ LdsE<V> lds[3 * R];
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / G), tid = threadIdx.x % G, b = tid % B, t = tid / B;
  const RowAt at = row_at<OWN>(a, logical_block(a.xcd), k, b, B);
  V *row = OWN ? a.buf + at.row : a.buf;  // written out: one form or the other spills (10 registers at N1 = 4096)
  const int64_t base = OWN ? 0 : at.row;
  V v[16];
#pragma unroll
  for (int i = 0; i < 16; i++) v[i] = row[base + t + TS * i];
  LdsE<V> *own = lds + k * R;
  fft_reg<V, -1, LOG2N1, B>(v, t, own + b, a.tw4096);
  if (OWN && at.set < 0) {
    const T *w = a.wt + at.wrow;
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const T ws = w[t + TS * s];
      v[s] = mk<V>(v[s].x * ws, v[s].y * ws);
    }
  } else {
    // H_kk, H_kp, H_kq: entry (i, j), i <= j, is the (3 i - i (i - 1) / 2 + j - i)-th
    const int p = k == 2 ? 0 : k + 1, q = k == 0 ? 2 : k - 1;  // the other two streams
    auto hrow = [&](int x, int y) {
      const int i = x < y ? x : y, l = x < y ? y : x;
      const int64_t e = 3 * i - i * (i - 1) / 2 + l - i;
      return OWN ? a.mix + at.wrow + e * a.g.N : a.mix + ((int64_t)at.set * 6 + e) * a.g.N + at.k2 * N1;
    };
    const T *hk = hrow(k, k), *hp = hrow(k, p), *hq = hrow(k, q);
    V *ek = reinterpret_cast<V *>(own);
    const V *ep = reinterpret_cast<const V *>(lds + p * R), *eq = reinterpret_cast<const V *>(lds + q * R);
#pragma unroll
    for (int h = 0; h < 16 / HB; h++) {
      __syncthreads();  // the FFT's (or the last half's) LDS reads are done
#pragma unroll
      for (int s = 0; s < HB; s++) ek[s * G + tid] = v[h * HB + s];
      __syncthreads();
#pragma unroll
      for (int s = 0; s < HB; s++) {
        const int k1 = t + TS * (h * HB + s);
        const V x = v[h * HB + s], xp = ep[s * G + tid], xq = eq[s * G + tid];
        const T wk = hk[k1], wp = hp[k1], wq = hq[k1];
        v[h * HB + s] = mk<V>(fma(wq, xq.x, fma(wp, xp.x, wk * x.x)), fma(wq, xq.y, fma(wp, xp.y, wk * x.y)));
      }
    }
  }
  fft_reg<V, +1, LOG2N1, B>(v, t, own + b, a.tw4096);
  if (OWN && !at.live) return;
  TwRun tr = tw_run<+1>(a.twlo64, a.twhi64, (int64_t)t * at.k2, (int64_t)TS * at.k2);
#pragma unroll
  for (int s = 0; s < 16; s++) row[base + t + TS * s] = cmul(v[s], tw_next<V>(tr));
}

// chi2 against each detector's own data spectrum: the forward half of
// k_row_mix (rows read, not written), then the residuals
// D_d - (X_0 + c_d X_1 + s_d X_2) of a set's detectors k, k + 3, ... in thread
// group k, D_d - X of a detector on its own.  A launch of its own before
// k_row_mix: with both in one kernel the spectra, the data and the mixed
// values together spilled 98-225 registers a lane (1533 us; now 515 + 286 us at
// 16 detectors x 2^24 samples).
template <int LOG2N1, bool OWN>
__global__ __launch_bounds__(3 * row_group<LOG2N1>()) void k_row_chi(OpArgs<double> a) {
  using V = double2;
  constexpr int G = row_group<LOG2N1>(), N1 = 1 << LOG2N1, TS = N1 / 16, B = G / TS, HB = 8;
  constexpr int R = LdsSize<LOG2N1, B>::value, NW = 3 * G / 64;
  static_assert(HB * G * sizeof(V) <= R * sizeof(double), "LDS");
  __shared__ double lds[3 * R];
  __shared__ double red[NW];
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / G), tid = threadIdx.x % G, b = tid % B, t = tid / B;
  const int64_t N = a.g.N, ppd = a.g.ppd, lb = logical_block(a.xcd);
  const RowAt at = row_at<OWN>(a, lb, k, b, B);
  const V *row = a.buf + at.row;
  V v[16];
#pragma unroll
  for (int i = 0; i < 16; i++) v[i] = row[t + TS * i];
  fft_reg<V, -1, LOG2N1, B>(v, t, lds + k * R + b, a.tw4096);
  const bool dc = at.k2 == 0;  // bins 0 and N/2 are counted twice by the reference's per-segment sum
  double chi = 0.0;
  if (OWN && at.set < 0) {
    const V *D = a.dspec + ((int64_t)at.det * ppd + at.j) * N + at.k2 * N1;
    const double *w = a.wt + at.wrow;
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const int k1 = t + TS * s;
      const V d = D[k1];
      const double rx = d.x - v[s].x, ry = d.y - v[s].y;
      double c = w[k1] * (rx * rx + ry * ry);
      if (dc && (k1 == 0 || k1 == N1 / 2)) c += c;
      chi += c;
    }
    if (!at.live) chi = 0.0;
  } else {
    V *own = reinterpret_cast<V *>(lds + k * R);
    const V *e0 = reinterpret_cast<const V *>(lds), *e1 = reinterpret_cast<const V *>(lds + R),
            *e2 = reinterpret_cast<const V *>(lds + 2 * R);
    const int d0 = a.sbeg[at.set] + k, d1 = a.sbeg[at.set + 1];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      __syncthreads();
#pragma unroll
      for (int s = 0; s < HB; s++) own[s * G + tid] = v[h * HB + s];
      __syncthreads();
#pragma unroll
      for (int g = 0; g < HB; g += 4) {  // four bins: their spectra stay in registers over the detectors
#pragma unroll 1
        for (int d = d0; d < d1; d += 3) {
          const SkyDet sd = a.sdet[d];
          const int64_t o = at.k2 * N1 + t + TS * (h * HB + g);
          const V *D = a.dspec + ((int64_t)sd.det * ppd + at.j) * N + o;
          const double *w = a.wt + (int64_t)sd.det * N + o;
          V dv[4];
          double wv[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            dv[s] = D[TS * s];
            wv[s] = w[TS * s];
          }
#pragma unroll
          for (int s = 0; s < 4; s++) {
            const int e = (g + s) * G + tid, k1 = t + TS * (h * HB + g + s);
            const double rx = dv[s].x - (e0[e].x + (sd.c * e1[e].x + sd.s * e2[e].x));
            const double ry = dv[s].y - (e0[e].y + (sd.c * e1[e].y + sd.s * e2[e].y));
            double c = wv[s] * (rx * rx + ry * ry);
            if (dc && (k1 == 0 || k1 == N1 / 2)) c += c;
            chi += c;
          }
        }
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) chi += __shfl_xor(chi, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = chi;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int i = 0; i < NW; i++) tot += red[i];
    a.chi2part[lb] = tot;
  }
}

// Row pass of the detectors on their own (the streams after the sets').
template <typename T, int LOG2N1>
__global__ __launch_bounds__(256) void k_row_own(OpArgs<T> a) {
  __shared__ LdsE<VT<T>> lds[kLds];
  __shared__ double red[4];
  row_body<T, LOG2N1, true>(a, logical_block(a.xcd), lds, red, a.mode);
}

// One step of the segmented scan for the sums [F, F + NV) of x (seg_step's
// rule on a shared line of sight's record, whose streams hold one or two sums).
template <int OFF, int NV, typename T>
__device__ __forceinline__ void seg_step_n(T (&x)[NV], int i, uint32_t m) {
  if constexpr (sizeof(T) == 8) {
    const T w = (((m << OFF) >> i) & ((1u << OFF) - 1u)) == 0u ? 1.0 : 0.0;
#pragma unroll
    for (int n = 0; n < NV; n++) x[n] = fma(row_shr<OFF>(x[n]), w, x[n]);
  } else {
    const bool pass = ((m >> i) & ((1u << OFF) - 1u)) == 0u;
#pragma unroll
    for (int n = 0; n < NV; n++) x[n] += row_shr<OFF>(pass ? x[n] : (T)0);
  }
}

// The run sums of one sample's z (run_record), PARTS of (z, z cos, z sin), at
// the stream's slot of the run's five-sum record.
template <typename T, int PARTS, typename A>
__device__ __forceinline__ void stream_record(const OpArgs<T> &a, const SkyStream &st, uint64_t meta, int i, T zv,
                                              A ang) {
  constexpr int NV = PARTS == 1 ? 1 : PARTS == 2 ? 2 : 3;
  const uint32_t m = (uint32_t)meta & 0xFFFFu;
  T x[NV];
  if constexpr (PARTS == 1) {
    x[0] = zv;
  } else {
    const VT<T> c = stream_cs(st.turn, ang);
    if constexpr (PARTS == 3) x[0] = zv;
    x[NV - 2] = zv * c.x;
    x[NV - 1] = zv * c.y;
  }
  seg_step_n<1>(x, i, m);
  seg_step_n<2>(x, i, m);
  seg_step_n<4>(x, i, m);
  seg_step_n<8>(x, i, m);
  if ((m >> i) & 1u) {
    T *r = a.rec + 5 * (int64_t)((uint32_t)(meta >> 16) + (uint32_t)__popc(m & ((1u << i) - 1u))) + st.slot;
#pragma unroll
    for (int n = 0; n < NV; n++) r[n] = x[n];
  }
}

// Inverse column pass of a stream writing its sums of the run records
// (col_inv_rec_body over streams: outputs parked in the LDS, loads in batches
// of SB rows, the first before the FFT).
template <typename T, int LOG2N2>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_col_inv_st(OpArgs<T> a) {
  using V = VT<T>;
  using A = decltype(stream_turn(a, 0));
  constexpr int N2 = 1 << LOG2N2, TS = N2 / 16, B = 256 / TS, SB = 8, NB = 16 / SB;
  static_assert(B >= 16, "a 16-lane row holds a piece");
  static_assert(LdsSize<LOG2N2, B>::value <= kLds && 4096 * sizeof(T) <= kLds * sizeof(LdsE<V>), "LDS");
  __shared__ LdsE<V> lds[kLds];
  if constexpr (sizeof(T) == 8) fill_turn_tab();  // complete at the barrier after the FFT
  const int tid = threadIdx.x, b = tid % B, t = tid / B, i = tid & 15;
  const int64_t N1 = a.g.N1, N = a.g.N;
  int vi;
  int64_t j, cb;
  stream_block(a, logical_block(a.xcd), N1 / B, vi, j, cb);
  const SkyStream st = a.vs[vi];
  const int64_t n1 = cb * B + b, step = N1 * (int64_t)TS;
  const int64_t at = 2 * j * N + n1 + N1 * (int64_t)t;        // in the line of sight's samples
  const int64_t g0 = (int64_t)st.det * a.g.nseg * N + at, m0 = (int64_t)st.set * a.g.nseg * N + at;
  const int nq = (2 * j + 1 < a.g.nseg ? 2 : 1) * NB;         // batches: segment a's rows, then b's
  A an[SB], bn[SB];
  uint64_t am[SB], bm[SB];
  auto fetch = [&](int q, A *pa, uint64_t *pm) {
    const int64_t o = (q >= NB ? N : 0) + step * (int64_t)((q % NB) * SB);
#pragma unroll
    for (int l = 0; l < SB; l++) pm[l] = a.rmeta[(m0 + o + step * l) >> 4];
    if (st.parts != 1) {
#pragma unroll
      for (int l = 0; l < SB; l++) pa[l] = stream_turn(a, g0 + o + step * l);
    }
  };
  const V *in = a.buf + ((int64_t)vi * a.g.ppd + j) * N;
  V v[16];
#pragma unroll
  for (int l = 0; l < 16; l++) v[l] = in[(int64_t)(t + TS * l) * N1 + n1];
  fetch(0, an, am);
  fft_reg<V, +1, LOG2N2, B>(v, t, lds + b, a.tw4096);
  __syncthreads();  // the FFT's last reads of its LDS are done
  T *tile = reinterpret_cast<T *>(lds);
#pragma unroll
  for (int s = 0; s < 16; s++) tile[s * 256 + tid] = v[s].x;
#pragma unroll 1
  for (int q = 0; q < nq; q++) {
    if (q + 1 < nq) fetch(q + 1, bn, bm);
    if (q == NB) {  // segment b: its outputs replace a's (own slots only)
#pragma unroll
      for (int s = 0; s < 16; s++) tile[s * 256 + tid] = v[s].y;
    }
    const T *z = tile + (q % NB) * SB * 256 + tid;
    if (st.parts == 1) {
#pragma unroll
      for (int l = 0; l < SB; l++) stream_record<T, 1>(a, st, am[l], i, z[l * 256], an[l]);
    } else if (st.parts == 2) {
#pragma unroll
      for (int l = 0; l < SB; l++) stream_record<T, 2>(a, st, am[l], i, z[l * 256], an[l]);
    } else {
#pragma unroll
      for (int l = 0; l < SB; l++) stream_record<T, 3>(a, st, am[l], i, z[l * 256], an[l]);
    }
#pragma unroll
    for (int l = 0; l < SB; l++) {
      an[l] = bn[l];
      am[l] = bm[l];
    }
  }
}

// H of set b at bin k = k2 + N2 k1, stored at k2 N1 + k1
__global__ __launch_bounds__(256) void k_build_mix(const double *spn, const SkyDet *sdet, const int32_t *sbeg, int nset,
                                                   int64_t N, int64_t N1, int64_t N2, double *mix, float *mix32) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= nset * N) return;
  const int64_t b = g / N, i = g - b * N, k2 = i / N1, k1 = i - k2 * N1, k = k2 + N2 * k1;
  const int64_t bin = k < N - k ? k : N - k;
  double h[6] = {0, 0, 0, 0, 0, 0};
  for (int d = sbeg[b]; d < sbeg[b + 1]; d++) {
    const SkyDet sd = sdet[d];
    const double w = spn[(int64_t)sd.det * (N / 2 + 1) + bin];
    h[0] += w;
    h[1] += w * sd.c;
    h[2] += w * sd.s;
    h[3] += w * sd.c * sd.c;
    h[4] += w * sd.c * sd.s;
    h[5] += w * sd.s * sd.s;
  }
#pragma unroll
  for (int n = 0; n < 6; n++) {
    mix[(b * 6 + n) * N + i] = h[n];
    if (mix32) mix32[(b * 6 + n) * N + i] = (float)h[n];
  }
}

__global__ __launch_bounds__(256) void k_same_pixels(const int32_t *pix, int64_t spd, const int32_t *lead,
                                                     int32_t *flag) {
  const int d = blockIdx.y, l = lead[d];
  if (l == d) return;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < spd && pix[d * spd + i] != pix[l * spd + i]) flag[d] = 1;
}

}  // namespace

// Column passes over streams: one block per (stream, pair, column block).
template <typename T>
int launch_col_fwd_streams(const OpArgs<T> &a, hipStream_t s) {
  const int64_t nb = (int64_t)a.nvs * a.g.ppd * (a.g.N / 4096);
#define CS(L) \
  case L: return launch1(k_col_fwd_st<T, L>, nb, s, a);
  switch (a.g.log2N2) {
    CS(4) CS(5) CS(6) CS(7) CS(8)
    default: return -2;
  }
#undef CS
}

// Whether the detectors on their own share the sets' row launch.  In small
// contexts a launch after it costs more than their rows (4 + 1 detectors x 4
// segments of 2^13 samples: 87 us an iteration with two launches, 72 with one,
// 79 with one stream per detector); in large ones the rows of one wave or two a
// stream lose to blocks of 256 threads (8 + 9 x 8 x 2^18: 894 us, 958 with one
// launch), and at N1 = 4096 the common kernel would spill 65 registers.
static bool row_merged(const PairGeom &g, int nvs, int nset) {
  return nvs > 3 * nset && g.log2N1 <= 11 && nvs * g.ppd * g.N < kStreamsSmall;
}

int64_t stream_row_blocks(const PairGeom &g, int nvs, int nset) {
  const int64_t rows = g.ppd * (g.N / 4096), n = rows * (g.log2N1 <= 10 ? 4 : g.log2N1 == 11 ? 2 : 1);
  const int64_t own = nvs - 3 * (int64_t)nset;
  return nset * n + (row_merged(g, nvs, nset) ? (own * n + 2) / 3 : own * rows);
}

template <typename T>
int launch_row_streams(const OpArgs<T> &a, hipStream_t s, int64_t *nblocks) {
  const bool chi = (a.mode & ROW_CHI2) != 0, merged = row_merged(a.g, a.nvs, a.nset);
  const int64_t nb = stream_row_blocks(a.g, a.nvs, a.nset);
  const int64_t nown = merged ? 0 : (a.nvs - 3 * (int64_t)a.nset) * a.g.ppd * (a.g.N / 4096), nmix = nb - nown;
  if (nblocks) *nblocks = nb;
  if (chi && sizeof(T) != 8) return -2;
#define RM1(L, OWN)                                                                     \
  do {                                                                                  \
    if constexpr (sizeof(T) == 8)                                                       \
      if (chi && launch1(k_row_chi<L, OWN>, nmix, s, a, 3 * row_group<L>())) return -1; \
    if (launch1(k_row_mix<T, L, OWN>, nmix, s, a, 3 * row_group<L>())) return -1;       \
  } while (0)
#define RM(L)                  \
  case L:                      \
    if (merged) RM1(L, true);  \
    else RM1(L, false);        \
    break;
  switch (a.g.log2N1) {
    RM(9) RM(10) RM(11)
    case 12: RM1(12, false); break;
    default: return -2;
  }
#undef RM
#undef RM1
  if (nown <= 0) return 0;
  OpArgs<T> o = a;
  o.g.npairs = nown / (a.g.N / 4096);
  o.g.pair0 = 0;
  o.chi2off = nmix;
  switch (a.g.log2N1) {
    case 9: return launch1(k_row_own<T, 9>, nown, s, o);
    case 10: return launch1(k_row_own<T, 10>, nown, s, o);
    case 11: return launch1(k_row_own<T, 11>, nown, s, o);
    case 12: return launch1(k_row_own<T, 12>, nown, s, o);
    default: return -2;
  }
}

template <typename T>
int launch_col_inv_streams(const OpArgs<T> &a, hipStream_t s) {
  const int64_t nb = (int64_t)a.nvs * a.g.ppd * (a.g.N / 4096);
#define CS(L) \
  case L: return launch1(k_col_inv_st<T, L>, nb, s, a);
  switch (a.g.log2N2) {
    CS(4) CS(5) CS(6) CS(7) CS(8)
    default: return -2;
  }
#undef CS
}

int launch_build_mix(const double *spn, const SkyDet *sdet, const int32_t *sbeg, int nset, int64_t N, int64_t N1,
                     int64_t N2, double *mix, float *mix32, hipStream_t s) {
  if (nset <= 0) return 0;
  hipLaunchKernelGGL(k_build_mix, dim3((unsigned)((nset * N + 255) / 256)), dim3(256), 0, s, spn, sdet, sbeg, nset, N,
                     N1, N2, mix, mix32);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_same_pixels(const int32_t *pix, int64_t spd, const int32_t *lead, int64_t ndet, int32_t *flag,
                       hipStream_t s) {
  if (ndet > 65535) return -2;
  hipLaunchKernelGGL(k_same_pixels, dim3((unsigned)((spd + 255) / 256), (unsigned)ndet), dim3(256), 0, s, pix, spd, lead,
                     flag);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template int launch_col_fwd_streams<double>(const OpArgs<double> &, hipStream_t);
template int launch_col_fwd_streams<float>(const OpArgs<float> &, hipStream_t);
template int launch_row_streams<double>(const OpArgs<double> &, hipStream_t, int64_t *);
template int launch_row_streams<float>(const OpArgs<float> &, hipStream_t, int64_t *);
template int launch_col_inv_streams<double>(const OpArgs<double> &, hipStream_t);
template int launch_col_inv_streams<float>(const OpArgs<float> &, hipStream_t);

