// ops_dev.h -- device helpers of the filter passes, shared by ops.hip (one
// stream per detector) and ops_streams.hip (shared lines of sight).
#pragma once
#include <type_traits>

#include "fft_core.h"
#include "kernels.h"
#include "turn.h"

using namespace sfft;

namespace {

template <typename T> using VT = typename Vec2<T>::type;

// pr is the launch-local pair; buffers of the four-step passes are indexed
// locally (a chunk of pairs reuses one buffer), samples and spectra globally.
__device__ __forceinline__ void pair_info(const PairGeom &g, int64_t pr, int &det, int64_t &ga,
                                          int64_t &gb) {
  pr += g.pair0;
  det = (int)(pr / g.ppd);
  const int64_t j = pr % g.ppd;
  ga = ((int64_t)det * g.nseg + 2 * j) * g.N;
  gb = (2 * j + 1 < g.nseg) ? ga + g.N : -1;
}

// P: Ps = S[m] + polard (S[npix+m] cos 2psi + S[2npix+m] sin 2psi), polard = 1
// (deproject, 2865-2868); the map is interleaved [npix][3] on the device.
// LEAK: the map is [npix][4] and Ps += S[3 npix + m] rfGal (2869-2870), the
// coefficient of the sample's detector g / spd.
template <typename T, bool LEAK = false>
__device__ __forceinline__ T gather_one(const OpArgs<T> &a, int64_t gi) {
  const int p = a.pix[gi];
  VT<T> c;
  if constexpr (sizeof(T) == 4) c = cs_of_turn(a.ang[gi]);
  else c = a.cs[gi];
  const T *m = a.map + (LEAK ? 4 : 3) * (int64_t)p;
  T v = m[0] + fma(m[1], c.x, m[2] * c.y);  // explicit: the same bits in every kernel
  if constexpr (LEAK) v = fma(m[3], a.relf[gi / a.spd], v);
  return v;
}

// A block's table of (cos, sin) of j/256 turn in LDS, for decoding 64-bit
// turns with cs_of_turn64_tab; a kernel that uses it calls fill_turn_tab with
// all of its 256 threads and then passes a barrier.
__shared__ double2 s_turn_tab[256];
__device__ __forceinline__ void fill_turn_tab() {
  s_turn_tab[threadIdx.x] = cs_of_turn64((uint64_t)threadIdx.x << 56);
}

// FP64 gather with the angle as a 64-bit turn (8 bytes a sample instead of
// 16), decoded through the block's table with TAB (the power-of-two column
// pass; the radix-3/5 passes, at the register limit, keep the series)
template <typename T, bool TAB>
__device__ __forceinline__ T gather_t64(const OpArgs<T> &a, int64_t gi) {
  const int p = a.pix[gi];
  const double2 c = TAB ? cs_of_turn64_tab(a.ang64[gi], s_turn_tab) : cs_of_turn64(a.ang64[gi]);
  const T *m = a.map + 3 * (int64_t)p;
  return m[0] + fma(m[1], (T)c.x, m[2] * (T)c.y);  // explicit: the same bits in every kernel
}

template <typename T, int SRC, bool TAB = false>
__device__ __forceinline__ T load_src(const OpArgs<T> &a, int64_t gi) {
  if constexpr (SRC == SRC_GATHER) return gather_one<T>(a, gi);
  else if constexpr (SRC == SRC_GATHER_T64) return gather_t64<T, TAB>(a, gi);
  else if constexpr (SRC == SRC_RNG) return (T)normal_at(a.seed, (uint64_t)gi);
  else if constexpr (SRC == SRC_PX) return a.px[gi];
  else return (T)a.tod[gi];
}

template <typename V, int DIR>
__device__ __forceinline__ V twN(const V *__restrict__ lo, const V *__restrict__ hi, int64_t j) {
  V w = cmul(lo[j & 4095], hi[j >> 12]);
  return DIR < 0 ? w : cconj(w);
}

// Angle of sample g in the operator's form: a turn (FP32) or (cos, sin) (FP64).
template <typename T> struct AngOf;
template <> struct AngOf<float> {
  using type = uint32_t;
  __device__ static type load(const OpArgs<float> &a, int64_t g) { return a.ang[g]; }
  __device__ static float2 cs(type v) { return cs_of_turn(v); }
};
template <> struct AngOf<double> {
  using type = double2;
  __device__ static type load(const OpArgs<double> &a, int64_t g) { return a.cs[g]; }
  __device__ static double2 cs(type v) { return v; }
};
// FP64 angles read as 64-bit turns
struct AngOf64 {
  using type = uint64_t;
  __device__ static type load(const OpArgs<double> &a, int64_t g) { return a.ang64[g]; }
  __device__ static double2 cs(type v) { return cs_of_turn64(v); }
};
// ... decoded through the block's table
struct AngOf64Tab {
  using type = uint64_t;
  __device__ static type load(const OpArgs<double> &a, int64_t g) { return a.ang64[g]; }
  __device__ static double2 cs(type v) { return cs_of_turn64_tab(v, s_turn_tab); }
};

// Outer four-step twiddles w_N^{DIR (j0 + dj s)}, s = 0, 1, ..., for one
// thread's outputs.  A lookup per output (twN) spreads a wave's 64 lanes over
// up to 64 lines of the 4096-entry table; a run reads w_N^{j0} and w_N^{dj}
// once from the FP64 tables and steps by FP64 multiplication (after 15 steps
// the error is ~1e-15, below the rounding of an FP32 twiddle and of the same
// order as the two-table product in FP64).
struct TwRun {
  double2 w, step;
};

template <int DIR>
__device__ __forceinline__ TwRun tw_run(const double2 *__restrict__ lo, const double2 *__restrict__ hi,
                                        int64_t j0, int64_t dj) {
  return TwRun{twN<double2, DIR>(lo, hi, j0), twN<double2, DIR>(lo, hi, dj)};
}

template <typename V>
__device__ __forceinline__ V tw_next(TwRun &r) {
  using S = decltype(V::x);
  const V w = mk<V>((S)r.w.x, (S)r.w.y);
  r.w = cmul(r.w, r.step);
  return w;
}

__device__ __forceinline__ double block_sum256(double v, double *red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) s = ((red[0] + red[1]) + (red[2] + red[3]));
  return s;
}

// Workgroups are dispatched to the 8 XCDs round-robin (block b on XCD b % 8),
// each XCD with its own L2.  With a.xcd set, XCD x takes one contiguous range
// of logical blocks instead, so neighbouring column blocks -- which read and
// write the two halves of the same 128-byte lines -- share an L2.
__device__ __forceinline__ int64_t logical_block(int xcd) {
  const int64_t b = blockIdx.x;
  if (!xcd) return b;
  const int64_t nb = gridDim.x, q = nb >> 3, r = nb & 7, x = b & 7, i = b >> 3;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// Output slot of sample g: its position in the pixel-sorted order when the
// context keeps z sorted (P^T then reads z contiguously), else g itself.
template <typename T>
__device__ __forceinline__ int64_t zslot(const OpArgs<T> &a, int64_t g) {
  return a.zpos ? (int64_t)a.zpos[g] : g;
}

// Relative calibration of the (detector, segment) block holding sample g
// (1 when the context has none): the filtered z of the block is scaled by
// it once more on the way out, N^-1 relCalib^2 of do_PtNd (2543-2545).
template <typename T>
__device__ __forceinline__ T seg_gain(const OpArgs<T> &a, int64_t g) {
  return a.gain ? a.gain[g / a.blk] : (T)1;
}

// The gathered values of segments ga and gb (gb < 0: none) times their gains:
// the model the recalibrated data are compared with (write_tfAS on S, 1252).
// In the column pass, where the values are in registers; a pass of its own that
// wrote the scaled P x took 17 us beside a column pass of 10 us at 4 detectors x
// 12 segments of 2^16 samples, one of 20 us now.
template <typename T, int SRC>
__device__ __forceinline__ void gather_gain(const OpArgs<T> &a, int64_t ga, int64_t gb, VT<T> (&v)[16]) {
  if constexpr (SRC == SRC_GATHER || SRC == SRC_GATHER_T64) {
    if (!a.gain) return;
    const T fa = seg_gain(a, ga), fb = gb >= 0 ? seg_gain(a, gb) : (T)0;
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = mk<VT<T>>(v[i].x * fa, gb >= 0 ? v[i].y * fb : v[i].y);
  }
}

constexpr int kLds = 4352;

// ---------------------------------------------------------------------- row
// OWN: the rows belong to the streams after the sets' of a context with shared
// lines of sight; weights and data spectra are those of the stream's detector.
template <typename T, int LOG2N1, bool OWN = false>
__device__ __forceinline__ void row_body(const OpArgs<T> &a, int64_t lb, LdsE<VT<T>> *lds, double *red, int mode) {
  using V = VT<T>;
  constexpr int N1 = 1 << LOG2N1, TS = N1 / 16, B = 256 / TS;
  static_assert(LdsSize<LOG2N1, B>::value <= kLds, "LDS");
  const int tid = threadIdx.x, b = tid % B, t = tid / B;
  const int64_t N = a.g.N, N2 = a.g.N2;
  const int64_t nrb = N2 / B;
  int64_t pr, rb;
  if (a.rowdet) {
    // consecutive blocks take the same rows of one detector's pairs, so the
    // detector's weight row is read from L2 by all but the first
    const int64_t ppd = a.g.ppd, per = ppd * nrb, r = lb % per;
    rb = r / ppd;
    pr = (lb / per) * ppd + r % ppd;
  } else {
    pr = lb / nrb;
    rb = lb % nrb;
  }
  const int64_t k2 = rb * B + b;
  int det;
  int64_t ga, gb;
  pair_info(a.g, pr, det, ga, gb);
  int64_t base = pr * N + k2 * N1;
  int64_t sbase = (pr + a.g.pair0) * N + k2 * N1;
  if constexpr (OWN) {
    base += 3 * (int64_t)a.nset * a.g.ppd * N;
    det = a.vs[3 * a.nset + det].det;
    sbase = ((int64_t)det * a.g.ppd + pr % a.g.ppd) * N + k2 * N1;
  }
  const T *w = a.wt + (int64_t)det * N + k2 * N1;
  V v[16];
  if (mode & ROW_SRC_WT) {
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = mk<V>(w[t + TS * i], (T)0);
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = a.buf[base + t + TS * i];
  }
  // the weights are loaded with the row, so their latency hides under the
  // forward FFT instead of stalling the filter
  T wf[16];
  if (mode & ROW_FILTER) {
#pragma unroll
    for (int s = 0; s < 16; s++) wf[s] = w[t + TS * s];
  }
  double chi = 0.0;
  if (mode & ROW_FWD) {
    fft_reg<V, -1, LOG2N1, B>(v, t, lds + b, a.tw4096);
    if (mode & ROW_STORE_D) {
#pragma unroll
      for (int s = 0; s < 16; s++) a.dspec[sbase + t + TS * s] = v[s];
    }
    if (mode & ROW_CHI2) {
#pragma unroll
      for (int s = 0; s < 16; s++) {
        const int k1 = t + TS * s;
        const V D = a.dspec[sbase + k1];
        const double rx = (double)D.x - (double)v[s].x, ry = (double)D.y - (double)v[s].y;
        double e = (double)w[k1] * (rx * rx + ry * ry);
        // bins 0 and N/2 are counted twice by the reference's per-segment sum
        if (k2 == 0 && (k1 == 0 || k1 == N1 / 2)) e += e;
        chi += e;
      }
    }
    if (mode & ROW_FILTER) {
#pragma unroll
      for (int s = 0; s < 16; s++) v[s] = mk<V>(v[s].x * wf[s], v[s].y * wf[s]);
    }
  }
  if (mode & ROW_INV) {
    fft_reg<V, +1, LOG2N1, B>(v, t, lds + b, a.tw4096);
    TwRun tr = tw_run<+1>(a.twlo64, a.twhi64, (int64_t)t * k2, (int64_t)TS * k2);  // j = n1 k2, n1 = t + TS s
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const int64_t n1 = t + TS * s;
      a.buf[base + n1] = cmul(v[s], tw_next<V>(tr));
    }
  }
  if (mode & ROW_CHI2) {
    const double tot = block_sum256(chi, red);
    if (tid == 0) a.chi2part[a.chi2off + lb] = tot;
  }
}

// Lane i of a 16-lane row reads lane i - OFF of the same row (DPP row_shr;
// lanes below OFF read 0).
template <int OFF>
__device__ __forceinline__ float row_shr(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x110 + OFF, 0xF,
                                                               0xF, true));
}
template <int OFF>
__device__ __forceinline__ double row_shr(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, 0x110 + OFF, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), 0x110 + OFF, 0xF, 0xF, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

template <typename K, typename A>
int launch1(K kern, int64_t nblocks, hipStream_t s, const A &a, int threads = 256) {
  if (nblocks <= 0) return 0;
  if (nblocks > 0x7fffffffLL) return -1;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(threads), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace
