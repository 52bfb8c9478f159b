// Oversampled FFT of the table NUFFT with the element-wise stages fused in (gfx950).
//
// Replaces fft_and_scale / ifft_and_scale (torchkbnufft/_nufft/fft.py:36-118) plus the
// SENSE expansion and coil combine (modules/kbnufft.py:182-183, 404-405):
//   forward : grid = FFT_K( pad_end( image * smaps * scaling_coef * scale ) )    (unnormalised)
//   adjoint : image = sum_c crop( IFFT_K(grid) ) * conj(scaling_coef) * conj(smaps_c) * scale
// as a sequence of one-dimensional passes over memory:
//   * the last-dimension pass reads contiguous lines; the forward one builds its input
//     from image * smaps * scaling (zero beyond im_size), the adjoint one writes the
//     cropped, deapodised, coil-combined image directly;
//   * every other dimension is a strided pass over a block of adjacent columns
//     (coalesced 64-128 B segments), which zero-pads (forward) or crops (adjoint).
// Intermediates therefore only hold im_size extents in the not-yet-transformed
// dimensions (half of the grid per dimension at 2x oversampling).
//
// One pass is a decimation-in-frequency FFT of two to four butterfly stages of radix up
// to 16.  The first stage's butterflies are loaded from memory straight into registers
// and the last stage's go straight to memory; only the values between stages cross LDS,
// one write and one read each, in place (a thread writes the addresses it read), with
// one barrier per stage.  64 images of 320 x 320 -> 640 x 640 (row pass 157 MB, column pass
// 315 MB, the filter's column pass 210 MB; a large copy runs at 5.1 TB/s): row pass 47 us
// forward and 60 us adjoint, column pass 84 and 77 us, filter 98 us.  Stockham passes of
// radices <= 8 with every value in LDS (six LDS writes and reads per element and nine
// barriers at length 640) and twiddles evaluated by each group took 69 and 57, 92 and 92,
// 148 us.  The vector units are busy 79 % of the filter's time, 52 to 54 % of the column passes'
// (which move 4.0 and 4.3 TB/s) and 28 to 53 % of the row passes': the filter is bound by the
// butterflies' arithmetic, the others by neither alone.
// Grid sizes whose prime factors are 2, 3 and 5 have compiled or runtime plans of these
// radices; the primes 7 to 17 add runtime butterflies of their own size, and a dimension with
// a larger prime is transformed as a convolution (chirp kernels below).
// Twiddles (double precision rounded to float) are put into LDS while the first stage's
// loads are in flight.  Only the forward transform is coded: the inverse swaps real and
// imaginary parts on the way in and out.
#include "tkbn_common.h"

namespace tkbn {

constexpr int kMaxStages = 6;

// ---------------------------------------------------------------------------
// radices of a length
// ---------------------------------------------------------------------------
struct RadixList {
  int n;  // stages; 0: a prime factor above 17
  int r[kMaxStages];
};

constexpr int kNumRadices = 14;
constexpr int kRadices[kNumRadices] = {17, 16, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// the shortest product of radices (in descending order) equal to K; among those of one
// length, the one whose smallest radix is largest (fewest butterflies, so fewest threads)
constexpr void search_radices(int K, int from, RadixList cur, RadixList& best) {
  if (K == 1) {
    const bool better = best.n == 0 || cur.n < best.n || (cur.n == best.n && cur.r[cur.n - 1] > best.r[best.n - 1]);
    if (cur.n > 0 && better) best = cur;
    return;
  }
  if (cur.n >= kMaxStages || (best.n > 0 && cur.n >= best.n)) return;
  for (int i = from; i < kNumRadices; ++i) {
    if (K % kRadices[i] == 0) {
      RadixList nxt = cur;
      nxt.r[nxt.n++] = kRadices[i];
      search_radices(K / kRadices[i], i, nxt, best);
    }
  }
}

// Stages of a transform of length K >= 1, at least two (a lone radix is followed by a
// radix of 1).  An even radix goes first and last where there are two: with half of the
// inputs zero (padding) or half of the outputs unused (cropping), half of that stage's
// butterfly inputs or outputs then drop out whole.
constexpr RadixList radix_list(int K) {
  RadixList best{0, {}};
  if (K == 1) return RadixList{2, {1, 1}};
  search_radices(K, 0, RadixList{0, {}}, best);
  if (best.n == 0) return best;
  if (best.n == 1) {
    best.r[best.n++] = 1;
    return best;
  }
  for (int end = 0; end < 2; ++end) {  // last place, then first place, from the evens left
    const int at = end == 0 ? best.n - 1 : 0;
    const int lo = 0, hi = end == 0 ? best.n : best.n - 1;
    for (int i = lo; i < hi; ++i) {
      if (best.r[i] % 2 == 0) {
        const int t = best.r[i];
        best.r[i] = best.r[at];
        best.r[at] = t;
        break;
      }
    }
  }
  return best;
}

// Runtime plan of one length: per stage s the block length Lb = K / (r_0 .. r_{s-1}),
// the butterflies per block nbs = Lb / r_s and per transform per = K / r_s.
struct FftPlan1D {
  int K;
  int n;
  int r[kMaxStages];
  int Lb[kMaxStages];
  int tw[kMaxStages];  // offset of the stage's twiddles
  int ntw;             // twiddles in all
  FastDiv nbs[kMaxStages], per[kMaxStages], rd[kMaxStages];
  FastDiv q1[kMaxStages];  // (r_1 .. r_{s-1}): a block's index / this = its first digit
};

// ---------------------------------------------------------------------------
// forward DFTs of R values in registers, x[k] = sum_n x[n] exp(-2 pi i n k / R)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 mul_mi(float2 a) { return make_float2(a.y, -a.x); }  // times -i
__device__ __forceinline__ float2 cswap(float2 a) { return make_float2(a.y, a.x); }

// sin(x) and cos(x) for |x| <= pi by their series (compile time; ~1e-15)
constexpr double cx_sin(double x) {
  double t = x, s = x;
  for (int n = 1; n < 20; ++n) {
    t *= -x * x / ((2 * n) * (2 * n + 1));
    s += t;
  }
  return s;
}
constexpr double cx_cos(double x) {
  double t = 1, s = 1;
  for (int n = 1; n < 20; ++n) {
    t *= -x * x / ((2 * n - 1) * (2 * n));
    s += t;
  }
  return s;
}
constexpr double kTwoPi = 6.283185307179586476925286766559;
// exp(-2 pi i m / R), |m| < R
constexpr double root_angle(int m, int R) {
  int q = m % R;
  if (2 * q > R) q -= R;
  return kTwoPi * q / R;
}
template <int M, int R>
__device__ __forceinline__ float2 mul_root(float2 a) {
  constexpr int m = M % R;
  if constexpr (m == 0) {
    return a;
  } else if constexpr (4 * m == R) {
    return mul_mi(a);
  } else if constexpr (2 * m == R) {
    return make_float2(-a.x, -a.y);
  } else if constexpr (4 * m == 3 * R) {
    return make_float2(-a.y, a.x);
  } else {
    constexpr float c = (float)cx_cos(root_angle(m, R)), s = (float)-cx_sin(root_angle(m, R));
    return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
  }
}

template <int R>
__device__ __forceinline__ void dft(float2* x);

// the multiple of A below A * B that is 1 modulo B
constexpr int unit_multiple(int A, int B) {
  int m = A;
  while (m % B != 1) m += A;
  return m;
}

// R = A * B: A-point DFTs over the inputs n2 + B n1, roots, B-point DFTs
template <int A, int B, int N2, int K1>
__device__ __forceinline__ void mul_roots_row(float2 (&y)[A]) {
  if constexpr (K1 < A) {
    y[K1] = mul_root<N2 * K1, A * B>(y[K1]);
    mul_roots_row<A, B, N2, K1 + 1>(y);
  }
}
template <int A, int B, int N2 = 0>
__device__ __forceinline__ void dft_rows(const float2* x, float2 (&y)[B][A]) {
  if constexpr (N2 < B) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) y[N2][n1] = x[N2 + B * n1];
    dft<A>(y[N2]);
    mul_roots_row<A, B, N2, 1>(y[N2]);
    dft_rows<A, B, N2 + 1>(x, y);
  }
}
template <int A, int B>
__device__ __forceinline__ void dft_ab(float2* x) {
  float2 y[B][A];
  dft_rows<A, B>(x, y);
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    float2 z[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) z[n2] = y[n2][k1];
    dft<B>(z);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) x[k1 + A * k2] = z[k2];
  }
}

// R = A * B without a common factor: A-point and B-point DFTs with no roots between them (Good,
// "The interaction algorithm and practical Fourier analysis", 1958): input B n1 + A n2, output
// congruent to k1 modulo A and to k2 modulo B.  The roots that dft_ab multiplies by cost
// roundings beside their work: 1000 = 10 * 10 * 10 was 5 to 14 % further from 64-bit values
// than passes of radices 8 and below, 216 = 6 * 6 * 6 7 to 12 %.
template <int A, int B>
__device__ __forceinline__ void dft_coprime(float2* x) {
  constexpr int R = A * B, E1 = unit_multiple(B, A), E2 = unit_multiple(A, B);
  float2 y[B][A];
#pragma unroll
  for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
    for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = x[(B * n1 + A * n2) % R];
    dft<A>(y[n2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    float2 z[B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) z[n2] = y[n2][k1];
    dft<B>(z);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) x[(E1 * k1 + E2 * k2) % R] = z[k2];
  }
}

// an odd prime P: x_k and x_{P-k} combined into sums and differences
template <int P, int Q, int K>
__device__ __forceinline__ void prime_terms(float2& u, float2& v, const float2* a, const float2* b) {
  if constexpr (K <= (P - 1) / 2) {
    constexpr float c = (float)cx_cos(root_angle(Q * K % P, P)), s = (float)cx_sin(root_angle(Q * K % P, P));
    u.x = fmaf(c, a[K].x, u.x);
    u.y = fmaf(c, a[K].y, u.y);
    v.x = fmaf(s, b[K].x, v.x);
    v.y = fmaf(s, b[K].y, v.y);
    prime_terms<P, Q, K + 1>(u, v, a, b);
  }
}
template <int P, int Q = 1>
__device__ __forceinline__ void prime_outputs(float2* x, float2 x0, const float2* a, const float2* b) {
  if constexpr (Q <= (P - 1) / 2) {
    float2 u = x0, v = make_float2(0.f, 0.f);
    prime_terms<P, Q, 1>(u, v, a, b);
    x[Q] = make_float2(u.x + v.y, u.y - v.x);  // u - i v
    x[P - Q] = make_float2(u.x - v.y, u.y + v.x);
    prime_outputs<P, Q + 1>(x, x0, a, b);
  }
}
template <int P>
__device__ __forceinline__ void dft_prime(float2* x) {
  constexpr int H = (P - 1) / 2;
  float2 a[H + 1], b[H + 1];
  const float2 x0 = x[0];
  float2 s = x0;
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    a[k] = cadd(x[k], x[P - k]);
    b[k] = csub(x[k], x[P - k]);
    s = cadd(s, a[k]);
  }
  prime_outputs<P>(x, x0, a, b);
  x[0] = s;
}

template <int R>
__device__ __forceinline__ void dft(float2* x) {
  if constexpr (R == 2) {
    const float2 a = x[0], b = x[1];
    x[0] = cadd(a, b);
    x[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const float2 t0 = cadd(x[0], x[2]), t1 = csub(x[0], x[2]);
    const float2 t2 = cadd(x[1], x[3]), t3 = mul_mi(csub(x[1], x[3]));
    x[0] = cadd(t0, t2);
    x[2] = csub(t0, t2);
    x[1] = cadd(t1, t3);
    x[3] = csub(t1, t3);
  } else if constexpr (R == 8) {
    float2 e[4] = {x[0], x[2], x[4], x[6]};
    float2 o[4] = {x[1], x[3], x[5], x[7]};
    dft<4>(e);
    dft<4>(o);
    const float r = 0.70710678118654752f;
    // w8 = (1 - i)/sqrt2, w8^2 = -i, w8^3 = (-1 - i)/sqrt2
    const float2 o1 = make_float2(r * (o[1].x + o[1].y), r * (o[1].y - o[1].x));
    const float2 o2 = mul_mi(o[2]);
    const float2 o3 = make_float2(r * (o[3].y - o[3].x), -r * (o[3].x + o[3].y));
    x[0] = cadd(e[0], o[0]);
    x[4] = csub(e[0], o[0]);
    x[1] = cadd(e[1], o1);
    x[5] = csub(e[1], o1);
    x[2] = cadd(e[2], o2);
    x[6] = csub(e[2], o2);
    x[3] = cadd(e[3], o3);
    x[7] = csub(e[3], o3);
  } else if constexpr (R == 3 || R == 5 || R == 7 || R == 11 || R == 13 || R == 17) {
    dft_prime<R>(x);
  } else if constexpr (R == 6) {
    dft_coprime<2, 3>(x);
  } else if constexpr (R == 9) {
    dft_ab<3, 3>(x);
  } else if constexpr (R == 10) {
    dft_coprime<2, 5>(x);
  } else if constexpr (R == 12) {
    dft_coprime<4, 3>(x);
  } else if constexpr (R == 16) {
    dft_ab<4, 4>(x);
  } else {
    static_assert(R == 1, "no butterfly of this radix");
  }
}

// ---------------------------------------------------------------------------
// stages
// ---------------------------------------------------------------------------
// Work-group barrier that orders LDS accesses only (global loads and stores stay in flight).
__device__ __forceinline__ void fft_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Lengths and dividers of a transform: compiled for its length (every division and
// stride is a constant) or from a runtime plan.  S: the stage as an integral constant or int.
template <int V>
struct Int {
  static constexpr int value = V;
};
constexpr int radices_before(const RadixList& L, int s) {
  int p = 1;
  for (int i = 0; i < s; ++i) p *= L.r[i];
  return p;
}

template <int KC>
struct StaticLen {
  static constexpr RadixList L = radix_list(KC);
  static constexpr int n = L.n;
  template <class S> __device__ static constexpr int Lb(S) { return KC / radices_before(L, S::value); }
  template <class S> __device__ static constexpr int nbs(S) { return KC / radices_before(L, S::value) / L.r[S::value]; }
  template <class S> __device__ static constexpr int per(S) { return KC / L.r[S::value]; }
  template <class S> __device__ static constexpr int tw(S) {
    int o = 0;
    for (int i = 0; i < S::value; ++i) o += KC / radices_before(L, i);
    return o;
  }
  template <class S> __device__ static int div_nbs(S s, int x) { return (unsigned)x / (unsigned)nbs(s); }
  template <class S> __device__ static int div_per(S s, int x) { return (unsigned)x / (unsigned)per(s); }
  // first digit of block blk of stage s
  template <class S> __device__ static int digit0(S, int blk) {
    return (unsigned)blk / (unsigned)(radices_before(L, S::value) / L.r[0]);
  }
  // LDS place of block f0 of the last stage (its digits reversed) and its first digit
  template <int S = 0>
  __device__ static void reverse(int f, int& blk, int& d0) {
    if constexpr (S == 0) blk = 0;
    if constexpr (S < L.n - 1) {
      const int q = (unsigned)f / (unsigned)L.r[S], d = f - q * L.r[S];
      if constexpr (S == 0) d0 = d;
      blk = blk * L.r[S] + d;
      reverse<S + 1>(q, blk, d0);
    }
  }
};

// Stage s of a runtime plan.  Its values are read once, here: a kernel argument with more
// than some hundred indexed uses is copied to scratch memory.
struct DynLen {
  const FftPlan1D& p;
  int r, lb, tw0;
  FastDiv fnbs, fper, fq1;
  __device__ __forceinline__ DynLen(const FftPlan1D& pl, int s)
      : p(pl), r(pl.r[s]), lb(pl.Lb[s]), tw0(pl.tw[s]), fnbs(pl.nbs[s]), fper(pl.per[s]), fq1(pl.q1[s]) {}
  __device__ int Lb(int) const { return lb; }
  __device__ int nbs(int) const { return (int)fnbs.d; }
  __device__ int per(int) const { return (int)fper.d; }
  __device__ int tw(int) const { return tw0; }
  __device__ int div_nbs(int, int x) const { return (int)fdiv(x, fnbs); }
  __device__ int div_per(int, int x) const { return (int)fdiv(x, fper); }
  __device__ int digit0(int, int blk) const { return (int)fdiv(blk, fq1); }
  __device__ void reverse(int f, int& blk, int& d0) const {
    blk = 0;
    for (int s = 0; s < p.n - 1; ++s) {
      const int q = (int)fdiv(f, p.rd[s]), d = f - q * p.r[s];
      if (s == 0) d0 = d;
      blk = blk * p.r[s] + d;
      f = q;
    }
  }
};

// Twiddles of every stage but the last, tw_s[q] = exp(-2 pi i q / Lb_s), q < Lb_s, to LDS.
// A compiled length has them as constant data (evaluated in double and rounded); a runtime
// length evaluates them in double precision.  Ends with a barrier.
constexpr int twiddles_of(const RadixList& L, int K) {
  int n = 0, len = K;
  for (int s = 0; s < L.n - 1; ++s) {
    n += len;
    len /= L.r[s];
  }
  return n;
}
template <int N>
struct TwTable {
  float v[2 * N];
};
template <int KC>
constexpr TwTable<twiddles_of(radix_list(KC), KC)> make_tw_table() {
  constexpr RadixList L = radix_list(KC);
  TwTable<twiddles_of(L, KC)> t{};
  int at = 0, len = KC;
  for (int s = 0; s < L.n - 1; ++s) {
    for (int q = 0; q < len; ++q) {
      const double a = root_angle(q, len);
      t.v[2 * (at + q)] = (float)cx_cos(a);
      t.v[2 * (at + q) + 1] = (float)-cx_sin(a);
    }
    at += len;
    len /= L.r[s];
  }
  return t;
}
template <int KC>
__device__ const TwTable<twiddles_of(radix_list(KC), KC)> kTwTable = make_tw_table<KC>();

template <int KC>
__device__ __forceinline__ void fill_twiddles(float2* tw, const FftPlan1D& pl) {
  if constexpr (KC > 0) {
    constexpr int n = twiddles_of(radix_list(KC), KC);
    for (int q = threadIdx.x; q < n; q += blockDim.x) tw[q] = make_float2(kTwTable<KC>.v[2 * q], kTwTable<KC>.v[2 * q + 1]);
  } else {
    for (int s = 0; s < pl.n - 1; ++s) {
      const DynLen len(pl, s);
      const int n = len.Lb(s);
      for (int q = threadIdx.x; q < n; q += blockDim.x) {
        double sn, cs;
        sincospi(2.0 * (double)q / (double)n, &sn, &cs);
        tw[len.tw(s) + q] = make_float2((float)cs, (float)-sn);
      }
    }
  }
  fft_barrier();
}

// Place of the transforms of a group in LDS.  Value idx of transform t: block digit 0 of
// idx is d0; the block of each first digit is one value longer than its K / r_0 values,
// which spreads the strided reads of the later stages over the banks.
//   COL: 1 << lgc transforms side by side (t fastest), LGC >= 0: lgc known at compile time
//   ROW: one after the other
template <bool COL, int LGC = -1>
struct LdsMap {
  int lgc_rt;
  int pitch;  // ROW: values per transform (K + r_0)
  static constexpr bool kCol = COL;
  __device__ __forceinline__ int lgc() const { return LGC >= 0 ? LGC : lgc_rt; }
  __device__ __forceinline__ int at(int t, int a) const { return COL ? (a << lgc()) + t : t * pitch + a; }
  __device__ __forceinline__ int step(int a) const { return COL ? a << lgc() : a; }
};

// Butterfly b of a stage over `nl` transforms: its transform t, place q among the
// transform's butterflies, LDS address of its value 0 and step between its values, and
// (not LAST) its twiddle index j.
template <int R, bool FIRST, bool LAST, class Map, class Len, class S>
__device__ __forceinline__ void butterfly_at(const Len& len, S s, const Map& map, int b, int& t, int& q, int& j,
                                             int& base, int& step) {
  const int per = len.per(s);
  if (Map::kCol) {
    q = b >> map.lgc();
    t = b & ((1 << map.lgc()) - 1);
  } else {
    t = len.div_per(s, b);
    q = b - t * per;
  }
  const int nbs = len.nbs(s);
  if constexpr (FIRST) {
    j = q;
    base = map.at(t, q);
    step = map.step(nbs + 1);
  } else if constexpr (!LAST) {
    const int blk = len.div_nbs(s, q);
    j = q - blk * nbs;
    base = map.at(t, blk * len.Lb(s) + len.digit0(s, blk) + j);
    step = map.step(nbs);
  } else {
    int blk, d0 = 0;
    len.reverse(q, blk, d0);
    j = 0;
    base = map.at(t, blk * R + d0);
    step = map.step(1);
  }
}

// One decimation-in-frequency stage.  FIRST: values from load.value(load.read(k, t), k, t),
// all reads of a butterfly issued before any is used; HIN: the inputs k >= K/2 are zero; with `fill` the twiddles
// of a compiled length are put into LDS once the first loads are issued.
// LAST: results to store(f, t, value, address of the butterfly's own LDS slot for it);
// HOUT: only f < K/2 are wanted.
template <int R, bool FIRST, bool LAST, bool HIN, bool HOUT, int KC, class Map, class Len, class S, class LoadF,
          class StoreF>
__device__ __forceinline__ void dif_stage(const FftPlan1D& pl, const Len& len, S s, const Map& map, int nl,
                                          float2* buf, float2* tw, int tid, LoadF load, bool fill, StoreF store) {
  const int total = nl * len.per(s);
  const float2* tws = tw + len.tw(s);
  float2 x[R];
  typename LoadF::Raw raw[R];
  int t = 0, q = 0, j = 0, base = 0, step = 0;
  auto take = [&](int b) {
    butterfly_at<R, FIRST, LAST>(len, s, map, b, t, q, j, base, step);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (!FIRST)
        x[i] = buf[base + i * step];
      else if (!(HIN && 2 * i >= R))
        raw[i] = load.read(q + i * len.nbs(s), t);
    }
  };
  int b = tid;
  if (b < total) take(b);
  if (FIRST && KC > 0 && fill) fill_twiddles<KC>(tw, pl);
  while (b < total) {
    if (FIRST) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        x[i] = (HIN && 2 * i >= R) ? make_float2(0.f, 0.f) : load.value(raw[i], q + i * len.nbs(s), t);
    }
    dft<R>(x);
    if (LAST) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (!(HOUT && R > 1 && 2 * i >= R)) store(q + i * len.per(s), t, x[i], base + i * step);
    } else {
      buf[base] = x[0];
#pragma unroll
      for (int i = 1; i < R; ++i) buf[base + i * step] = cmul(x[i], tws[i * j]);
    }
    b += blockDim.x;
    if (b < total) take(b);
  }
}

// The decimation-in-time counterpart, for a transform that follows a DIF one directly:
// takes the values in the DIF's order (digits reversed) and ends in natural order.
//   TURN: the DIF's last butterfly, mid.value(mid.read(f, t), value) of its results, and this
//         transform's first one, in registers
//   END : results of stage 0 to store(k, t, value); HOUT: only k < K/2 are wanted
template <int R, bool TURN, bool END, bool HOUT, class Map, class Len, class S, class MidF, class StoreF>
__device__ __forceinline__ void dit_stage(const Len& len, S s, const Map& map, int nl, float2* buf,
                                          const float2* tw, int tid, MidF mid, StoreF store) {
  const int total = nl * len.per(s);
  const float2* tws = tw + len.tw(s);
  for (int b = tid; b < total; b += blockDim.x) {
    int t, q, j, base, step;
    butterfly_at<R, END, TURN>(len, s, map, b, t, q, j, base, step);
    float2 x[R], m[R];
    if (TURN) {
#pragma unroll
      for (int i = 0; i < R; ++i) m[i] = mid.read(q + i * len.per(s), t);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) x[i] = buf[base + i * step];
    if (TURN) {
      dft<R>(x);
#pragma unroll
      for (int i = 0; i < R; ++i) x[i] = mid.value(m[i], x[i]);
    } else {
#pragma unroll
      for (int i = 1; i < R; ++i) x[i] = cmul(x[i], tws[i * j]);
    }
    dft<R>(x);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (END) {
        if (!(HOUT && R > 1 && 2 * i >= R)) store(q + i * len.nbs(s), t, x[i]);
      } else {
        buf[base + i * step] = x[i];
      }
    }
  }
}

// (KC < 0: a runtime plan with primes above 5; their butterflies cost the other sizes'
// kernels registers: 167 -> 215 in the first pass)
#define TKBN_FOR_RADIX(r, CALL)                                                                   \
  switch (r) {                                                                                    \
    case 17: if constexpr (KC < 0) { CALL(17); } break;                                           \
    case 16: CALL(16); break;                                                                     \
    case 13: if constexpr (KC < 0) { CALL(13); } break;                                           \
    case 12: CALL(12); break;                                                                     \
    case 11: if constexpr (KC < 0) { CALL(11); } break;                                           \
    case 10: CALL(10); break;                                                                     \
    case 9: CALL(9); break;                                                                       \
    case 8: CALL(8); break;                                                                       \
    case 7: if constexpr (KC < 0) { CALL(7); } break;                                             \
    case 6: CALL(6); break;                                                                       \
    case 5: CALL(5); break;                                                                       \
    case 4: CALL(4); break;                                                                       \
    case 3: CALL(3); break;                                                                       \
    case 2: CALL(2); break;                                                                       \
    default: CALL(1); break;                                                                      \
  }

struct NoStore {
  __device__ void operator()(int, int, float2, int) const {}
};
// A stage's source: read() issues the loads, value() combines what they brought.
struct NoLoad {
  using Raw = float2;
  __device__ Raw read(int, int) const { return make_float2(0.f, 0.f); }
  __device__ float2 value(Raw v, int, int) const { return v; }
};
struct NoMid {
  __device__ float2 read(int, int) const { return make_float2(0.f, 0.f); }
  __device__ float2 value(float2, float2 v) const { return v; }
};
// column `t` of a block of columns, the first n rows (SWAP: real and imaginary exchanged);
// places past the block read its first value
struct ColLoad {
  const float2* s;
  int64_t inner;
  int n, nc;
  bool swap;
  using Raw = float2;
  __device__ __forceinline__ Raw read(int k, int t) const {
    return s[(int64_t)(k < n ? k : 0) * inner + (t < nc ? t : 0)];
  }
  __device__ __forceinline__ float2 value(Raw v, int k, int t) const {
    if (k >= n || t >= nc) return make_float2(0.f, 0.f);
    return swap ? cswap(v) : v;
  }
};
// line t of consecutive lines `pitch` apart, real and imaginary exchanged
struct LineLoad {
  const float2* s;
  int64_t pitch;
  using Raw = float2;
  __device__ __forceinline__ Raw read(int k, int t) const { return s[t * pitch + k]; }
  __device__ __forceinline__ float2 value(Raw v, int, int) const { return cswap(v); }
};

// All DIF stages but the last (LDS then holds the last stage's inputs, behind a barrier).
template <int KC, bool HIN, int S = 0, class Map, class LoadF>
__device__ __forceinline__ void dif_head_c(const FftPlan1D& pl, const Map& map, int nl, float2* buf,
                                           float2* tw, int tid, LoadF load, bool fill) {
  using Len = StaticLen<KC>;
  if constexpr (S < Len::n - 1) {
    dif_stage<Len::L.r[S], S == 0, false, HIN, false, KC>(pl, Len{}, Int<S>{}, map, nl, buf, tw, tid, load, fill,
                                                               NoStore{});
    fft_barrier();
    dif_head_c<KC, HIN, S + 1>(pl, map, nl, buf, tw, tid, load, fill);
  }
}
template <int KC, class Map, class LoadF>
__device__ __forceinline__ void dif_head_d(const FftPlan1D& pl, const Map& map, int nl, float2* buf,
                                           float2* tw, int tid, LoadF load, bool fill) {
  if (fill) fill_twiddles<0>(tw, pl);
  {
    const DynLen len(pl, 0);
#define TKBN_CALL(R) \
  dif_stage<R, true, false, false, false, 0>(pl, len, 0, map, nl, buf, tw, tid, load, fill, NoStore{})
    TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
  }
  fft_barrier();
  for (int s = 1; s < pl.n - 1; ++s) {
    const DynLen len(pl, s);
#define TKBN_CALL(R) \
  dif_stage<R, false, false, false, false, 0>(pl, len, s, map, nl, buf, tw, tid, NoLoad{}, false, NoStore{})
    TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
    fft_barrier();
  }
}

// A whole forward transform of `nl` lines or columns: store(f, t, value, own LDS slot).
// fill: put the twiddles into LDS first (behind the first loads).
// KC > 0: compiled for length KC.
template <int KC, bool HIN, bool HOUT, class Map, class LoadF, class StoreF>
__device__ __forceinline__ void dif_fft(const FftPlan1D& pl, const Map& map, int nl, float2* buf,
                                        float2* tw, int tid, LoadF load, bool fill, StoreF store) {
  if constexpr (KC > 0) {
    using Len = StaticLen<KC>;
    dif_head_c<KC, HIN>(pl, map, nl, buf, tw, tid, load, fill);
    dif_stage<Len::L.r[Len::n - 1], false, true, false, HOUT, KC>(pl, Len{}, Int<Len::n - 1>{}, map, nl, buf, tw,
                                                                      tid, NoLoad{}, false, store);
  } else {
    dif_head_d<KC>(pl, map, nl, buf, tw, tid, load, fill);
    const int s = pl.n - 1;
    const DynLen len(pl, s);
#define TKBN_CALL(R) \
  dif_stage<R, false, true, false, false, 0>(pl, len, s, map, nl, buf, tw, tid, NoLoad{}, false, store)
    TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
  }
}

// A transform, mid.value(mid.read(f, t), value) of every result, and a second transform of those:
// store(k, t, value).
template <int KC, bool HOUT, int S, class Map, class StoreF>
__device__ __forceinline__ void dit_tail_c(const Map& map, int nl, float2* buf, const float2* tw, int tid,
                                           StoreF store) {
  using Len = StaticLen<KC>;
  const NoMid none{};
  fft_barrier();
  dit_stage<Len::L.r[S], false, S == 0, HOUT>(Len{}, Int<S>{}, map, nl, buf, tw, tid, none, store);
  if constexpr (S > 0) dit_tail_c<KC, HOUT, S - 1>(map, nl, buf, tw, tid, store);
}
template <int KC, bool HIN, bool HOUT, class Map, class LoadF, class MidF, class StoreF>
__device__ __forceinline__ void dif_dit(const FftPlan1D& pl, const Map& map, int nl, float2* buf,
                                        float2* tw, int tid, LoadF load, bool fill, MidF mid, StoreF store) {
  const auto drop = [](int, int, float2) {};
  const NoMid none{};
  if constexpr (KC > 0) {
    using Len = StaticLen<KC>;
    dif_head_c<KC, HIN>(pl, map, nl, buf, tw, tid, load, fill);
    dit_stage<Len::L.r[Len::n - 1], true, false, false>(Len{}, Int<Len::n - 1>{}, map, nl, buf, tw, tid, mid, drop);
    dit_tail_c<KC, HOUT, Len::n - 2>(map, nl, buf, tw, tid, store);
  } else {
    dif_head_d<KC>(pl, map, nl, buf, tw, tid, load, fill);
    {
      const DynLen len(pl, pl.n - 1);
#define TKBN_CALL(R) dit_stage<R, true, false, false>(len, pl.n - 1, map, nl, buf, tw, tid, mid, drop)
      TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
    }
    for (int s = pl.n - 2; s > 0; --s) {
      fft_barrier();
      const DynLen len(pl, s);
#define TKBN_CALL(R) dit_stage<R, false, false, false>(len, s, map, nl, buf, tw, tid, none, drop)
      TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
    }
    fft_barrier();
    const DynLen len(pl, 0);
#define TKBN_CALL(R) dit_stage<R, false, true, false>(len, 0, map, nl, buf, tw, tid, none, store)
    TKBN_FOR_RADIX(len.r, TKBN_CALL)
#undef TKBN_CALL
  }
}

// ---------------------------------------------------------------------------
// geometry of the passes
// ---------------------------------------------------------------------------
struct FftGeom {
  int ndim;
  int N[3];         // image size
  int K[3];         // grid size
  int64_t B, C;     // batch, coils
  int image_coils;  // forward: coils of the image (1 with smaps, else C)
  int out_coils;    // adjoint: 1 with smaps (combined), else C
  float scale;
  FastDiv fQ, fC;  // lines per (b, c), coils
};
struct FftPlans {
  FftPlan1D d[3];
  int chirp_m[3];  // convolution length of a dimension whose extent has no plan, else 0
};

constexpr int kFftMaxThreads = 1024;
constexpr int kFftLdsBudget = 60 * 1024;  // largest group (twiddles + transforms)
constexpr int kFftLdsGoal = 50 * 1024;    // three groups per CU
constexpr int kFftMaxLines = 16;          // transforms per group

// LDS of a group with nl transforms of length K
constexpr int64_t fft_lds_bytes(int K, int64_t nl) {
  const RadixList L = radix_list(K);
  return (twiddles_of(L, K) + nl * (K + L.r[0])) * 8;
}
// log2 of the columns per group: 16 or 8 (128 or 64 B of a row), fewer only where LDS holds
// no more
constexpr int cols_log2(int K) {
  int lg = 4;
  while (lg > 3 && fft_lds_bytes(K, 1 << lg) > kFftLdsGoal) --lg;
  while (lg > 0 && fft_lds_bytes(K, 1 << lg) > kFftLdsBudget) --lg;
  return lg;
}

// ---------------------------------------------------------------------------
// last-dimension pass (contiguous lines).  One group: `lpg` lines.
//   MODE 0: forward first pass, input = image * smaps * scaling * scale (n < N), zero pad
// (scaling == NULL: unit apodisation, used by the FFT filter)
//   MODE 1: adjoint last pass, output = sum_c crop * conj(scaling) * scale * conj(smaps_c)
//   MODE 2: adjoint last pass without smaps, output = crop * conj(scaling) * scale per coil
// In MODE 0 and 2 lines run over (b, c, n_0..n_{d-2}); MODE 0 writes the extents
// (N_0..N_{d-2}, K_{d-1}).  In MODE 1 lines run over (b, n_0..n_{d-2}) of the image, one per
// group, which loops over the coils, `lpg` at a time.
// ---------------------------------------------------------------------------
// Values of image * smaps * scaling * scale along the lines (b, c, q) from line0 on.
struct ImageLoad {
  const FftGeom& g;
  const float2 *src, *smaps, *scaling;
  int64_t line0, Q, P;
  int N;
  struct Raw {
    float2 v, sm, sc;
  };
  __device__ __forceinline__ Raw read(int k, int t) const {
    const uint32_t line = (uint32_t)(line0 + t);  // < 2^31 (checked on the host)
    const uint32_t bc = fdiv(line, g.fQ);
    const int64_t n = (int64_t)(line - bc * (uint32_t)Q) * N + (k < N ? k : 0);
    const int64_t ib = g.image_coils == 1 ? (int64_t)fdiv(bc, g.fC) : (int64_t)bc;
    // absent operands read the image in their place, so that no branch parts the loads
    Raw r;
    const float2* im = src + ib * P + n;
    const float2* sm = smaps ? smaps + (int64_t)bc * P + n : im;
    const float2* sc = scaling ? scaling + n : im;
    r.v = *im;
    r.sm = *sm;
    r.sc = *sc;
    return r;
  }
  __device__ __forceinline__ float2 value(const Raw& r, int k, int) const {
    if (k >= N) return make_float2(0.f, 0.f);
    float2 v = r.v;
    if (smaps) v = cmul(v, r.sm);
    if (scaling) v = cmul(v, r.sc);
    v.x *= g.scale;
    v.y *= g.scale;
    return v;
  }
};

// The runtime form of MODE 0 holds up to three operands of 16 values: 512 threads leave it
// the registers.
constexpr int last_max_threads(int mode, int kc) { return mode == 0 && kc <= 0 ? 512 : kFftMaxThreads; }
// KC > 0: the last grid extent is KC and 2 N <= KC (compiled passes, halved first or last stage).
template <int MODE, int KC>
__global__ void __launch_bounds__((last_max_threads(MODE, KC)))
    fft_last_kernel(const FftGeom g, const FftPlan1D pl, const float2* __restrict__ src, const float2* __restrict__ smaps,
                    const float2* __restrict__ scaling, float2* __restrict__ dst, int lpg) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int D = g.ndim;
  const int K = KC > 0 ? KC : pl.K, N = g.N[D - 1];
  const LdsMap<false> map{0, KC > 0 ? K + StaticLen<KC>::L.r[0] : K + pl.r[0]};
  float2* tw = reinterpret_cast<float2*>(smem);
  float2* buf = tw + pl.ntw;

  int64_t Q = 1;  // spatial lines of the image: prod N[0..D-2]
  for (int d = 0; d < D - 1; ++d) Q *= g.N[d];
  const int64_t P = Q * N;  // image elements per (b, c)

  if constexpr (MODE == 0) {
    const int64_t line0 = (int64_t)blockIdx.x * lpg;
    const int64_t nlines = g.B * g.C * Q;
    const int nl = (int)(line0 + lpg <= nlines ? lpg : nlines - line0);
    dif_fft<KC, true, false>(
        pl, map, nl, buf, tw, threadIdx.x,
        ImageLoad{g, src, smaps, scaling, line0, Q, P, N},
        true, [&](int f, int t, float2 v, int) { dst[(line0 + t) * K + f] = v; });
  } else if constexpr (MODE == 2) {
    const int64_t line0 = (int64_t)blockIdx.x * lpg;
    const int64_t nlines = g.B * g.C * Q;
    const int nl = (int)(line0 + lpg <= nlines ? lpg : nlines - line0);
    dif_fft<KC, false, true>(
        pl, map, nl, buf, tw, threadIdx.x, LineLoad{src + line0 * K, K},
        true,
        [&](int f, int t, float2 v, int) {
          if (f < N) {
            v = cswap(v);
            if (scaling) {
              const uint32_t line = (uint32_t)(line0 + t);
              const int64_t q = line - fdiv(line, g.fQ) * (uint32_t)Q;
              v = cmul_conj(v, scaling[q * N + f]);
            }
            v.x *= g.scale;
            v.y *= g.scale;
            dst[(line0 + t) * N + f] = v;
          }
        });
  } else {
    const int64_t line = blockIdx.x;
    const int64_t b = fdiv((uint32_t)line, g.fQ), q = line - b * Q;
    // the output n of this thread (the host launches at least N threads) and the LDS slot
    // where the last stage leaves it
    const int n = threadIdx.x;
    int slot;
    {
      const int nn = min(n, N - 1);
      int blk, d0 = 0, i;
      if constexpr (KC > 0) {
        using Len = StaticLen<KC>;
        constexpr int R = Len::L.r[Len::n - 1];
        i = Len::div_per(Int<Len::n - 1>{}, nn);
        Len::reverse(nn - i * Len::per(Int<Len::n - 1>{}), blk, d0);
        slot = blk * R + d0 + i;
      } else {
        const DynLen len(pl, pl.n - 1);
        i = len.div_per(pl.n - 1, nn);
        len.reverse(nn - i * len.per(pl.n - 1), blk, d0);
        slot = blk * len.r + d0 + i;
      }
    }
    float2 acc = make_float2(0.f, 0.f);
    for (int64_t c0 = 0; c0 < g.C; c0 += lpg) {
      const int nc = (int)(c0 + lpg <= g.C ? lpg : g.C - c0);
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));  // keeps the stages' index arithmetic inside the loop
      dif_fft<KC, false, true>(
          pl, map, nc, buf, tw, tid,
          LineLoad{src + ((b * g.C + c0) * Q + q) * K, Q * K},
          c0 == 0,
          // the product with the coil's map goes back to the butterfly's own LDS slot
          [&](int f, int t, float2 v, int own) {
            if (f < N) {
              const float2 sm = smaps[((b * g.C + c0 + t) * Q + q) * N + f];
              v = cswap(v);
              if (scaling) v = cmul_conj(v, scaling[q * N + f]);
              v.x *= g.scale;
              v.y *= g.scale;
              buf[own] = cmul_conj(v, sm);
            }
          });
      fft_barrier();
      if (n < N)
        for (int t = 0; t < nc; ++t) acc = cadd(acc, buf[map.at(t, slot)]);
      fft_barrier();  // the next coils overwrite the lines
    }
    if (n < N) dst[(b * Q + q) * N + n] = acc;
  }
}

// Work item of a column pass.  Groups are dealt to the 8 XCDs round-robin; each XCD takes a
// contiguous range of (row, column block) items instead, so neighbouring column blocks,
// which share cache lines, meet in one L2.  The grid is a multiple of 8: a bijection.
__device__ __forceinline__ int64_t xcd_contiguous_item() {
  const int64_t per_xcd = gridDim.x >> 3;
  return (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
}

// ---------------------------------------------------------------------------
// pass along dimension d < ndim-1 (strided).  The array is viewed as
// (rows = b*c*outer, len, inner) with len = n_in (input) / n_out (output) and inner
// the product of the extents after d.  One group: 1 << lgc adjacent inner columns of one row.
// Forward: n_in = N[d] zero-padded to K; adjoint (INV): n_out = N[d] (crop).
// ---------------------------------------------------------------------------
// KC > 0: the length is KC and 2 N[d] <= KC.  KC = 0: `inv` says the direction.
template <bool INV, int KC>
__global__ void __launch_bounds__(kFftMaxThreads)
    fft_mid_kernel(const FftPlan1D pl, int64_t rows, int n_in, int n_out, int64_t inner, int lgc, int inv,
                   const float2* __restrict__ src, float2* __restrict__ dst) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const bool swap = KC > 0 ? INV : inv != 0;
  float2* tw = reinterpret_cast<float2*>(smem);
  float2* buf = tw + pl.ntw;
  const int lg = KC > 0 ? cols_log2(KC) : lgc;
  const int ncol = 1 << lg;
  const int64_t item = xcd_contiguous_item();
  const int64_t chunks = (inner + ncol - 1) >> lg;
  const int64_t row = item / chunks;
  const int64_t col0 = (item - row * chunks) << lg;
  if (row >= rows) return;
  const int nc = (int)(col0 + ncol <= inner ? ncol : inner - col0);
  const float2* s = src + row * (int64_t)n_in * inner + col0;
  float2* o = dst + row * (int64_t)n_out * inner + col0;
  dif_fft<KC, !INV, INV>(
      pl, LdsMap<true, (KC > 0 ? cols_log2(KC) : -1)>{lgc, 0}, ncol, buf, tw, threadIdx.x,
      ColLoad{s, inner, n_in, nc, swap},
      true,
      [&](int f, int t, float2 v, int) {
        if (f < n_out && t < nc) o[(int64_t)f * inner + t] = swap ? cswap(v) : v;
      });
}

// ---------------------------------------------------------------------------
// FFT filter along dimension 0 (the Toeplitz normal operator's middle): for a block
// of adjacent columns of one (b, c) row, zero-pad the n image rows to K, transform,
// multiply by the kernel (K x inner, one per batch item or shared), transform back
// and keep the first n rows, in place.  The padded grid never reaches memory, and the
// forward transform's last butterfly, the product and the inverse's first butterfly stay
// in registers.
// ---------------------------------------------------------------------------
// times the kernel's values, real and imaginary exchanged for the inverse
struct KernelMul {
  const float2* k;
  int64_t inner;
  int nc;
  __device__ __forceinline__ float2 read(int f, int t) const { return k[(int64_t)f * inner + (t < nc ? t : 0)]; }
  __device__ __forceinline__ float2 value(float2 m, float2 v) const { return cswap(cmul(v, m)); }
};
template <int KC>
__global__ void __launch_bounds__(kFftMaxThreads)
    fft_filter_kernel(const FftPlan1D pl, int64_t rows, int n, int64_t inner, int lgc,
                      const float2* __restrict__ kern, int64_t rows_per_kern, float2* data) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float2* tw = reinterpret_cast<float2*>(smem);
  float2* buf = tw + pl.ntw;
  const int ncol = 1 << (KC > 0 ? cols_log2(KC) : lgc);
  // the rows of one column block follow each other: they share the kernel's columns, which
  // an XCD's L2 then reads once (all of it per row otherwise: 3.3 MB at 640 x 640)
  const int64_t item = xcd_contiguous_item();
  const int64_t chunk = item / rows;
  const int64_t row = item - chunk * rows;
  const int64_t col0 = chunk * ncol;
  if (col0 >= inner) return;
  const int nc = (int)(col0 + ncol <= inner ? ncol : inner - col0);
  float2* d = data + row * (int64_t)n * inner + col0;
  const int64_t K = KC > 0 ? KC : pl.K;
  const float2* kr = kern + (rows_per_kern > 0 ? row / rows_per_kern : 0) * K * inner + col0;
  dif_dit<KC, true, true>(
      pl, LdsMap<true, (KC > 0 ? cols_log2(KC) : -1)>{lgc, 0}, ncol, buf, tw, threadIdx.x,
      ColLoad{d, inner, n, nc, false},
      true,
      KernelMul{kr, inner, nc},
      [&](int k, int t, float2 v) {
        if (k < n && t < nc) d[(int64_t)k * inner + t] = cswap(v);
      });
}

// ---------------------------------------------------------------------------
// A length K with a prime factor above 17, as a convolution (Bluestein, "A linear filtering approach to the
// computation of discrete Fourier transform", 1970): with c[n] = exp(-i pi n^2 / K),
//   X[k] = c[k] sum_n (x[n] c[n]) conj(c[k - n]),
// a circular convolution of length M >= n_in + n_out - 1, M one of the compiled lengths.  A
// group transforms its lines to length M, multiplies by the spectrum H of conj(c) and
// transforms back, all in LDS (dif_dit); the zero padding, the crop and the apodisation
// cost no pass of their own.  Bound as the passes above by LDS and memory together; the two
// transforms of 1.3 to 2 K values take about three times the LDS work of a smooth length.
// 39 images, 217 x 181 -> 434 x 362 (2 * 7 * 31 and 2 * 181; M = 768 and 576), forward and
// adjoint: row passes 28 and 24 us, column passes 42 and 43 us, chirps 7 us a call, against
// 219 us each way for the pad or crop kernel, rocFFT's own convolutions of the unpruned grid
// and its transposes.
// c and H are written by one small kernel of the same call (chirp_prep_kernel), evaluated in
// double and rounded once.
// ---------------------------------------------------------------------------
constexpr int kMaxChirpM = 1280;  // chirp_prep_kernel's LDS

struct ChirpDim {
  int K, M, n_in, n_out;
  float2 *c, *h;
};
struct ChirpDims {
  ChirpDim d[3];
};

// blockIdx.y: dimension.  A block sums 32 values of H, 32 threads each.
__global__ void __launch_bounds__(1024) chirp_prep_kernel(const ChirpDims dims) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ double2 part[32][33];
  const ChirpDim q = blockIdx.y == 0 ? dims.d[0] : blockIdx.y == 1 ? dims.d[1] : dims.d[2];
  const int f0 = blockIdx.x * 32;
  if (f0 >= q.M) return;
  double2* const w = reinterpret_cast<double2*>(smem);  // exp(-2 pi i p / M)
  double2* const h = w + q.M;                           // conj(c) around the circle
  const auto chirp = [&](int n) {  // exp(i pi n^2 / K)
    double s, c;
    sincospi((double)((int64_t)n * n % (2 * q.K)) / (double)q.K, &s, &c);
    return make_double2(c, s);
  };
  for (int p = threadIdx.x; p < q.M; p += blockDim.x) {
    double s, c;
    sincospi(2. * (double)p / (double)q.M, &s, &c);
    w[p] = make_double2(c, -s);
    h[p] = p < q.n_out ? chirp(p) : p > q.M - q.n_in ? chirp(q.M - p) : make_double2(0., 0.);
  }
  if (threadIdx.x < 32 && f0 + (int)threadIdx.x < q.K) {
    const double2 e = chirp(f0 + threadIdx.x);
    q.c[f0 + threadIdx.x] = make_float2((float)e.x, (float)-e.y);
  }
  __syncthreads();
  const int o = threadIdx.x & 31, r = threadIdx.x >> 5;
  const int f = f0 + o < q.M ? f0 + o : q.M - 1;
  int at = f * r % q.M;
  const int step = f * 32 % q.M;
  double2 sum = make_double2(0., 0.);
  for (int p = r; p < q.M; p += 32) {
    const double2 a = h[p], b = w[at];
    sum.x += a.x * b.x - a.y * b.y;
    sum.y += a.x * b.y + a.y * b.x;
    at += step;
    if (at >= q.M) at -= q.M;
  }
  part[r][o] = sum;
  __syncthreads();
  if (r == 0 && f0 + o < q.M) {
    for (int k = 1; k < 32; ++k) {
      sum.x += part[k][o].x;
      sum.y += part[k][o].y;
    }
    q.h[f] = make_float2((float)(sum.x / q.M), (float)(sum.y / q.M));
  }
}

// a source times the chirp
template <class Load>
struct ChirpLoad {
  Load l;
  const float2* c;
  int n;
  struct Raw {
    typename Load::Raw v;
    float2 c;
  };
  __device__ __forceinline__ Raw read(int k, int t) const {
    Raw r;
    r.v = l.read(k, t);
    r.c = c[k < n ? k : 0];
    return r;
  }
  __device__ __forceinline__ float2 value(const Raw& r, int k, int t) const { return cmul(l.value(r.v, k, t), r.c); }
};
// line t of consecutive lines of n values, real and imaginary exchanged, zeros past the end
struct PaddedLineLoad {
  const float2* s;
  int n;
  using Raw = float2;
  __device__ __forceinline__ Raw read(int k, int t) const { return s[(int64_t)t * n + (k < n ? k : 0)]; }
  __device__ __forceinline__ float2 value(Raw v, int k, int) const { return k < n ? cswap(v) : make_float2(0.f, 0.f); }
};
// times the spectrum, real and imaginary exchanged for the way back
struct SpectrumMul {
  const float2* h;
  __device__ __forceinline__ float2 read(int f, int) const { return h[f]; }
  __device__ __forceinline__ float2 value(float2 m, float2 v) const { return cswap(cmul(v, m)); }
};

// KC > 0: M = KC, of which the first half takes all inputs (forward) or outputs (inverse)
constexpr int chirp_max_threads(bool inv) { return inv ? kFftMaxThreads : 512; }
template <bool INV, int KC>
__global__ void __launch_bounds__((chirp_max_threads(INV)))
    chirp_last_kernel(const FftGeom g, const FftPlan1D pl, const ChirpDim cd, const float2* __restrict__ src,
                      const float2* __restrict__ smaps, const float2* __restrict__ scaling, float2* __restrict__ dst,
                      int lpg) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int D = g.ndim;
  const int M = KC > 0 ? KC : pl.K, N = g.N[D - 1], K = cd.K;
  const LdsMap<false> map{0, KC > 0 ? M + StaticLen<KC>::L.r[0] : M + pl.r[0]};
  float2* tw = reinterpret_cast<float2*>(smem);
  float2* buf = tw + pl.ntw;
  const float2* const c = cd.c;
  int64_t Q = 1;
  for (int d = 0; d < D - 1; ++d) Q *= g.N[d];
  const int64_t line0 = (int64_t)blockIdx.x * lpg;
  const int64_t nlines = g.B * g.C * Q;
  const int nl = (int)(line0 + lpg <= nlines ? lpg : nlines - line0);
  if constexpr (!INV) {
    dif_dit<KC, true, false>(
        pl, map, nl, buf, tw, threadIdx.x,
        ChirpLoad<ImageLoad>{ImageLoad{g, src, smaps, scaling, line0, Q, Q * N, N}, c, N}, true, SpectrumMul{cd.h},
        [&](int k, int t, float2 v) {
          if (k < K) dst[(line0 + t) * K + k] = cmul(cswap(v), c[k]);
        });
  } else {
    dif_dit<KC, false, true>(
        pl, map, nl, buf, tw, threadIdx.x, ChirpLoad<PaddedLineLoad>{PaddedLineLoad{src + line0 * K, K}, c, K}, true,
        SpectrumMul{cd.h}, [&](int k, int t, float2 v) {
          if (k < N) {
            v = cswap(cmul(cswap(v), c[k]));
            if (scaling) {
              const uint32_t line = (uint32_t)(line0 + t);
              const int64_t q = line - fdiv(line, g.fQ) * (uint32_t)Q;
              v = cmul_conj(v, scaling[q * N + k]);
            }
            v.x *= g.scale;
            v.y *= g.scale;
            dst[(line0 + t) * N + k] = v;
          }
        });
  }
}

template <bool INV, int KC>
__global__ void __launch_bounds__(kFftMaxThreads)
    chirp_mid_kernel(const FftPlan1D pl, const ChirpDim cd, int64_t rows, int64_t inner, int lgc,
                     const float2* __restrict__ src, float2* __restrict__ dst) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float2* tw = reinterpret_cast<float2*>(smem);
  float2* buf = tw + pl.ntw;
  const float2* const c = cd.c;
  const int lg = KC > 0 ? cols_log2(KC) : lgc;
  const int ncol = 1 << lg;
  const int64_t item = xcd_contiguous_item();
  const int64_t chunks = (inner + ncol - 1) >> lg;
  const int64_t row = item / chunks;
  const int64_t col0 = (item - row * chunks) << lg;
  if (row >= rows) return;
  const int nc = (int)(col0 + ncol <= inner ? ncol : inner - col0);
  const float2* s = src + row * (int64_t)cd.n_in * inner + col0;
  float2* o = dst + row * (int64_t)cd.n_out * inner + col0;
  const int n_out = cd.n_out;
  dif_dit<KC, !INV, INV>(
      pl, LdsMap<true, (KC > 0 ? cols_log2(KC) : -1)>{lgc, 0}, ncol, buf, tw, threadIdx.x,
      ChirpLoad<ColLoad>{ColLoad{s, inner, cd.n_in, nc, INV}, c, cd.n_in}, true, SpectrumMul{cd.h},
      [&](int k, int t, float2 v) {
        if (k < n_out && t < nc) {
          v = cmul(cswap(v), c[k]);
          o[(int64_t)k * inner + t] = INV ? cswap(v) : v;
        }
      });
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static bool smooth5(int64_t n) {
  for (int p : {2, 3, 5})
    while (n % p == 0) n /= p;
  return n == 1;
}

static bool factorize(int K, FftPlan1D* pl) {
  const RadixList L = radix_list(K);
  if (L.n == 0) return false;
  pl->K = K;
  pl->n = L.n;
  pl->ntw = 0;
  int ns = 1;
  for (int s = 0; s < L.n; ++s) {
    pl->r[s] = L.r[s];
    pl->Lb[s] = K / ns;
    pl->tw[s] = pl->ntw;
    if (s < L.n - 1) pl->ntw += K / ns;
    pl->nbs[s] = make_fastdiv((uint32_t)(K / ns / L.r[s]));
    pl->per[s] = make_fastdiv((uint32_t)(K / L.r[s]));
    pl->rd[s] = make_fastdiv((uint32_t)L.r[s]);
    pl->q1[s] = make_fastdiv((uint32_t)(s > 0 ? ns / L.r[0] : 1));
    ns *= L.r[s];
  }
  return true;
}

// threads of a group: one butterfly of the first stage each, as far as they go
static unsigned fft_threads(const FftPlan1D& pl, int64_t nl, int64_t at_least) {
  int64_t n = nl * (pl.K / pl.r[0]);
  n = n > at_least ? n : at_least;
  n = ceil_div(n, 64) * 64;
  return (unsigned)(n > kFftMaxThreads ? kFftMaxThreads : n);
}

// Transforms per group: as many as leave three groups per CU (a group alternates between
// memory and LDS, so the others fill its gaps), fewer when the launch would not give every
// CU two groups.
static int fft_lines(const FftPlan1D& pl, int64_t total) {
  int64_t n = kFftMaxLines;
  while (n > 1 && fft_lds_bytes(pl.K, n) > kFftLdsGoal) --n;
  while (n > 1 && ceil_div(total, n) < 512) n = (n + 1) / 2;
  return (int)n;
}
constexpr int kMaxK = 2048;

// Lengths of the convolutions: all but the last two are compiled.
#define TKBN_CHIRP_COMPILED_SIZES(X) X(192) X(256) X(320) X(384) X(480) X(576) X(640) X(768) X(1024)
static int chirp_length(int need) {
#define TKBN_CHIRP_FIT(M) \
  if (need <= M) return M;
  TKBN_CHIRP_COMPILED_SIZES(TKBN_CHIRP_FIT)
#undef TKBN_CHIRP_FIT
  return need <= 1152 ? 1152 : kMaxChirpM;
}

// `any`: extents may hold the primes 7 to 17 too (butterflies of those sizes in the runtime
// plan: a convolution was up to 1.6 times further from 64-bit values, 63^2 -> 126^2 adjoint
// 2.41e-7 against 1.51e-7), and any larger one (the convolution)
static int check_fft(int32_t ndim, const int64_t* im, const int64_t* gs, FftGeom* g, FftPlans* plans, bool any) {
  TKBN_REQUIRE(ndim >= 1 && ndim <= 3, TKBN_ERR_UNSUPPORTED, "ndim %d not in 1..3", ndim);
  TKBN_REQUIRE(im && gs, TKBN_ERR_INVALID, "NULL size array");
  g->ndim = ndim;
  for (int d = 0; d < 3; ++d) {
    g->N[d] = 1;
    g->K[d] = 1;
  }
  for (int d = 0; d < ndim; ++d) {
    TKBN_REQUIRE(im[d] >= 1 && gs[d] >= im[d], TKBN_ERR_INVALID, "dim %d: need 1 <= im_size <= grid_size", d);
    plans->chirp_m[d] = 0;
    TKBN_REQUIRE(any || (gs[d] <= kMaxK && smooth5(gs[d])), TKBN_ERR_UNSUPPORTED,
                 "grid size %lld is not a product of 2, 3, 5 up to %d", (long long)gs[d], kMaxK);
    if (!(gs[d] <= kMaxK && factorize((int)gs[d], &plans->d[d]))) {
      TKBN_REQUIRE(im[d] + gs[d] - 1 <= kMaxChirpM, TKBN_ERR_UNSUPPORTED,
                   "grid size %lld needs a convolution of more than %d values", (long long)gs[d], kMaxChirpM);
      plans->chirp_m[d] = chirp_length((int)(im[d] + gs[d] - 1));
      TKBN_REQUIRE(factorize(plans->chirp_m[d], &plans->d[d]), TKBN_ERR_UNSUPPORTED, "no convolution length");
    }
    g->N[d] = (int)im[d];
    g->K[d] = (int)gs[d];
  }
  // one thread of the coil-combining pass per output of a line
  TKBN_REQUIRE(g->N[ndim - 1] <= kFftMaxThreads, TKBN_ERR_UNSUPPORTED, "last image dim must be <= %d",
               kFftMaxThreads);
  return TKBN_OK;
}

// dividers of the last-dimension pass; the index arithmetic there is 32-bit
static int set_divs(FftGeom* g) {
  const int D = g->ndim;
  int64_t Q = 1;
  for (int d = 0; d < D - 1; ++d) Q *= g->N[d];
  TKBN_REQUIRE(g->B * g->C * Q < (1LL << 31) && g->B * g->C > 0, TKBN_ERR_UNSUPPORTED,
               "too many FFT lines (batch * coils * image lines must be < 2^31)");
  g->fQ = make_fastdiv((uint32_t)Q);
  g->fC = make_fastdiv((uint32_t)g->C);
  return TKBN_OK;
}

// Grid extents whose passes are compiled for their length (others use the runtime plan).
#define TKBN_FFT_COMPILED_SIZES(X) \
  X(128) X(160) X(192) X(256) X(288) X(320) X(384) X(400) X(480) X(512) X(576) X(640) X(768) X(1024)

// lines: (b, c, q) for MODE 0 and 2; MODE 1 has one group per (b, q), which loops over coils
template <int MODE>
static int launch_last(const FftGeom& g, const FftPlan1D& pl, const float2* src, const float2* smaps, const float2* scaling, float2* dst,
                       hipStream_t s) {
  const int D = g.ndim;
  int64_t Q = 1;
  for (int d = 0; d < D - 1; ++d) Q *= g.N[d];
  int lpg;
  int64_t groups;
  if (MODE == 1) {
    lpg = kFftMaxLines;
    while (lpg > 1 && (lpg > g.C || fft_lds_bytes(pl.K, lpg) > kFftLdsGoal)) --lpg;
    lpg = (int)ceil_div(g.C, ceil_div(g.C, lpg));  // rounds of equal size
    groups = g.B * Q;
  } else {
    lpg = fft_lines(pl, g.B * g.C * Q);
    groups = ceil_div(g.B * g.C * Q, lpg);
  }
  const int kc = !smooth5(pl.K) ? -1 : 2 * g.N[D - 1] <= pl.K ? pl.K : 0;  // compiled, if in the list below
  unsigned threads = fft_threads(pl, lpg, MODE == 1 ? g.N[D - 1] : 0);
  const size_t lds = (size_t)fft_lds_bytes(pl.K, lpg);
  const dim3 grid((unsigned)groups), block(threads);
  switch (kc) {
#define TKBN_LAST(KV)                                                                                  \
  case KV:                                                                                             \
    fft_last_kernel<MODE, KV><<<grid, block, lds, s>>>(g, pl, src, smaps, scaling, dst, lpg);              \
    break;
    TKBN_FFT_COMPILED_SIZES(TKBN_LAST)
#undef TKBN_LAST
    case -1:
      threads = threads < (unsigned)last_max_threads(MODE, -1) ? threads : (unsigned)last_max_threads(MODE, -1);
      fft_last_kernel<MODE, -1><<<grid, dim3(threads), lds, s>>>(g, pl, src, smaps, scaling, dst, lpg);
      break;
    default:
      threads = threads < (unsigned)last_max_threads(MODE, 0) ? threads : (unsigned)last_max_threads(MODE, 0);
      fft_last_kernel<MODE, 0><<<grid, dim3(threads), lds, s>>>(g, pl, src, smaps, scaling, dst, lpg);
  }
  TKBN_LAUNCH_CHECK("fft_last_kernel");
  return TKBN_OK;
}

static int launch_mid(bool inv, const FftPlan1D& pl, int64_t rows, int n_in, int n_out, int64_t inner,
                      const float2* src, float2* dst, hipStream_t s) {
  const int lgc = cols_log2(pl.K);
  const int64_t groups = ceil_div(rows * ceil_div(inner, 1 << lgc), 8) * 8;  // see xcd_contiguous_item
  TKBN_REQUIRE(groups < (1LL << 31), TKBN_ERR_INVALID, "too many FFT columns");
  const size_t lds = (size_t)fft_lds_bytes(pl.K, 1 << lgc);
  const dim3 grid((unsigned)groups), block(fft_threads(pl, 1 << lgc, 0));
  switch (!smooth5(pl.K) ? -1 : 2 * (inv ? n_out : n_in) <= pl.K ? pl.K : 0) {
#define TKBN_MID(KV)                                                                                            \
  case KV:                                                                                                      \
    if (inv)                                                                                                    \
      fft_mid_kernel<true, KV><<<grid, block, lds, s>>>(pl, rows, n_in, n_out, inner, lgc, 1, src, dst);        \
    else                                                                                                        \
      fft_mid_kernel<false, KV><<<grid, block, lds, s>>>(pl, rows, n_in, n_out, inner, lgc, 0, src, dst);       \
    break;
    TKBN_FFT_COMPILED_SIZES(TKBN_MID)
#undef TKBN_MID
    case -1:
      fft_mid_kernel<false, -1><<<grid, block, lds, s>>>(pl, rows, n_in, n_out, inner, lgc, inv ? 1 : 0, src, dst);
      break;
    default:
      fft_mid_kernel<false, 0><<<grid, block, lds, s>>>(pl, rows, n_in, n_out, inner, lgc, inv ? 1 : 0, src, dst);
  }
  TKBN_LAUNCH_CHECK("fft_mid_kernel");
  return TKBN_OK;
}

static int launch_filter(const FftPlan1D& pl, int64_t rows, int n, int64_t inner, const float2* kern,
                         int64_t rows_per_kern, float2* data, hipStream_t s) {
  const int lgc = cols_log2(pl.K);
  const int64_t groups = ceil_div(rows * ceil_div(inner, 1 << lgc), 8) * 8;
  TKBN_REQUIRE(groups < (1LL << 31), TKBN_ERR_INVALID, "too many FFT columns");
  const size_t lds = (size_t)fft_lds_bytes(pl.K, 1 << lgc);
  const dim3 grid((unsigned)groups), block(fft_threads(pl, 1 << lgc, 0));
  switch (2 * n <= pl.K ? pl.K : 0) {
#define TKBN_FILT(KV)                                                                                     \
  case KV:                                                                                                \
    fft_filter_kernel<KV><<<grid, block, lds, s>>>(pl, rows, n, inner, lgc, kern, rows_per_kern, data);   \
    break;
    TKBN_FFT_COMPILED_SIZES(TKBN_FILT)
#undef TKBN_FILT
    default:
      fft_filter_kernel<0><<<grid, block, lds, s>>>(pl, rows, n, inner, lgc, kern, rows_per_kern, data);
  }
  TKBN_LAUNCH_CHECK("fft_filter_kernel");
  return TKBN_OK;
}

// Lines of the last dimension: as many as fft_lines says of their convolutions.
template <bool INV>
static int launch_chirp_last(const FftGeom& g, const FftPlan1D& pl, const ChirpDim& cd, const float2* src,
                             const float2* smaps, const float2* scaling, float2* dst, hipStream_t s) {
  int64_t Q = 1;
  for (int d = 0; d < g.ndim - 1; ++d) Q *= g.N[d];
  const int lpg = fft_lines(pl, g.B * g.C * Q);
  unsigned threads = fft_threads(pl, lpg, 0);
  threads = threads < (unsigned)chirp_max_threads(INV) ? threads : (unsigned)chirp_max_threads(INV);
  const size_t lds = (size_t)fft_lds_bytes(pl.K, lpg);
  const dim3 grid((unsigned)ceil_div(g.B * g.C * Q, lpg)), block(threads);
  switch (cd.M) {
#define TKBN_CHIRP(MV)                                                                                       \
  case MV: chirp_last_kernel<INV, MV><<<grid, block, lds, s>>>(g, pl, cd, src, smaps, scaling, dst, lpg); break;
    TKBN_CHIRP_COMPILED_SIZES(TKBN_CHIRP)
#undef TKBN_CHIRP
    default: chirp_last_kernel<INV, 0><<<grid, block, lds, s>>>(g, pl, cd, src, smaps, scaling, dst, lpg);
  }
  TKBN_LAUNCH_CHECK("chirp_last_kernel");
  return TKBN_OK;
}

template <bool INV>
static int launch_chirp_mid(const FftPlan1D& pl, const ChirpDim& cd, int64_t rows, int64_t inner, const float2* src,
                            float2* dst, hipStream_t s) {
  const int lgc = cols_log2(pl.K);
  const int64_t groups = ceil_div(rows * ceil_div(inner, 1 << lgc), 8) * 8;  // see xcd_contiguous_item
  TKBN_REQUIRE(groups < (1LL << 31), TKBN_ERR_INVALID, "too many FFT columns");
  const size_t lds = (size_t)fft_lds_bytes(pl.K, 1 << lgc);
  const dim3 grid((unsigned)groups), block(fft_threads(pl, 1 << lgc, 0));
  switch (cd.M) {
#define TKBN_CHIRP(MV) \
  case MV: chirp_mid_kernel<INV, MV><<<grid, block, lds, s>>>(pl, cd, rows, inner, lgc, src, dst); break;
    TKBN_CHIRP_COMPILED_SIZES(TKBN_CHIRP)
#undef TKBN_CHIRP
    default: chirp_mid_kernel<INV, 0><<<grid, block, lds, s>>>(pl, cd, rows, inner, lgc, src, dst);
  }
  TKBN_LAUNCH_CHECK("chirp_mid_kernel");
  return TKBN_OK;
}

// elements of the chirps and spectra
static int64_t chirp_elements(const FftGeom& g, const FftPlans& plans) {
  int64_t n = 0;
  for (int d = 0; d < g.ndim; ++d)
    if (plans.chirp_m[d]) n += g.K[d] + plans.chirp_m[d];
  return n;
}
// lays them out at `p` and fills them
static int launch_chirp_prep(const FftGeom& g, const FftPlans& plans, bool inv, float2* p, ChirpDim (&cd)[3],
                             hipStream_t s) {
  ChirpDims dims{};
  int n = 0, mmax = 0;
  for (int d = 0; d < g.ndim; ++d) {
    const int M = plans.chirp_m[d];
    if (!M) continue;
    cd[d] = ChirpDim{g.K[d], M, inv ? g.K[d] : g.N[d], inv ? g.N[d] : g.K[d], p, p + g.K[d]};
    p += g.K[d] + M;
    dims.d[n++] = cd[d];
    mmax = M > mmax ? M : mmax;
  }
  if (n == 0) return TKBN_OK;
  chirp_prep_kernel<<<dim3((unsigned)ceil_div(mmax, 32), (unsigned)n), dim3(1024), (size_t)mmax * 32, s>>>(dims);
  TKBN_LAUNCH_CHECK("chirp_prep_kernel");
  return TKBN_OK;
}

// elements of the intermediate after the last-dim pass (forward) / before it (adjoint),
// and after/before each middle pass; ws holds two ping-pong buffers
static void ws_sizes(const FftGeom& g, int64_t* a, int64_t* b) {
  const int D = g.ndim;
  const int64_t BC = g.B * g.C;
  // forward sequence: [N0..N_{D-2}, K_{D-1}] -> [.., K_{D-2}, K_{D-1}] -> ... final = grid
  int64_t sz[3] = {0, 0, 0};
  int e[3];
  for (int d = 0; d < D; ++d) e[d] = g.N[d];
  e[D - 1] = g.K[D - 1];
  int idx = 0;
  for (int d = D - 1; d >= 1; --d) {  // arrays that are not the final grid
    int64_t n = BC;
    for (int k = 0; k < D; ++k) n *= e[k];
    sz[idx++] = n;
    e[d - 1] = g.K[d - 1];
  }
  *a = idx > 0 ? sz[0] : 0;
  *b = idx > 1 ? sz[1] : 0;
}

static int fft_supported(int32_t ndim, const int64_t* im_size, const int64_t* grid_size, bool any) {
  FftGeom g;
  FftPlans plans;
  return check_fft(ndim, im_size, grid_size, &g, &plans, any);
}

static int64_t fft_workspace_bytes(int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                                   int64_t coils, bool any) {
  FftGeom g;
  FftPlans plans;
  if (check_fft(ndim, im_size, grid_size, &g, &plans, any) != TKBN_OK) return -1;
  g.B = batch;
  g.C = coils;
  int64_t a, b;
  ws_sizes(g, &a, &b);
  return (a + b + chirp_elements(g, plans)) * 8 + 256;
}

static int fft_grid_fwd(bool any, int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, int64_t image_coils, const void* image, const void* smaps,
                      const void* scaling_coef, double scale, void* grid, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  FftGeom g;
  FftPlans plans;
  TKBN_REQUIRE(dtype == TKBN_F32, TKBN_ERR_UNSUPPORTED, "fused FFT is complex64 only");
  int st = check_fft(ndim, im_size, grid_size, &g, &plans, any);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(batch >= 0 && coils >= 0, TKBN_ERR_INVALID, "negative batch/coils");
  TKBN_REQUIRE(image_coils == 1 || image_coils == coils, TKBN_ERR_INVALID, "image_coils must be 1 or coils");
  TKBN_REQUIRE(smaps != nullptr || image_coils == coils, TKBN_ERR_INVALID, "without smaps image_coils must equal coils");
  if (batch == 0 || coils == 0) return TKBN_OK;
  TKBN_REQUIRE(image && scaling_coef && grid, TKBN_ERR_INVALID, "NULL data pointer");
  g.B = batch;
  g.C = coils;
  g.image_coils = (int)image_coils;
  g.out_coils = (int)coils;
  g.scale = (float)scale;
  st = set_divs(&g);
  if (st != TKBN_OK) return st;
  int64_t wa, wb;
  ws_sizes(g, &wa, &wb);
  const int64_t need = (wa + wb + chirp_elements(g, plans)) * 8;
  TKBN_REQUIRE(workspace_bytes >= need && (need == 0 || workspace), TKBN_ERR_WORKSPACE,
               "workspace of %lld bytes needed", (long long)need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int D = ndim;
  float2* bufa = static_cast<float2*>(workspace);
  float2* bufb = bufa + wa;
  ChirpDim cd[3];
  st = launch_chirp_prep(g, plans, false, bufb + wb, cd, s);
  if (st != TKBN_OK) return st;
  // pass 1: last dimension with fused apodisation / SENSE / zero-pad
  const float2 *im = static_cast<const float2*>(image), *sm = static_cast<const float2*>(smaps),
               *sc = static_cast<const float2*>(scaling_coef);
  float2* first = D == 1 ? static_cast<float2*>(grid) : bufa;
  st = plans.chirp_m[D - 1] ? launch_chirp_last<false>(g, plans.d[D - 1], cd[D - 1], im, sm, sc, first, s)
                            : launch_last<0>(g, plans.d[D - 1], im, sm, sc, first, s);
  if (st != TKBN_OK) return st;
  // remaining dimensions, innermost first
  int e[3];
  for (int d = 0; d < D; ++d) e[d] = g.N[d];
  e[D - 1] = g.K[D - 1];
  float2* cur = bufa;
  for (int d = D - 2; d >= 0; --d) {
    int64_t outer = g.B * g.C, inner = 1;
    for (int k = 0; k < d; ++k) outer *= e[k];
    for (int k = d + 1; k < D; ++k) inner *= e[k];
    float2* out = d == 0 ? static_cast<float2*>(grid) : (cur == bufa ? bufb : bufa);
    st = plans.chirp_m[d] ? launch_chirp_mid<false>(plans.d[d], cd[d], outer, inner, cur, out, s)
                          : launch_mid(false, plans.d[d], outer, g.N[d], g.K[d], inner, cur, out, s);
    if (st != TKBN_OK) return st;
    e[d] = g.K[d];
    cur = out;
  }
  return TKBN_OK;
}

static int fft_grid_adj(bool any, int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, const void* grid, const void* smaps, const void* scaling_coef, double scale,
                      void* image, void* workspace, int64_t workspace_bytes, void* stream) {
  FftGeom g;
  FftPlans plans;
  TKBN_REQUIRE(dtype == TKBN_F32, TKBN_ERR_UNSUPPORTED, "fused FFT is complex64 only");
  int st = check_fft(ndim, im_size, grid_size, &g, &plans, any);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(batch >= 0 && coils >= 0, TKBN_ERR_INVALID, "negative batch/coils");
  if (batch == 0 || coils == 0) return TKBN_OK;
  TKBN_REQUIRE(grid && (any || scaling_coef) && image, TKBN_ERR_INVALID, "NULL data pointer");
  g.B = batch;
  g.C = coils;
  g.image_coils = (int)coils;
  g.out_coils = smaps ? 1 : (int)coils;
  g.scale = (float)scale;
  st = set_divs(&g);
  if (st != TKBN_OK) return st;
  int64_t wa, wb;
  ws_sizes(g, &wa, &wb);
  const int64_t need = (wa + wb + chirp_elements(g, plans)) * 8;
  TKBN_REQUIRE(workspace_bytes >= need && (need == 0 || workspace), TKBN_ERR_WORKSPACE,
               "workspace of %lld bytes needed", (long long)need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int D = ndim;
  float2* bufa = static_cast<float2*>(workspace);
  float2* bufb = bufa + wa;
  TKBN_REQUIRE(!(smaps && plans.chirp_m[D - 1]), TKBN_ERR_UNSUPPORTED,
               "coil maps need a last grid size without prime factors above 17");
  ChirpDim cd[3];
  st = launch_chirp_prep(g, plans, true, bufb + wb, cd, s);
  if (st != TKBN_OK) return st;
  // outer dimensions first (inverse, cropping), mirror of the forward sequence
  int e[3];
  for (int d = 0; d < D; ++d) e[d] = g.K[d];
  const float2* cur = static_cast<const float2*>(grid);
  // the forward wrote bufa after the last-dim pass; the adjoint ends reading bufa
  for (int d = 0; d <= D - 2; ++d) {
    int64_t outer = g.B * g.C, inner = 1;
    for (int k = 0; k < d; ++k) outer *= e[k];
    for (int k = d + 1; k < D; ++k) inner *= e[k];
    // choose the buffer so that the last middle pass lands in bufa
    const int remaining = (D - 2) - d;  // passes after this one
    float2* out = (remaining % 2 == 0) ? bufa : bufb;
    st = plans.chirp_m[d] ? launch_chirp_mid<true>(plans.d[d], cd[d], outer, inner, cur, out, s)
                          : launch_mid(true, plans.d[d], outer, g.K[d], g.N[d], inner, cur, out, s);
    if (st != TKBN_OK) return st;
    e[d] = g.N[d];
    cur = out;
  }
  if (smaps)
    return launch_last<1>(g, plans.d[D - 1], cur, static_cast<const float2*>(smaps), static_cast<const float2*>(scaling_coef),
                          static_cast<float2*>(image), s);
  if (plans.chirp_m[D - 1])
    return launch_chirp_last<true>(g, plans.d[D - 1], cd[D - 1], cur, nullptr, static_cast<const float2*>(scaling_coef),
                                   static_cast<float2*>(image), s);
  return launch_last<2>(g, plans.d[D - 1], cur, nullptr, static_cast<const float2*>(scaling_coef), static_cast<float2*>(image), s);
}

}  // namespace tkbn

using namespace tkbn;

extern "C" {

int tkbn_fft_supported(int32_t ndim, const int64_t* im_size, const int64_t* grid_size) {
  return fft_supported(ndim, im_size, grid_size, false);
}
int tkbn_fft_any_supported(int32_t ndim, const int64_t* im_size, const int64_t* grid_size) {
  return fft_supported(ndim, im_size, grid_size, true);
}
int64_t tkbn_fft_workspace_bytes(int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                                 int64_t coils) {
  return fft_workspace_bytes(ndim, im_size, grid_size, batch, coils, false);
}
int64_t tkbn_fft_any_workspace_bytes(int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                                     int64_t coils) {
  return fft_workspace_bytes(ndim, im_size, grid_size, batch, coils, true);
}
int tkbn_fft_grid_fwd(int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, int64_t image_coils, const void* image, const void* smaps,
                      const void* scaling_coef, double scale, void* grid, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  return fft_grid_fwd(false, dtype, ndim, im_size, grid_size, batch, coils, image_coils, image, smaps, scaling_coef, scale,
                      grid, workspace, workspace_bytes, stream);
}
int tkbn_fft_grid_adj(int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, const void* grid, const void* smaps, const void* scaling_coef, double scale,
                      void* image, void* workspace, int64_t workspace_bytes, void* stream) {
  return fft_grid_adj(false, dtype, ndim, im_size, grid_size, batch, coils, grid, smaps, scaling_coef, scale, image,
                      workspace, workspace_bytes, stream);
}
int tkbn_fft_any_grid_fwd(int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, int64_t image_coils, const void* image, const void* smaps,
                      const void* scaling_coef, double scale, void* grid, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  return fft_grid_fwd(true, dtype, ndim, im_size, grid_size, batch, coils, image_coils, image, smaps, scaling_coef, scale,
                      grid, workspace, workspace_bytes, stream);
}
int tkbn_fft_any_grid_adj(int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                      int64_t coils, const void* grid, const void* smaps, const void* scaling_coef, double scale,
                      void* image, void* workspace, int64_t workspace_bytes, void* stream) {
  return fft_grid_adj(true, dtype, ndim, im_size, grid_size, batch, coils, grid, smaps, scaling_coef, scale, image,
                      workspace, workspace_bytes, stream);
}

int tkbn_fft_filter(int32_t dtype, int32_t ndim, const int64_t* im_size, const int64_t* grid_size, int64_t batch,
                    int64_t coils, int64_t image_coils, const void* image, const void* smaps, const void* kernel,
                    int32_t kernel_batched, double scale_fwd, double scale_adj, void* out, void* workspace,
                    int64_t workspace_bytes, void* stream) {
  FftGeom g;
  FftPlans plans;
  TKBN_REQUIRE(dtype == TKBN_F32, TKBN_ERR_UNSUPPORTED, "fused FFT is complex64 only");
  int st = check_fft(ndim, im_size, grid_size, &g, &plans, false);
  if (st != TKBN_OK) return st;
  TKBN_REQUIRE(ndim >= 2, TKBN_ERR_UNSUPPORTED, "the fused FFT filter needs at least two dimensions");
  TKBN_REQUIRE(batch >= 0 && coils >= 0, TKBN_ERR_INVALID, "negative batch/coils");
  TKBN_REQUIRE(image_coils == 1 || image_coils == coils, TKBN_ERR_INVALID, "image_coils must be 1 or coils");
  TKBN_REQUIRE(smaps != nullptr || image_coils == coils, TKBN_ERR_INVALID, "without smaps image_coils must equal coils");
  if (batch == 0 || coils == 0) return TKBN_OK;
  TKBN_REQUIRE(image && kernel && out, TKBN_ERR_INVALID, "NULL data pointer");
  g.B = batch;
  g.C = coils;
  g.image_coils = (int)image_coils;
  g.out_coils = smaps ? 1 : (int)coils;
  st = set_divs(&g);
  if (st != TKBN_OK) return st;
  int64_t wa, wb;
  ws_sizes(g, &wa, &wb);
  TKBN_REQUIRE(workspace_bytes >= (wa + wb) * 8 && (wa + wb == 0 || workspace), TKBN_ERR_WORKSPACE,
               "workspace of %lld bytes needed", (long long)((wa + wb) * 8));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int D = ndim;
  float2* bufa = static_cast<float2*>(workspace);
  float2* bufb = bufa + wa;
  // forward: last dimension (SENSE expansion, zero pad, scale_fwd), then dimensions
  // D-2 .. 1 zero-padded; dimension 0 is transformed, filtered and transformed back
  // in place; then dimensions 1 .. D-2 and the last one inverse with crop and coil
  // combine (scale_adj)
  g.scale = (float)scale_fwd;
  st = launch_last<0>(g, plans.d[D - 1], static_cast<const float2*>(image), static_cast<const float2*>(smaps), nullptr, bufa, s);
  if (st != TKBN_OK) return st;
  int e[3];
  for (int d = 0; d < D; ++d) e[d] = g.N[d];
  e[D - 1] = g.K[D - 1];
  float2* cur = bufa;
  for (int d = D - 2; d >= 1; --d) {
    int64_t outer = g.B * g.C, inner = 1;
    for (int k = 0; k < d; ++k) outer *= e[k];
    for (int k = d + 1; k < D; ++k) inner *= e[k];
    float2* nxt = cur == bufa ? bufb : bufa;
    st = launch_mid(false, plans.d[d], outer, g.N[d], g.K[d], inner, cur, nxt, s);
    if (st != TKBN_OK) return st;
    e[d] = g.K[d];
    cur = nxt;
  }
  {
    int64_t inner = 1;
    for (int k = 1; k < D; ++k) inner *= e[k];
    st = launch_filter(plans.d[0], g.B * g.C, g.N[0], inner, static_cast<const float2*>(kernel),
                       kernel_batched ? g.C : 0, cur, s);
    if (st != TKBN_OK) return st;
  }
  for (int d = 1; d <= D - 2; ++d) {
    int64_t outer = g.B * g.C, inner = 1;
    for (int k = 0; k < d; ++k) outer *= e[k];
    for (int k = d + 1; k < D; ++k) inner *= e[k];
    float2* nxt = cur == bufa ? bufb : bufa;
    st = launch_mid(true, plans.d[d], outer, g.K[d], g.N[d], inner, cur, nxt, s);
    if (st != TKBN_OK) return st;
    e[d] = g.N[d];
    cur = nxt;
  }
  g.scale = (float)scale_adj;
  if (smaps)
    return launch_last<1>(g, plans.d[D - 1], cur, static_cast<const float2*>(smaps), nullptr, static_cast<float2*>(out), s);
  return launch_last<2>(g, plans.d[D - 1], cur, nullptr, nullptr, static_cast<float2*>(out), s);
}

}  // extern "C"
