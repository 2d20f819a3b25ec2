// Device and host parts that the FFT passes share (gfx950): the LDS transforms
// of P pencils of any length, the block maps of row and strided passes, and
// the plans that size their workgroups.  Passes: pmx_fft.hip, pmx_lpt.hip.
#pragma once
#include "pmx_internal.h"

#define FFT_CAP 8192                 // complex values per strided workgroup, fixed lengths
#define PFFT_CAP 4096                // Poisson x pass (8 columns of 512, three 40 KB workgroups
                                     // per CU; 16 columns measured slower)
#define RFFT_CAP 4096                // row passes
// Kernels for lengths known only at run time: up to 512 threads of eight
// values (gen_tpb); their TPB argument is 0, the launch's own block size.
// With 16 values a thread the stages' addresses and twiddles spilled.
#define GEN_CAP 4096
#define GEN_MAXV 8
#define GEN_TPB 0
#define GEN_MAXTPB (GEN_CAP / GEN_MAXV)

template <int TPB>
__device__ __forceinline__ int tpb() {
  return TPB ? TPB : (int)blockDim.x;
}

// Complex products inside the transforms may fuse into FMAs (the file is
// otherwise built with separate roundings).
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
#pragma clang fp contract(fast)
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a w (DIR < 0) or a conj(w) (DIR > 0)
template <int DIR>
__device__ __forceinline__ float2 cmul_dir(float2 a, float2 w) {
#pragma clang fp contract(fast)
  return DIR < 0 ? make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x)
                 : make_float2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// multiply by -i (forward, DIR<0) or +i (inverse)
template <int DIR>
__device__ __forceinline__ float2 mul_mi(float2 a) {
  return DIR < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

template <int DIR>
__device__ __forceinline__ float2 twiddle(const float2* __restrict__ tw, int m) {
  float2 w = tw[m];
  if (DIR > 0) w.y = -w.y;
  return w;
}

template <int DIR>
__device__ __forceinline__ void dft2(float2* v) {
  float2 a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <int DIR>
__device__ __forceinline__ void dft4(float2* v) {
  float2 t0 = cadd(v[0], v[2]);
  float2 t1 = csub(v[0], v[2]);
  float2 t2 = cadd(v[1], v[3]);
  float2 t3 = mul_mi<DIR>(csub(v[1], v[3]));
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3);
  v[3] = csub(t1, t3);
}

template <int DIR>
__device__ __forceinline__ void dft8(float2* v) {
  const float h = 0.70710678118654752440f;
  float2 e[4] = {v[0], v[2], v[4], v[6]};
  float2 o[4] = {v[1], v[3], v[5], v[7]};
  dft4<DIR>(e);
  dft4<DIR>(o);
  // w8^q for q = 0..3 with w8 = exp(DIR * i pi/4)
  float2 o1 = DIR < 0 ? make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x))
                      : make_float2(h * (o[1].x - o[1].y), h * (o[1].y + o[1].x));
  float2 o2 = mul_mi<DIR>(o[2]);
  float2 o3 = DIR < 0 ? make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y))
                      : make_float2(-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y));
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}

// Odd radices: with a_q = v_q + v_{R-q}, b_q = v_q - v_{R-q} for q = 1..(R-1)/2,
// X_r and X_{R-r} = v_0 + sum_q cos(2 pi q r / R) a_q -+ i sum_q sin(2 pi q r / R) b_q
// (exp(-2 pi i q r / R) forward).
template <int R>
struct OddTab;
template <>
struct OddTab<3> {
  static constexpr float c[1] = {-0.4999999999999998f};
  static constexpr float s[1] = {0.8660254037844387f};
};
template <>
struct OddTab<5> {
  static constexpr float c[2] = {0.30901699437494745f, -0.8090169943749473f};
  static constexpr float s[2] = {0.9510565162951535f, 0.5877852522924732f};
};
template <>
struct OddTab<7> {
  static constexpr float c[3] = {0.6234898018587336f, -0.22252093395631434f, -0.900968867902419f};
  static constexpr float s[3] = {0.7818314824680298f, 0.9749279121818236f, 0.43388373911755823f};
};

template <int R, int DIR>
__device__ __forceinline__ void dft_odd(float2* v) {
#pragma clang fp contract(fast)
  constexpr int K = (R - 1) / 2;
  float2 a[K], b[K];
  const float2 x0 = v[0];
  float2 sum = x0;
#pragma unroll
  for (int q = 1; q <= K; ++q) {
    a[q - 1] = cadd(v[q], v[R - q]);
    b[q - 1] = csub(v[q], v[R - q]);
    sum = cadd(sum, a[q - 1]);
  }
  v[0] = sum;
#pragma unroll
  for (int r = 1; r <= K; ++r) {
    float2 m = x0, d = make_float2(0.f, 0.f);
#pragma unroll
    for (int q = 1; q <= K; ++q) {
      const int t = (q * r) % R;
      const float c = t <= K ? OddTab<R>::c[t - 1] : OddTab<R>::c[R - t - 1];
      const float e = t <= K ? OddTab<R>::s[t - 1] : -OddTab<R>::s[R - t - 1];
      m.x += c * a[q - 1].x;
      m.y += c * a[q - 1].y;
      d.x += e * b[q - 1].x;
      d.y += e * b[q - 1].y;
    }
    d = mul_mi<DIR>(d);
    v[r] = cadd(m, d);
    v[R - r] = csub(m, d);
  }
}

// Radix 2 N with N odd (Good-Thomas): input N n1 + 2 n2 mod 2N, output
// N k1 + (N + 1) k2 mod 2N, no twiddles.
template <int N, int DIR>
__device__ __forceinline__ void dft_2odd(float2* v) {
  float2 e[N], o[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    e[i] = cadd(v[(2 * i) % (2 * N)], v[(N + 2 * i) % (2 * N)]);
    o[i] = csub(v[(2 * i) % (2 * N)], v[(N + 2 * i) % (2 * N)]);
  }
  dft_odd<N, DIR>(e);
  dft_odd<N, DIR>(o);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    v[((N + 1) * k) % (2 * N)] = e[k];
    v[(N + (N + 1) * k) % (2 * N)] = o[k];
  }
}

// Radix 9 as 3 x 3.
template <int DIR>
__device__ __forceinline__ void dft9(float2* v) {
  // exp(-2 pi i m / 9), m = 1, 2, 4
  const float2 w1 = make_float2(0.76604444311897803520f, -0.64278760968653932632f);
  const float2 w2 = make_float2(0.17364817766693034885f, -0.98480775301220805937f);
  const float2 w4 = make_float2(-0.93969262078590838405f, -0.34202014332566873304f);
  float2 u[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) u[i][j] = v[i + 3 * j];
    dft_odd<3, DIR>(u[i]);
  }
  u[1][1] = cmul_dir<DIR>(u[1][1], w1);
  u[1][2] = cmul_dir<DIR>(u[1][2], w2);
  u[2][1] = cmul_dir<DIR>(u[2][1], w2);
  u[2][2] = cmul_dir<DIR>(u[2][2], w4);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    float2 t[3] = {u[0][j], u[1][j], u[2][j]};
    dft_odd<3, DIR>(t);
#pragma unroll
    for (int k = 0; k < 3; ++k) v[j + 3 * k] = t[k];
  }
}

template <int R, int DIR>
__device__ __forceinline__ void dftR(float2* v) {
  if constexpr (R == 2) dft2<DIR>(v);
  else if constexpr (R == 4) dft4<DIR>(v);
  else if constexpr (R == 8) dft8<DIR>(v);
  else if constexpr (R == 9) dft9<DIR>(v);
  else if constexpr (R % 2 == 0) dft_2odd<R / 2, DIR>(v);
  else dft_odd<R, DIR>(v);
}

// i / d by a multiply, exact while i * d < 2^32 (the callers' i and d are
// below 2^16)
struct FastDiv {
  unsigned d, m;
  __device__ __forceinline__ explicit FastDiv(int d_)
      : d((unsigned)d_), m(d_ > 1 ? 0xffffffffu / (unsigned)d_ + 1u : 0u) {}
  __device__ __forceinline__ int operator()(int i) const {
    return d > 1 ? (int)__umulhi((unsigned)i, m) : i;
  }
};

// LDS layouts of P pencils of length n:
//   ROWS (pencil-major):  element (p, j) at p*(n + n/8) + j + j/8; the gap
//                         after every 8 elements spreads the stride-R stage
//                         writes over the banks
//   COLS (interleaved):   element (p, j) at j*P + p
// Work items are mapped so that consecutive lanes touch consecutive words.
enum { ROWS = 0, COLS = 1 };

template <int LAY>
__device__ __forceinline__ int lidx(int p, int j, int n, int P) {
  return LAY == ROWS ? p * (n + (n >> 3)) + j + (j >> 3) : j * P + p;
}

// LDS elements needed for P pencils of length n in a layout
__host__ __device__ constexpr int lds_elems(int lay, int n, int P) {
  return lay == ROWS ? P * (n + (n >> 3)) : P * n;
}

__host__ __device__ constexpr int ilog2c(int n) { return n <= 1 ? 0 : 1 + ilog2c(n >> 1); }

// Lengths with compile-time kernels, by the code LN: 2^LN for 6..10, and
// 3 2^(LN - 32) for 37..40 (96, 192, 384, 768: the meshes of 1.5 cells a
// particle).  With run-time stages, divisions and addresses the passes of
// 192^3 took: Poisson x 90 us (now 28), the inverse y pair 67 (22), y 31 (13),
// c2r 39 (29).
__host__ __device__ constexpr bool ct_three(int ln) { return ln >= 32; }
__host__ __device__ constexpr int ct_n(int ln) { return ct_three(ln) ? 3 << (ln - 32) : 1 << ln; }
__host__ __device__ constexpr int pow2_floor(int n) { return n < 2 ? 1 : 2 * pow2_floor(n / 2); }

// Columns per workgroup of a strided pass of fixed length: 16 (128-byte
// segments of a row), fewer when they exceed cap values; and its threads, of
// v values each.  A 64^3 or 128^3 mesh has 33 or 65 columns, which blocks
// filled to cap (128 and 64 columns) left half empty and too few.
__host__ __device__ constexpr int ct_cols(int ln, int cap) {
  return cap / ct_n(ln) >= 16 ? 16 : pow2_floor(cap / ct_n(ln));
}
__host__ __device__ constexpr int ct_tpb(int ln, int cols, int v) { return cols * ct_n(ln) / v; }
// Values per thread of the y and plain x passes: 16, and 8 where more
// wavefronts on the few blocks of a small mesh count (inverse of 128^3: 9.6
// -> 8.5 us, the pair of components 10.8 -> 9.7; 256^3 25.0 -> 24.4 and 42.7
// -> 41.1; but 512^3 251 -> 256 and 413 -> 433).  The forward passes keep 16:
// with 8 the compiler contracts other products into FMAs, and results would
// move by a rounding.
// Lengths 3 2^k take 12, which their first (4) and last (6) radix divide.
__host__ __device__ constexpr int fft_v(int dir, int ln) {
  return ct_three(ln) ? 12 : (dir > 0 && ln <= 8 ? 8 : 16);
}
// Poisson x pass
__host__ __device__ constexpr int pfft_v(int ln) { return ct_three(ln) ? 12 : 8; }

// Rows per workgroup of a row pass of fixed length: RFFT_CAP values, or
// a quarter of that (3/8 for 3 2^k: whole wavefronts) for meshes whose row
// blocks would leave CUs idle.  The workgroup has eight values per thread.
__host__ __device__ constexpr int ct_rows(int lh, bool small) {
  return pow2_floor((small ? (ct_three(lh) ? RFFT_CAP * 3 / 8 : RFFT_CAP / 4) : RFFT_CAP) / ct_n(lh));
}
__host__ __device__ constexpr int ct_row_tpb(int lh, bool small) {
  return ct_rows(lh, small) * ct_n(lh) / 8;
}

// One Stockham stage of radix R (n a power of two, Ns the size of the
// sub-transforms already done): reads x[j + r n/R], twiddles by
// w_{Ns R}^{(j mod Ns) r}, and writes the radix-R DFT to
// (j - j mod Ns) R + j mod Ns + r Ns.  Twiddle powers are built from at most
// three table reads (w, w^2, w^4) with at most two extra products; all reads
// of a stage are issued before the arithmetic.
template <int R, int DIR, int LAY, int MAXV, int TPB>
__device__ __forceinline__ void fft_stage(float2* s, int n, int P, int Ns, int lnb, int lP,
                                          const float2* __restrict__ tw, int tws) {
  constexpr int NG = MAXV / R;
  const int nb = n / R;
  const int total = P * nb;
  const int step = n / (Ns * R);
  float2 v[MAXV];
  float2 w1[NG], w2[NG], w4[NG];
  int mm[NG];
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    int idx = threadIdx.x + it * tpb<TPB>();
    mm[it] = 0;
    if (idx < total) {
      int p = LAY == ROWS ? (idx >> lnb) : (idx & (P - 1));
      int j = LAY == ROWS ? (idx & (nb - 1)) : (idx >> lP);
      int m = (j & (Ns - 1)) * step * tws;
      mm[it] = m;
      w1[it] = twiddle<DIR>(tw, m);
      if (R >= 4) w2[it] = twiddle<DIR>(tw, 2 * m);
      if (R == 8) w4[it] = twiddle<DIR>(tw, 4 * m);
#pragma unroll
      for (int r = 0; r < R; ++r) v[it * R + r] = s[lidx<LAY>(p, j + r * nb, n, P)];
    }
  }
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      if (mm[it] != 0) {
        float2* u = &v[it * R];
        u[1] = cmul(u[1], w1[it]);
        if (R >= 4) {
          float2 w3 = cmul(w2[it], w1[it]);
          u[2] = cmul(u[2], w2[it]);
          u[3] = cmul(u[3], w3);
          if (R == 8) {
            u[4] = cmul(u[4], w4[it]);
            u[5] = cmul(u[5], cmul(w4[it], w1[it]));
            u[6] = cmul(u[6], cmul(w4[it], w2[it]));
            u[7] = cmul(u[7], cmul(w4[it], w3));
          }
        }
      }
      dftR<R, DIR>(&v[it * R]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      int p = LAY == ROWS ? (idx >> lnb) : (idx & (P - 1));
      int j = LAY == ROWS ? (idx & (nb - 1)) : (idx >> lP);
      int k = j & (Ns - 1);
      int o = (j - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) s[lidx<LAY>(p, o + r * Ns, n, P)] = v[it * R + r];
    }
  }
  __syncthreads();
}

// One Stockham stage of radix R for a length n that is no power of two: as
// fft_stage, with divisions by the run-time sub-transform sizes and every
// twiddle power read from the table.
template <int R, int DIR, int LAY, int MAXV, int TPB>
__device__ __forceinline__ void fft_mix_stage(float2* s, int n, int P, int Ns, int lP,
                                              const float2* __restrict__ tw, int tws) {
  constexpr int NG = (MAXV + R - 1) / R;
  const int nb = n / R;
  const int total = P * nb;
  const int step = nb / Ns * tws;
  const FastDiv dnb(nb), dNs(Ns);
  float2 v[NG * R];
  int ob[NG], pp[NG];
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      const int p = LAY == ROWS ? dnb(idx) : (idx & (P - 1));
      const int j = LAY == ROWS ? idx - p * nb : (idx >> lP);
      const int k = j - dNs(j) * Ns;
      pp[it] = p;
      ob[it] = (j - k) * R + k;
      const int m = k * step;
#pragma unroll
      for (int r = 0; r < R; ++r) v[it * R + r] = s[lidx<LAY>(p, j + r * nb, n, P)];
      if (Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[it * R + r] = cmul_dir<DIR>(v[it * R + r], tw[r * m]);
      }
      dftR<R, DIR>(&v[it * R]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    if ((int)threadIdx.x + it * tpb<TPB>() < total) {
#pragma unroll
      for (int r = 0; r < R; ++r) s[lidx<LAY>(pp[it], ob[it] + r * Ns, n, P)] = v[it * R + r];
    }
  }
  __syncthreads();
}

// The stage of a prime radix R >= 11: the twiddles in place, then outputs r
// and R - r of a butterfly together (dft_odd's sums), (R + 1) / 2 work items
// each of (R - 1) / 2 terms.
template <int DIR, int LAY, int MAXV, int TPB>
__device__ __forceinline__ void fft_prime_stage(float2* s, int n, int P, int Ns, int R, int lP,
                                                const float2* __restrict__ tw, int tws) {
#pragma clang fp contract(fast)
  constexpr int NG = (MAXV * 6 + 10) / 11;  // (R + 1) / (2 R) <= 6 / 11 items per value
  const int nb = n / R, K = (R - 1) / 2;
  const FastDiv dnb(nb), dn(n), dNs(Ns);
  if (Ns > 1) {
    const int step = nb / Ns * tws;
    for (int idx = threadIdx.x; idx < P * n; idx += tpb<TPB>()) {
      const int p = LAY == ROWS ? dn(idx) : (idx & (P - 1));
      const int e = LAY == ROWS ? idx - p * n : (idx >> lP);
      const int q = dnb(e), j = e - q * nb;
      const int k = j - dNs(j) * Ns;
      float2* x = s + lidx<LAY>(p, e, n, P);
      *x = cmul_dir<DIR>(*x, tw[q * k * step]);
    }
    __syncthreads();
  }
  const int per = nb * (K + 1), total = P * per;
  const FastDiv dper(per);
  float2 u[NG], v[NG];
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      const int p = LAY == ROWS ? dper(idx) : (idx & (P - 1));
      const int e = LAY == ROWS ? idx - p * per : (idx >> lP);
      const int r = dnb(e), j = e - r * nb;
      float2 m = s[lidx<LAY>(p, j, n, P)], d = make_float2(0.f, 0.f);
      int t = 0;
#pragma unroll 2
      for (int q = 1; q <= K; ++q) {
        t += r;
        if (t >= R) t -= R;
        const float2 w = tw[t * nb * tws];  // (cos, -sin)
        const float2 a = s[lidx<LAY>(p, j + q * nb, n, P)];
        const float2 b = s[lidx<LAY>(p, j + (R - q) * nb, n, P)];
        m.x += w.x * (a.x + b.x);
        m.y += w.x * (a.y + b.y);
        d.x -= w.y * (a.x - b.x);
        d.y -= w.y * (a.y - b.y);
      }
      d = mul_mi<DIR>(d);
      u[it] = cadd(m, d);
      v[it] = csub(m, d);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      const int p = LAY == ROWS ? dper(idx) : (idx & (P - 1));
      const int e = LAY == ROWS ? idx - p * per : (idx >> lP);
      const int r = dnb(e), j = e - r * nb;
      const int k = j - dNs(j) * Ns, o = (j - k) * R + k;
      s[lidx<LAY>(p, o + r * Ns, n, P)] = u[it];
      if (r) s[lidx<LAY>(p, o + (R - r) * Ns, n, P)] = v[it];
    }
  }
  __syncthreads();
}

// Smallest prime factor of m that is at least 11 (m has no smaller one).
__device__ __forceinline__ int prime_factor(int m) {
  for (int q = 11; q * q <= m; q += 2)
    if (m % q == 0) return q;
  return m;
}

// Mixed-radix FFT of P pencils of any length: radices 8, 4, then 6 and 10
// (which take a remaining factor 2 along), 2, 9, 3, 5 and 7, then the primes
// from 11 up.
template <int DIR, int LAY, int MAXV, int TPB>
__device__ __forceinline__ void fft_mixed(float2* s, int n, int P, int lP,
                                          const float2* __restrict__ tw, int tws) {
#define PMX_STAGE(R) fft_mix_stage<R, DIR, LAY, MAXV, TPB>(s, n, P, Ns, lP, tw, tws), Ns *= R, rem /= R
  int Ns = 1, rem = n;
  while (rem > 1) {
    if (rem % 8 == 0) PMX_STAGE(8);
    else if (rem % 4 == 0) PMX_STAGE(4);
    else if (rem % 6 == 0) PMX_STAGE(6);
    else if (rem % 10 == 0) PMX_STAGE(10);
    else if (rem % 2 == 0) PMX_STAGE(2);
    else if (rem % 9 == 0) PMX_STAGE(9);
    else if (rem % 3 == 0) PMX_STAGE(3);
    else if (rem % 5 == 0) PMX_STAGE(5);
    else if (rem % 7 == 0) PMX_STAGE(7);
    else {
      const int R = prime_factor(rem);
      fft_prime_stage<DIR, LAY, MAXV, TPB>(s, n, P, Ns, R, lP, tw, tws);
      Ns *= R;
      rem /= R;
    }
  }
#undef PMX_STAGE
}

// Unnormalised in-LDS FFT of P pencils (exp(DIR 2 pi i jk/n)).  POW2
// selects the power-of-two stages or the mixed-radix ones.  tw
// is a table of exp(-2 pi i m/(n tws)); tws > 1 reuses a longer table.
// Callers synchronise before it; it ends with a barrier.
template <int DIR, int LAY, bool POW2, int MAXV, int TPB>
__device__ __forceinline__ void lds_fft(float2* s, int n, int P, const float2* __restrict__ tw,
                                        int tws = 1) {
  if (n == 1) return;
  const int lP = __ffs(P) - 1;
  if (!POW2) {
    fft_mixed<DIR, LAY, MAXV, TPB>(s, n, P, lP, tw, tws);
    return;
  }
  int Ns = 1;
  while (Ns < n) {
    int rem = n / Ns;
    if (rem % 8 == 0) {
      fft_stage<8, DIR, LAY, MAXV, TPB>(s, n, P, Ns, __ffs(n / 8) - 1, lP, tw, tws);
      Ns *= 8;
    } else if (rem % 4 == 0) {
      fft_stage<4, DIR, LAY, MAXV, TPB>(s, n, P, Ns, __ffs(n / 4) - 1, lP, tw, tws);
      Ns *= 4;
    } else {
      fft_stage<2, DIR, LAY, MAXV, TPB>(s, n, P, Ns, __ffs(n / 2) - 1, lP, tw, tws);
      Ns *= 2;
    }
  }
}

// ----------------------------------------- compile-time length FFTs --
// The same Stockham stages with N, P and the stage size NS known at compile
// time (N and P powers of two): index arithmetic folds to shifts and
// immediate LDS offsets, and the bounds tests go when the butterflies fill
// the workgroup.  COLS blocks read every twiddle power from the table (the
// pencils of a wave share a twiddle, so the reads broadcast); ROWS blocks
// build w^3, w^5..w^7 from w, w^2, w^4 as lds_fft does.  In both layouts
// element x of pencil p sits at lidx(p, x); the R inputs of a butterfly are
// a fixed stride apart, and so are its R outputs except for ROWS stages
// with 1 < NS < 8, which compute each address.
//
// REG (COLS): the first (REG & 1) stage takes its inputs from reg, the last
// (REG & 2) leaves its outputs there, both in the order of ColMap (element e
// of a thread is row j0 + e js): a butterfly's inputs j + r N/R of the first
// stage and outputs of the last are the rows that its thread loads and
// stores, so half of a transform's LDS traffic and three of its barriers go.
// Poisson x pass, same bits: 128^3 15.0 -> 13.2 us, 256^3 53 -> 45, 512^3 470
// -> 455 (there bound by memory).
template <int R, int DIR, int LAY, int N, int P, int NS, int TPB, int TWS, int REG = 0>
__device__ __forceinline__ void ct_stage(float2* s, const float2* __restrict__ tw,
                                         float2* reg = nullptr) {
  constexpr int NB = N / R, TOTAL = P * NB;
  constexpr int NG = (TOTAL + TPB - 1) / TPB;
  constexpr bool FULL = TOTAL % TPB == 0;
  constexpr int LP = ilog2c(P);
  constexpr int STEP = N / (NS * R) * TWS;
  constexpr bool SEP_IN = LAY == COLS || NB % 8 == 0;
  constexpr bool SEP_OUT = LAY == COLS || NS % 8 == 0 || NS == 1;
  constexpr int SIN = LAY == ROWS ? NB + (NB >> 3) : NB * P;
  constexpr int SOUT = LAY == ROWS ? NS + (NS >> 3) : NS * P;
  constexpr bool ALLTW = LAY == COLS || R == 6;
  float2 v[NG * R];
  float2 w[NG][R > 1 ? R - 1 : 1];
  int ob[NG];
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (FULL || idx < TOTAL) {
      const int p = LAY == ROWS ? (unsigned)idx / NB : idx & (P - 1);
      const int j = LAY == ROWS ? (unsigned)idx % NB : idx >> LP;
      const int k = j & (NS - 1);
      ob[it] = lidx<LAY>(p, (j - k) * R + k, N, P);
      const int ib = lidx<LAY>(p, j, N, P);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (REG & 1) v[it * R + r] = reg[it + r * NG];
        else v[it * R + r] = SEP_IN ? s[ib + r * SIN] : s[lidx<LAY>(p, j + r * NB, N, P)];
      }
      if (NS > 1) {
        const int m = k * STEP;
        if (ALLTW) {
#pragma unroll
          for (int r = 1; r < R; ++r) w[it][r - 1] = tw[r * m];
        } else {
          w[it][0] = tw[m];
          if constexpr (R >= 4) w[it][1] = tw[2 * m];
          if constexpr (R == 8) w[it][3] = tw[4 * m];
        }
      }
    }
  }
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (FULL || idx < TOTAL) {
      float2* u = &v[it * R];
      if (NS > 1) {
        if constexpr (!ALLTW) {
          if constexpr (R >= 4) w[it][2] = cmul(w[it][1], w[it][0]);
          if constexpr (R == 8) {
            w[it][4] = cmul(w[it][3], w[it][0]);
            w[it][5] = cmul(w[it][3], w[it][1]);
            w[it][6] = cmul(w[it][3], w[it][2]);
          }
        }
#pragma unroll
        for (int r = 1; r < R; ++r) u[r] = cmul_dir<DIR>(u[r], w[it][r - 1]);
      }
      dftR<R, DIR>(u);
    }
  }
  if constexpr (REG & 2) {
#pragma unroll
    for (int it = 0; it < NG; ++it)
#pragma unroll
      for (int r = 0; r < R; ++r) reg[it + r * NG] = v[it * R + r];
    return;
  }
  if constexpr (!(REG & 1)) __syncthreads();
#pragma unroll
  for (int it = 0; it < NG; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (FULL || idx < TOTAL) {
      if (SEP_OUT) {
#pragma unroll
        for (int r = 0; r < R; ++r) s[ob[it] + r * SOUT] = v[it * R + r];
      } else {
        const int p = (unsigned)idx / NB, j = (unsigned)idx % NB;
        const int k = j & (NS - 1), o = (j - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) s[lidx<LAY>(p, o + r * NS, N, P)] = v[it * R + r];
      }
    }
  }
  __syncthreads();
}

// Radix of the stage after NS: 8 (then 4 or 2) for powers of two; 4, then 8
// or 4, and 6 last for 3 2^k, so that every NS is a power of two.
__host__ __device__ constexpr int ct_radix(int n, int ns) {
  return n % 3      ? (n / ns % 8 == 0 ? 8 : (n / ns % 4 == 0 ? 4 : 2))
         : ns == 1  ? 4
         : n / ns == 6 ? 6
                    : (n / ns / 6 % 8 == 0 && n / ns != 96 ? 8 : (n / ns / 6 % 4 == 0 ? 4 : 2));
}

template <int DIR, int LAY, int N, int P, int NS, int TPB, int TWS>
__device__ __forceinline__ void ct_fft(float2* s, const float2* __restrict__ tw) {
  if constexpr (NS < N) {
    constexpr int R = ct_radix(N, NS);
    ct_stage<R, DIR, LAY, N, P, NS, TPB, TWS>(s, tw);
    ct_fft<DIR, LAY, N, P, NS * R, TPB, TWS>(s, tw);
  }
}

// The same from and to registers (N >= 64: at least two stages).
template <int DIR, int N, int P, int NS, int TPB>
__device__ __forceinline__ void ct_fft_reg(float2* reg, float2* s, const float2* __restrict__ tw) {
  if constexpr (NS < N) {
    constexpr int R = ct_radix(N, NS);
    ct_stage<R, DIR, COLS, N, P, NS, TPB, 1, (NS == 1 ? 1 : 0) | (NS * R == N ? 2 : 0)>(s, tw, reg);
    ct_fft_reg<DIR, N, P, NS * R, TPB>(reg, s, tw);
  }
}

// FFT of P pencils of length n: the compile-time path when LN > 0
// (n = ct_n(LN), P = 2^LP), else lds_fft.
template <int DIR, int LAY, bool POW2, int LN, int LP, int MAXV, int TPB, int TWS = 1>
__device__ __forceinline__ void fft_run(float2* s, int n, int P, const float2* __restrict__ tw) {
  if constexpr (LN > 0)
    ct_fft<DIR, LAY, ct_n(LN), 1 << LP, 1, TPB, TWS>(s, tw);
  else
    lds_fft<DIR, LAY, POW2, MAXV, TPB>(s, n, P, tw, TWS);
}

static inline bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }

// -------------------------------------------------- batched transfers --
// Global <-> LDS traffic goes through registers in unrolled batches of up to
// MAXV values per thread, so a thread's loads are all in flight at once
// instead of waiting out the memory latency one element at a time.
template <int MAXV, int TPB, class LD, class ST>
__device__ __forceinline__ void batch_copy(int total, LD ld, ST st) {
  float2 r[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) r[it] = ld(idx);
  }
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) st(idx, r[it]);
  }
}

// Copies the twiddle table tw[0, n) to LDS (no barrier).
template <int TPB>
__device__ __forceinline__ void stage_twiddles(float2* stw, const float2* __restrict__ tw, int n) {
  for (int base = 0; base < n; base += 4 * tpb<TPB>())
    batch_copy<4, TPB>(n - base, [&](int i) { return tw[base + i]; },
                       [&](int i, float2 v) { stw[base + i] = v; });
}

// Logical block of a pass: the XCD-contiguous remap of the hardware block
// index, in reverse when rev is set.  Consecutive passes of a transform run
// in opposite directions, so that each first reads what the pass before it
// wrote last, while that is still in the last-level cache.
__device__ __forceinline__ unsigned pass_block(unsigned lin, unsigned nb, int rev) {
  const unsigned l = pmx_xcd_block(lin, nb);
  return rev ? nb - 1 - l : l;
}

// Element k <= H of the r2c of a row from its half-length transform (see
// z_r2c_half_k).
__device__ __forceinline__ float2 r2c_half_x(const float2* s, const float2* stw, int p, int k, int H,
                                             int P) {
  float2 zk = s[lidx<ROWS>(p, k == H ? 0 : k, H, P)];
  float2 zm = s[lidx<ROWS>(p, k == 0 ? 0 : H - k, H, P)];
  zm.y = -zm.y;
  float2 e = make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y + zm.y));
  float2 dd = csub(zk, zm);
  float2 o = make_float2(0.5f * dd.y, -0.5f * dd.x);
  return cadd(e, cmul(stw[k], o));
}

// Splits a block's value index into row and position (by a constant when LH).
template <int LH>
struct RowSplit {
  int H;
  FastDiv d;
  __device__ __forceinline__ explicit RowSplit(int H_) : H(H_), d(LH ? 1 : H_) {}
  __device__ __forceinline__ int row(int idx) const { return LH ? (unsigned)idx / ct_n(LH) : d(idx); }
  __device__ __forceinline__ int col(int idx, int p) const {
    return LH ? (unsigned)idx % ct_n(LH) : idx - p * H;
  }
};

// Half-length c2r of a block's np rows (blk, rows of rsc complex values) into
// the real pairs r of each thread, times scale (see z_c2r_half_k).  The first
// barrier inside also covers the staging of stw and earlier reads of s.
template <int LH, bool SM, bool POW2, int MAXV, int TPB>
__device__ __forceinline__ void c2r_half_rows(float2 (&r)[MAXV], const float2* __restrict__ blk,
                                              int rsc, float2* s, const float2* stw,
                                              const RowSplit<LH>& rsp, int H, int P, int np) {
  constexpr int PC = LH ? ct_rows(LH, SM) : 1;
  const int total = np * H;
  // X[k] and X[H-k] per thread: both loads of the batch are issued first
  float2 xa[MAXV], xb[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    const int p = rsp.row(idx);
    if (idx < total) {
      const float2* row = blk + __umul24(p, rsc);
      const int k = rsp.col(idx, p);
      xa[it] = row[k];
      xb[it] = row[H - k];
    }
  }
  __syncthreads();  // the twiddle table is read below
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (idx < total) {
      const int p = rsp.row(idx), k = rsp.col(idx, p);
      float2 a = xa[it], b = xb[it];
      if (k == 0) {
        a.y = 0.f;
        b.y = 0.f;
      }
      b.y = -b.y;
      float2 sum = cadd(a, b);
      float2 dif = csub(a, b);
      float2 t = cmul_dir<1>(dif, stw[k]);
      s[lidx<ROWS>(p, k, H, P)] = make_float2(sum.x - t.y, sum.y + t.x);
    }
  }
  __syncthreads();
  fft_run<1, ROWS, POW2, LH, ilog2c(PC), MAXV, TPB, 2>(s, H, np, stw);
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    const int p = rsp.row(idx);
    if (idx < total) r[it] = s[lidx<ROWS>(p, rsp.col(idx, p), H, P)];
  }
}

// Half-length r2c of a block's rows, held as real pairs in s, to blk.
template <int LH, bool SM, bool POW2, int MAXV, int TPB>
__device__ __forceinline__ void r2c_half_rows(float2* __restrict__ blk, int rsc, float2* s,
                                              const float2* stw, const RowSplit<LH>& rsp, int H,
                                              int P, int np) {
  constexpr int PC = LH ? ct_rows(LH, SM) : 1;
  const int total = np * H;
  fft_run<-1, ROWS, POW2, LH, ilog2c(PC), MAXV, TPB, 2>(s, H, np, stw);
  {
    float2 r[MAXV];
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      const int p = rsp.row(idx);
      if (idx < total) r[it] = r2c_half_x(s, stw, p, rsp.col(idx, p), H, P);
    }
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      const int p = rsp.row(idx);
      if (idx < total) blk[__umul24(p, rsc) + rsp.col(idx, p)] = r[it];
    }
    // X[H] of each row
    for (int p = threadIdx.x; p < np; p += tpb<TPB>()) blk[__umul24(p, rsc) + H] = r2c_half_x(s, stw, p, H, H, P);
  }
}

// rev: the pass runs its blocks in the reverse order (pass_block)
struct Fields3 {
  float2* f[3];
  int rev;
};
// One side of a strided pass: element j of pencil (o, c) of field i at
// f[i] + o * os + j * es + c.
struct Side3 {
  float2* f[3];
  long long es, os;
};

// Block coordinates of a (gx, gy, gz) grid after the XCD-contiguous remap
// of the linear block index: neighbouring column blocks, which share the
// 128-byte lines of a row, then run on one XCD close together and meet in
// its L2.
__device__ __forceinline__ void xcd_block3(int& bx, int& by, int& bz, int rev) {
  const unsigned nb = gridDim.x * gridDim.y * gridDim.z;
  const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const unsigned l = pass_block(lin, nb, rev);
  bx = l % gridDim.x;
  by = (l / gridDim.x) % gridDim.y;
  bz = l / (gridDim.x * gridDim.y);
}

// A thread's share of an n x B block of columns (B a power of two dividing
// TPB): its it-th element is (row j0 + it*js, column b), at LDS index
// threadIdx.x + it*TPB in the COLS layout.
struct ColMap {
  int b, j0, js;
};
template <int TPB>
__device__ __forceinline__ ColMap col_map(int lB) {
  ColMap m;
  m.b = threadIdx.x & ((1 << lB) - 1);
  m.j0 = threadIdx.x >> lB;
  m.js = tpb<TPB>() >> lB;
  return m;
}

// FFT of a block of columns held in registers in the order of cm, through
// the LDS block s, which no thread may still be reading on entry (and some
// may on return).  The staging of the twiddles need not be waited for.
// REGS false: the first and last stage go through LDS as well (fewer
// registers at once).
template <int DIR, bool POW2, int LN, int LP, int MAXV, int TPB, bool REGS = true>
__device__ __forceinline__ void fft_cols(float2 (&r)[MAXV], float2* s, int n, int P,
                                         const float2* __restrict__ tw, const ColMap& cm) {
  if constexpr (LN > 0 && REGS) {
    ct_fft_reg<DIR, ct_n(LN), 1 << LP, 1, TPB>(r, s, tw);
  } else {
#pragma unroll
    for (int it = 0; it < MAXV; ++it)
      if (cm.j0 + it * cm.js < n) s[threadIdx.x + it * tpb<TPB>()] = r[it];
    __syncthreads();
    fft_run<DIR, COLS, POW2, LN, LP, MAXV, TPB>(s, n, P, tw);
#pragma unroll
    for (int it = 0; it < MAXV; ++it)
      if (cm.j0 + it * cm.js < n) r[it] = s[threadIdx.x + it * tpb<TPB>()];
  }
}

// Source of a Poisson x pass other than its own buffer (poisson_x_k).
struct SpecSrc {
  const float2* modes;
  const float2* f;
  float vol, ca, cb;
};

struct KTab {
  const float* k[3];
  const float* km[3];
};

// -------------------------------------------------------------- plans --
#define PMX_LDS_MAX (160 * 1024)     // LDS a gfx950 workgroup may allocate

// A pencil block must fit the per-thread batches (total <= cap) and LDS.
static inline int fft_fits(const char* who, int n, int total, int cap, size_t lds) {
  PMX_REQUIRE_CODE(total <= cap && lds <= PMX_LDS_MAX, PMX_EUNSUP,
                   "%s: axis of length %d needs %d values and %zu bytes of LDS per workgroup "
                   "(limits %d and %d)", who, n, total, lds, cap, PMX_LDS_MAX);
  return PMX_OK;
}

static inline size_t lds_bytes(int n, int P, int lay = COLS) {
  return (size_t)lds_elems(lay, n, P) * sizeof(float2);
}

// the twiddle table staged after the data block
static inline size_t tw_bytes(int n) { return (size_t)n * sizeof(float2); }


// Code of a length that has compile-time kernels, else 0.
static inline int ct_code(int n) {
  for (int l = 6; l <= 10; ++l)
    if (n == ct_n(l)) return l;
  for (int l = 37; l <= 40; ++l)
    if (n == ct_n(l)) return l;
  return 0;
}

// Threads of a run-time-length workgroup of `total` values.
static inline int gen_tpb(int total) {
  const int t = (total + GEN_MAXV - 1) / GEN_MAXV;
  return t < 64 ? 64 : (t + 63) / 64 * 64;
}

// Fewest workgroups of a pass before its blocks are made smaller: four per CU.
#define FFT_MIN_WGS 1024

// The z pass of n2 over nrows rows: even n2 as half-length transforms, of
// compile-time length (code lh) when there are kernels and the row blocks come out
// even, else (and for odd n2, two rows a pencil) at run time.  rows: rows per
// workgroup.  Meshes of few rows take smaller blocks (sm): a 128^3 mesh has
// 256 row blocks of 4096 values, one per CU, and their load, barrier and
// store phases then follow each other with nothing to overlap.
struct RowPlan {
  bool half, sm;
  int lh, P, len, rows, tpb;
  size_t lds;
};

static inline RowPlan row_plan(int n2, long long nrows) {
  RowPlan r;
  r.half = n2 >= 4 && (n2 & 1) == 0;
  r.len = r.half ? n2 / 2 : n2;
  r.lh = r.half ? ct_code(r.len) : 0;
  r.sm = false;
  if (r.lh) {
    r.sm = nrows / ct_rows(r.lh, false) < FFT_MIN_WGS;
    r.P = ct_rows(r.lh, r.sm);
    r.tpb = ct_row_tpb(r.lh, r.sm);
    if (nrows % r.P) r.lh = 0;
  }
  if (!r.lh) {
    r.P = 1;
    while (2 * r.P * r.len <= GEN_CAP / 2) r.P *= 2;
    const int per = r.half ? 1 : 2;
    while (r.P > 1 && r.P * r.len > GEN_CAP / 8 && nrows / (per * r.P) < FFT_MIN_WGS) r.P /= 2;
  }
  if (!r.lh) r.tpb = gen_tpb(r.P * r.len);
  r.rows = r.half ? r.P : 2 * r.P;
  r.lds = lds_bytes(r.len, r.P, ROWS) + tw_bytes(n2);
  return r;
}

// Columns per workgroup of a strided pass of length n without compile-time
// variants: 16 (128-byte segments), fewer when they exceed GEN_CAP values or
// would leave CUs idle.
static inline int gen_cols(int n, int ncol, long long nouter) {
  int B = 16;
  while (B > 1 && B * n > GEN_CAP) B /= 2;
  while (B > 4 && B * n > GEN_CAP / 4 && (ncol + B - 1) / B * nouter < FFT_MIN_WGS / 2) B /= 2;
  return B;
}

// CALL(L) with L the compile-time code ln (0: generic kernels)
#define PMX_CT_SWITCH(ln, CALL) \
  do {                          \
    switch (ln) {               \
      case 6: CALL(6); break;   \
      case 7: CALL(7); break;   \
      case 8: CALL(8); break;   \
      case 9: CALL(9); break;   \
      case 10: CALL(10); break; \
      case 37: CALL(37); break; \
      case 38: CALL(38); break; \
      case 39: CALL(39); break; \
      case 40: CALL(40); break; \
      default: CALL(0);         \
    }                           \
  } while (0)

static inline KTab ktab(const pmx_ctx* c) {
  KTab kt;
  for (int a = 0; a < 3; ++a) {
    kt.k[a] = c->k[a];
    kt.km[a] = c->km[a];
  }
  return kt;
}

// axis 1 (y) or axis 0 (x) complex FFT of nf spectra, from src (rows of
// srow) to dst (rows of drow)
int pmx_strided_from_to(pmx_ctx* c, float2* const* src, int srow, float2* const* dst, int drow,
                        int nf, int axis, int dir, int rev);
// c2r of one padded spectrum to a dense mesh
int pmx_c2r_dense(pmx_ctx* c, float* out, float2* f, float scale, int rev = 0);
int pmx_poisson_x(pmx_ctx* c, float2* const* f, int adjoint, const SpecSrc* src = nullptr, int rev = 0);
