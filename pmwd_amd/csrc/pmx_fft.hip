// Hand-written 3D real FFTs and the fused Poisson/gradient solve (gfx950).
//
// Layout: a real mesh lives in "padded" rows of rs = 2*(n2/2+1) floats so the
// r2c/c2r row passes run in place; the complex mesh is (n0, n1, n2h) float2 in rows of n2p >= n2h.
// Each kernel stages P pencils of length n in LDS (pencil-major for the
// contiguous row passes, interleaved for the strided passes) and runs a
// Stockham autosort FFT: radix 8/4/2 stages for powers of two, mixed radices
// for other lengths (pmx_fft.h).
//
// Pass order (forward): z r2c (rows, contiguous) -> y (strided) -> x
// (strided).  The x pass of the Poisson solve does forward x FFT, Green's
// function, -ik_d and the inverse x FFT for the three components, so the
// inverse ends with y (strided) and z c2r (rows).
#include "pmx_fft.h"

#include <algorithm>

// ------------------------------------------------------------ z passes --
// Up to three meshes of one row pass: block b works on field b / nblk, in the
// block order of pass_block (rev per field).  fold: the halo shells of field
// i lie i * hstride floats into the halo.  o: the real side, rows of ors
// floats that an r2c reads and a c2r writes (f itself when in place; dense
// caller meshes save the copy into or out of the padded layout).
struct RowFields {
  float* f[3];
  float* o[3];
  int ors;
  int rev[3];
  unsigned nblk;
  long long hstride;
};
__device__ __forceinline__ int row_field(unsigned nblk, int rev0, int rev1, int rev2, unsigned& blk) {
  const unsigned i = blockIdx.x / nblk;
  blk = pass_block(blockIdx.x - i * nblk, nblk, i == 0 ? rev0 : (i == 1 ? rev1 : rev2));
  return (int)i;
}
#define PMX_ROW_FIELD(rf, blk) row_field((rf).nblk, (rf).rev[0], (rf).rev[1], (rf).rev[2], blk)
#define PMX_ROW_DATA(rf, i) ((i) == 0 ? (rf).f[0] : ((i) == 1 ? (rf).f[1] : (rf).f[2]))
#define PMX_ROW_REAL(rf, i) ((i) == 0 ? (rf).o[0] : ((i) == 1 ? (rf).o[1] : (rf).o[2]))

// In-place r2c of padded rows by a length-n2 complex FFT (odd n2; even ones
// take z_r2c_half_k): two rows a and b are transformed as z = a + i b, and
//   A[k] = (Z[k] + conj Z[n2-k]) / 2,  B[k] = -i (Z[k] - conj Z[n2-k]) / 2.
// PRE applies (x - 1) * coef on load (gravity.py:52-54).  A block takes P
// pairs of rows.  LDS: the P pencils, then the n2-entry twiddle table.
template <int PRE, bool POW2>
__global__ void __launch_bounds__(GEN_MAXTPB, 4) z_r2c_k(RowFields rf, long long nrows, int n2, int rs,
                                                      int P, float coef,
                                                      const float2* __restrict__ tw,
                                                      const float* __restrict__ fcoef) {
  extern __shared__ float2 s[];
  if (PRE && fcoef) coef = fcoef[0];
  float2* stw = s + lds_elems(ROWS, n2, P);
  unsigned blk;
  const int field = PMX_ROW_FIELD(rf, blk);
  float* data = PMX_ROW_DATA(rf, field);
  const float* real = PMX_ROW_REAL(rf, field);
  const long long row0 = (long long)blk * 2 * P;
  const int nr = (int)((nrows - row0) < 2 * P ? (nrows - row0) : 2 * P);
  const int np = (nr + 1) / 2;
  const FastDiv dn(n2);
  stage_twiddles<GEN_TPB>(stw, tw, n2);
  batch_copy<GEN_MAXV, GEN_TPB>(
      np * n2,
      [&](int idx) {
        const int p = dn(idx), j = idx - p * n2;
        const float* r = real + (row0 + 2 * p) * rf.ors + j;
        float2 v = make_float2(r[0], 2 * p + 1 < nr ? r[rf.ors] : 0.f);
        if (PRE) {
          v.x = v.x - 1.f;
          v.x = v.x * coef;
          v.y = v.y - 1.f;
          v.y = v.y * coef;
        }
        return v;
      },
      [&](int idx, float2 v) {
        const int p = dn(idx);
        s[lidx<ROWS>(p, idx - p * n2, n2, P)] = v;
      });
  __syncthreads();
  lds_fft<-1, ROWS, POW2, GEN_MAXV, GEN_TPB>(s, n2, np, stw);
  const int n2h = n2 / 2 + 1;
  float2* out = reinterpret_cast<float2*>(data);
  const int rsc = rs / 2;
  const FastDiv dh(n2h);
  for (int idx = threadIdx.x; idx < np * n2h; idx += tpb<GEN_TPB>()) {
    const int p = dh(idx), k = idx - p * n2h;
    const float2 z = s[lidx<ROWS>(p, k, n2, P)];
    float2 m = s[lidx<ROWS>(p, k ? n2 - k : 0, n2, P)];
    m.y = -m.y;
    float2* o = out + (row0 + 2 * p) * rsc + k;
    o[0] = make_float2(0.5f * (z.x + m.x), 0.5f * (z.y + m.y));
    if (2 * p + 1 < nr) o[rsc] = make_float2(0.5f * (z.y - m.y), -0.5f * (z.x - m.x));
  }
}

// In-place c2r of padded rows with a final scale (odd n2), two rows a time:
// Z = A + i B over the full spectra rebuilt from the halves (X[n-k] = conj
// X[k]), Im X[0] and (even n2) Im X[n2/2] dropped as irfft does; the inverse
// is a + i b.
template <bool POW2>
__global__ void __launch_bounds__(GEN_MAXTPB, 4) z_c2r_k(RowFields rf, long long nrows, int n2, int rs,
                                                      int P, float scale,
                                                      const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  float2* stw = s + lds_elems(ROWS, n2, P);
  unsigned blk;
  const int field = PMX_ROW_FIELD(rf, blk);
  const float* data = PMX_ROW_DATA(rf, field);
  float* real = PMX_ROW_REAL(rf, field);
  const long long row0 = (long long)blk * 2 * P;
  const int nr = (int)((nrows - row0) < 2 * P ? (nrows - row0) : 2 * P);
  const int np = (nr + 1) / 2;
  const float2* in = reinterpret_cast<const float2*>(data);
  const int rsc = rs / 2;
  const int half = n2 / 2;
  const FastDiv dn(n2);
  stage_twiddles<GEN_TPB>(stw, tw, n2);
  batch_copy<GEN_MAXV, GEN_TPB>(
      np * n2,
      [&](int idx) {
        const int p = dn(idx), k = idx - p * n2;
        const int kk = k <= half ? k : n2 - k;
        const float2* r = in + (row0 + 2 * p) * rsc + kk;
        float2 a = r[0], b = make_float2(0.f, 0.f);
        if (2 * p + 1 < nr) b = r[rsc];
        if (kk == 0 || 2 * kk == n2) a.y = b.y = 0.f;
        return k <= half ? make_float2(a.x - b.y, a.y + b.x) : make_float2(a.x + b.y, b.x - a.y);
      },
      [&](int idx, float2 v) {
        const int p = dn(idx);
        s[lidx<ROWS>(p, idx - p * n2, n2, P)] = v;
      });
  __syncthreads();
  lds_fft<1, ROWS, POW2, GEN_MAXV, GEN_TPB>(s, n2, np, stw);
  for (int idx = threadIdx.x; idx < np * n2; idx += tpb<GEN_TPB>()) {
    const int p = dn(idx), j = idx - p * n2;
    const float2 v = s[lidx<ROWS>(p, j, n2, P)];
    float* r = real + (row0 + 2 * p) * rf.ors + j;
    r[0] = v.x * scale;
    if (2 * p + 1 < nr) r[rf.ors] = v.y * scale;
  }
}

// Half-length r2c for even n2, H = n2/2: the row is read as H complex values z[m] = x[2m] + i x[2m+1],
// Z = FFT_H(z), and for k = 0..H:  X[k] = E + w^k O,  E = (Z[k] + conj Z[H-k])/2,
// O = -i (Z[k] - conj Z[H-k])/2,  w = exp(-2 pi i/n2)  (Z[H] = Z[0]).
// PRE applies (x - 1) * coef on load.  LH > 0 fixes H = ct_n(LH) and
// P = ct_rows(LH, SM) at compile time (the launch then holds whole blocks);
// LH = 0 takes any H, POW2 telling whether it is a power of two.
// The deposit's halo shells of one channel for a row pass that folds them
// in on load (16^3 tiles; n1 the y extent of the mesh).
struct FoldIn {
  const float* halo;
  int shell, ntx, nty, ntz, n1;
};

// Row (x, y), z cells 2m and 2m+1: each cell on a low face of its tile gets
// the fold's shell sum added, as fold_k adds it to the mesh.
__device__ __forceinline__ float2 fold_pair(float2 v, const FoldIn& fi, int x, int y, int m) {
  const int lx = x & 15, ly = y & 15, z = 2 * m, lz = z & 15;
  if (lx == 0 || ly == 0 || lz == 0)
    v.x = v.x + pmx_fold_sum16(fi.halo, fi.shell, fi.ntx, fi.nty, fi.ntz, x >> 4, y >> 4, z >> 4,
                               lx, ly, lz);
  if (lx == 0 || ly == 0)
    v.y = v.y + pmx_fold_sum16(fi.halo, fi.shell, fi.ntx, fi.nty, fi.ntz, x >> 4, y >> 4, z >> 4,
                               lx, ly, lz + 1);
  return v;
}

// The fold terms of a block of P rows (x plane x, rows y = y0 + p, pairs
// z = 2m, 2m + 1; 2H cells a row), staged in LDS.  A cell takes
// pmx_fold_sum16's terms; by the faces its row lies on (lx = x % 16,
// ly = y % 16, lz = z % 16):
//   lx != 0, ly != 0: S = 4 on cells with lz = 0;
//   lx == 0, ly != 0 (a face row): S = 1 on every cell, then S = 4, 5 when lz = 0;
//   lx != 0, ly == 0 (a face row): S = 2 on every cell, then S = 4, 6 when lz = 0;
//   lx == 0, ly == 0 (a corner row, 1 in 256): fold_pair.
// T[p * 2H + z] holds the face rows' S = 1 or S = 2 term, loaded straight into
// LDS (the rows' FFT buffer, before the rows go there), and Z0[p + P tz] the
// S = 4 term and Z1[p + P tz] the S = 5 or S = 6 term of cell (p, 16 tz),
// one each per thread (P * H / 8 <= TPB of them).  All of it is issued before
// the row loads, so no wait falls between two of them.
template <int P, int TPB, int H>
__device__ __forceinline__ void fold_tables(const FoldIn& fi, int x, int y0, float* T, float& z0,
                                            float& z1) {
  typedef __attribute__((address_space(1))) const void gptr;
  typedef __attribute__((address_space(3))) void lptr;
  constexpr int lP = ilog2c(P);
  const int lx = x & 15, tx = x >> 4, txm = tx == 0 ? fi.ntx - 1 : tx - 1;
  auto tile = [&](int nx, int ny, int nz) {
    return fi.halo + (long long)((nx * fi.nty + ny) * fi.ntz + nz) * fi.shell;
  };
  const int j = (int)threadIdx.x;
  z0 = z1 = 0.f;
  if (j < P * (H >> 3)) {
    const int y = y0 + (j & (P - 1)), tz = j >> lP, ly = y & 15, ty = y >> 4;
    const int tym = ty == 0 ? fi.nty - 1 : ty - 1, tzm = tz == 0 ? fi.ntz - 1 : tz - 1;
    if (lx != 0 || ly != 0) {
      z0 = tile(tx, ty, tzm)[561 + lx * 16 + ly];
      if (lx == 0)
        z1 = tile(txm, ty, tzm)[ly * 17 + 16];
      else if (ly == 0)
        z1 = tile(tx, tym, tzm)[289 + lx * 17 + 16];
    }
  }
  // a wave's 64 entries lie in one row (2H a multiple of 64), so the face-row
  // test is wave-uniform; lane l of a wave writes the LDS word at its base plus l
  static_assert(2 * H % 64 == 0 && TPB % 64 == 0 && P * (H >> 3) <= TPB, "fold tables");
  constexpr int n2 = 2 * H;
  const int wave0 = j & ~63;
  for (int e0 = 0; e0 < P * n2; e0 += TPB) {
    const int e = e0 + j;
    if (e >= P * n2) break;
    const int p = (unsigned)e / n2, z = (unsigned)e % n2;
    const int y = y0 + p, ly = y & 15, ty = y >> 4;
    if ((lx == 0) == (ly == 0)) continue;
    const float* src = lx == 0 ? tile(txm, ty, z >> 4) + ly * 17 + (z & 15)
                               : tile(tx, ty == 0 ? fi.nty - 1 : ty - 1, z >> 4) + 289 + lx * 17 + (z & 15);
    __builtin_amdgcn_global_load_lds((gptr*)src, (lptr*)(T + e0 + wave0), 4, 0, 0);
  }
}

// Adds the fold (fold_tables' terms, in pmx_fold_sum16's order) to a block's
// NV values per thread (row p = idx / H, pair m = idx % H).
template <int NV, int TPB, int P, int H>
__device__ __forceinline__ void fold_rows(float2 (&r)[NV], const FoldIn& fi, int x, int y0, int total,
                                          const float* T, const float* Z0, const float* Z1) {
  const int lx = x & 15;
#pragma unroll
  for (int it = 0; it < NV; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    if (idx >= total) continue;
    const int p = (unsigned)idx / H, y = y0 + p, m = (unsigned)idx % H;
    const int ly = y & 15, z = 2 * m, lz = z & 15, k = (m >> 3) * P + p;
    if (lx == 0 && ly == 0) {
      r[it] = fold_pair(r[it], fi, x, y, m);
    } else if (lx == 0 || ly == 0) {
      const float* t = T + p * 2 * H + z;
      float sx = 0.f;
      sx += t[0];
      if (lz == 0) {
        sx += Z0[k];
        sx += Z1[k];
      }
      r[it].x = r[it].x + sx;
      float sy = 0.f;
      sy += t[1];
      r[it].y = r[it].y + sy;
    } else if (lz == 0) {
      float sx = 0.f;
      sx += Z0[k];
      r[it].x = r[it].x + sx;
    }
  }
}

// FOLD (with LH > 0, 16^3 tiles, P | n1): the density is the deposit's tile
// interiors plus the fold of fi.halo, added here on load (192^3: 27 us, where
// the pass and a fold pass took 18 + 33; 512^3: 243).
template <int PRE, int LH, bool SM, bool FOLD, bool POW2>
__global__ void __launch_bounds__(LH ? ct_row_tpb(LH, SM) : GEN_MAXTPB, 4)
    z_r2c_half_k(RowFields rf, long long nrows, int n2, int rs, int P_, float coef,
                 const float2* __restrict__ tw, FoldIn fi, const float* __restrict__ fcoef) {
  extern __shared__ float2 s[];
  // 1.5 Omega_m from the device factor table when the call has one
  if (PRE && fcoef) coef = fcoef[0];
  constexpr int PC = LH ? ct_rows(LH, SM) : 1;
  constexpr int TPB = LH ? ct_row_tpb(LH, SM) : GEN_TPB;
  constexpr int MAXV = LH ? PC * ct_n(LH) / TPB : GEN_MAXV;
  const int H = LH ? ct_n(LH) : n2 >> 1;
  const int P = LH ? PC : P_;
  const RowSplit<LH> rsp(H);
  float2* stw = s + lds_elems(ROWS, H, P);
  unsigned bk;
  const int field = PMX_ROW_FIELD(rf, bk);
  const long long row0 = (long long)bk * P;
  const int np = LH ? PC : (int)((nrows - row0) < P ? (nrows - row0) : P);
  const int rsc = rs / 2;
  float2* blk = reinterpret_cast<float2*>(PMX_ROW_DATA(rf, field)) + row0 * rsc;
  const int orc = rf.ors / 2;
  const float2* src = reinterpret_cast<const float2*>(PMX_ROW_REAL(rf, field)) + row0 * orc;
  const int total = np * H;
  if (FOLD) fi.halo += field * rf.hstride;
  stage_twiddles<TPB>(stw, tw, 2 * H);
  // the block's rows lie in one x plane when folding
  const int fx = FOLD ? (int)row0 / fi.n1 : 0;
  const int fy0 = FOLD ? (int)row0 - fx * fi.n1 : 0;
  {
    // the block's fold terms (fold_tables), issued before the row loads, in
    // the rows' buffer: T (P * 2H floats), then Z0 and Z1 (P * H / 8 each) in
    // what the rows' padding leaves (P * (H + H / 8) float2 in all)
    float* T = reinterpret_cast<float*>(s);
    float* Z0 = T + PC * 2 * H;
    float* Z1 = Z0 + PC * (H >> 3);
    float z0 = 0.f, z1 = 0.f;
    if constexpr (FOLD) fold_tables<PC, TPB, ct_n(LH)>(fi, fx, fy0, T, z0, z1);
    float2 r[MAXV];
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      const int p = rsp.row(idx);
      if (idx < total) r[it] = src[__umul24(p, orc) + rsp.col(idx, p)];
    }
    if constexpr (FOLD) {
      if ((int)threadIdx.x < PC * (H >> 3)) {
        Z0[threadIdx.x] = z0;
        Z1[threadIdx.x] = z1;
      }
      __builtin_amdgcn_s_waitcnt(0);  // T's loads into LDS have landed
      __syncthreads();
      fold_rows<MAXV, TPB, PC, ct_n(LH)>(r, fi, fx, fy0, total, T, Z0, Z1);
      __syncthreads();  // T is read before the rows take its place
    }
    if (PRE) {
#pragma unroll
      for (int it = 0; it < MAXV; ++it) {
        r[it].x = r[it].x - 1.f;
        r[it].x = r[it].x * coef;
        r[it].y = r[it].y - 1.f;
        r[it].y = r[it].y * coef;
      }
    }
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      const int p = rsp.row(idx);
      if (idx < total) s[lidx<ROWS>(p, rsp.col(idx, p), H, P)] = r[it];
    }
  }
  __syncthreads();
  r2c_half_rows<LH, SM, POW2, MAXV, TPB>(blk, rsc, s, stw, rsp, H, P, np);
}

// Half-length c2r (inverse of the above) with a final scale:
// Z[k] = (X[k] + conj X[H-k]) + i w^-k (X[k] - conj X[H-k]) for k < H with
// Im X[0] = Im X[H] = 0 (as irfft), z = IFFT_H(Z), x[2m] + i x[2m+1] = z[m].
// LH, SM and POW2 as in z_r2c_half_k.
template <int LH, bool SM, bool POW2>
__global__ void __launch_bounds__(LH ? ct_row_tpb(LH, SM) : GEN_MAXTPB, 4)
    z_c2r_half_k(RowFields rf, long long nrows, int n2, int rs, int P_, float scale,
                 const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int PC = LH ? ct_rows(LH, SM) : 1;
  constexpr int TPB = LH ? ct_row_tpb(LH, SM) : GEN_TPB;
  constexpr int MAXV = LH ? PC * ct_n(LH) / TPB : GEN_MAXV;
  const int H = LH ? ct_n(LH) : n2 >> 1;
  const int P = LH ? PC : P_;
  const RowSplit<LH> rsp(H);
  float2* stw = s + lds_elems(ROWS, H, P);
  unsigned bk;
  const int field = PMX_ROW_FIELD(rf, bk);
  const long long row0 = (long long)bk * P;
  const int np = LH ? PC : (int)((nrows - row0) < P ? (nrows - row0) : P);
  const int rsc = rs / 2;
  const float2* blk = reinterpret_cast<const float2*>(PMX_ROW_DATA(rf, field)) + row0 * rsc;
  const int orc = rf.ors / 2;
  float2* dst = reinterpret_cast<float2*>(PMX_ROW_REAL(rf, field)) + row0 * orc;
  const int total = np * H;
  stage_twiddles<TPB>(stw, tw, 2 * H);
  float2 r[MAXV];
  c2r_half_rows<LH, SM, POW2, MAXV, TPB>(r, blk, rsc, s, stw, rsp, H, P, np);
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int idx = threadIdx.x + it * tpb<TPB>();
    const int p = rsp.row(idx);
    if (idx < total)
      dst[__umul24(p, orc) + rsp.col(idx, p)] = make_float2(r[it].x * scale, r[it].y * scale);
  }
}

// ------------------------------------------------------ strided passes --
// FFT along a strided axis of complex (outer, n, ncol) views, from one side
// to the other (the same one in place).  A workgroup takes B consecutive
// columns, so each of its loads is B contiguous float2.
// LDS: the n x B block, then the n-entry twiddle table.  LN > 0 fixes
// n = ct_n(LN) and B = ct_cols(LN, FFT_CAP) at compile time.
template <int DIR, bool POW2, int LN>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, FFT_CAP), fft_v(DIR, LN)) : GEN_MAXTPB, 4) strided_fft_k(Side3 si, Side3 so, int rev,
                                                         int n_, int ncol, int B_,
                                                         const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int BC = LN ? ct_cols(LN, FFT_CAP) : 1;
  constexpr int TPB = LN ? ct_tpb(LN, BC, fft_v(DIR, LN)) : GEN_TPB;
  constexpr int MAXV = LN ? BC * ct_n(LN) / TPB : GEN_MAXV;
  const int n = LN ? ct_n(LN) : n_;
  const int B = LN ? BC : B_;
  const int lB = LN ? ilog2c(BC) : __ffs(B_) - 1;
  float2* stw = s + n * B;
  int bx, by, bz;
  xcd_block3(bx, by, bz, rev);
  const int c0 = bx * B;
  const int nb = ncol - c0 < B ? ncol - c0 : B;
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  const float2* g = (bz == 0 ? si.f[0] : (bz == 1 ? si.f[1] : si.f[2])) + (long long)by * si.os +
                    c0 + cm.b + (long long)cm.j0 * si.es;
  const long long gs = (long long)cm.js * si.es;
  stage_twiddles<TPB>(stw, tw, n);
  float2 r[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    r[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n) r[it] = g[it * gs];
  }
  fft_cols<DIR, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n, B, stw, cm);
  float2* d = (bz == 0 ? so.f[0] : (bz == 1 ? so.f[1] : so.f[2])) + (long long)by * so.os + c0 +
              cm.b + (long long)cm.j0 * so.es;
  const long long ds = (long long)cm.js * so.es;
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n) d[it * ds] = r[it];
}

// x pass of the Poisson solve (gravity.py:56-66): forward FFT along x of
// c0, pot = -src/k^2 (k=0 -> 0), g_d = (-i km_d) pot, inverse FFT along x.
// km_1 (one value per y row) and km_2 (one per kz column) are constant along
// x, so the y and z components share one inverse transform h =
// IFFT_x(-i pot), stored to c_1 (y_inv_seq_k scales it by km_1 and km_2 for
// the two components); the x component (-i km_0 pot) is transformed on its
// own and stored to c_0.  The two inverse transforms run one after the
// other in the same LDS block, h kept in registers meanwhile.  Pencils along
// axis 0 of (n0,n1,n2h); blockIdx.y = y index, blockIdx.x = block of B kz
// columns.  LDS: the n0 x B block, the n0-entry twiddle table, then the k_0
// and km_0 tables.  The run-time kernels are held to 128 VGPRs, two blocks a
// CU: at 150 x 180 x 210 that spills a few and takes 69 us instead of 85.
// KIN: the source.  0: rows of n2p of f[0] after the y pass; 1: the full
// spectrum sp.modes (rows of n2h) over sp.vol; 2: sp.ca times that plus sp.cb
// times the x transform of sp.f (rows of n2p).
template <bool POW2, int LN, int KIN = 0>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, PFFT_CAP), pfft_v(LN)) : GEN_MAXTPB, LN ? 1 : 4) poisson_x_k(Fields3 fl, int n0_, int n1, int n2h, int n2p,
                                                       int B_, KTab kt, const float2* __restrict__ tw,
                                                       SpecSrc sp) {
  extern __shared__ float2 s[];
  constexpr int BC = LN ? ct_cols(LN, PFFT_CAP) : 1;
  constexpr int TPB = LN ? ct_tpb(LN, BC, pfft_v(LN)) : GEN_TPB;
  constexpr int MAXV = LN ? BC * ct_n(LN) / TPB : GEN_MAXV;
  const int n0 = LN ? ct_n(LN) : n0_;
  const int B = LN ? BC : B_;
  const int lB = LN ? ilog2c(BC) : __ffs(B_) - 1;
  float2* stw = s + n0 * B;
  float* sk = reinterpret_cast<float*>(stw + n0);
  float* skm = sk + n0;
  const long long es = (long long)n1 * n2p;
  int bx, y, bz;
  xcd_block3(bx, y, bz, fl.rev);
  const int c0 = bx * B;
  const int nb = n2h - c0 < B ? n2h - c0 : B;
  const long long off = (long long)y * n2p + c0;
  stage_twiddles<TPB>(stw, tw, n0);
  for (int i = threadIdx.x; i < n0; i += tpb<TPB>()) {
    sk[i] = kt.k[0][i];
    skm[i] = kt.km[0][i];
  }
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  float2* g0 = fl.f[0] + off + cm.b + (long long)cm.j0 * es;
  float2* g1 = fl.f[1] + off + cm.b + (long long)cm.j0 * es;
  const long long gs = (long long)cm.js * es;
  const long long ms = (long long)cm.js * n1 * n2h;
  const float2* gm = nullptr;
  if constexpr (KIN != 0) gm = sp.modes + ((long long)cm.j0 * n1 + y) * n2h + c0 + cm.b;
  float2 r[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    r[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n0) {
      if constexpr (KIN == 0) r[it] = g0[it * gs];
      if constexpr (KIN == 1) r[it] = gm[it * ms];
      if constexpr (KIN == 2) r[it] = sp.f[off + cm.b + (long long)cm.j0 * es + it * gs];
    }
  }
  float2 m[MAXV];
  if constexpr (KIN == 2) {
#pragma unroll
    for (int it = 0; it < MAXV; ++it)
      if (live && cm.j0 + it * cm.js < n0) m[it] = gm[it * ms];
  }
  if constexpr (KIN != 1) fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n0, B, stw, cm);
  else __syncthreads();  // the tables are read below
  const float ky = kt.k[1][y];
  const float kz = live ? kt.k[2][c0 + cm.b] : 0.f;
  float2 h[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    h[it] = make_float2(0.f, 0.f);
    if (live && j < n0) {
      float2 v = r[it];
      if constexpr (KIN == 1) v = make_float2(v.x / sp.vol, v.y / sp.vol);
      if constexpr (KIN == 2)
        v = make_float2(sp.ca * (m[it].x / sp.vol) + sp.cb * v.x, sp.ca * (m[it].y / sp.vol) + sp.cb * v.y);
      float kx = sk[j];
      float k2 = kx * kx;
      k2 = k2 + ky * ky;
      k2 = k2 + kz * kz;
      // pot = -v / k^2, h = -i pot = (pot.y, -pot.x)
      if (k2 != 0.f) {
        const float q = 1.f / k2;
        h[it] = make_float2(-(v.y * q), v.x * q);
      }
    }
  }
  // x component: IFFT_x(km_0 h) to c_0
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    if (j < n0) {
      const float kmx = skm[j];
      r[it] = make_float2(kmx * h[it].x, kmx * h[it].y);
    }
  }
  __syncthreads();
  fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n0, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n0) g0[it * gs] = r[it];
  __syncthreads();
  // h to c_1
  fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(h, s, n0, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n0) g1[it * gs] = h[it];
}

// Adjoint x pass: acc = sum_d (-i km_d) laplace(FFT_x c_d); inverse FFT
// along x; stored to c0.  Transpose of the three force components.  As km_1
// and km_2 are constant along x, FFT_x(km_1 c_1 + km_2 c_2) replaces the two
// transforms of c_1 and c_2; y_fwd_seq_k leaves that combination in c_1.
// The forward transforms of c_0 and c_1 run one after the other in the same
// LDS block (the first result kept in registers), then the inverse of the
// sum.  LDS as poisson_x_k.
template <bool POW2, int LN>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, PFFT_CAP), pfft_v(LN)) : GEN_MAXTPB, LN ? 1 : 4) poisson_x_adj_k(Fields3 fl, int n0_, int n1, int n2h, int n2p,
                                                           int B_, KTab kt, const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int BC = LN ? ct_cols(LN, PFFT_CAP) : 1;
  constexpr int TPB = LN ? ct_tpb(LN, BC, pfft_v(LN)) : GEN_TPB;
  constexpr int MAXV = LN ? BC * ct_n(LN) / TPB : GEN_MAXV;
  const int n0 = LN ? ct_n(LN) : n0_;
  const int B = LN ? BC : B_;
  const int lB = LN ? ilog2c(BC) : __ffs(B_) - 1;
  float2* stw = s + n0 * B;
  float* sk = reinterpret_cast<float*>(stw + n0);
  float* skm = sk + n0;
  const long long es = (long long)n1 * n2p;
  int bx, y, bz;
  xcd_block3(bx, y, bz, fl.rev);
  const int c0 = bx * B;
  const int nb = n2h - c0 < B ? n2h - c0 : B;
  const long long off = (long long)y * n2p + c0;
  stage_twiddles<TPB>(stw, tw, n0);
  for (int i = threadIdx.x; i < n0; i += tpb<TPB>()) {
    sk[i] = kt.k[0][i];
    skm[i] = kt.km[0][i];
  }
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  float2* g0 = fl.f[0] + off + cm.b + (long long)cm.j0 * es;
  const float2* g1 = fl.f[1] + off + cm.b + (long long)cm.j0 * es;
  const long long gs = (long long)cm.js * es;
  float2 x0[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    x0[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n0) x0[it] = g0[it * gs];
  }
  float2 yz[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    yz[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n0) yz[it] = g1[it * gs];
  }
  fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB>(x0, s, n0, B, stw, cm);
  __syncthreads();
  fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB>(yz, s, n0, B, stw, cm);
  const float ky = kt.k[1][y];
  const float kz = live ? kt.k[2][c0 + cm.b] : 0.f;
  float2 acc[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    acc[it] = make_float2(0.f, 0.f);
    if (live && j < n0) {
      float kx = sk[j];
      float k2 = kx * kx;
      k2 = k2 + ky * ky;
      k2 = k2 + kz * kz;
      if (k2 != 0.f) {
        const float kmx = skm[j];
        const float2 w = yz[it];
        float sx = kmx * x0[it].x + w.x, sy = kmx * x0[it].y + w.y;
        // pot = -sum / k^2, acc = -i pot = (pot.y, -pot.x)
        const float q = 1.f / k2;
        acc[it] = make_float2(-(sy * q), sx * q);
      }
    }
  }
  __syncthreads();
  fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(acc, s, n0, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n0) g0[it * gs] = acc[it];
}

// y passes of the gradient components, paired (pencils along axis 1 of
// (n0,n1,n2h); blockIdx.y = x row, blockIdx.x = block of B
// kz columns, 128-byte segments at n = 512; LDS: the n x B block, then the
// twiddle table).  The two transforms run one after the other in the same
// LDS block.
//
// Inverse: from h = IFFT_x(-i pot) in c_1, the y and z force components
// IFFT_y(km_1 h) to c_1 and IFFT_y(km_2 h) to c_2 -- the products and
// transforms of a separate y pass over km_1 h and km_2 h, with h read once
// and kept in registers.  BOTH: the x
// component's inverse (c_0 in place) runs in the same launch (pmx_fft_yinv).
//
// Forward (adjoint path, y_fwd_seq_k): FFT_y of c_1 (kept in registers) and
// of c_2, then their combination km_1 FFT_y(c_1) + km_2 FFT_y(c_2) to c_1
// for poisson_x_adj_k.
template <bool POW2, int LN, int BOTH>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, FFT_CAP), fft_v(1, LN)) : GEN_MAXTPB, LN ? 2 : 4) y_inv_seq_k(Fields3 fl, int n_, long long es,
                                                        long long ostride, int ncol, int B_,
                                                        KTab kt, const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int BC = LN ? ct_cols(LN, FFT_CAP) : 1;
  constexpr int TPB = LN ? ct_tpb(LN, BC, fft_v(1, LN)) : GEN_TPB;
  constexpr int MAXV = LN ? BC * ct_n(LN) / TPB : GEN_MAXV;
  const int n = LN ? ct_n(LN) : n_;
  const int B = LN ? BC : B_;
  const int lB = LN ? ilog2c(BC) : __ffs(B_) - 1;
  float2* stw = s + n * B;
  int bx, by, bz;
  xcd_block3(bx, by, bz, fl.rev);
  // BOTH: odd rows of the grid are the x component's (alternating, so that
  // every XCD's share of the blocks holds as many pairs)
  const bool xc = BOTH && (by & 1);
  by >>= BOTH;
  const int c0 = bx * B;
  const int nb = ncol - c0 < B ? ncol - c0 : B;
  const long long off = (long long)by * ostride + c0;
  stage_twiddles<TPB>(stw, tw, n);
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  const float kmz = live ? kt.km[2][c0 + cm.b] : 0.f;
  float2* g1 = (xc ? fl.f[0] : fl.f[1]) + off + cm.b + (long long)cm.j0 * es;
  float2* g2 = fl.f[2] + off + cm.b + (long long)cm.j0 * es;
  const long long gs = (long long)cm.js * es;
  float2 h[MAXV], r[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    h[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n) h[it] = g1[it * gs];
  }
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    if (j < n) {
      const float kmy = kt.km[1][j];
      r[it] = xc ? h[it] : make_float2(kmy * h[it].x, kmy * h[it].y);
    }
  }
  fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n) g1[it * gs] = r[it];
  if (xc) return;
#pragma unroll
  for (int it = 0; it < MAXV; ++it) h[it] = make_float2(kmz * h[it].x, kmz * h[it].y);
  __syncthreads();
  fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(h, s, n, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n) g2[it * gs] = h[it];
}

//
// Workgroups of 512 threads keep to 128 registers, so that two share a CU; of
// the 512-long axis the transforms then go through LDS at both ends, which
// fits without spilling (the cap alone spills 14).  The axis' forward passes
// in a force and its gradient, from registers without the cap, with it, and
// now: 512^3 1090, 1080, 1054 us; 128 x 1024 x 128 195, 186, 186; 128 x 768 x
// 128 155, 146, 146.
constexpr int yfwd_tpb(int ln) { return ln ? ct_tpb(ln, ct_cols(ln, FFT_CAP), fft_v(-1, ln)) : GEN_MAXTPB; }
template <bool POW2, int LN>
__global__ void __launch_bounds__(yfwd_tpb(LN), yfwd_tpb(LN) == 512 ? 4 : 2) y_fwd_seq_k(Fields3 fl, int n_, long long es,
                                                        long long ostride, int ncol, int B_,
                                                        KTab kt, const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int BC = LN ? ct_cols(LN, FFT_CAP) : 1;
  constexpr int TPB = LN ? ct_tpb(LN, BC, fft_v(-1, LN)) : GEN_TPB;
  constexpr bool REGS = LN != 9;
  constexpr int MAXV = LN ? BC * ct_n(LN) / TPB : GEN_MAXV;
  const int n = LN ? ct_n(LN) : n_;
  const int B = LN ? BC : B_;
  const int lB = LN ? ilog2c(BC) : __ffs(B_) - 1;
  float2* stw = s + n * B;
  int bx, by, bz;
  xcd_block3(bx, by, bz, fl.rev);
  const int c0 = bx * B;
  const int nb = ncol - c0 < B ? ncol - c0 : B;
  const long long off = (long long)by * ostride + c0;
  stage_twiddles<TPB>(stw, tw, n);
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  const float kmz = live ? kt.km[2][c0 + cm.b] : 0.f;
  float2* g1 = fl.f[1] + off + cm.b + (long long)cm.j0 * es;
  const float2* g2 = fl.f[2] + off + cm.b + (long long)cm.j0 * es;
  const long long gs = (long long)cm.js * es;
  float2 a[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    a[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n) a[it] = g1[it * gs];
  }
  float2 c[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    c[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n) c[it] = g2[it * gs];
  }
  fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB, REGS>(a, s, n, B, stw, cm);
  __syncthreads();
  fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB, REGS>(c, s, n, B, stw, cm);
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    if (j < n) {
      const float kmy = kt.km[1][j];
      a[it] = make_float2(kmy * a[it].x + kmz * c[it].x, kmy * a[it].y + kmz * c[it].y);
    }
  }
#pragma unroll
  for (int it = 0; it < MAXV; ++it)
    if (live && cm.j0 + it * cm.js < n) g1[it * gs] = a[it];
}

// ------------------------------------------------------------- copies --
// dst rows of dst_rs floats <- src rows of src_rs floats, n2 valid columns
__global__ void copy_rows_k(float* __restrict__ dst, int dst_rs, const float* __restrict__ src,
                            int src_rs, long long nrows, int n2) {
  long long total = nrows * n2;
  for (long long i = (long long)blockIdx.x * PMX_TPB + threadIdx.x; i < total;
       i += (long long)gridDim.x * PMX_TPB) {
    long long r = i / n2;
    int j = (int)(i - r * n2);
    dst[r * dst_rs + j] = src[r * src_rs + j];
  }
}

// copies n0*n1 rows of ncols floats between row strides (ncols <= 0: n2)
int pmx_copy_rows(pmx_ctx* c, float* dst, int dst_rs, const float* src, int src_rs, int ncols) {
  if (ncols <= 0) ncols = c->n[2];
  long long nrows = (long long)c->n[0] * c->n[1];
  long long total = nrows * ncols;
  unsigned nblk = (unsigned)((total + PMX_TPB - 1) / PMX_TPB);
  if (nblk > 65536u * 4) nblk = 65536u * 4;
  copy_rows_k<<<nblk, PMX_TPB, 0, c->stream>>>(dst, dst_rs, src, src_rs, nrows, ncols);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// ------------------------------------------------------------ drivers --
int pmx_fold_deferrable(const pmx_ctx* c) {
  if (!c->fold_on_load) return 0;
  const TileGeom& t = c->tg;
  if (t.tx != 16 || t.ty != 16 || t.tz != 16) return 0;
  if (c->n[0] % 16 || c->n[1] % 16 || c->n[2] % 16) return 0;
  const RowPlan r = row_plan(c->n[2], (long long)c->n[0] * c->n[1]);
  return r.lh > 0 && c->n[1] % r.P == 0;
}

static RowFields row_fields(const pmx_ctx* c, float* const* f, int nf, const int* rev, unsigned nblk,
                            long long hstride, float* const* real, int ors) {
  RowFields rf;
  for (int i = 0; i < 3; ++i) {
    rf.f[i] = f[i < nf ? i : 0];
    rf.o[i] = real ? real[i < nf ? i : 0] : rf.f[i];
    rf.rev[i] = rev[i < nf ? i : 0];
  }
  rf.ors = real ? ors : c->rs;
  rf.nblk = nblk;
  rf.hstride = hstride;
  return rf;
}

// Whether a row pass can read or write a dense (n0, n1, n2) mesh in place of
// the padded layout: even n2 moves the rows as float2.
static bool dense_rows_ok(const pmx_ctx* c, const void* p) {
  return (c->n[2] & 1) || (reinterpret_cast<uintptr_t>(p) & 7) == 0;
}

// r2c of nf padded real meshes in place (real: from meshes of ors floats a
// row); pre applies (x - 1) * coef.  With halo (pmx_fold_deferrable must
// hold; one channel's shells per mesh) the deposit's fold is added on load.
int pmx_fft_r2c_rows(pmx_ctx* c, float* const* f, int nf, int pre, float coef, const float* halo,
                     const int* rev, const float* const* real, int ors) {
  const long long nrows = (long long)c->n[0] * c->n[1];
  const int n2 = c->n[2];
  const RowPlan r = row_plan(n2, nrows);
  if (int rc = fft_fits("z r2c", n2, r.len * r.P, GEN_CAP, r.lds)) return rc;
  const unsigned nblk = (unsigned)((nrows + r.rows - 1) / r.rows);
  const FoldIn fi = {halo, c->tg.shell, c->tg.ntx, c->tg.nty, c->tg.ntz, c->n[1]};
  const RowFields rf = row_fields(c, f, nf, rev, nblk, c->ntiles * c->tg.shell,
                                  const_cast<float* const*>(real), ors);
  const float* fc = pre ? c->dfac : nullptr;
  PMX_REQUIRE(!halo || pmx_fold_deferrable(c), "z r2c: no fold on load for this mesh");
  pmx_tic(c, PMX_T_ZR2C);
  const unsigned grid = nblk * (unsigned)nf;
#define R2C(PRE, L, SM, FOLD, P2)                                                        \
  z_r2c_half_k<PRE, L, SM, FOLD, P2><<<grid, r.tpb, r.lds, c->stream>>>(                 \
      rf, nrows, n2, c->rs, r.P, coef, c->tw[2], fi, fc)
#define R2C_SM(L, SM)                                   \
  do {                                                  \
    if (halo && pre) R2C(1, L, SM, (L > 0), true);      \
    else if (halo) R2C(0, L, SM, (L > 0), true);        \
    else if (pre) R2C(1, L, SM, false, true);           \
    else R2C(0, L, SM, false, true);                    \
  } while (0)
#define R2C_HALF(L)                       \
  if (r.sm && L) R2C_SM(L, (L > 0));      \
  else R2C_SM(L, false)
#define R2C_FULL(PRE, P2)                                                              \
  z_r2c_k<PRE, P2><<<grid, r.tpb, r.lds, c->stream>>>(rf, nrows, n2, c->rs, r.P, coef, c->tw[2], fc)
  if (r.lh || (r.half && is_pow2(r.len))) {
    PMX_CT_SWITCH(r.lh, R2C_HALF);
  } else if (r.half) {
    if (pre) R2C(1, 0, false, false, false);
    else R2C(0, 0, false, false, false);
  } else if (is_pow2(n2)) {
    if (pre) R2C_FULL(1, true);
    else R2C_FULL(0, true);
  } else {
    if (pre) R2C_FULL(1, false);
    else R2C_FULL(0, false);
  }
#undef R2C_FULL
#undef R2C_HALF
#undef R2C_SM
#undef R2C
  pmx_toc(c, PMX_T_ZR2C);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// c2r of nf padded meshes with a final scale, in place (real: to meshes of
// ors floats a row).
int pmx_fft_c2r_rows(pmx_ctx* c, float* const* f, int nf, float scale, const int* rev,
                     float* const* real, int ors) {
  const long long nrows = (long long)c->n[0] * c->n[1];
  const int n2 = c->n[2];
  const RowPlan r = row_plan(n2, nrows);
  if (int rc = fft_fits("z c2r", n2, r.len * r.P, GEN_CAP, r.lds)) return rc;
  const unsigned nblk = (unsigned)((nrows + r.rows - 1) / r.rows);
  const RowFields rf = row_fields(c, f, nf, rev, nblk, 0, real, ors);
  const unsigned grid = nblk * (unsigned)nf;
  pmx_tic(c, PMX_T_ZC2R);
#define C2R(L, SM, P2)                                                                         \
  z_c2r_half_k<L, SM, P2><<<grid, r.tpb, r.lds, c->stream>>>(rf, nrows, n2, c->rs, r.P, scale, \
                                                             c->tw[2])
#define C2R_HALF(L)                    \
  if (r.sm && L) C2R(L, (L > 0), true); \
  else C2R(L, false, true)
#define C2R_FULL(P2) \
  z_c2r_k<P2><<<grid, r.tpb, r.lds, c->stream>>>(rf, nrows, n2, c->rs, r.P, scale, c->tw[2])
  if (r.lh || (r.half && is_pow2(r.len))) {
    PMX_CT_SWITCH(r.lh, C2R_HALF);
  } else if (r.half) {
    C2R(0, false, false);
  } else if (is_pow2(n2)) {
    C2R_FULL(true);
  } else {
    C2R_FULL(false);
  }
#undef C2R_FULL
#undef C2R_HALF
#undef C2R
  pmx_toc(c, PMX_T_ZC2R);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

int pmx_fft_r2c_inplace(pmx_ctx* c, float* const* f, int nf, int pre, float coef, const float* halo,
                        const int* rev) {
  return pmx_fft_r2c_rows(c, f, nf, pre, coef, halo, rev, nullptr, 0);
}
int pmx_fft_c2r_inplace(pmx_ctx* c, float* const* f, int nf, float scale, const int* rev) {
  return pmx_fft_c2r_rows(c, f, nf, scale, rev, nullptr, 0);
}
// One mesh.
int pmx_fft_r2c_inplace(pmx_ctx* c, float* buf, int pre, float coef, const float* halo, int rev) {
  return pmx_fft_r2c_inplace(c, &buf, 1, pre, coef, halo, &rev);
}
int pmx_fft_c2r_inplace(pmx_ctx* c, float* buf, float scale, int rev) {
  return pmx_fft_c2r_inplace(c, &buf, 1, scale, &rev);
}
// One dense caller mesh to or from padded rows.
static int r2c_dense(pmx_ctx* c, float2* f, const float* in, int pre = 0, float coef = 0.f, int rev = 0) {
  float* b = reinterpret_cast<float*>(f);
  if (!dense_rows_ok(c, in)) {
    if (int rc = pmx_copy_rows(c, b, c->rs, in, c->n[2])) return rc;
    return pmx_fft_r2c_inplace(c, b, pre, coef, nullptr, rev);
  }
  return pmx_fft_r2c_rows(c, &b, 1, pre, coef, nullptr, &rev, &in, c->n[2]);
}
int pmx_c2r_dense(pmx_ctx* c, float* out, float2* f, float scale, int rev) {
  float* b = reinterpret_cast<float*>(f);
  if (!dense_rows_ok(c, out)) {
    if (int rc = pmx_fft_c2r_inplace(c, b, scale, rev)) return rc;
    return pmx_copy_rows(c, out, c->n[2], b, c->rs);
  }
  return pmx_fft_c2r_rows(c, &b, 1, scale, &rev, &out, c->n[2]);
}

// The axis pencils of spectra whose rows are row complex values long.
static Side3 strided_side(const pmx_ctx* c, float2* const* f, int nf, int axis, int row) {
  Side3 s;
  for (int i = 0; i < 3; ++i) s.f[i] = f[i < nf ? i : 0];
  const long long plane = (long long)c->n[1] * row;
  s.es = axis == 1 ? row : plane;
  s.os = axis == 1 ? plane : row;
  return s;
}

int pmx_strided_from_to(pmx_ctx* c, float2* const* src, int srow, float2* const* dst, int drow,
                           int nf, int axis, int dir, int rev) {
  const Side3 si = strided_side(c, src, nf, axis, srow);
  const Side3 so = strided_side(c, dst, nf, axis, drow);
  const int n = c->n[axis];
  const int ncol = c->n2h;
  const unsigned nouter = axis == 1 ? c->n[0] : c->n[1];
  const int ln = ct_code(n);
  const int B = ln ? ct_cols(ln, FFT_CAP) : gen_cols(n, ncol, (long long)nouter * nf);
  const int tpb = ln ? ct_tpb(ln, B, fft_v(dir, ln)) : gen_tpb(n * B);
  dim3 grid((ncol + B - 1) / B, nouter, nf);
  size_t lds = lds_bytes(n, B) + tw_bytes(n);
  if (int rc = fft_fits("strided FFT", n, n * B, ln ? FFT_CAP : GEN_CAP, lds)) return rc;
  const bool p2 = is_pow2(n);
  const int cls = axis == 1 ? (dir < 0 ? PMX_T_YFWD : PMX_T_YINV) : PMX_T_OTHER;
  pmx_tic(c, cls);
#define STRIDED(L)                                                                                  \
  if (dir < 0 && (L || p2))                                                                         \
    strided_fft_k<-1, true, L><<<grid, tpb, lds, c->stream>>>(si, so, rev, n, ncol, B, c->tw[axis]); \
  else if (dir < 0)                                                                                 \
    strided_fft_k<-1, false, 0><<<grid, tpb, lds, c->stream>>>(si, so, rev, n, ncol, B, c->tw[axis]); \
  else if (L || p2)                                                                                 \
    strided_fft_k<1, true, L><<<grid, tpb, lds, c->stream>>>(si, so, rev, n, ncol, B, c->tw[axis]);  \
  else                                                                                              \
    strided_fft_k<1, false, 0><<<grid, tpb, lds, c->stream>>>(si, so, rev, n, ncol, B, c->tw[axis])
  PMX_CT_SWITCH(ln, STRIDED);
#undef STRIDED
  pmx_toc(c, cls);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// the same in place on spectra of the padded layout
int pmx_fft_strided(pmx_ctx* c, float2* const* f, int nf, int axis, int dir, int rev) {
  return pmx_strided_from_to(c, f, c->n2p, f, c->n2p, nf, axis, dir, rev);
}

// Paired y pass of the gradient's y and z components: dir > 0 turns h in
// f[1] into the two force components in f[1] and f[2] (y_inv_seq_k; both:
// and inverts f[0]); dir < 0 turns the cotangents in f[1] and f[2] into km_1
// FFT_y(f[1]) + km_2 FFT_y(f[2]) in f[1] (y_fwd_seq_k).
static int pmx_fft_ypair(pmx_ctx* c, float2* const* f, int dir, int rev, int both = 0) {
  Fields3 fl = {{f[0], f[1], f[2]}, rev};
  const int n = c->n[1];
  const int ncol = c->n2h;
  const int ln = ct_code(n);
  const int B = ln ? ct_cols(ln, FFT_CAP) : gen_cols(n, ncol, c->n[0]);
  const int tpb = ln ? ct_tpb(ln, B, fft_v(dir, ln)) : gen_tpb(n * B);
  const long long es = c->n2p, ostride = (long long)n * c->n2p;
  dim3 grid((ncol + B - 1) / B, c->n[0] << both, 1);
  const size_t lds = lds_bytes(n, B) + tw_bytes(n);
  if (int rc = fft_fits("paired y FFT", n, n * B, ln ? FFT_CAP : GEN_CAP, lds)) return rc;
  const KTab kt = ktab(c);
  const bool p2 = is_pow2(n);
  const int cls = dir < 0 ? PMX_T_YFWD : PMX_T_YINV;
  pmx_tic(c, cls);
#define YINV1(P2, L, BOTH) \
  y_inv_seq_k<P2, L, BOTH><<<grid, tpb, lds, c->stream>>>(fl, n, es, ostride, ncol, B, kt, c->tw[1])
#define YINV(P2, L)        \
  do {                     \
    if (both) YINV1(P2, L, 1); \
    else YINV1(P2, L, 0);  \
  } while (0)
#define YPAIR(L)                                                                                  \
  if (dir < 0 && (L || p2))                                                                       \
    y_fwd_seq_k<true, L><<<grid, tpb, lds, c->stream>>>(fl, n, es, ostride, ncol, B, kt, c->tw[1]); \
  else if (dir < 0)                                                                               \
    y_fwd_seq_k<false, 0><<<grid, tpb, lds, c->stream>>>(fl, n, es, ostride, ncol, B, kt, c->tw[1]); \
  else if (L || p2)                                                                               \
    YINV(true, L); \
  else                                                                                            \
    YINV(false, 0)
  PMX_CT_SWITCH(ln, YPAIR);
#undef YPAIR
#undef YINV
#undef YINV1
  pmx_toc(c, cls);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// The inverse y passes of the three components after poisson_x_k.  Meshes of
// few blocks take them in one launch (128^3, 640 blocks: 18.4 -> 12.3 us);
// larger ones keep one mesh's and the pair's streams apart (256^3, 2304
// blocks: 63 against 67; 512^3: 664 against 687, and their z pass 679 against
// 730, as the pair's meshes are then the last ones written).
int pmx_fft_yinv(pmx_ctx* c, float2* const* f, int rev) {
  const int ln = ct_code(c->n[1]);
  const int B = ln ? ct_cols(ln, FFT_CAP) : gen_cols(c->n[1], c->n2h, c->n[0]);
  if ((long long)((c->n2h + B - 1) / B) * c->n[0] < 2 * FFT_MIN_WGS)
    return pmx_fft_ypair(c, f, 1, rev, 1);
  if (int rc = pmx_fft_strided(c, f, 1, 1, 1, rev)) return rc;
  return pmx_fft_ypair(c, f, 1, 1 - rev);
}

int pmx_poisson_x(pmx_ctx* c, float2* const* f, int adjoint, const SpecSrc* src, int rev) {
  Fields3 fl = {{f[0], f[1], f[2]}, rev};
  const int n0 = c->n[0];
  const int ln = ct_code(n0);
  const int B = ln ? ct_cols(ln, PFFT_CAP) : gen_cols(n0, c->n2h, c->n[1]);
  const int tpb = ln ? ct_tpb(ln, B, pfft_v(ln)) : gen_tpb(n0 * B);
  dim3 grid((c->n2h + B - 1) / B, c->n[1], 1);
  // the data block, the twiddles, then the k_0 and km_0 tables
  size_t lds = lds_bytes(n0, B) + tw_bytes(n0) + 2 * (size_t)n0 * sizeof(float);
  if (int rc = fft_fits("Poisson x pass", n0, n0 * B, PFFT_CAP, lds)) return rc;
  const bool p2 = is_pow2(n0);
  const KTab kt = ktab(c);
  pmx_tic(c, PMX_T_POISSON);
  const SpecSrc sp = src ? *src : SpecSrc{};
  const int kin = !src ? 0 : (src->f ? 2 : 1);
#define PXF(P2, L, K)                                                                              \
  poisson_x_k<P2, L, K><<<grid, tpb, lds, c->stream>>>(fl, n0, c->n[1], c->n2h, c->n2p, B, kt, c->tw[0], sp)
#define PX(L)                                                                                             \
  if (adjoint && (L || p2))                                                                               \
    poisson_x_adj_k<true, L><<<grid, tpb, lds, c->stream>>>(fl, n0, c->n[1], c->n2h, c->n2p, B, kt, c->tw[0]); \
  else if (adjoint)                                                                                       \
    poisson_x_adj_k<false, 0><<<grid, tpb, lds, c->stream>>>(fl, n0, c->n[1], c->n2h, c->n2p, B, kt, c->tw[0]); \
  else if (kin == 1 && (L || p2)) PXF(true, L, 1);                                                        \
  else if (kin == 1) PXF(false, 0, 1);                                                                    \
  else if (kin == 2 && (L || p2)) PXF(true, L, 2);                                                        \
  else if (kin == 2) PXF(false, 0, 2);                                                                    \
  else if (L || p2) PXF(true, L, 0);                                                                      \
  else PXF(false, 0, 0)
  PMX_CT_SWITCH(ln, PX);
#undef PX
#undef PXF
  pmx_toc(c, PMX_T_POISSON);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// Full forward Poisson on the context buffers: cbuf[0] holds the density in
// the padded real layout (deferred: its tile interiors, the fold of c->halo
// still to add); on return cbuf[0..2] hold the three force meshes (padded
// real layout), scaled 1/M.
int pmx_poisson_ctx(pmx_ctx* c, float coef, int deferred) {
  int rc;
  float2* f[3] = {c->cbuf[0], c->cbuf[1], c->cbuf[2]};
  const float* halo = deferred && pmx_fold_deferrable(c) ? c->halo : nullptr;
  // block directions alternate from pass to pass (pass_block), the first
  // against the deposit's and the last against the gather's; the z passes
  // run y's components first, the x component last
  if ((rc = pmx_fft_r2c_inplace(c, (float*)f[0], 1, coef, halo, 1))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, -1, 0))) return rc;
  if ((rc = pmx_poisson_x(c, f, 0, nullptr, 1))) return rc;
  if ((rc = pmx_fft_yinv(c, f, 0))) return rc;
  float scale = (float)(1.0 / (double)c->M);
  float* z[3] = {(float*)f[1], (float*)f[2], (float*)f[0]};
  const int rev[3] = {0, 1, 1};
  return pmx_fft_c2r_inplace(c, z, 3, scale, rev);
}

// Adjoint Poisson on the context buffers: cbuf[0..2] hold the three
// cotangent meshes (padded real; deferred: with the folds of c->halo's three
// channels still to add); on return cbuf[0] holds the density cotangent
// (padded real) times `scale_out`.
int pmx_poisson_adj_ctx(pmx_ctx* c, float scale_out, int deferred) {
  float2* f[3] = {c->cbuf[0], c->cbuf[1], c->cbuf[2]};
  return pmx_poisson_adj_bufs(c, f, scale_out, deferred);
}

// The same on three other mesh buffers of the context's layout.
int pmx_poisson_adj_bufs(pmx_ctx* c, float2* const* f, float scale_out, int deferred) {
  int rc;
  const bool fold = deferred && pmx_fold_deferrable(c);
  // block directions alternate as in pmx_poisson_ctx
  float* z[3] = {(float*)f[0], (float*)f[1], (float*)f[2]};
  const int rev[3] = {1, 1, 1};
  if ((rc = pmx_fft_r2c_inplace(c, z, 3, 0, 0.f, fold ? c->halo : nullptr, rev))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, -1, 0))) return rc;
  if ((rc = pmx_fft_ypair(c, f, -1, 0))) return rc;
  if ((rc = pmx_poisson_x(c, f, 1, nullptr, 1))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, 1, 0))) return rc;
  if ((rc = pmx_fft_c2r_inplace(c, (float*)f[0], scale_out, 1))) return rc;
  return PMX_OK;
}

// Dense complex meshes are rows of n2h float2.
static bool dense_spec_ok(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; }

// The dense caller meshes are the first pass's source and the last pass's
// destination, which saves two copies (the one r2c in white noise to 2LPT at
// 256^3: 2475 -> 2403 us for the whole).  Pointers that the passes' float2
// accesses cannot take still go through the copies.
extern "C" int pmx_rfftn(pmx_ctx* c, const float* in, float* out_c) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && in && out_c, "pmx_rfftn: NULL argument");
  int rc;
  float2* f[1] = {c->cbuf[0]};
  float2* o[1] = {reinterpret_cast<float2*>(out_c)};
  if ((rc = r2c_dense(c, f[0], in))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, -1))) return rc;
  if (dense_spec_ok(out_c)) return pmx_strided_from_to(c, f, c->n2p, o, c->n2h, 1, 0, -1, 0);
  if ((rc = pmx_fft_strided(c, f, 1, 0, -1))) return rc;
  return pmx_copy_rows(c, out_c, 2 * c->n2h, (const float*)f[0], c->rs, 2 * c->n2h);
}

extern "C" int pmx_irfftn(pmx_ctx* c, const float* in_c, float* out) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && in_c && out, "pmx_irfftn: NULL argument");
  int rc;
  float2* f[1] = {c->cbuf[0]};
  float2* in[1] = {reinterpret_cast<float2*>(const_cast<float*>(in_c))};
  if (dense_spec_ok(in_c)) {
    if ((rc = pmx_strided_from_to(c, in, c->n2h, f, c->n2p, 1, 0, 1, 0))) return rc;
  } else {
    if ((rc = pmx_copy_rows(c, (float*)f[0], c->rs, in_c, 2 * c->n2h, 2 * c->n2h))) return rc;
    if ((rc = pmx_fft_strided(c, f, 1, 0, 1))) return rc;
  }
  if ((rc = pmx_fft_strided(c, f, 1, 1, 1))) return rc;
  return pmx_c2r_dense(c, out, f[0], (float)(1.0 / (double)c->M));
}

extern "C" int pmx_poisson_grad(pmx_ctx* c, const float* dens, float coef, float* grad) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && dens && grad, "pmx_poisson_grad: NULL argument");
  int rc;
  if ((rc = pmx_copy_rows(c, (float*)c->cbuf[0], c->rs, dens, c->n[2]))) return rc;
  if ((rc = pmx_poisson_ctx(c, coef))) return rc;
  for (int d = 0; d < 3; ++d)
    if ((rc = pmx_copy_rows(c, grad + (long long)d * c->M, c->n[2], (const float*)c->cbuf[d], c->rs)))
      return rc;
  return PMX_OK;
}

extern "C" int pmx_poisson_grad_adj(pmx_ctx* c, const float* grad_cot, float coef, float* dens_cot) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && grad_cot && dens_cot, "pmx_poisson_grad_adj: NULL argument");
  int rc;
  for (int d = 0; d < 3; ++d)
    if ((rc = pmx_copy_rows(c, (float*)c->cbuf[d], c->rs, grad_cot + (long long)d * c->M, c->n[2])))
      return rc;
  // dens_cot = -coef * sum_d L_d(grad_cot_d), L_d = irfftn (-ik_d) laplace rfftn
  if ((rc = pmx_poisson_adj_ctx(c, (float)(-(double)coef / (double)c->M), 0))) return rc;
  return pmx_copy_rows(c, dens_cot, c->n[2], (const float*)c->cbuf[0], c->rs);
}

// ------------------------------------------------------- power spectrum --
// pmwd/spec_util.py:47-147: per complex cell of the r2c layout, |k| from
// fftfreq(shape, None) in float32 (the integer frequency divided by the
// extent in float64, then rounded, as jnp.fft.fftfreq), P = |F|^2 or
// F conj(G) in float32 (optionally deconvolved by sinc^-deconv per axis),
// the weight N = 2 (1 on the kz = 0 and, for an even n2, Nyquist planes),
// and the bin of |k| among the float64 edges (right: edge < k counts; else
// edge <= k).
//
// |k| and the bin are the same for the cells (+-kx, +-ky) of a kz, so a
// thread takes such a group (1, 2 or 4 cells) at once, and L groups of
// consecutive |ky| one after the other: their sums of k N, Re P N, Im P N and
// N stay in registers (float64) until the bin changes and then go to the
// workgroup's bins in LDS (float64 atomic adds: their order within a
// workgroup is not fixed).  Lanes run along kz, so the loads are whole lines.
// A second kernel adds the workgroups' partials, 32 threads to a sum.
// 512^3, 28 bins: 168 us, 3.2 TB/s of spectrum read (more loads in flight, copies
// of the bins in LDS and fewer edge searches changed nothing); one cell a
// thread with three LDS atomics each took 1190 us, and the sums of the 1024
// partials by one thread each 236 us (now 12).
#define PS_TPB 256
#define PS_BLOCKS 1024
#define PS_RED 32

// |fftfreq| of the index of least magnitude j <= n/2
__device__ __forceinline__ float ps_freq(int j, int n) { return (float)((double)j / (double)n); }

__device__ __forceinline__ float ps_sinc(float x) {
  if (x == 0.f) return 1.f;
  const float px = 3.14159265358979323846f * x;
  return sinf(px) / px;
}

// F and, with CROSS, G: (n0, n1, n2p) spectra, n2h columns used.  nc1: chunks
// of L |ky| values.
template <bool CROSS>
__global__ void __launch_bounds__(PS_TPB)
    powspec_bin_k(const float2* __restrict__ F, const float2* __restrict__ G, int n0, int n1,
                  int n2, int n2h, int n2p, const double* __restrict__ edges, int nedges, int right,
                  int deconv, int L, int nc1, double* __restrict__ part) {
  extern __shared__ double ps_sh[];
  double* acc = ps_sh;                 // 4 * nedges
  double* e = ps_sh + 4 * nedges;      // nedges
  const int h0 = n0 / 2 + 1, h1 = n1 / 2 + 1;
  float* tfy = reinterpret_cast<float*>(e + nedges);  // |fy|, then sinc^-deconv
  float* tsy = tfy + h1;
  for (int i = threadIdx.x; i < 4 * nedges; i += PS_TPB) acc[i] = 0.0;
  for (int i = threadIdx.x; i < nedges; i += PS_TPB) e[i] = edges[i];
  for (int i = threadIdx.x; i < h1; i += PS_TPB) {
    const float fy = ps_freq(i, n1);
    tfy[i] = fy;
    if (deconv) tsy[i] = powf(ps_sinc(fy), (float)-deconv);
  }
  __syncthreads();
  const unsigned total = (unsigned)h0 * nc1 * n2h;
  for (unsigned u = blockIdx.x * PS_TPB + threadIdx.x; u < total; u += gridDim.x * PS_TPB) {
    const unsigned r = u / (unsigned)n2h;
    const int kz = (int)(u - r * n2h);
    const int kx = (int)(r / (unsigned)nc1);
    const int y0 = (int)(r - (unsigned)kx * nc1) * L;
    const int y1 = y0 + L < h1 ? y0 + L : h1;
    const bool x2 = kx != 0 && 2 * kx != n0;  // -kx is another cell
    const float fx = ps_freq(kx, n0), fz = ps_freq(kz, n2);
    float sx = 1.f, sz = 1.f;
    if (deconv) {
      sx = powf(ps_sinc(fx), (float)-deconv);
      sz = powf(ps_sinc(fz), (float)-deconv);
    }
    const float w = (kz == 0 || ((n2 & 1) == 0 && kz == n2 / 2)) ? 1.f : 2.f;
    const long long pa = (long long)kx * n1 * n2p + kz;
    const long long pb = (long long)(x2 ? n0 - kx : kx) * n1 * n2p + kz;
    int bin = nedges;
    double ak = 0.0, ar = 0.0, ai = 0.0, an = 0.0;
    auto flush = [&]() {
      if (bin >= nedges) return;
      atomicAdd(&acc[bin], ak);
      atomicAdd(&acc[nedges + bin], ar);
      if (CROSS) atomicAdd(&acc[2 * nedges + bin], ai);
      atomicAdd(&acc[3 * nedges + bin], an);
    };
#pragma unroll 2
    for (int ky = y0; ky < y1; ++ky) {
      const bool y2 = ky != 0 && 2 * ky != n1;
      const long long ra = (long long)ky * n2p, rb = (long long)(y2 ? n1 - ky : ky) * n2p;
      const long long at[4] = {pa + ra, pa + rb, pb + ra, pb + rb};
      float2 f[4], g[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool on = ((q & 1) == 0 || y2) && ((q & 2) == 0 || x2);
        f[q] = g[q] = make_float2(0.f, 0.f);
        if (on) {
          f[q] = F[at[q]];
          if (CROSS) g[q] = G[at[q]];
        }
      }
      const float fy = tfy[ky];
      const float k = sqrtf((fx * fx + fy * fy) + fz * fz);
      // number of edges below k (right) or at most k (left-inclusive bins)
      const double kd = (double)k;
      int lo = 0, hi = nedges;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const bool below = right ? (e[mid] < kd) : (e[mid] <= kd);
        if (below) lo = mid + 1;
        else hi = mid;
      }
      if (lo != bin) {
        flush();
        bin = lo;
        ak = ar = ai = an = 0.0;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (((q & 1) && !y2) || ((q & 2) && !x2)) continue;
        float pr, pi = 0.f;
        if (CROSS) {
          pr = f[q].x * g[q].x + f[q].y * g[q].y;
          pi = f[q].y * g[q].x - f[q].x * g[q].y;
        } else {
          pr = f[q].x * f[q].x + f[q].y * f[q].y;
        }
        if (deconv) {
          const float sy = tsy[ky];
          pr = ((pr * sx) * sy) * sz;
          pi = ((pi * sx) * sy) * sz;
        }
        ar += (double)(pr * w);
        if (CROSS) ai += (double)(pi * w);
      }
      const double mult = (double)((x2 ? 2 : 1) * (y2 ? 2 : 1));
      ak += mult * (double)(k * w);
      an += mult * (double)w;
    }
    flush();
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 4 * nedges; i += PS_TPB)
    part[(long long)blockIdx.x * 4 * nedges + i] = acc[i];
}

// out[i] = the sum over blocks of part[b * m + i]: PS_RED threads to an i,
// each over every PS_RED-th block in order, then their sums in order.
__global__ void __launch_bounds__(PS_TPB)
    powspec_reduce_k(const double* __restrict__ part, int nblocks, int m, double* __restrict__ out) {
  constexpr int W = PS_TPB / PS_RED;
  __shared__ double sh[PS_TPB];
  const int col = threadIdx.x % W, row = threadIdx.x / W;
  const int i = blockIdx.x * W + col;
  double s = 0.0;
  if (i < m)
    for (int b = row; b < nblocks; b += PS_RED) s += part[(long long)b * m + i];
  sh[threadIdx.x] = s;
  __syncthreads();
  if (row || i >= m) return;
  for (int r = 1; r < PS_RED; ++r) s += sh[r * W + col];
  out[i] = s;
}

// r2c of a caller mesh into context buffer cb (padded layout, all axes)
static int ps_r2c(pmx_ctx* c, const float* in, int cb) {
  int rc;
  float2* f[1] = {c->cbuf[cb]};
  if ((rc = r2c_dense(c, f[0], in))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, -1))) return rc;
  return pmx_fft_strided(c, f, 1, 0, -1);
}

extern "C" int pmx_powspec(pmx_ctx* c, const float* f, const float* g, int nedges,
                           const double* edges, int right, int deconv, double* out) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && f && edges && out, "pmx_powspec: NULL argument");
  PMX_REQUIRE(nedges >= 1 && nedges <= 2048, "pmx_powspec: 1..2048 bin edges");
  PMX_REQUIRE(deconv >= 0 && deconv <= 16, "pmx_powspec: deconv must be in 0..16");
  int rc;
  // the binned sums are read back on the host
  if ((rc = pmx_no_capture(c, "pmx_powspec"))) return rc;
  const int m = 4 * nedges;
  // partial sums of the workgroups, then the reduced sums and the edges
  const long long need = (long long)PS_BLOCKS * m + m + nedges;
  if ((rc = pmx_ensure_red(c, need))) return rc;
  double* part = c->red;
  double* sums = c->red + (long long)PS_BLOCKS * m;
  double* dedges = sums + m;
  PMX_CHECK_HIP(hipMemcpyAsync(dedges, edges, (size_t)nedges * sizeof(double),
                               hipMemcpyHostToDevice, c->stream));
  if ((rc = ps_r2c(c, f, 1))) return rc;
  if (g && (rc = ps_r2c(c, g, 2))) return rc;
  // Groups of |ky| per thread: 8 let a sum stay in registers over a run; a
  // small mesh takes fewer, down to one, before it leaves threads without work.
  const int h0 = c->n[0] / 2 + 1, h1 = c->n[1] / 2 + 1;
  int L = 8;
  while (L > 1 && (long long)h0 * ((h1 + L - 1) / L) * c->n2h < PS_BLOCKS * PS_TPB) L /= 2;
  const int nc1 = (h1 + L - 1) / L;
  const long long units = (long long)h0 * nc1 * c->n2h;
  const int nblk = (int)std::min<long long>((units + PS_TPB - 1) / PS_TPB, PS_BLOCKS);
  const size_t lds = (size_t)(m + nedges) * sizeof(double) + 2 * (size_t)h1 * sizeof(float);
#define PS_BIN(CROSS)                                                                              \
  powspec_bin_k<CROSS><<<nblk, PS_TPB, lds, c->stream>>>(                                          \
      c->cbuf[1], c->cbuf[2], c->n[0], c->n[1], c->n[2], c->n2h, c->n2p, dedges, nedges, right,    \
      deconv, L, nc1, part)
  if (g) PS_BIN(true);
  else PS_BIN(false);
#undef PS_BIN
  PMX_LAUNCH_CHECK();
  constexpr int W = PS_TPB / PS_RED;
  powspec_reduce_k<<<(m + W - 1) / W, PS_TPB, 0, c->stream>>>(part, nblk, m, sums);
  PMX_LAUNCH_CHECK();
  PMX_CHECK_HIP(hipMemcpyAsync(out, sums, (size_t)m * sizeof(double), hipMemcpyDeviceToHost,
                               c->stream));
  PMX_CHECK_HIP(hipStreamSynchronize(c->stream));
  return PMX_OK;
}
