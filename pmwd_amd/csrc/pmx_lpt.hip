// 2LPT initial conditions on the particle grid (pmwd/lpt.py:13-212), their
// adjoint, and the linear modes, with the library's FFT passes.
//
// The displacement is -i k irfftn of D1 pot_1 + D2 pot_2 and the velocity of
// v1 pot_1 + v2 pot_2 (v = a^2 H D'), pot_1 = -modes / (V_cell k^2), pot_2 =
// -rfftn(L) / k^2 with the strain source L = s00 s22 + s00 s11 + s11 s22 -
// s01^2 - s02^2 - s12^2 (lpt.py:40-76, in that order), s_ij =
// irfftn(-k_i k_j pot_1) with Nyquist zeroed for i != j (lpt.py:13-37).  Each
// transform's first and last pass reads and writes what the physics needs:
//   x: lpt_x_k forms three strain spectra from one read of the modes and
//      transforms them; poisson_x_k sums the two potentials on load
//   z: lpt_rows_k transforms the rows of three fields and combines them in
//      registers, to L and its r2c, to the strains' cotangents, or to the
//      particles' displacements and velocities, each written once
// so a strain costs under five mesh reads or writes instead of ten and no particle
// array is read back.  The passes are bound by memory (3.5 to 8 TB/s, the
// larger where a mesh stays in cache).  White noise to 2LPT at 256^3: 2403 ->
// 1190 us; with its gradient at 128^3 (before: tensor ops) 5000 -> 636 us.
// Odd n2 (rows in pairs, no half-length transform) keeps separate z passes.
#include "pmx_fft.h"

// ------------------------------------------------------------- x passes --
// The strain spectra f * pot, f = -k_i k_j, of set 0 (i = j = o) or set 1
// (01, 02, 12; Nyquist zeroed), o = 0..2.
__device__ __forceinline__ float strain_f(int set, int o, float kx, float ky, float kz, float mx,
                                          float my, float mz) {
  if (set == 0) {
    const float k = o == 0 ? kx : (o == 1 ? ky : kz);
    return -k * k;
  }
  return -(o == 2 ? my : mx) * (o == 0 ? my : mz);
}

// From the modes (rows of n2h) to the three fields of a set, transformed
// along x.  One read of the modes serves the three: pot stays in registers.
// 8 values a thread, as poisson_x_k.
template <bool POW2, int LN>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, PFFT_CAP), pfft_v(LN)) : GEN_MAXTPB)
    lpt_x_k(Fields3 fl, const float2* __restrict__ modes, int n0_, int n1, int n2h, int n2p, int B_,
            KTab kt, const float2* __restrict__ tw, float cell_vol, int set) {
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
  int bx, y, bz;
  xcd_block3(bx, y, bz, fl.rev);
  const int c0 = bx * B;
  const int nb = n2h - c0 < B ? n2h - c0 : B;
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  stage_twiddles<TPB>(stw, tw, n0);
  for (int i = threadIdx.x; i < n0; i += tpb<TPB>()) {
    sk[i] = kt.k[0][i];
    skm[i] = kt.km[0][i];
  }
  const float2* g = modes + ((long long)cm.j0 * n1 + y) * n2h + c0 + cm.b;
  const long long gs = (long long)cm.js * n1 * n2h;
  float2 pot[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    pot[it] = make_float2(0.f, 0.f);
    if (live && cm.j0 + it * cm.js < n0) pot[it] = g[it * gs];
  }
  __syncthreads();
  const float ky = kt.k[1][y], my = kt.km[1][y];
  const float kz = live ? kt.k[2][c0 + cm.b] : 0.f, mz = live ? kt.km[2][c0 + cm.b] : 0.f;
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    if (!live || j >= n0) continue;
    const float kx = sk[j];
    float k2 = kx * kx;
    k2 = k2 + ky * ky;
    k2 = k2 + kz * kz;
    const float2 m = make_float2(pot[it].x / cell_vol, pot[it].y / cell_vol);
    pot[it] = k2 != 0.f ? make_float2(-m.x / k2, -m.y / k2) : make_float2(0.f, 0.f);
  }
  const long long es = (long long)n1 * n2p;
  const long long o0 = (long long)y * n2p + c0 + cm.b + (long long)cm.j0 * es;
  for (int o = 0; o < 3; ++o) {
    float2 r[MAXV];
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int j = cm.j0 + it * cm.js;
      if (j >= n0) continue;
      const float f = strain_f(set, o, sk[j], ky, kz, skm[j], my, mz);
      r[it] = make_float2(f * pot[it].x, f * pot[it].y);
    }
    if (o) __syncthreads();
    fft_cols<1, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n0, B, stw, cm);
    float2* d = (o == 0 ? fl.f[0] : (o == 1 ? fl.f[1] : fl.f[2])) + o0;
#pragma unroll
    for (int it = 0; it < MAXV; ++it)
      if (live && cm.j0 + it * cm.js < n0) d[(long long)it * cm.js * es] = r[it];
  }
}

// Adjoint: the x transforms of three fields, each times its factor (sets 0
// and 1: -k_i k_j; set 2: i km_o), summed; out (rows of n2h) (+)= the sum
// times -w scale / k^2, w = 2 on the last axis' interior columns (those that
// stand for two of the full spectrum), 0 at k = 0.
template <bool POW2, int LN>
__global__ void __launch_bounds__(LN ? ct_tpb(LN, ct_cols(LN, PFFT_CAP), pfft_v(LN)) : GEN_MAXTPB)
    lpt_x_adj_k(Fields3 fl, float2* __restrict__ out, int n0_, int n1, int n2, int n2h, int n2p,
                int B_, KTab kt, const float2* __restrict__ tw, float scale, int set, int first) {
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
  int bx, y, bz;
  xcd_block3(bx, y, bz, fl.rev);
  const int c0 = bx * B;
  const int nb = n2h - c0 < B ? n2h - c0 : B;
  const ColMap cm = col_map<TPB>(lB);
  const bool live = cm.b < nb;
  stage_twiddles<TPB>(stw, tw, n0);
  for (int i = threadIdx.x; i < n0; i += tpb<TPB>()) {
    sk[i] = kt.k[0][i];
    skm[i] = kt.km[0][i];
  }
  const float ky = kt.k[1][y], my = kt.km[1][y];
  const float kz = live ? kt.k[2][c0 + cm.b] : 0.f, mz = live ? kt.km[2][c0 + cm.b] : 0.f;
  const long long es = (long long)n1 * n2p;
  const long long o0 = (long long)y * n2p + c0 + cm.b + (long long)cm.j0 * es;
  float2 t[MAXV];
#pragma unroll
  for (int it = 0; it < MAXV; ++it) t[it] = make_float2(0.f, 0.f);
  for (int o = 0; o < 3; ++o) {
    const float2* g = (o == 0 ? fl.f[0] : (o == 1 ? fl.f[1] : fl.f[2])) + o0;
    float2 r[MAXV];
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      r[it] = make_float2(0.f, 0.f);
      if (live && cm.j0 + it * cm.js < n0) r[it] = g[(long long)it * cm.js * es];
    }
    if (o) __syncthreads();
    fft_cols<-1, POW2, LN, ilog2c(BC), MAXV, TPB>(r, s, n0, B, stw, cm);
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int j = cm.j0 + it * cm.js;
      if (j >= n0) continue;
      const float2 v = r[it];
      if (set == 2) {
        const float km = o == 0 ? skm[j] : (o == 1 ? my : mz);
        t[it].x -= km * v.y;
        t[it].y += km * v.x;
      } else {
        const float f = strain_f(set, o, sk[j], ky, kz, skm[j], my, mz);
        t[it].x += f * v.x;
        t[it].y += f * v.y;
      }
    }
  }
  if (!live) return;
  const int col = c0 + cm.b;
  const float w = col == 0 || 2 * col == n2 ? scale : 2.f * scale;
  float2* d = out + ((long long)cm.j0 * n1 + y) * n2h + col;
#pragma unroll
  for (int it = 0; it < MAXV; ++it) {
    const int j = cm.j0 + it * cm.js;
    if (j >= n0) continue;
    const float kx = sk[j];
    float k2 = kx * kx;
    k2 = k2 + ky * ky;
    k2 = k2 + kz * kz;
    float2 v = make_float2(0.f, 0.f);
    if (k2 != 0.f) v = make_float2(-(t[it].x * w) / k2, -(t[it].y * w) / k2);
    float2* q = d + (long long)it * cm.js * n1 * n2h;
    if (!first) v = cadd(v, *q);
    *q = v;
  }
}

// ------------------------------------------------------------- z passes --
// What a z pass makes of the rows of three fields.
enum {
  LPT_DIAG,      // L = s00 s22 + s00 s11 + s11 s22
  LPT_OFF,       // L -= s01^2 + s02^2 + s12^2, then its r2c
  LPT_DIAG_ADJ,  // the fields' r2c after s_ii = Lc (the other two's sum)
  LPT_OFF_ADJ,   // the fields' r2c after s_ij = -2 Lc s_ij
  LPT_MOVE       // particles
};

// Particle p = grid cell p (C order): o[i] (3 floats a particle) = base +
// coef[i] * field.  The base is what the array holds, zero, or the Lagrangian
// grid's displacements (grid: n0 + n1 + n2 per-axis values).
enum { BASE_OWN, BASE_ZERO, BASE_GRID };
struct LptOut {
  float* o[2];
  float coef[2];
  int base[2];
  int n;
  const float* grid;
};

struct LptRows {
  float2* f[3];
  float* L;   // the source, or its cotangent, in padded rows
  float scale;
  LptOut out;
};

__device__ __forceinline__ float lpt_diag(float a, float b, float c) {
  float l = a * c;
  l = l + a * b;
  return l + b * c;
}

template <int OP, int LH, bool SM, bool POW2>
__global__ void __launch_bounds__(LH ? ct_row_tpb(LH, SM) : GEN_MAXTPB, 4)
    lpt_rows_k(LptRows q, long long nrows, int n0, int n1, int n2, int rs, int P_,
               const float2* __restrict__ tw) {
  extern __shared__ float2 s[];
  constexpr int PC = LH ? ct_rows(LH, SM) : 1;
  constexpr int TPB = LH ? ct_row_tpb(LH, SM) : GEN_TPB;
  constexpr int MAXV = LH ? PC * ct_n(LH) / TPB : GEN_MAXV;
  const int H = LH ? ct_n(LH) : n2 >> 1;
  const int P = LH ? PC : P_;
  const RowSplit<LH> rsp(H);
  float2* stw = s + lds_elems(ROWS, H, P);
  const long long row0 = (long long)pass_block(blockIdx.x, gridDim.x, 0) * P;
  const int np = LH ? PC : (int)((nrows - row0) < P ? (nrows - row0) : P);
  const int rsc = rs / 2;
  const int total = np * H;
  stage_twiddles<TPB>(stw, tw, 2 * H);
  float2 v[3][MAXV];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    c2r_half_rows<LH, SM, POW2, MAXV, TPB>(v[i], q.f[i] + row0 * rsc, rsc, s, stw, rsp, H, P, np);
#pragma unroll
    for (int it = 0; it < MAXV; ++it) v[i][it] = make_float2(v[i][it].x * q.scale, v[i][it].y * q.scale);
  }
  float2* L = reinterpret_cast<float2*>(q.L) + row0 * rsc;
  if constexpr (OP == LPT_DIAG || OP == LPT_OFF) {
    if constexpr (OP == LPT_OFF) __syncthreads();  // s is read
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      if (idx >= total) continue;
      const int p = rsp.row(idx), m = rsp.col(idx, p);
      float2* g = L + __umul24(p, rsc) + m;
      if constexpr (OP == LPT_DIAG) {
        *g = make_float2(lpt_diag(v[0][it].x, v[1][it].x, v[2][it].x),
                         lpt_diag(v[0][it].y, v[1][it].y, v[2][it].y));
      } else {
        float2 l = *g;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          l.x = l.x - v[i][it].x * v[i][it].x;
          l.y = l.y - v[i][it].y * v[i][it].y;
        }
        s[lidx<ROWS>(p, m, H, P)] = l;
      }
    }
    if constexpr (OP == LPT_OFF) {
      __syncthreads();
      r2c_half_rows<LH, SM, POW2, MAXV, TPB>(L, rsc, s, stw, rsp, H, P, np);
    }
  }
  if constexpr (OP == LPT_DIAG_ADJ || OP == LPT_OFF_ADJ) {
    float2 l[MAXV];
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      const int p = rsp.row(idx);
      if (idx < total) l[it] = L[__umul24(p, rsc) + rsp.col(idx, p)];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      __syncthreads();  // s is read
#pragma unroll
      for (int it = 0; it < MAXV; ++it) {
        const int idx = threadIdx.x + it * tpb<TPB>();
        if (idx >= total) continue;
        const int p = rsp.row(idx);
        float2 t;
        if constexpr (OP == LPT_DIAG_ADJ) {
          const float2 a = v[(i + 1) % 3][it], b = v[(i + 2) % 3][it];
          t = make_float2(l[it].x * (a.x + b.x), l[it].y * (a.y + b.y));
        } else {
          t = make_float2(-2.f * l[it].x * v[i][it].x, -2.f * l[it].y * v[i][it].y);
        }
        s[lidx<ROWS>(p, rsp.col(idx, p), H, P)] = t;
      }
      __syncthreads();
      r2c_half_rows<LH, SM, POW2, MAXV, TPB>(q.f[i] + row0 * rsc, rsc, s, stw, rsp, H, P, np);
    }
  }
  if constexpr (OP == LPT_MOVE) {
#pragma unroll
    for (int it = 0; it < MAXV; ++it) {
      const int idx = threadIdx.x + it * tpb<TPB>();
      if (idx >= total) continue;
      const int p = rsp.row(idx), m = rsp.col(idx, p);
      const long long row = row0 + p;
      const int x = (int)(row / n1), y = (int)(row - (long long)x * n1);
      float2 b[3] = {};  // the cells' three components one after the other
      if (q.out.base[0] == BASE_GRID) {
        const float bx = q.out.grid[x], by = q.out.grid[n0 + y];
        const float* bz = q.out.grid + n0 + n1 + 2 * m;
        b[0] = make_float2(bx, by);
        b[1] = make_float2(bz[0], bx);
        b[2] = make_float2(by, bz[1]);
      }
      const float g[6] = {v[0][it].x, v[1][it].x, v[2][it].x, v[0][it].y, v[1][it].y, v[2][it].y};
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        if (a >= q.out.n) break;
        float2* o = reinterpret_cast<float2*>(q.out.o[a]) + 3 * (row * H + m);
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          float2 u = make_float2(0.f, 0.f);
          if (q.out.base[a] == BASE_OWN) u = o[e];
          if (q.out.base[a] == BASE_GRID) u = b[e];
          u.x = u.x + q.out.coef[a] * g[2 * e];
          u.y = u.y + q.out.coef[a] * g[2 * e + 1];
          o[e] = u;
        }
      }
    }
  }
}

// The same for rows that the half-length transform does not take (odd n2,
// or particle arrays off float2 alignment), on the transformed meshes.
__global__ void __launch_bounds__(PMX_TPB)
    lpt_cells_k(LptRows q, int op, int n0, int n1, int n2, int rs, long long total) {
  const long long t = (long long)blockIdx.x * PMX_TPB + threadIdx.x;
  if (t >= total) return;
  const long long row = t / n2;
  const int z = (int)(t - row * n2);
  const long long i = row * rs + z;
  float* f[3] = {(float*)q.f[0], (float*)q.f[1], (float*)q.f[2]};
  const float v[3] = {f[0][i], f[1][i], f[2][i]};
  if (op == LPT_DIAG) {
    q.L[i] = lpt_diag(v[0], v[1], v[2]);
  } else if (op == LPT_OFF) {
    float l = q.L[i];
    for (int d = 0; d < 3; ++d) l = l - v[d] * v[d];
    q.L[i] = l;
  } else if (op == LPT_DIAG_ADJ) {
    for (int d = 0; d < 3; ++d) f[d][i] = q.L[i] * (v[(d + 1) % 3] + v[(d + 2) % 3]);
  } else if (op == LPT_OFF_ADJ) {
    for (int d = 0; d < 3; ++d) f[d][i] = -2.f * q.L[i] * v[d];
  } else {
    const int x = (int)(row / n1), y = (int)(row - (long long)x * n1);
    for (int a = 0; a < q.out.n; ++a)
      for (int d = 0; d < 3; ++d) {
        float* o = q.out.o[a] + 3 * t + d;
        float b = 0.f;
        if (q.out.base[a] == BASE_OWN) b = *o;
        if (q.out.base[a] == BASE_GRID) b = q.out.grid[d == 0 ? x : (d == 1 ? n0 + y : n0 + n1 + z)];
        *o = b + q.out.coef[a] * v[d];
      }
  }
}

// f[d] (padded rows) = a ga + b gb of the (N,3) cotangents, N = M cells; a
// workgroup's rows of both move through LDS.
__global__ void __launch_bounds__(PMX_TPB)
    lpt_cot_k(float* __restrict__ f0, float* __restrict__ f1, float* __restrict__ f2,
              float* __restrict__ ga, float* __restrict__ gb, float a, float b, long long n, int n2,
              int rs) {
  constexpr int T3 = 3 * PMX_TPB;
  __shared__ __align__(16) float sh[2 * T3];
  const long long b0 = (long long)blockIdx.x * PMX_TPB;
  const int cnt = (int)(n - b0 < PMX_TPB ? n - b0 : PMX_TPB);
  pmx_stage_in3<2, PMX_TPB>(sh, {{ga, gb}}, b0, cnt);
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= cnt) return;
  const long long p = b0 + q;
  const long long row = p / n2;
  const long long i = row * rs + (p - row * n2);
  f0[i] = a * sh[3 * q] + b * sh[T3 + 3 * q];
  f1[i] = a * sh[3 * q + 1] + b * sh[T3 + 3 * q + 1];
  f2[i] = a * sh[3 * q + 2] + b * sh[T3 + 3 * q + 2];
}

// The Lagrangian grid's (N,3) rows from per-axis values (n0 + n1 + n2 of T),
// 16 bytes a thread: the K particles that those touch, then each element
// picked from them.  Bound by its writes; 256^3's int16 rows 22 us, 64
// with a table load an element.  I: 32-bit where it holds the element count.
template <class T, class I>
__global__ void __launch_bounds__(PMX_TPB)
    lpt_grid_k(T* __restrict__ out, const T* __restrict__ tab, int n0, int n1, int n2, I total) {
  constexpr int V = 16 / sizeof(T), K = (V + 4) / 3;
  const I e0 = ((I)blockIdx.x * PMX_TPB + threadIdx.x) * V;
  if (e0 >= total) return;
  const I p = e0 / 3, row = p / n2;
  const int d = (int)(e0 - 3 * p);
  int z = (int)(p - row * n2);
  int x = (int)(row / n1), y = (int)(row - (I)x * n1);
  T c[K][3];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    c[k][0] = tab[x];
    c[k][1] = tab[n0 + y];
    c[k][2] = tab[n0 + n1 + z];
    if (++z == n2) {
      z = 0;
      if (++y == n1) {
        y = 0;
        x = x + 1 < n0 ? x + 1 : 0;  // past the last particle
      }
    }
  }
  __align__(16) T v[V];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    // element d + e of the particles, d = 0, 1 or 2
    const T a = c[e / 3][e % 3], b = c[(e + 1) / 3][(e + 1) % 3], g = c[(e + 2) / 3][(e + 2) % 3];
    v[e] = d == 0 ? a : (d == 1 ? b : g);
  }
  if (e0 + V <= total) {
    *reinterpret_cast<uint4*>(out + e0) = *reinterpret_cast<const uint4*>(v);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e)
      if (e0 + e < total) out[e0 + e] = v[e];
  }
}

// ------------------------------------------------------------- drivers --
// lpt_x_k and lpt_x_adj_k: (adj) out += from f, else f from in.
static int lpt_x(pmx_ctx* c, float2* const* f, int set, const float* in, float cell_vol, float* out,
                 float scale, int first) {
  const Fields3 fl = {{f[0], f[1], f[2]}, 0};
  const int n0 = c->n[0];
  const int ln = ct_code(n0);
  const int B = ln ? ct_cols(ln, PFFT_CAP) : gen_cols(n0, c->n2h, c->n[1]);
  const int tpb = ln ? ct_tpb(ln, B, pfft_v(ln)) : gen_tpb(n0 * B);
  const dim3 grid((c->n2h + B - 1) / B, c->n[1], 1);
  const size_t lds = lds_bytes(n0, B) + tw_bytes(n0) + 2 * (size_t)n0 * sizeof(float);
  if (int rc = fft_fits("2LPT x pass", n0, n0 * B, PFFT_CAP, lds)) return rc;
  const bool p2 = is_pow2(n0);
  const KTab kt = ktab(c);
  pmx_tic(c, PMX_T_OTHER);
#define LX1(P2, L)                                                                          \
  if (in)                                                                                   \
    lpt_x_k<P2, L><<<grid, tpb, lds, c->stream>>>(fl, (const float2*)in, n0, c->n[1], c->n2h, \
                                                  c->n2p, B, kt, c->tw[0], cell_vol, set);  \
  else                                                                                      \
    lpt_x_adj_k<P2, L><<<grid, tpb, lds, c->stream>>>(fl, (float2*)out, n0, c->n[1], c->n[2], \
                                                      c->n2h, c->n2p, B, kt, c->tw[0], scale, set, first)
#define LX(L)                \
  if (L || p2) {             \
    LX1(true, L);            \
  } else {                   \
    LX1(false, 0);           \
  }
  PMX_CT_SWITCH(ln, LX);
#undef LX
#undef LX1
  pmx_toc(c, PMX_T_OTHER);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

template <int OP>
static int lpt_rows_fused(pmx_ctx* c, const LptRows& q, const RowPlan& r) {
  const long long nrows = (long long)c->n[0] * c->n[1];
  const unsigned nblk = (unsigned)((nrows + r.rows - 1) / r.rows);
  pmx_tic(c, PMX_T_OTHER);
#define LROWS(L, SM, P2)                                                                        \
  lpt_rows_k<OP, L, SM, P2><<<nblk, r.tpb, r.lds, c->stream>>>(q, nrows, c->n[0], c->n[1],      \
                                                               c->n[2], c->rs, r.P, c->tw[2])
#define LROWS_P2(L) LROWS(L, (L > 0), true)
  if (r.lh || is_pow2(r.len)) {
    PMX_CT_SWITCH(r.lh, LROWS_P2);
  } else {
    LROWS(0, false, false);
  }
#undef LROWS_P2
#undef LROWS
  pmx_toc(c, PMX_T_OTHER);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

static int lpt_rows(pmx_ctx* c, int op, LptRows q) {
  const long long nrows = (long long)c->n[0] * c->n[1];
  RowPlan r = row_plan(c->n[2], nrows);
  // three fields' rows in registers leave few wavefronts a CU: small blocks
  // keep more of them at different phases (256^3: LPT_DIAG 80 -> 69 us,
  // LPT_OFF 103 -> 97, LPT_MOVE 118 -> 110)
  if (r.lh && !r.sm) {
    r.sm = true;
    r.P = r.rows = ct_rows(r.lh, true);
    r.tpb = ct_row_tpb(r.lh, true);
    r.lds = lds_bytes(r.len, r.P, ROWS) + tw_bytes(c->n[2]);
  }
  q.scale = (float)(1.0 / (double)c->M);
  bool fused = r.half;
  if (op == LPT_MOVE)
    for (int a = 0; a < q.out.n; ++a) fused = fused && ((uintptr_t)q.out.o[a] & 7) == 0;
  int rc;
  if (fused) {
    if ((rc = fft_fits("2LPT z pass", c->n[2], r.len * r.P, GEN_CAP, r.lds))) return rc;
    switch (op) {
      case LPT_DIAG: return lpt_rows_fused<LPT_DIAG>(c, q, r);
      case LPT_OFF: return lpt_rows_fused<LPT_OFF>(c, q, r);
      case LPT_DIAG_ADJ: return lpt_rows_fused<LPT_DIAG_ADJ>(c, q, r);
      case LPT_OFF_ADJ: return lpt_rows_fused<LPT_OFF_ADJ>(c, q, r);
      default: return lpt_rows_fused<LPT_MOVE>(c, q, r);
    }
  }
  float* f[3] = {(float*)q.f[0], (float*)q.f[1], (float*)q.f[2]};
  const int rev[3] = {0, 0, 0};
  if ((rc = pmx_fft_c2r_inplace(c, f, 3, q.scale, rev))) return rc;
  pmx_tic(c, PMX_T_OTHER);
  lpt_cells_k<<<pmx_blocks(c->M), PMX_TPB, 0, c->stream>>>(q, op, c->n[0], c->n[1], c->n[2], c->rs, c->M);
  pmx_toc(c, PMX_T_OTHER);
  PMX_LAUNCH_CHECK();
  if (op == LPT_OFF) return pmx_fft_r2c_inplace(c, q.L, 0, 0.f);
  if (op == LPT_DIAG_ADJ || op == LPT_OFF_ADJ)
    return pmx_fft_r2c_inplace(c, f, 3, 0, 0.f, nullptr, rev);
  return PMX_OK;
}

// The strains of a set from the modes, up to their z pass.
static int strains(pmx_ctx* c, float2* const* f, int set, const float* modes, float cell_vol) {
  if (int rc = lpt_x(c, f, set, modes, cell_vol, nullptr, 0.f, 0)) return rc;
  return pmx_fft_strided(c, f, 3, 1, 1);
}

// out = base + coef * (-i k pot of src) on the grid, f[0..2] as scratch
static int lpt_move(pmx_ctx* c, float2* const* f, const SpecSrc& src, const LptOut& out) {
  int rc;
  if ((rc = pmx_poisson_x(c, f, 0, &src))) return rc;
  if ((rc = pmx_fft_yinv(c, f, 0))) return rc;
  return lpt_rows(c, LPT_MOVE, {{f[0], f[1], f[2]}, nullptr, 0.f, out});
}

static int ensure_lbuf(pmx_ctx* c) {
  if (c->lbuf) return PMX_OK;
  return pmx_dev_alloc(c, (void**)&c->lbuf, (size_t)c->Mc * sizeof(float2));
}

static int lpt_forward(pmx_ctx* c, const float* modes, float cell_vol, int order, const float* fac,
                       const float* grid, float* disp, float* vel) {
  int rc;
  // every allocation before the first write to disp and vel
  if (order > 1 && (rc = ensure_lbuf(c))) return rc;
  float2* f[3] = {c->cbuf[0], c->cbuf[1], c->cbuf[2]};
  const float2* m = (const float2*)modes;
  const int bd = grid ? BASE_GRID : BASE_OWN, bv = grid ? BASE_ZERO : BASE_OWN;
  if (order == 1)
    return lpt_move(c, f, {m, nullptr, cell_vol, 1.f, 0.f},
                    {{disp, vel}, {fac[0], fac[1]}, {bd, bv}, 2, grid});
  const LptRows q = {{f[0], f[1], f[2]}, (float*)c->lbuf, 0.f, {}};
  if ((rc = strains(c, f, 0, modes, cell_vol))) return rc;
  if ((rc = lpt_rows(c, LPT_DIAG, q))) return rc;
  if ((rc = strains(c, f, 1, modes, cell_vol))) return rc;
  if ((rc = lpt_rows(c, LPT_OFF, q))) return rc;
  float2* l[1] = {c->lbuf};
  if ((rc = pmx_fft_strided(c, l, 1, 1, -1))) return rc;
  if ((rc = lpt_move(c, f, {m, c->lbuf, cell_vol, fac[0], fac[2]},
                     {{disp, nullptr}, {1.f, 0.f}, {bd, 0}, 1, grid})))
    return rc;
  return lpt_move(c, f, {m, c->lbuf, cell_vol, fac[1], fac[3]},
                  {{vel, nullptr}, {1.f, 0.f}, {bv, 0}, 1, grid});
}

extern "C" int pmx_lpt(pmx_ctx* c, const float* modes, float cell_vol, int order,
                       const float* fac, float* disp, float* vel) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && order >= 0 && order <= 2, "pmx_lpt: bad argument (order %d)", order);
  if (order == 0) return PMX_OK;
  PMX_REQUIRE(modes && fac && disp && vel, "pmx_lpt: NULL pointer");
  PMX_REQUIRE(cell_vol > 0.f, "pmx_lpt: cell volume must be positive");
  return lpt_forward(c, modes, cell_vol, order, fac, nullptr, disp, vel);
}

extern "C" int pmx_lpt_grid(pmx_ctx* c, const float* modes, float cell_vol, int order,
                            const float* fac, const float* dtab, float* disp, float* vel) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && order >= 1 && order <= 2, "pmx_lpt_grid: bad argument (order %d)", order);
  PMX_REQUIRE(modes && fac && dtab && disp && vel, "pmx_lpt_grid: NULL pointer");
  PMX_REQUIRE(cell_vol > 0.f, "pmx_lpt_grid: cell volume must be positive");
  return lpt_forward(c, modes, cell_vol, order, fac, dtab, disp, vel);
}

extern "C" int pmx_lpt_vjp(pmx_ctx* c, const float* modes, float cell_vol, int order,
                           const float* fac, const float* disp_cot, const float* vel_cot,
                           float* modes_cot) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && order >= 1 && order <= 2, "pmx_lpt_vjp: bad argument (order %d)", order);
  PMX_REQUIRE((modes || order == 1) && fac && disp_cot && vel_cot && modes_cot,
              "pmx_lpt_vjp: NULL pointer");
  PMX_REQUIRE(cell_vol > 0.f, "pmx_lpt_vjp: cell volume must be positive");
  int rc;
  if (order > 1 && (rc = ensure_lbuf(c))) return rc;
  float2* f[3] = {c->cbuf[0], c->cbuf[1], c->cbuf[2]};
  const int rev[3] = {0, 0, 0};
  const float scale = (float)(1.0 / ((double)c->M * (double)cell_vol));
  auto cot = [&](float2* const* g, float a, float b) {
    pmx_tic(c, PMX_T_OTHER);
    lpt_cot_k<<<pmx_blocks(c->M), PMX_TPB, 0, c->stream>>>(
        (float*)g[0], (float*)g[1], (float*)g[2], const_cast<float*>(disp_cot),
        const_cast<float*>(vel_cot), a, b, c->M, c->n[2], c->rs);
    pmx_toc(c, PMX_T_OTHER);
    PMX_LAUNCH_CHECK();
    return PMX_OK;
  };
  // modes_cot (+)= the set's terms of the three fields after their z pass
  auto add = [&](int set, int first) {
    if (int r = pmx_fft_strided(c, f, 3, 1, -1)) return r;
    return lpt_x(c, f, set, nullptr, 0.f, modes_cot, scale, first);
  };
  if (order > 1) {
    // the source's cotangent, minus the adjoint of -i k laplace
    float2* g[3] = {c->lbuf, c->cbuf[1], c->cbuf[2]};
    if ((rc = cot(g, fac[2], fac[3]))) return rc;
    if ((rc = pmx_poisson_adj_bufs(c, g, (float)(-1.0 / (double)c->M), 0))) return rc;
    const LptRows q = {{f[0], f[1], f[2]}, (float*)c->lbuf, 0.f, {}};
    for (int set = 0; set < 2; ++set) {
      if ((rc = strains(c, f, set, modes, cell_vol))) return rc;
      if ((rc = lpt_rows(c, set ? LPT_OFF_ADJ : LPT_DIAG_ADJ, q))) return rc;
      if ((rc = add(set, set == 0))) return rc;
    }
  }
  if ((rc = cot(f, fac[0], fac[1]))) return rc;
  float* z[3] = {(float*)f[0], (float*)f[1], (float*)f[2]};
  if ((rc = pmx_fft_r2c_inplace(c, z, 3, 0, 0.f, nullptr, rev))) return rc;
  return add(2, order == 1);
}

extern "C" int pmx_grid(const int16_t* ptab, const float* dtab, int n0, int n1, int n2,
                        int16_t* pmid, float* disp, void* stream) {
  PMX_REQUIRE(n0 > 0 && n1 > 0 && n2 > 0, "pmx_grid: extents must be positive");
  PMX_REQUIRE((!pmid || ptab) && (!disp || dtab), "pmx_grid: NULL table");
  PMX_REQUIRE((((uintptr_t)pmid | (uintptr_t)disp) & 15) == 0, "pmx_grid: arrays must be 16-byte aligned");
  const long long total = 3LL * n0 * n1 * n2;
  hipStream_t st = (hipStream_t)stream;
#define GRID(T, V, out, tab)                                                                      \
  do {                                                                                            \
    const unsigned nb = pmx_blocks((total + V - 1) / V);                                          \
    if (total < (1LL << 32) - PMX_TPB * V)                                                        \
      lpt_grid_k<T, unsigned><<<nb, PMX_TPB, 0, st>>>(out, tab, n0, n1, n2, (unsigned)total);     \
    else                                                                                          \
      lpt_grid_k<T, long long><<<nb, PMX_TPB, 0, st>>>(out, tab, n0, n1, n2, total);              \
  } while (0)
  if (pmid) GRID(int16_t, 8, pmid, ptab);
  if (disp) GRID(float, 4, disp, dtab);
#undef GRID
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// ------------------------------------------------------- linear modes --
// modes.py:67-117 on an r2c spectrum in place: m *= scale, then m *=
// sqrt(V P(|k|)) in float32, P evaluated in float64 as boltzmann.py:399-455
// with the transfer table interpolated linearly (numpy.interp, clamped):
// P = amp (k / k_pivot)^n_s (q T(k))^2 d2, amp = 0.32 A_s k_pivot,
// q = pi (c/H_0)^2 / Omega_m, d2 = D(a)^2 or 1; |k| is formed in float32 from
// the float32 wavevectors.
struct PowerPar {
  const double* tk;   // transfer table k (ascending) and T on the device
  const double* tT;
  int ntab;
  double amp, k_pivot, n_s, q, vol, d2;
};

__device__ __forceinline__ double interp_table(double x, const double* __restrict__ xp,
                                               const double* __restrict__ fp, int n) {
  if (x <= xp[0]) return fp[0];
  if (x >= xp[n - 1]) return fp[n - 1];
  // first index with xp[i] > x (searchsorted right), at least 1
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (xp[mid] > x) hi = mid;
    else lo = mid + 1;
  }
  const int i = lo < 1 ? 1 : (lo > n - 1 ? n - 1 : lo);
  const double x0 = xp[i - 1], x1 = xp[i], f0 = fp[i - 1], f1 = fp[i];
  const double t = (x - x0) / (x1 - x0);
  return f0 + t * (f1 - f0);
}

// dst (rows of drow) = src (rows of srow) * scale * sqrt(V P(|k|)), times
// inner on the last axis' interior columns.  |k| is that of the cells
// (+-kx, +-ky) of a kz, so a thread takes the group: the float64 power and
// table search (256^3: 122 us, of which 46 remain) are done once for up to four.
__global__ void __launch_bounds__(PMX_TPB)
    linear_modes_k(const float2* src, int srow, float2* dst, int drow,
                   int n0, int n1, int n2, int n2h, unsigned total, float scale, float inner,
                   KTab kt, PowerPar pp) {
  const unsigned t = blockIdx.x * PMX_TPB + threadIdx.x;
  if (t >= total) return;
  const unsigned h1 = n1 / 2 + 1;
  const unsigned r = t / (unsigned)n2h;
  const int kz = (int)(t - r * n2h);
  const int x = (int)(r / h1);
  const int y = (int)(r - (unsigned)x * h1);
  const float kx = kt.k[0][x], ky = kt.k[1][y], kk = kt.k[2][kz];
  float k2 = kx * kx;
  k2 = k2 + ky * ky;
  k2 = k2 + kk * kk;
  const double k = (double)sqrtf(k2);
  const double T = interp_table(k, pp.tk, pp.tT, pp.ntab);
  const double qT = pp.q * T;
  double P = pp.amp * pow(k / pp.k_pivot, pp.n_s) * (qT * qT);
  if (pp.d2 != 1.0) P = P * pp.d2;
  const float fac = (float)sqrt(P * pp.vol);
  const float sc = kz == 0 || 2 * kz == n2 ? scale : scale * inner;
  const int xs[2] = {x, x == 0 || 2 * x == n0 ? -1 : n0 - x};
  const int ys[2] = {y, y == 0 || 2 * y == n1 ? -1 : n1 - y};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int xx = xs[q >> 1], yy = ys[q & 1];
    if (xx < 0 || yy < 0) continue;
    const long long row = (long long)xx * n1 + yy;
    float2 m = src[row * srow + kz];
    m.x = m.x * sc;
    m.y = m.y * sc;
    dst[row * drow + kz] = make_float2(m.x * fac, m.y * fac);
  }
}

static int linear_modes(pmx_ctx* c, const float2* src, float2* dst, int drow,
                        float scale, float inner, const double* tk, const double* tT, int ntab,
                        const double* par) {
  // the transfer table goes to the context's table scratch, then the stream
  // waits for nothing else (the copy is from pageable host memory)
  const size_t tb = (size_t)2 * ntab * sizeof(double);
  if (c->tab_cap < tb) {
    if (c->tab) pmx_dev_free(c, (void**)&c->tab, c->tab_cap);
    c->tab_cap = 0;
    if (int rc = pmx_dev_alloc(c, (void**)&c->tab, tb)) return rc;
    c->tab_cap = tb;
  }
  PMX_CHECK_HIP(hipMemcpyAsync(c->tab, tk, ntab * sizeof(double), hipMemcpyHostToDevice,
                               c->stream));
  PMX_CHECK_HIP(hipMemcpyAsync(c->tab + ntab, tT, ntab * sizeof(double), hipMemcpyHostToDevice,
                               c->stream));
  PowerPar pp = {c->tab, c->tab + ntab, ntab, par[0], par[1], par[2], par[3], par[4], par[5]};
  const unsigned total = (unsigned)(c->n[0] / 2 + 1) * (c->n[1] / 2 + 1) * c->n2h;
  pmx_tic(c, PMX_T_OTHER);
  linear_modes_k<<<pmx_blocks(total), PMX_TPB, 0, c->stream>>>(
      src, c->n2h, dst, drow, c->n[0], c->n[1], c->n[2], c->n2h, total, scale, inner, ktab(c), pp);
  pmx_toc(c, PMX_T_OTHER);
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

extern "C" int pmx_linear_modes(pmx_ctx* c, float* modes, float scale, const double* tk,
                                const double* tT, int ntab, const double* par) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && modes && tk && tT && par && ntab >= 2, "pmx_linear_modes: bad argument");
  return linear_modes(c, (const float2*)modes, (float2*)modes, c->n2h, scale, 1.f, tk, tT, ntab, par);
}

extern "C" int pmx_linear_modes_vjp(pmx_ctx* c, const float* cot, float scale, const double* tk,
                                    const double* tT, int ntab, const double* par, float* white_cot) {
  PMX_ENTRY(c);
  PMX_REQUIRE(c && cot && tk && tT && par && white_cot && ntab >= 2,
              "pmx_linear_modes_vjp: bad argument");
  int rc;
  float2* f[1] = {c->cbuf[0]};
  // the adjoint of the r2c: M irfftn of the spectrum with its interior halved
  if ((rc = linear_modes(c, (const float2*)cot, f[0], c->n2p, scale, 0.5f, tk, tT, ntab, par))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 0, 1))) return rc;
  if ((rc = pmx_fft_strided(c, f, 1, 1, 1))) return rc;
  return pmx_c2r_dense(c, white_cot, f[0], 1.f);
}
