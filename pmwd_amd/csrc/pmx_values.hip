// CIC of per-particle values and mesh readouts at the default geometry (3D,
// no offset, output cells the mesh's own): the gather, the adjoints of gather
// and scatter with respect to positions and values, and the scatter of one to
// three value channels.  Other geometries and channel counts take the
// kernels of pmx_generic.hip, whose float operations these repeat.
#include "pmx_internal.h"

// Lower and upper cell indices per axis and the flat index of corner j.
struct CicCorners {
  int row[4];  // flat index of (x, y) corner (jx + 2 jy) at z = 0
  int z[2];
};

__device__ __forceinline__ CicCorners cic_corners(const CicAxis ax[3], const MeshGeom& g) {
  CicCorners c;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int x = (j & 1) ? ax[0].hi : ax[0].lo, y = (j & 2) ? ax[1].hi : ax[1].lo;
    c.row[j] = (x * g.n1 + y) * g.n2;
  }
  c.z[0] = ax[2].lo;
  c.z[1] = ax[2].hi;
  return c;
}

// Loads the block's particles through LDS; false for threads beyond the end.
__device__ __forceinline__ bool load_block(const int16_t* __restrict__ pmid,
                                           const float* __restrict__ disp, long long b0, int cnt,
                                           const MeshGeom& g, CicAxis ax[3]) {
  __shared__ __align__(16) float sd[3 * PMX_TPB];
  __shared__ __align__(16) int16_t sp[3 * PMX_TPB];
  pmx_stage_in3<1, PMX_TPB>(sd, {{disp}}, b0, cnt);
  pmx_stage_pmid<PMX_TPB>(sp, pmid, b0, cnt);
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= cnt) return false;
  const int pm[3] = {sp[3 * q], sp[3 * q + 1], sp[3 * q + 2]};
  const float dp[3] = {sd[3 * q], sd[3 * q + 1], sd[3 * q + 2]};
  cic_setup(pm, dp, g, ax);
  return true;
}

// Gather (gather.py:33-77): out[i] = val + sum_j mesh[c_j] w_j, NC channels
// interleaved.  One particle a thread in the caller's order, whose neighbours
// read neighbouring cells; an XCD takes a contiguous eighth of the particles,
// so the rows they share stay in its L2.  Bound by those reads: 16.8 M
// particles on a 256^3 mesh take 251 us, 1028 in the any-geometry kernel,
// whose run-time corner loops keep their arrays in scratch memory.
template <int NC>
__global__ void __launch_bounds__(PMX_TPB)
    cic_gather_k(MeshGeom g, const int16_t* __restrict__ pmid, const float* __restrict__ disp,
                 long long n, const float* __restrict__ mesh, const float* __restrict__ val,
                 float vs, float* __restrict__ out) {
  const long long b0 = (long long)pmx_xcd_block(blockIdx.x, gridDim.x) * PMX_TPB;
  const int cnt = (int)(n - b0 < PMX_TPB ? n - b0 : PMX_TPB);
  CicAxis ax[3];
  if (!load_block(pmid, disp, b0, cnt, g, ax)) return;
  const long long i = b0 + threadIdx.x;
  const CicCorners c = cic_corners(ax, g);
  float m[8][NC];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float* p = mesh + (long long)(c.row[j & 3] + c.z[j >> 2]) * NC;
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) m[j][ch] = p[ch];
  }
#pragma unroll
  for (int ch = 0; ch < NC; ++ch) {
    float t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) t[j] = m[j][ch] * pmx_w(ax, j);
    const float v = val ? val[i * NC + ch] : vs;
    out[i * NC + ch] = v + pmx_tree8(t);
  }
}

// Position and value cotangents (scatter.py:86-121, gather.py:80-116) of
// values v (per particle, or vs) against a mesh f: disp_cot = sum_j (f[c_j].v)
// grad w_j / cell and, when wanted, val_cot = sum_j f[c_j] w_j.  Laid out as
// the gather; disp_cot leaves through LDS in 16-byte stores.  16.8 M
// particles, one channel on a 512^3 mesh: 415 us (1543 in the any-geometry
// kernel); three channels with both cotangents on 256^3: 631 us (3263).
template <int NC>
__global__ void __launch_bounds__(PMX_TPB)
    cic_adj_k(MeshGeom g, const int16_t* __restrict__ pmid, const float* __restrict__ disp,
              long long n, const float* __restrict__ f, const float* __restrict__ val, float vs,
              float* __restrict__ disp_cot, float* __restrict__ val_cot) {
  __shared__ __align__(16) float so[3 * PMX_TPB];
  const long long b0 = (long long)pmx_xcd_block(blockIdx.x, gridDim.x) * PMX_TPB;
  const int cnt = (int)(n - b0 < PMX_TPB ? n - b0 : PMX_TPB);
  CicAxis ax[3];
  if (load_block(pmid, disp, b0, cnt, g, ax)) {
    const long long i = b0 + threadIdx.x;
    const CicCorners c = cic_corners(ax, g);
    float m[8][NC], v[NC];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* p = f + (long long)(c.row[j & 3] + c.z[j >> 2]) * NC;
#pragma unroll
      for (int ch = 0; ch < NC; ++ch) m[j][ch] = p[ch];
    }
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) v[ch] = val ? val[i * NC + ch] : vs;
    if (disp_cot) {
      float gd[3][8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float dc = 0.f;
#pragma unroll
        for (int ch = 0; ch < NC; ++ch) dc = dc + m[j][ch] * v[ch];
        float gw[3];
        pmx_wgrad(ax, j, gw);
#pragma unroll
        for (int a = 0; a < 3; ++a) gd[a][j] = dc * gw[a];
      }
#pragma unroll
      for (int a = 0; a < 3; ++a)
        so[3 * threadIdx.x + a] = pmx_div_cell(pmx_tree8(gd[a]), g.cell, g.inv_cell);
    }
    if (val_cot) {
#pragma unroll
      for (int ch = 0; ch < NC; ++ch) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = m[j][ch] * pmx_w(ax, j);
        val_cot[i * NC + ch] = pmx_tree8(t);
      }
    }
  }
  if (!disp_cot) return;
  __syncthreads();
  pmx_stage_out3<1, PMX_TPB>({{disp_cot}}, so, b0, cnt);
}

// Scatter of NC value channels: one workgroup per tile adds v*w of the tile's
// binned records (values read at the particle's index) to float64 sums in LDS
// over the tile and its +1 shell, then to the interleaved mesh: cells that no
// other tile reaches by a plain read and write, the low faces and the shell
// (which the tiles share) by float32 atomics, 1538 of a tile's 4913 cells
// (atomicAdd, as the any-geometry kernel: the mesh is the caller's memory).
// Float64 sums rather than the density deposit's fixed-point ones: values may
// be of any magnitude, infinite or NaN, and each contribution keeps its
// float32 rounding.  They take about 20 ps a particle and channel, the integer
// ones of a tile-ordered deposit 5; how much of that is the adds, the values'
// way through pidx or the LDS a workgroup holds has not been told apart.  The
// any-geometry kernel is bound by its global float32 atomics, 24
// per particle: 16.8 M particles, three channels on a 256^3 mesh, 17.5 ms
// against 1.0 ms here; one channel 0.5 ms.
// Three channels take 118 KB of LDS, one workgroup of 1024 threads per CU;
// one channel 39 KB, four of 512.
template <int NC>
struct ValTpb {
  static constexpr int v = NC == 1 ? 512 : 1024;
};

template <int NC>
__global__ void __launch_bounds__(ValTpb<NC>::v)
    deposit_vals_k(const float4* __restrict__ rec, const uint32_t* __restrict__ pidx,
                   const uint32_t* __restrict__ tile_start, const uint32_t* __restrict__ tile_count,
                   MeshGeom g, TileGeom tg, const float* __restrict__ val, float vs,
                   float* __restrict__ mesh) {
  constexpr int TPB = ValTpb<NC>::v;
  extern __shared__ double acc[];
  int o[3], s[3], ti[3];
  const int t = (int)pmx_xcd_block(blockIdx.x, gridDim.x);
  tile_origin(t, tg, g, o, s, ti);
  const int LY = s[1] + 1, LZ = s[2] + 1, sxy = LY * LZ;
  const int ltot = (s[0] + 1) * sxy;
  const uint32_t start = tile_start[t], cnt = tile_count[t];
  if (cnt == 0u) return;
  for (int i = threadIdx.x; i < NC * ltot; i += TPB) acc[i] = 0.0;
  __syncthreads();
  // the next round's record and values are loaded before this round's sums
  float4 rn;
  float vn[NC];
  auto fetch = [&](uint32_t q) {
    if (q < cnt) {
      rn = rec[start + q];
      const long long p = pidx[start + q];
#pragma unroll
      for (int ch = 0; ch < NC; ++ch) vn[ch] = val ? val[p * NC + ch] : vs;
    }
  };
  fetch(threadIdx.x);
  for (uint32_t q = threadIdx.x; q < cnt; q += TPB) {
    const float4 r = rn;
    float v[NC];
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) v[ch] = vn[ch];
    fetch(q + TPB);
    int lx, ly, lz;
    pmx_unpack_local(r.w, lx, ly, lz);
    if (lx >= s[0] || ly >= s[1] || lz >= s[2]) continue;
    const float d[3] = {r.x, r.y, r.z};
    const CicFrac fr = pmx_frac_of_d(d);
    const int b = (lx * LY + ly) * LZ + lz;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = (fr.w[0][j & 1] * fr.w[1][(j >> 1) & 1]) * fr.w[2][j >> 2];
      const int li = b + ((j & 1) ? sxy : 0) + ((j & 2) ? LZ : 0) + (j >> 2);
#pragma unroll
      for (int ch = 0; ch < NC; ++ch) unsafeAtomicAdd(&acc[ch * ltot + li], (double)(v[ch] * w));
    }
  }
  __syncthreads();
  // lanes run over a row's cells and channels, which are contiguous in the mesh
  const int row = LZ * NC;
  for (int i = threadIdx.x; i < ltot * NC; i += TPB) {
    const int rr = i / row, e = i - rr * row;
    const int qz = NC == 1 ? e : e / NC, ch = e - qz * NC;
    const int qx = rr / LY, qy = rr - qx * LY;
    const double a = acc[ch * ltot + rr * LZ + qz];
    int x = o[0] + qx, y = o[1] + qy, z = o[2] + qz;
    if (x >= g.n0) x -= g.n0;
    if (y >= g.n1) y -= g.n1;
    if (z >= g.n2) z -= g.n2;
    float* m = mesh + (((long long)x * g.n1 + y) * g.n2 + z) * NC + ch;
    const bool shared = qx == 0 || qy == 0 || qz == 0 || qx == s[0] || qy == s[1] || qz == s[2];
    if (a != 0.0) {
      if (shared)
        atomicAdd(m, (float)a);
      else
        *m = *m + (float)a;
    }
  }
}

// Whether g is the context's own mesh with enmesh's default arguments.
static bool default_geom(const pmx_ctx* c, const pmx_cic_geom* g) {
  if (g->out_cell_size > 0 || g->cell_size != c->cell) return false;
  for (int a = 0; a < 3; ++a)
    if (g->mesh_shape[a] != c->n[a] || g->out_shape[a] != c->n[a] || g->offset[a] != 0.0)
      return false;
  return true;
}

static MeshGeom plain_geom(const pmx_ctx* c) {
  MeshGeom g = pmx_geom_padded(c);
  g.rs = c->n[2];
  return g;
}

#define VAL_SWITCH(nchan, CALL) \
  do {                          \
    if ((nchan) == 1) CALL(1);  \
    else if ((nchan) == 2) CALL(2); \
    else CALL(3);               \
  } while (0)

bool pmx_values_fit(const pmx_ctx* c, const pmx_cic_geom* g, int nchan) {
  return nchan <= 3 && default_geom(c, g);
}

int pmx_values_gather(pmx_ctx* c, const int16_t* pmid, const float* disp, long long n,
                      const float* mesh, int nchan, const float* val, float vs, float* out) {
  const MeshGeom g = plain_geom(c);
#define CALL(NC)                                                                               \
  cic_gather_k<NC><<<pmx_blocks(n), PMX_TPB, 0, c->stream>>>(g, pmid, disp, n, mesh, val, vs, out)
  VAL_SWITCH(nchan, CALL);
#undef CALL
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

int pmx_values_adj(pmx_ctx* c, const int16_t* pmid, const float* disp, long long n, const float* f,
                   int nchan, const float* val, float vs, float* disp_cot, float* val_cot) {
  const MeshGeom g = plain_geom(c);
#define CALL(NC)                                                                             \
  cic_adj_k<NC><<<pmx_blocks(n), PMX_TPB, 0, c->stream>>>(g, pmid, disp, n, f, val, vs, disp_cot, \
                                                          val_cot)
  VAL_SWITCH(nchan, CALL);
#undef CALL
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

static int deposit_vals(pmx_ctx* c, const float* val, float vs, int nchan, float* mesh) {
  const MeshGeom g = plain_geom(c);
  const TileGeom& tg = c->tg;
  const size_t lds =
      (size_t)(tg.tx + 1) * (tg.ty + 1) * (tg.tz + 1) * sizeof(double) * (size_t)nchan;
#define CALL(NC)                                                                               \
  deposit_vals_k<NC><<<(unsigned)c->ntiles, ValTpb<NC>::v, lds, c->stream>>>(                  \
      c->rec, c->pidx, c->tile_start, c->tile_count, g, tg, val, vs, mesh)
  pmx_tic(c, PMX_T_DEPOSIT);
  VAL_SWITCH(nchan, CALL);
  pmx_toc(c, PMX_T_DEPOSIT);
#undef CALL
  PMX_LAUNCH_CHECK();
  return PMX_OK;
}

// Whether n particles' values go by tiles.  Binning is five launches more than
// one of float atomics and costs what it costs however few the channels; then
// one workgroup takes a tile, whether it holds few particles or many.  So the
// atomics win for few particles, for few tiles (idle CUs) and for sparse ones
// (a sum cleared and flushed for little).  Timed over meshes of 16^3 to 512^3
// and 32768 to 16 M particles in random and in cell order, 1 and 3 channels,
// atomics against tiles, us:
//   131072 on 64^3 (64 tiles)  46-68 / 45-49 (1), 135-172 / 57-64 (3);
//   131072 on 48^3 (27 tiles)  40-68 / 48 (1), 122-170 / 67-69 (3);
//   131072 on 32^3 (8 tiles)   45-78 / 61-81 (1), 110-170 / 110-170 (3);
//   1e6 on 16^3 (1 tile)  696-1557 / 1414-3660 (1), 1504-2251 / 3968-10795 (3);
//   131072 on 192^3 (76 a tile)  66-68 / 69-82 (1), 175-177 / 131-140 (3);
//   300000 on 256^3 (73 a tile)  132-141 / 116-132 (1), 387-392 / 253-268 (3);
//   1e6 on 512^3 (31 a tile)  487-517 / 639-695 (1), 1410-1438 / 1674-1735 (3);
//   16 M on 256^3  2988-6134 / 708-1326 (1), 13596-18552 / 1271-1714 (3).
// PMX_VALUES_MIN (c->values_min >= 0) puts a particle count in the rule's place.
static bool values_tiled(const pmx_ctx* c, long long n, int nchan) {
  if (c->values_min >= 0) return n >= c->values_min;
  const long long tiles = nchan > 1 ? 27 : 64, per = nchan > 1 ? 64 : 96;
  return n >= PMX_VALUES_MIN && c->ntiles >= tiles && n >= per * c->ntiles;
}

// The context with c->vbin for its binning scratch (c itself is left alone).
static pmx_ctx with_vbin(const pmx_ctx* c) {
  const BinScratch& b = c->vbin;
  pmx_ctx v = *c;
  v.ptcl_cap = b.ptcl_cap;
  v.rec_cap = b.rec_cap;
  v.caps_n = b.caps_n;
  v.scan_tmp_cap = b.scan_tmp_cap;
  v.caps_valid = b.caps_valid;
  v.rec = b.rec;
  v.pidx = b.pidx;
  v.tile_count = b.tile_count;
  v.tile_start = b.tile_start;
  v.tile_cap = b.tile_cap;
  v.flags = b.flags;
  v.scan_tmp = b.scan_tmp;
  return v;
}

// The binned scatter; false where the caller scatters without it.  It runs on
// scratch of its own (c->vbin), so that a graph captured over any call of the
// context neither loses what it addresses when that scratch grows nor meets
// it while it replays; under capture, and where there is no room for the
// scratch, it is not taken.  Threads that queue on one stream take turns.
bool pmx_values_scatter(pmx_ctx* c, const int16_t* pmid, const float* disp, long long n,
                        const float* val, float vs, int nchan, float* mesh, int* rc) {
  if (!values_tiled(c, n, nchan) || n >= (1LL << 32) - 2048 || pmx_capturing(c)) return false;
  const VbinTurn turn(c);
  if (pmx_ensure_vbin(c, n) != PMX_OK) return false;
  pmx_ctx v = with_vbin(c);
  *rc = pmx_bin_particles(&v, pmid, disp, n);
  c->vbin.caps_valid = v.caps_valid;
  c->vbin.caps_n = v.caps_n;
  if (*rc == PMX_OK) *rc = deposit_vals(&v, val, vs, nchan, mesh);
  return true;
}
