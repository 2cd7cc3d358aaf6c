/*
 * Multigrid preconditioner of the mixed form's inner FP32 sweep on large
 * grids (included by bb_solver.hip).  Jacobi-PCG needs hundreds of iterations
 * because it moves information one cell per iteration; one V-cycle moves it
 * across the box, and PCG with it needs about 10 to 18 iterations for the
 * reference's 1e-8 from phi = 0, with any number of spheres (256^3 with 500:
 * 440 with the Jacobi factor).  What a solve must reach does not change: the
 * FP64 residual of the masked operator under the reference's test.
 *
 * z = M^-1 r is one V-cycle on the cell-centred 7-point operator, symmetric
 * and positive, so PCG stays PCG:
 *   down   x = w r (never stored), d = r - A x, r_c = P^T d
 *   up     x = w r + P z_c,        z = x + w (r - A x)
 * with P the trilinear cell-centred interpolation (3/4, 1/4 per direction;
 * wrapped at a periodic face, the cell itself beyond a wall) and A
 * rediscretised on each level.  A level coarsens the directions whose spacing
 * is within 1.5 of the smallest (a channel's wall-normal direction first), so
 * a point smoother does.  A coarse cell is fluid when more than 3/4 of its
 * cells are; particle cells hold 0 on every level as they do on the grid.
 * The last level, at most MG_LAST_MAX cells, is a Chebyshev polynomial of its
 * operator in one workgroup.
 *
 * One kernel per level and direction of travel.  On the grid itself they are
 * bound by LDS and instruction issue (the vectors of 256^3 stay in the last
 * level cache), on the coarse levels by the latency of their few planes.
 * 256^3 with 500 spheres, us per V-cycle: down 46 on the grid, 13, 9 and 9 on
 * the levels below, the last level 10, up 9, 9, 16 and 47; as four kernels
 * per level (defect, restriction, x, z) 238 in all.  With the search and the
 * update an iteration takes some 290 us against 105 with the Jacobi factor,
 * and a timestep of that box 76 ms against 280; with particles the V-cycle has
 * to be asked for, though (bb_mg = 2).  Without them, where it is the default, a
 * timestep of a 256x128x128 channel takes 2.7 ms against 17 (27.5 kernel by
 * kernel), a solve of 128^3 1.7 ms against 10.2.
 */
#ifndef BB_MG_H
#define BB_MG_H

#define MG_LEVELS 10
#define MG_LAST 4096                  /* cells below which no level coarsens */
#define MG_LAST_MAX 16384             /* cells of the last level at most */
#define MG_OMEGA 0.8f                 /* damping of the Jacobi smoother */
#define MG_WGS 512                    /* workgroups of a level, at least */

/* One level: its cells and strides (cell (0, 0, 0) at the arrays' start),
 * 1/h^2, periodic directions, fluid mask (NULL: all fluid); vec: rows whose
 * runs of four cells can be loaded at once. */
struct MGLevel {
  int nx, ny, nz;
  int sy, sz;
  int perx, pery, perz;
  int vec;
  float hx, hy, hz;                   /* 1/dx^2, ... */
  const uint8_t *m;
};

/* The smoother's weight w: MG_OMEGA over the diagonal away from walls (beside a wall,
 * where the diagonal is smaller, it damps more; as many iterations). */
__device__ inline float mg_w(const MGLevel &L)
{
  return MG_OMEGA / (2.f * (L.hx + L.hy + L.hz));
}

/* A workgroup of the two level kernels: fine cells [x0, x0 + 64) by [y0, y0 +
 * 32) of planes [z0, z1), planes in turn.  Thread t owns the run of four cells
 * 4 (t % 16) of row t / 16; the runs around the tile go to the first threads.
 * z0 is even.  In LDS a row is 72 cells, cell 0 at place 4. */
#define MG_TX 64
#define MG_TY 32
#define MG_P 72

static int mg_planes(const MGLevel &L)
{
  const long t = (long) ((L.nx + MG_TX - 1) / MG_TX) *
                 ((L.ny + MG_TY - 1) / MG_TY);
  int zc = 32;
  while (zc > 2 && t * ((L.nz + zc - 1) / zc) < MG_WGS) zc /= 2;
  return zc;
}

static unsigned mg_groups(const MGLevel &L, int zc)
{
  return (unsigned) (((L.nx + MG_TX - 1) / MG_TX) *
                     ((L.ny + MG_TY - 1) / MG_TY) * ((L.nz + zc - 1) / zc));
}

struct MGBox { int x0, y0, z0, z1; };

__device__ inline MGBox mg_box(const MGLevel &L, int zc)
{
  const int ntx = (L.nx + MG_TX - 1) / MG_TX;
  const int nty = (L.ny + MG_TY - 1) / MG_TY;
  const int b = (int) tile_of_block((long) ntx * nty * ((L.nz + zc - 1) / zc));
  MGBox B;
  B.x0 = b % ntx * MG_TX;
  B.y0 = b / ntx % nty * MG_TY;
  B.z0 = b / (ntx * nty) * zc;
  B.z1 = min(B.z0 + zc, L.nz);
  return B;
}

/* The cell that stands at index g: itself, the wrapped one past a periodic
 * end, else the last (not used there: a wall's face weight is 0, and past the
 * ragged end of a row nothing is stored).  Always in [0, n). */
__device__ inline int mg_wrap(int g, int n, int per)
{
  if (g < 0) g = per ? g + n : 0;
  else if (g >= n) g = per ? g - n : n - 1;
  return min(max(g, 0), n - 1);
}

/* A run of four cells: offsets in the plane, weights of the faces in x and y,
 * place in LDS.  VEC: the four cells are consecutive and of one row (or the
 * run lies past its end), so one offset and the outer faces are enough. */
template <bool VEC> struct MGRun {
  unsigned o[VEC ? 1 : 4];
  float f[VEC ? 2 : 5], fs, fn;
  int p;
};

template <bool VEC>
__device__ inline MGRun<VEC> mg_run(const MGLevel &L, const MGBox &B, int lx,
  int ly, int halo)
{
  MGRun<VEC> R;
  const int y = mg_wrap(B.y0 + ly, L.ny, L.pery);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int x = mg_wrap(B.x0 + lx + e, L.nx, L.perx);
    if (e == 0) R.f[0] = x > 0 || L.perx ? L.hx : 0.f;
    const float f = x < L.nx - 1 || L.perx ? L.hx : 0.f;
    if (!VEC) R.f[e + 1] = f;
    else if (e == 3) R.f[1] = f;
    if (!VEC || e == 0)
      R.o[e] = (unsigned) ((VEC ? min(x, L.nx - 4) : x) + y * L.sy);
  }
  R.fs = y > 0 || L.pery ? L.hy : 0.f;
  R.fn = y < L.ny - 1 || L.pery ? L.hy : 0.f;
  R.p = (ly + halo) * MG_P + lx + 4;
  return R;
}

struct MG4 { float v[4]; };

/* The run at o of a plane; its mask, a byte per cell. */
template <int N>
__device__ inline MG4 mg_load(const float *plane, const unsigned (&o)[N])
{
  MG4 a;
  if constexpr (N == 1) {
    const float4 t = *(const float4 *) ((const char *) plane + 4u * o[0]);
    a.v[0] = t.x; a.v[1] = t.y; a.v[2] = t.z; a.v[3] = t.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      a.v[e] = *(const float *) ((const char *) plane + 4u * o[e]);
  }
  return a;
}

template <int N>
__device__ inline unsigned mg_load_mask(const MGLevel &L, size_t plane,
  const unsigned (&o)[N])
{
  if (L.m == NULL) return ~0u;
  const uint8_t *m = L.m + plane;
  if constexpr (N == 1)
    return *(const unsigned *) (m + o[0]);
  else
    return m[o[0]] | (unsigned) m[o[1]] << 8 | (unsigned) m[o[2]] << 16 |
           (unsigned) m[o[3]] << 24;
}
__device__ inline bool mg_fl(unsigned m, int e)
{
  return (m >> (8 * e) & 255u) != 0;
}

__device__ inline MG4 mg_get(const float *s)
{
  const float4 t = *(const float4 *) s;
  return {{t.x, t.y, t.z, t.w}};
}
__device__ inline void mg_put(float *s, const MG4 &a)
{
  *(float4 *) s = make_float4(a.v[0], a.v[1], a.v[2], a.v[3]);
}

__device__ inline float mg_fz(const MGLevel &L, int k, int up)
{
  return L.perz || k != (up ? L.nz - 1 : 0) ? L.hz : 0.f;
}

/* A of a run: its own values c, the plane in LDS at s (the run's place), the
 * runs below and above with their face weights. */
template <bool VEC>
__device__ inline MG4 mg_lap(const MGRun<VEC> &R, const MGLevel &L,
  const MG4 &c, const float *s, const MG4 &b, float fb, const MG4 &u, float fa)
{
  const MG4 S = mg_get(s - MG_P), N = mg_get(s + MG_P);
  float d[5];
  d[0] = R.f[0] * (c.v[0] - s[-1]);
#pragma unroll
  for (int e = 1; e < 4; e++)
    d[e] = (VEC ? L.hx : R.f[VEC ? 0 : e]) * (c.v[e] - c.v[e - 1]);
  d[4] = R.f[VEC ? 1 : 4] * (s[4] - c.v[3]);
  MG4 a;
#pragma unroll
  for (int e = 0; e < 4; e++)
    a.v[e] = (d[e] - d[e + 1]) + (R.fs * (c.v[e] - S.v[e]) +
             R.fn * (c.v[e] - N.v[e])) + (fb * (c.v[e] - b.v[e]) +
             fa * (c.v[e] - u.v[e]));
  return a;
}

/* Down: r_c = P^T (r - w A r), scaled by the ratio of the cells' volumes, in
 * fluid coarse cells.  Three planes of r pass through LDS with a halo of two
 * cells, the defect of one plane with one; a thread gathers a run of the
 * coarse row below its fine ones, and each coarse plane's sum over its four
 * fine ones stays in registers.  256^3 to 128^3: 46 us (92 MB); a kernel for
 * the defect and one that gathers it: 93; one cell per thread and its weights
 * by table: 62. */
template <bool CX, bool CY, bool CZ, bool VEC>
__global__ void __launch_bounds__(TILE_THREADS, VEC ? 4 : 1)
mg_down_kernel(const CGState *st, MGLevel L, MGLevel C, int zc,
  const float *__restrict__ r, float *__restrict__ rc)
{
  constexpr bool XY = CX || CY;         /* the defect needs its neighbours */
  constexpr int NR = 4 * 16 + 2 * (MG_TY + 4);  /* runs around the tile of r */
  constexpr int ND = 2 * 16 + 2 * (MG_TY + 2);  /* of the defect */
  __shared__ __attribute__((aligned(16))) float s_r[3][(MG_TY + 4) * MG_P];
  __shared__ __attribute__((aligned(16))) float s_d[XY ? (MG_TY + 2) * MG_P : 4];
  if (st->done | st->inner_done) return;
  const MGBox B = mg_box(L, zc);
  const float w = mg_w(L);
  const int t = threadIdx.x, i = t & 15, j = t >> 4;

  const MGRun<VEC> own = mg_run<VEC>(L, B, 4 * i, j, 2);
  const int tr = t - 64, td = t - 32;
  const MGRun<VEC> hr = t < 64
    ? mg_run<VEC>(L, B, 4 * i, j < 2 ? j - 2 : MG_TY + j - 2, 2)
    : mg_run<VEC>(L, B, tr & 1 ? MG_TX : -4, min(tr >> 1, MG_TY + 3) - 2, 2);
  const MGRun<VEC> hd = t < 32
    ? mg_run<VEC>(L, B, 4 * i, j ? MG_TY : -1, 2)
    : mg_run<VEC>(L, B, td & 1 ? MG_TX : -4, min(td >> 1, MG_TY + 1) - 1, 2);

  /* the coarse run: fine rows dy, first coarse cell and row */
  const bool out = j < (CY ? MG_TY / 2 : MG_TY);
  const int fy = CY ? 2 * (j & (MG_TY / 2 - 1)) : j;
  int dy[CY ? 4 : 1];
#pragma unroll
  for (int q = 0; q < (CY ? 4 : 1); q++) {
    int g = B.y0 + fy + (CY ? q - 1 : 0);
    if (CY && !L.pery) g = min(max(g, 0), L.ny - 1);
    dy[q] = (min(g - B.y0, MG_TY) + 1) * MG_P + 4 * i + 4;
  }
  const int gx = B.x0 + 4 * i;
  const bool w0 = CX && !L.perx && gx == 0, w2 = CX && !L.perx && gx + 2 >= L.nx,
             w4 = CX && !L.perx && gx + 4 >= L.nx;
  constexpr int NC = CX ? 2 : 4;
  const int cx = CX ? gx / 2 : gx, cy = CY ? (B.y0 + fy) / 2 : B.y0 + fy;
  const bool oky = out && cy < C.ny;
  const unsigned oc = (unsigned) (min(cx, C.nx - 1) + min(cy, C.ny - 1) * C.sy);

  /* fine planes whose defect is needed */
  const int ka = CZ && (B.z0 > 0 || L.perz) ? B.z0 - 1 : B.z0;
  const int kb = CZ && (B.z1 < L.nz || L.perz) ? B.z1 : B.z1 - 1;
  auto at = [&](int k) {
    return (size_t) mg_wrap(k, L.nz, L.perz) * (size_t) L.sz;
  };
  /* two planes of loads are in flight: on a coarse level nothing but their
   * latency counts (one: 14 us instead of 10) */
  struct In { MG4 o, h; unsigned m, mh; } in[2];
  auto load = [&](int k, In &v) {
    const size_t q = at(k);
    v.o = mg_load(r + q, own.o);
    if (t < NR) v.h = mg_load(r + q, hr.o);
  };
  auto mask = [&](int k, In &v) {
    const size_t q = at(k);
    v.m = mg_load_mask(L, q, own.o);
    if (XY && t < ND) v.mh = mg_load_mask(L, q, hd.o);
  };
  auto put = [&](const In &v, float *s) {
    mg_put(s + own.p, v.o);
    if (t < NR) mg_put(s + hr.p, v.h);
  };
  float *sb = s_r[0], *sc = s_r[1], *sa = s_r[2];
  MG4 b, c;
  {
    In v, u;
    load(ka - 1, v);
    load(ka, u);
    load(ka + 1, in[0]);
    mask(ka, in[0]);
    load(min(ka + 2, kb + 1), in[1]);
    mask(min(ka + 1, kb), in[1]);
    put(v, sb);
    put(u, sc);
    b = v.o;
    c = u.o;
  }
  float cur[NC], prev[NC];
#pragma unroll
  for (int n = 0; n < NC; n++) cur[n] = prev[n] = 0.f;
  const float scale = (CX ? 0.5f : 1.f) * (CY ? 0.5f : 1.f) * (CZ ? 0.5f : 1.f);
  auto store = [&](int kc) {
    const size_t o = (size_t) kc * (size_t) C.sz;
#pragma unroll
    for (int n = 0; n < NC; n++)
      if (oky && cx + n < C.nx)
        rc[o + oc + n] = C.m == NULL || C.m[o + oc + n] ? scale * prev[n] : 0.f;
  };
  /* v: plane k + 1 and the masks of plane k */
  auto step = [&](int k, In &v) {
    const MG4 u = v.o;
    const unsigned m = v.m, mr = v.mh;
    put(v, sa);
    load(min(k + 3, kb + 1), v);
    mask(min(k + 2, kb), v);
    __syncthreads();
    const int kw = mg_wrap(k, L.nz, L.perz);
    const float fb = mg_fz(L, kw, 0), fa = mg_fz(L, kw, 1);
    MG4 d = mg_lap(own, L, c, sc + own.p, b, fb, u, fa);
#pragma unroll
    for (int e = 0; e < 4; e++)
      d.v[e] = mg_fl(m, e) ? c.v[e] - w * d.v[e] : 0.f;
    float g[NC];
    if constexpr (XY) {
      mg_put(s_d + own.p - MG_P, d);
      if (t < ND) {
        const MG4 h = mg_get(sc + hd.p);
        d = mg_lap(hd, L, h, sc + hd.p, mg_get(sb + hd.p), fb,
                   mg_get(sa + hd.p), fa);
#pragma unroll
        for (int e = 0; e < 4; e++)
          d.v[e] = mg_fl(mr, e) ? h.v[e] - w * d.v[e] : 0.f;
        mg_put(s_d + hd.p - MG_P, d);
      }
      __syncthreads();
#pragma unroll
      for (int n = 0; n < NC; n++) g[n] = 0.f;
      if (out) {
#pragma unroll
        for (int q = 0; q < (CY ? 4 : 1); q++) {
          const float wy = !CY ? 1.f : (q == 0 || q == 3 ? 0.25f : 0.75f);
          const MG4 a = mg_get(s_d + dy[q]);
          if constexpr (CX) {
            const float l = w0 ? a.v[0] : s_d[dy[q] - 1];
            const float h = w4 ? a.v[3] : s_d[dy[q] + 4];
            const float n2 = w2 ? a.v[1] : a.v[2];
            g[0] += wy * (0.75f * (a.v[0] + a.v[1]) + 0.25f * (l + n2));
            g[1] += wy * (0.75f * (a.v[2] + a.v[3]) + 0.25f * (a.v[1] + h));
          } else {
#pragma unroll
            for (int n = 0; n < NC; n++) g[n] += wy * a.v[n];
          }
        }
      }
    } else {
#pragma unroll
      for (int n = 0; n < NC; n++) g[n] = d.v[n];
      __syncthreads();                  /* before sb is written again */
    }
    if (!CZ) {
#pragma unroll
      for (int n = 0; n < NC; n++) prev[n] = g[n];
      store(k);
    } else if (k & 1) {
      /* the second plane of coarse k / 2, and a quarter to the next */
      const float wk = !L.perz && k == L.nz - 1 ? 1.f : 0.75f;
#pragma unroll
      for (int n = 0; n < NC; n++) {
        prev[n] = cur[n] + wk * g[n];
        cur[n] = 0.25f * g[n];
      }
    } else {
      const float wk = !L.perz && k == 0 ? 1.f : 0.75f;
#pragma unroll
      for (int n = 0; n < NC; n++) {
        prev[n] += 0.25f * g[n];
        cur[n] += wk * g[n];
      }
      if (k > B.z0) store(k / 2 - 1);
    }
    b = c;
    c = u;
    float *sw = sb;
    sb = sc;
    sc = sa;
    sa = sw;
  };
  for (int k = ka; k <= kb; k += 2) {
    step(k, in[0]);
    if (k < kb) step(k + 1, in[1]);
  }
  /* the last coarse plane below a wall has no fourth plane */
  if (CZ && kb < B.z1) store(B.z1 / 2 - 1);
}

/* Up: x = w r + P z_c and z = x + w (r - A x) in fluid cells, 0 in the others;
 * on the grid itself (gpart) the workgroups' partials of (r, z) in FP64.  x
 * passes through LDS with a halo of one cell, planes k - 1 to k + 1 and the
 * one being written; each coarse plane is interpolated in x and y once.
 * 256^3: 47 us (159 MB); a kernel for x and one for z: 86; one cell per thread:
 * 90. */
template <bool CX, bool CY, bool CZ, bool VEC>
__global__ void __launch_bounds__(TILE_THREADS, VEC ? 4 : 1)
mg_up_kernel(const CGState *st, MGLevel L, MGLevel C, int zc,
  const float *__restrict__ r, const float *__restrict__ zcoarse,
  float *__restrict__ z, double *__restrict__ gpart)
{
  constexpr int NH = 2 * 16 + 2 * MG_TY;        /* runs around the tile */
  __shared__ __attribute__((aligned(16))) float s_x[4][(MG_TY + 2) * MG_P];
  if (st->done | st->inner_done) return;
  const MGBox B = mg_box(L, zc);
  const float w = mg_w(L);
  const int t = threadIdx.x, i = t & 15, j = t >> 4, th = t - 32;
  const bool ring = t < NH;
  const int hx = t < 32 ? 4 * i : (th & 1 ? MG_TX : -4);
  const int hy = t < 32 ? (j ? MG_TY : -1) : min(th >> 1, MG_TY - 1);
  const MGRun<VEC> own = mg_run<VEC>(L, B, 4 * i, j, 1),
                   h = mg_run<VEC>(L, B, hx, hy, 1);

  /* the coarse cells that a run interpolates from: offsets in x (CX: the one
   * beside, the two that it lies in, the other beside; else its own four) and
   * rows */
  struct Src { unsigned x[4], y0, y1; };
  auto src = [&](int lx, int ly) {
    Src S;
    const int gx = B.x0 + lx;
#pragma unroll
    for (int e = 0; e < 4; e++)
      S.x[e] = (unsigned) mg_wrap((CX ? (gx >> 1) - 1 : gx) + e, C.nx, C.perx);
    if (VEC) {
      if (CX) S.x[1] = min(S.x[1], (unsigned) C.nx - 2u);
      else S.x[0] = min(S.x[0], (unsigned) C.nx - 4u);
    }
    const int y = B.y0 + ly;
    S.y0 = (unsigned) (mg_wrap(CY ? y >> 1 : y, C.ny, C.pery) * C.sy);
    S.y1 = (unsigned) (mg_wrap(CY ? (y >> 1) + (y & 1 ? 1 : -1) : y, C.ny,
                               C.pery) * C.sy);
    return S;
  };
  const Src co = src(4 * i, j), ch = src(hx, hy);
  auto at = [](const float *p, unsigned o) {
    return (const float *) ((const char *) p + 4u * o);
  };
  auto row = [&](const float *p, const Src &S, unsigned y) {
    MG4 a;
    if constexpr (CX) {
      const float l = *at(p, S.x[0] + y), h = *at(p, S.x[3] + y);
      float2 m;
      if constexpr (VEC) m = *(const float2 *) at(p, S.x[1] + y);
      else m = make_float2(*at(p, S.x[1] + y), *at(p, S.x[2] + y));
      a.v[0] = 0.75f * m.x + 0.25f * l;
      a.v[1] = 0.75f * m.x + 0.25f * m.y;
      a.v[2] = 0.75f * m.y + 0.25f * m.x;
      a.v[3] = 0.75f * m.y + 0.25f * h;
    } else if constexpr (VEC) {
      const unsigned o[1] = {S.x[0] + y};
      a = mg_load(p, o);
    } else {
      const unsigned o[4] = {S.x[0] + y, S.x[1] + y, S.x[2] + y, S.x[3] + y};
      a = mg_load(p, o);
    }
    return a;
  };
  /* coarse plane k interpolated in x and y */
  auto plane = [&](int k, const Src &S) {
    const float *p = zcoarse + (size_t) mg_wrap(k, C.nz, C.perz) * (size_t) C.sz;
    MG4 a = row(p, S, S.y0);
    if constexpr (CY) {
      const MG4 q = row(p, S, S.y1);
#pragma unroll
      for (int e = 0; e < 4; e++) a.v[e] = 0.75f * a.v[e] + 0.25f * q.v[e];
    }
    return a;
  };
  struct In { MG4 o, h; unsigned m, mh; } in[2];
  auto load = [&](int k, In &v) {
    const size_t q = (size_t) mg_wrap(k, L.nz, L.perz) * (size_t) L.sz;
    v.o = mg_load(r + q, own.o);
    v.m = mg_load_mask(L, q, own.o);
    if (ring) {
      v.h = mg_load(r + q, h.o);
      v.mh = mg_load_mask(L, q, h.o);
    }
  };
  /* of the plane in the making: the coarse plane that it lies in, the one on
   * its side, the next of them read ahead (the tile's run, the ring's) */
  MG4 po, ph, so, sh = {}, no, nh = {};
  auto ahead = [&](int k) {
    no = plane(k, co);
    if (ring) nh = plane(k, ch);
  };
  auto next = [&](int k) {
    if (CZ && (k & 1)) {
      so = no;
      sh = nh;
    } else {
      so = po;
      sh = ph;
      po = no;
      ph = nh;
    }
  };
  auto make = [&](const In &v, float *s) {
    MG4 x;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float p = CZ ? 0.75f * po.v[e] + 0.25f * so.v[e] : po.v[e];
      x.v[e] = mg_fl(v.m, e) ? w * v.o.v[e] + p : 0.f;
    }
    mg_put(s + own.p, x);
    if (ring) {
      MG4 y;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float p = CZ ? 0.75f * ph.v[e] + 0.25f * sh.v[e] : ph.v[e];
        y.v[e] = mg_fl(v.mh, e) ? w * v.h.v[e] + p : 0.f;
      }
      mg_put(s + h.p, y);
    }
    return x;
  };
  const int z0 = B.z0;
  MG4 xb, xc, rc;
  unsigned mc;
  {
    In v, u;
    load(z0 - 1, v);
    load(z0, u);
    ahead(CZ ? z0 / 2 - 1 : z0 - 1);
    po = no;
    ph = nh;
    ahead(CZ ? z0 / 2 : z0);
    so = no;
    sh = nh;
    load(z0 + 1, in[0]);
    load(min(z0 + 2, B.z1), in[1]);
    xb = make(v, s_x[0]);
    next(z0);
    ahead(CZ ? z0 / 2 + 1 : z0 + 1);
    xc = make(u, s_x[1]);
    rc = u.o;
    mc = u.m;
  }
  const int gx = B.x0 + 4 * i;
  const bool oky = B.y0 + j < L.ny;
  double acc = 0.0;
  /* v: plane k + 1 */
  auto step = [&](int k, In &v) {
    const int ib = k - z0;              /* s_x[ib & 3] holds plane k - 1 */
    next(k + 1);
    const MG4 xa = make(v, s_x[(ib + 2) & 3]), ra = v.o;
    const unsigned ma = v.m;
    load(min(k + 3, B.z1), v);
    if (!CZ) ahead(k + 2);
    else if (k & 1) ahead((k + 3) / 2);
    __syncthreads();
    MG4 a = mg_lap(own, L, xc, s_x[(ib + 1) & 3] + own.p, xb, mg_fz(L, k, 0),
                   xa, mg_fz(L, k, 1));
#pragma unroll
    for (int e = 0; e < 4; e++)
      a.v[e] = mg_fl(mc, e) ? xc.v[e] + w * (rc.v[e] - a.v[e]) : 0.f;
    float *o = z + (size_t) k * (size_t) L.sz;
    if (oky && gx + 3 < L.nx) {
      if constexpr (VEC)
        *(float4 *) ((char *) o + 4u * own.o[0]) =
          make_float4(a.v[0], a.v[1], a.v[2], a.v[3]);
      else
#pragma unroll
        for (int e = 0; e < 4; e++) o[own.o[e]] = a.v[e];
      acc += ((double) rc.v[0] * (double) a.v[0] +
              (double) rc.v[1] * (double) a.v[1]) +
             ((double) rc.v[2] * (double) a.v[2] +
              (double) rc.v[3] * (double) a.v[3]);
    } else if (!VEC && oky) {
#pragma unroll
      for (int e = 0; e < 3; e++)
        if (gx + e < L.nx) {
          o[own.o[VEC ? 0 : e]] = a.v[e];
          acc += (double) rc.v[e] * (double) a.v[e];
        }
    }
    xb = xc;
    xc = xa;
    rc = ra;
    mc = ma;
  };
  for (int k = z0; k < B.z1; k += 2) {
    step(k, in[0]);
    if (k + 1 < B.z1) step(k + 1, in[1]);
  }
  if (gpart) tile_partial(acc, gpart, tile_of_block(gridDim.x));
}

/* The last level in one workgroup: z = q(A) r, q the Chebyshev polynomial of
 * degree `degree` that makes 1 - t q(t) smallest on [lmin, lmax].  A system
 * without particles is singular (constants): the mean is taken out.  Q cells
 * per thread. */
template <int Q>
__global__ void __launch_bounds__(1024)
mg_last_kernel(const CGState *st, MGLevel L, float lmin, float lmax,
  int degree, int singular, const float *__restrict__ r,
  float *__restrict__ z)
{
  __shared__ float s_d[1024 * Q];
  __shared__ float s_sum[16];
  if (st->done | st->inner_done) return;
  const int n = L.nx * L.ny * L.nz, t = threadIdx.x, s2 = L.nx * L.ny;
  float res[Q], x[Q], d[Q];
  /* which of a cell's six neighbours lie in the box (bits 0 to 5: west, east,
   * south, north, below, above), and bit 6 in a fluid cell; a level of
   * MG_LAST_MAX cells may be that long in one direction */
  int at[Q];
  float sum = 0.f;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int c = t + 1024 * q;
    const bool on = c < n && (L.m == NULL || L.m[c]);
    res[q] = on ? r[c] : 0.f;
    sum += res[q];
    const int cx = c % L.nx, cy = (c / L.nx) % L.ny, cz = c / s2;
    at[q] = (cx > 0) | (cx < L.nx - 1) << 1 | (cy > 0) << 2 |
            (cy < L.ny - 1) << 3 | (cz > 0) << 4 | (cz < L.nz - 1) << 5 |
            on << 6;
  }
  if (singular) {
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, WAVE);
    if ((t & 63) == 0) s_sum[t >> 6] = sum;
    __syncthreads();
    float tot = 0.f;
    for (int i = 0; i < 16; i++) tot += s_sum[i];
#pragma unroll
    for (int q = 0; q < Q; q++)
      if (at[q] >> 6) res[q] -= tot / (float) n;
  }
  const float th = 0.5f * (lmax + lmin), de = 0.5f * (lmax - lmin);
  const float sg = th / de;
  float rho = 1.f / sg;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    x[q] = 0.f;
    d[q] = res[q] / th;
  }
  for (int it = 1; it < degree; it++) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++) s_d[t + 1024 * q] = d[q];
    __syncthreads();
    const float rn = 1.f / (2.f * sg - rho);
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int i = t + 1024 * q;
      const int f = at[q];
      const float c = d[q];
      float a = 0.f;
      if (f >> 6) {
        /* beyond a wall: the cell itself, no difference */
        const int w = f & 1 ? i - 1 : (L.perx ? i + L.nx - 1 : i);
        const int e = f & 2 ? i + 1 : (L.perx ? i - L.nx + 1 : i);
        const int s = f & 4 ? i - L.nx : (L.pery ? i + s2 - L.nx : i);
        const int o = f & 8 ? i + L.nx : (L.pery ? i - s2 + L.nx : i);
        const int b = f & 16 ? i - s2 : (L.perz ? i + n - s2 : i);
        const int u = f & 32 ? i + s2 : (L.perz ? i - n + s2 : i);
        a = L.hx * ((c - s_d[w]) + (c - s_d[e]))
          + L.hy * ((c - s_d[s]) + (c - s_d[o]))
          + L.hz * ((c - s_d[b]) + (c - s_d[u]));
      }
      x[q] += c;
      res[q] -= a;
      d[q] = rn * rho * c + 2.f * rn / de * res[q];
    }
    rho = rn;
  }
#pragma unroll
  for (int q = 0; q < Q; q++)
    if (t + 1024 * q < n) z[t + 1024 * q] = x[q] + d[q];
}

/* A coarse cell is fluid when more than 3/4 of its cells are. */
__global__ void __launch_bounds__(256)
mg_mask_kernel(MGLevel F, MGLevel C, int cx, int cy, int cz,
  uint8_t *__restrict__ m)
{
  const int x = blockIdx.x * 64 + (threadIdx.x & 63);
  const int y = blockIdx.y * 4 + (threadIdx.x >> 6), z = blockIdx.z;
  if (x >= C.nx || y >= C.ny) return;
  int s = 0;
  for (int q = 0; q < (1 << (cx + cy + cz)); q++) {
    const int qx = cx & q, qy = cy & (q >> cx), qz = cz & (q >> (cx + cy));
    s += F.m[(unsigned) (((x << cx) + qx) + ((y << cy) + qy) * F.sy) +
             (unsigned) ((z << cz) + qz) * (unsigned) F.sz] != 0;
  }
  m[(unsigned) (x + y * C.sy) + (unsigned) z * (unsigned) C.sz] =
    4 * s > 3 << (cx + cy + cz);
}

/* A sweep that starts with no direction: beta multiplies zeros. */
__global__ void mg_start_kernel(CGState *st)
{
  st->mg = 1;
  st->rzs[0] = st->rzs[1] = 1.;
}

/* The singular system (no particles) fixes phi up to a constant.  The Jacobi
 * form keeps the mean of D phi, D the diagonal; so does this: tile partials
 * of D e, and phi += e less that mean (sd: the sum of D), e = 0. */
__global__ void __launch_bounds__(TILE_THREADS)
mg_mean_kernel(DevDom D, InvMTab T, const float *__restrict__ e,
  double *__restrict__ gpart)
{
  TILE_PROLOGUE
  double acc = 0.0;
  if (colok)
    for (int k = k0; k <= k1; k++)
      acc += (double) e[gidx(C, x, j, k)] / invm_at(T, D, x, j, k);
  tile_partial(acc, gpart, tile);
}

__global__ void __launch_bounds__(TILE_THREADS)
mg_fold_kernel(DevDom D, const double *__restrict__ mpart, long ntiles,
  double sd, double *__restrict__ phi, float *__restrict__ e)
{
  const double mean = tile_block_sum(mpart, ntiles) / sd;
  TILE_PROLOGUE
  if (!colok) return;
  for (int k = k0; k <= k1; k++) {
    long c = gidx(C, x, j, k);
    phi[c] += (double) e[c] - mean;
    e[c] = 0.f;
  }
}

/* The test that ends an inner sweep (cg_continue's, on the (r, D^-1 r) that
 * the update kernel left: search and update go by (r, z)). */
__global__ void __launch_bounds__(TILE_THREADS)
mg_check_kernel(CGState *st, int q, const double *__restrict__ rpart, long n)
{
  if (st->done | st->inner_done) return;
  const double s = tile_block_sum(rpart, n);
  if (threadIdx.x != 0) return;
  st->rz1 = s;
  if (s <= st->tol2*st->sp_rhs || s <= st->relup*st->rz_ref || isnan(s)) {
    st->q = q;
    st->nan_flag = isnan(s) ? 1 : 0;
    st->inner_done = 1;
  }
}

#endif
