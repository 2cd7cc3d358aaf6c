/*
 * The whole PCG sweep in one launch, for grids whose CG vectors fit the
 * register files of the chip (included by bb_solver.hip, whose operators,
 * CG state and stopping test it uses).
 *
 * One 512-thread workgroup per CU holds NT tiles of 64 x 8 x 8 cells stacked
 * in z: lane x, wavefront y, and each thread the 8 NT cells of its column, r,
 * p, A p and phi in registers from the first iteration to the last.  Per
 * iteration a workgroup reads the residual of the cells around its tiles
 * (and forms their search direction itself, with the arithmetic their owner
 * uses), passes the direction to its own neighbours through LDS, and meets
 * the other workgroups twice, at the two dot products.
 *
 * What bounds an iteration that is launched kernel by kernel on these grids
 * is latency, not bytes: two launches, in each of them the reduction of every
 * tile partial at the start, and the gap between them (64^3: 10.1 + 7.2 us of
 * kernels where 40 B per cell take 2 us; 16^3: 9.2 + 6.8 us and gaps).  Here
 * the two meetings are most of what is left: 1.2 us each with 4 workgroups,
 * 2.8 us with 64, 3.7 us with 256 (a meeting alone); then one trip to memory
 * for the cells around, and with many cells per thread the arithmetic.  The
 * host reads the state once per sweep instead of once per 16 iterations.
 * Microseconds per iteration, kernel by kernel -> in one launch:
 *   FP64: cavity 16^3 17 -> 5.7, 32^3 28 -> 5.9; channel 65 x 33 x 31
 *   33 -> 7.8; spheres 64^3 18 -> 8.3, 128^3 34 -> 16.2 (two tiles);
 *   FP32: channel 150 x 130 x 94 44 -> 17.6, 256 x 128 x 128 34 -> 21.7
 *   (four tiles; without the V-cycle that it takes by default).
 *
 * A meeting: each workgroup stores its tile partials into its slots of the
 * current set by 8-byte device-scope stores, and every thread waits for the
 * slots it adds up; a slot that nobody has written holds MEET_EMPTY.  The
 * sets take turns (MEET_SETS): a workgroup that publishes meeting s has seen
 * every slot of s - 1, so all have left s - 2, whose slots its owners set back
 * to MEET_EMPTY for s + 2.  Data that crosses workgroups (boundary r and phi)
 * is stored and loaded at device scope too, and a workgroup's stores have
 * completed (s_waitcnt vmcnt(0) in every wavefront, then the barrier) before
 * it publishes the meeting after which others read them.  The launch is
 * cooperative, so all workgroups are resident; every wait gives up after
 * a number of polls (seconds) all the same, and the host then starts again
 * kernel by kernel from phi = 0, or from the phi that it finds: workgroups that
 * ended the sweep have stored theirs by then, which the stopping test allows.
 *
 * Arithmetic, dot-product order and stopping test are those of the search and
 * update kernels: same bits, same iteration counts.
 */
#ifndef BB_RESIDENT_H
#define BB_RESIDENT_H

typedef unsigned long long u64;
#define MEET_EMPTY 0xffffffffffffffffull
#define MEET_SETS 4
#define MEET_SLOTS 1024               /* tiles of the largest grid */

template <typename V>
__device__ inline V dev_load(const V *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename V>
__device__ inline void dev_store(V *p, V v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* Every store of this wavefront has completed. */
__device__ inline void stores_done(void)
{
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

__global__ void __launch_bounds__(256) meet_clear_kernel(u64 *slots)
{
  slots[blockIdx.x * 256 + threadIdx.x] = MEET_EMPTY;
}

/* The state a sweep starts from and leaves. */
template <typename V> struct Sweep {
  V *r;                               /* residual in, boundary exchange */
  V *phi;                             /* phi (plain) or e (mixed) */
  V *pa, *pb;                         /* direction of odd and even iterations */
  const double *rhs;                  /* plain: b of the refreshed residual */
  const uint8_t *fluid;
  u64 *slots;
  const double *rpart;                /* tile partials of (r, z) so far */
  int q0, first;                      /* iterations done; start with p = z */
  int qmax;                           /* last iteration allowed */
  int spins;                          /* polls before a wait gives up */
  double rhs_min;                     /* plain: no sweep for (b, b) below it */
};

/* total = canonical sum of the slots of set `m & 3` once all `n` are there;
 * false: gave up.  s_v: 512 doubles of LDS, s_bad: set by whoever gives up
 * (cleared before the sweep). */
__device__ inline bool meet(u64 *slots, unsigned m, int n, int most,
  double *s_v, int *s_bad, double *total)
{
  const int t = threadIdx.x;
  const u64 *set = slots + (size_t) (m & (MEET_SETS - 1)) * MEET_SLOTS;
  double a = 0.0, b = 0.0;
  bool bad = false;
  if (t < n) {
    u64 w;
    int spins = 0;
    while ((w = dev_load(&set[t])) == MEET_EMPTY)
      if (++spins > most) { bad = true; break; }
    a = 0.0 + __longlong_as_double((long long) w);
  }
  if (t + TILE_THREADS < n) {
    u64 w;
    int spins = 0;
    while ((w = dev_load(&set[t + TILE_THREADS])) == MEET_EMPTY)
      if (++spins > most) { bad = true; break; }
    b = 0.0 + __longlong_as_double((long long) w);
  }
  s_v[t] = a + b;
  if (bad) *s_bad = 1;
  __syncthreads();
  if (*s_bad) return false;
  /* the halving tree over 512 values, every wavefront for itself: steps
   * 256, 128 and 64 between the eight values of a lane, then the lanes */
  const int l = t & (WAVE - 1);
  double v = ((s_v[l] + s_v[l + 256]) + (s_v[l + 128] + s_v[l + 384])) +
             ((s_v[l + 64] + s_v[l + 320]) + (s_v[l + 192] + s_v[l + 448]));
  v = tree_step<32>(v);
  v = tree_step<16>(v);
  v = tree_step<8>(v);
  v = tree_step<4>(v);
  v = tree_step<2>(v);
  v = tree_step<1>(v);
  *total = lane_get(v, 0);
  return true;
}

/* Publishes the row values s_w[tile][row] of this workgroup's `nt` tiles
 * for meeting m, and frees the slots of meeting m + 2.  Called by all
 * threads between two barriers; `stride` is the distance of stacked tiles in
 * the tile numbering. */
__device__ inline void publish(u64 *slots, unsigned m, int tile0, int stride,
  int nt, const double (*s_w)[TILE_Y])
{
  const int t = threadIdx.x;
  if (t >= nt) return;
  u64 *set = slots + (size_t) (m & (MEET_SETS - 1)) * MEET_SLOTS;
  u64 *next = slots + (size_t) ((m + 2) & (MEET_SETS - 1)) * MEET_SLOTS;
  const double *w = s_w[t];
  const double v = ((w[0] + w[1]) + (w[2] + w[3])) +
                   ((w[4] + w[5]) + (w[6] + w[7]));
  const int s = tile0 + t * stride;
  /* the slot freed at the last publication is free for all before this
   * one can be seen; long done, it costs no wait here */
  stores_done();
  dev_store(&set[s], isnan(v) ? 0x7ff8000000000000ull
                              : (u64) __double_as_longlong(v));
  dev_store(&next[s], (u64) MEET_EMPTY);
}

/* x where bit i of `live` is set, else +0. */
template <typename V>
__device__ inline V keep(V x, unsigned live, int i)
{
  const int m = ((int) (live << (31 - i))) >> 31;
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(float, __builtin_bit_cast(int, x) & m);
  } else {
    typedef int I2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(double, __builtin_bit_cast(I2, x) & m);
  }
}

template <typename V, bool MIXED, bool MASK, int NT>
__global__ void __launch_bounds__(TILE_THREADS)
resident_kernel(DevDom D, CoefT<V> K, InvMT<V> T, CGState *st, int ntiles,
  Sweep<V> S)
{
  constexpr int KZ = TILE_Z * NT;
  constexpr int NY = KZ / 4;          /* y halo entries per thread */
  constexpr int GR = sizeof(V) == 8 ? 2 : 4;   /* cells in flight at once */
  /* the largest columns (16 FP64 or 32 FP32 cells) keep phi in LDS, which a
   * thread reads and writes once per iteration */
  constexpr bool FAR = KZ * sizeof(V) >= 128;
  __shared__ V s_phi[FAR ? KZ * TILE_THREADS : 1];
  constexpr int RX = LX + 1;          /* a column for threads without a cell */
  __shared__ V s_p[KZ * LY * RX];     /* direction (or phi) and its halo */
  __shared__ V s_invm[27];
  __shared__ double s_v[TILE_THREADS];
  __shared__ double s_w[NT][TILE_Y];
  __shared__ int s_bad;
  if (st->done | st->inner_done) return;
  const int t = threadIdx.x;
  const int lane = t & (WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  if (!MIXED && st->sp_rhs < S.rhs_min) {
    if (blockIdx.x == 0 && t == 0) st->done = 1;
    return;
  }
  if (t < 27) s_invm[t] = T.v[t];
  if (t == 0) s_bad = 0;
  for (int e = t; e < KZ * LY * RX; e += TILE_THREADS) s_p[e] = 0;

  const Grid &C = D.cc;
  const unsigned sz0 = (unsigned) C.sz;
  const int ntx = (D.nx + TILE_X - 1) / TILE_X;
  const int nty = (D.ny + TILE_Y - 1) / TILE_Y;
  const int ntz = (D.nz + TILE_Z - 1) / TILE_Z;
  const int g = blockIdx.x;
  const int tx = g % ntx, ty = (g / ntx) % nty, tz = g / (ntx * nty) * NT;
  const int nt = ntz - tz < NT ? ntz - tz : NT;
  const int tile0 = tx + ntx * (ty + nty * tz), stride = ntx * nty;
  const int xb = tx * TILE_X, jb = ty * TILE_Y, k0 = tz * TILE_Z + 1;
  /* cells of this workgroup in x, y and z */
  const int w = D.nx - xb < TILE_X ? D.nx - xb : TILE_X;
  const int h = D.ny - jb < TILE_Y ? D.ny - jb : TILE_Y;
  const int kn0 = D.nz - k0 + 1 < KZ ? D.nz - k0 + 1 : KZ;
  const int x = xb + lane + 1, j = jb + wv + 1;
  const bool colok = lane < w && wv < h;
  const unsigned c0 = colok ? (unsigned) gidx(C, x, j, k0) : 0u;
  const int wxy = wcount(x, D.nx, D.perx) + 3 * wcount(j, D.ny, D.pery);
  /* the column in s_p; threads without one write beside the plane */
  const int own0 = (wv + 1) * RX + (colok ? lane + 1 : LX);

  /* the cells around: one below and above the column, NY beside a y face,
   * at most one beside an x face.  Beyond a wall face stands the cell itself:
   * its direction is formed from the same values, so the difference across
   * the face is 0, which is what the face's weight 0 makes of it. */
  const int kb = k0 == 1 ? (D.perz ? D.nz : 1) : k0 - 1;
  const int kt = k0 + kn0 - 1 == D.nz ? (D.perz ? 1 : D.nz) : k0 + kn0;
  const unsigned ozb = colok ? (unsigned) gidx(C, x, j, kb) : 0u;
  const unsigned ozt = colok ? (unsigned) gidx(C, x, j, kt) : 0u;
  const int izb = wxy + 9 * wcount(kb, D.nz, D.perz);
  const int izt = wxy + 9 * wcount(kt, D.nz, D.perz);
  const int yside = wv & 1, yi = wv >> 1;          /* planes yi + 4 m */
  const int yj = yside ? (jb + h == D.ny ? (D.pery ? 1 : D.ny) : jb + h + 1)
                       : (jb == 0 ? (D.pery ? D.ny : 1) : jb);
  const bool yok = lane < w;
  const unsigned oy = yok ? (unsigned) gidx(C, x, yj, k0 + yi) : 0u;
  const int iy = wcount(x, D.nx, D.perx) + 3 * wcount(yj, D.ny, D.pery);
  const int xside = t & 1, xrow = (t >> 1) & (TILE_Y - 1), xi = t >> 4;
  const int xx = xside ? (xb + w == D.nx ? (D.perx ? 1 : D.nx) : xb + w + 1)
                       : (xb == 0 ? (D.perx ? D.nx : 1) : xb);
  const bool xok = xi < kn0 && xrow < h;
  const unsigned ox = xok ? (unsigned) gidx(C, xx, jb + xrow + 1, k0 + xi) : 0u;
  const int ix = wcount(xx, D.nx, D.perx)
               + 3 * wcount(jb + xrow + 1, D.ny, D.pery)
               + 9 * wcount(k0 + xi, D.nz, D.perz);

  /* own cells */
  V r[KZ], p[KZ], ap[KZ], phi_r[FAR ? 1 : KZ];
  auto phi = [&](int i) -> V & {
    return FAR ? s_phi[i * TILE_THREADS + t] : phi_r[FAR ? 0 : i];
  };
  unsigned live = 0;                   /* bit i: a fluid cell of the domain */
  V *const pold = (S.q0 & 1) ? S.pa : S.pb;
#pragma unroll
  for (int i = 0; i < KZ; i++) {
    const bool in = colok && i < kn0;
    const unsigned c = in ? c0 + i * sz0 : 0u;
    /* offset 0 holds no cell: a load for every lane, kept or not */
    const V rv = ld32(S.r, c), pv = ld32(S.phi, c), dv = ld32(pold, c);
    r[i] = in ? rv : (V) 0;
    phi(i) = in ? pv : (V) 0;
    p[i] = in && !S.first ? dv : (V) 0;
    ap[i] = 0;
    if (in && (!MASK || S.fluid[c])) live |= 1u << i;
    if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
  }
  V pzb = 0, pzt = 0, px = 0, py[NY];
  if (!S.first) {
    pzb = colok ? pold[ozb] : (V) 0;
    pzt = colok ? pold[ozt] : (V) 0;
    px = xok ? pold[ox] : (V) 0;
  }
#pragma unroll
  for (int m = 0; m < NY; m++)
    py[m] = !S.first && yok && yi + 4 * m < kn0 ? pold[oy + 4 * m * sz0] : (V) 0;

  /* stopping test and beta at the start (cg_continue) */
  const double limit = st->tol2 * st->sp_rhs;
  const double relstop = st->relup * st->rz_ref;
  double rz = st->rzs[(S.q0 + 1) & 1], rzprev = st->rzs[S.q0 & 1];
  double beta64 = 0.;
  V *const yrow = s_p + (yside ? h + 1 : 0) * RX + lane + 1;
  V *const xcell = s_p + (xi * LY + xrow + 1) * RX + (xside ? w + 1 : 0);
  bool stop = false;
  double s = rz;
  if (!S.first) {
    s = tile_block_sum(S.rpart, ntiles);
    stop = s <= limit || isnan(s) || (MIXED && s <= relstop);
    beta64 = s / rzprev;
    rz = s;
  }
  __syncthreads();                     /* s_invm, s_p, s_bad */
  /* Jacobi factors of the column: inside, and on a plane with a wall face */
  V m2 = s_invm[wxy + 18], m1 = s_invm[wxy + 9 * wcount(1, D.nz, 0)];
  bool first = S.first != 0;
  int q = S.q0;
  unsigned meeting = 0;
  bool lost = false;
  /* planes of the column with a wall face */
  const int zlo = !D.perz && k0 == 1 ? 0 : -1;
  const int zhi0 = !D.perz && k0 + kn0 - 1 == D.nz ? kn0 - 1 : -1;
  const bool edge = colok && (wv == 0 || wv == h - 1 || lane == 0 ||
                              lane == w - 1);
  /* the cells that other workgroups (or this one, around a periodic box)
   * read: every plane at the edge, else the first and the last */
  auto store_boundary = [&](V *out, auto f, unsigned sz, int kn) {
    if (edge) {
#pragma unroll
      for (int i = 0; i < KZ; i++)
        if (i < kn) dev_store(out + c0 + i * sz, f(i));
    } else if (colok) {
#pragma unroll
      for (int i = 0; i < KZ; i++)
        if (i == 0 || i == kn - 1) dev_store(out + c0 + i * sz, f(i));
    }
  };

  while (!stop && q < S.qmax) {
    q++;
    const V beta = (V) beta64;
    /* offsets formed anew in each iteration: kept across it they would take
     * a register per cell */
    unsigned sz = (unsigned) C.sz;
    int kn = kn0, zhi = zhi0;
    int at = (wv + 1) * RX + lane + 1, own = own0;
    asm volatile("" : "+s"(sz), "+s"(kn), "+s"(zhi), "+v"(at), "+v"(own));
    auto wall_z = [&](int i) { return (i == 0 && zlo == 0) || i == zhi; };
    /* (-A) f of cell i from the column, the cells beside it in LDS and the
     * planes below and above the column */
    auto lap = [&](int i, auto f, V below, V above) {
      const V *c = s_p + at + i * LY * RX;
      const V fc = f(i);
      const V dn = i == 0 ? below : f(i > 0 ? i - 1 : 0);
      const V up = i == KZ - 1 ? above : f(i < KZ - 1 ? i + 1 : 0);
      return -K.idx2 * ((c[1] - fc) - (fc - c[-1]))
             -K.idy2 * ((c[RX] - fc) - (fc - c[-RX]))
             -K.idz2 * ((up - fc) - (fc - dn));
    };
    /* search direction: around, then own cells */
    {
      const V rb = colok ? dev_load(S.r + ozb) : (V) 0;
      const V rt = colok ? dev_load(S.r + ozt) : (V) 0;
      const V rx = xok ? dev_load(S.r + ox) : (V) 0;
      V ry[NY];
#pragma unroll
      for (int m = 0; m < NY; m++)
        ry[m] = yok && yi + 4 * m < kn ? dev_load(S.r + oy + 4 * m * sz)
                                       : (V) 0;
      if (first) {
#pragma unroll
        for (int i = 0; i < KZ; i++) {
          p[i] = r[i]*(wall_z(i) ? m1 : m2);
          s_p[own + i * LY * RX] = p[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < KZ; i++) {
          const V z = r[i]*(wall_z(i) ? m1 : m2);
          p[i] = z + beta*p[i];
          s_p[own + i * LY * RX] = p[i];
          if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
      const V zb = rb*s_invm[izb], zt = rt*s_invm[izt], zx = rx*s_invm[ix];
      pzb = first ? zb : zb + beta*pzb;
      pzt = first ? zt : zt + beta*pzt;
      px = first ? zx : zx + beta*px;
      if (xok) *xcell = px;
#pragma unroll
      for (int m = 0; m < NY; m++)
        if (yok && yi + 4 * m < kn) {
          const int i = yi + 4 * m;
          const V z = ry[m]*s_invm[iy + 9 * wcount(k0 + i, D.nz, D.perz)];
          py[m] = first ? z : z + beta*py[m];
          yrow[i * LY * RX] = py[m];
        }
    }
    /* a column that ends early has the cell above it as its next cell */
    if (kn < KZ) {
#pragma unroll
      for (int i = 1; i < KZ; i++)
        if (i == kn) p[i] = pzt;
    }
    __syncthreads();
    /* A p and the tile partials of (p, A p) */
    double acc[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = 0.0;
#pragma unroll
    for (int i = 0; i < KZ; i++) {
      /* 0 in particle cells and outside the domain: r stays 0 there */
      ap[i] = keep(lap(i, [&](int m) { return p[m]; }, pzb, pzt), live, i);
      acc[i / TILE_Z] += (double) p[i] * (double) ap[i];
      /* the reads of four cells in flight, not of all */
      if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int n = 0; n < NT; n++) {
      double v = tree_step<32>(acc[n]);
      v = tree_step<16>(v);
      v = tree_step<8>(v);
      v = tree_step<4>(v);
      v = tree_step<2>(v);
      v = tree_step<1>(v);
      if (lane == 0) s_w[n][wv] = v;
    }
    __syncthreads();
    publish(S.slots, meeting, tile0, stride, nt, s_w);
    double pap;
    if (!meet(S.slots, meeting, ntiles, S.spins, s_v, &s_bad, &pap)) { lost = true; break; }
    meeting++;
    const V alpha = (V) (rz / pap);
    /* per-cell flags and factors formed again, not kept from above */
    asm volatile("" : "+v"(live), "+v"(m1), "+v"(m2), "+s"(kn), "+s"(zhi));
    const bool refresh = !MIXED && q % 50 == 0;
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = 0.0;
    if (!refresh) {
#pragma unroll
      for (int i = 0; i < KZ; i++) {
        phi(i) += alpha*p[i];
        const V rr = r[i] - alpha*ap[i];
        r[i] = rr;
        const V z = rr*(wall_z(i) ? m1 : m2);
        acc[i / TILE_Z] += (double) rr * (double) z;
        if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      /* the true residual b - (-A) phi, phi of the cells around read from
       * memory */
#pragma unroll
      for (int i = 0; i < KZ; i++) {
        const V f = phi(i) + alpha*p[i];
        phi(i) = f;
        s_p[own + i * LY * RX] = f;
      }
      store_boundary(S.phi, phi, sz, kn);
      if (lane < TILE_Y && wv < NT) s_w[wv][lane] = 0.0;
      stores_done();
      __syncthreads();
      publish(S.slots, meeting, tile0, stride, nt, s_w);
      double none;
      if (!meet(S.slots, meeting, ntiles, S.spins, s_v, &s_bad, &none)) { lost = true; break; }
      meeting++;
      const V fb = colok ? dev_load(S.phi + ozb) : (V) 0;
      const V ft = colok ? dev_load(S.phi + ozt) : (V) 0;
      if (xok) *xcell = dev_load(S.phi + ox);
#pragma unroll
      for (int m = 0; m < NY; m++)
        if (yok && yi + 4 * m < kn)
          yrow[(yi + 4 * m) * LY * RX] = dev_load(S.phi + oy + 4 * m * sz);
      if (kn < KZ) {
#pragma unroll
        for (int i = 1; i < KZ; i++)
          if (i == kn) phi(i) = ft;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < KZ; i++) {
        const bool in = colok && i < kn;
        const V a = lap(i, phi, fb, ft);
        const V rr = in ? (V) (S.rhs[c0 + i * sz] - a) : (V) 0;
        r[i] = keep(rr, live, i);
        const V z = r[i]*(wall_z(i) ? m1 : m2);
        acc[i / TILE_Z] += (double) rr * (double) z;
        if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    /* boundary cells for the workgroups around, tile partials of (r, z) */
    store_boundary(S.r, [&](int m) { return r[m]; }, sz, kn);
#pragma unroll
    for (int n = 0; n < NT; n++) {
      double v = tree_step<32>(acc[n]);
      v = tree_step<16>(v);
      v = tree_step<8>(v);
      v = tree_step<4>(v);
      v = tree_step<2>(v);
      v = tree_step<1>(v);
      if (lane == 0) s_w[n][wv] = v;
    }
    stores_done();
    __syncthreads();
    publish(S.slots, meeting, tile0, stride, nt, s_w);
    if (!meet(S.slots, meeting, ntiles, S.spins, s_v, &s_bad, &s)) { lost = true; break; }
    meeting++;
    stop = s <= limit || isnan(s) || (MIXED && s <= relstop);
    beta64 = s / rz;
    rzprev = rz;
    rz = s;
    first = false;
  }
  if (lost) {
    if (t == 0) st->lost = 1;
    return;
  }
  V *const pout = (q & 1) ? S.pa : S.pb;
  unsigned sz1 = (unsigned) C.sz;
  asm volatile("" : "+s"(sz1));
#pragma unroll
  for (int i = 0; i < KZ; i++) {
    if (colok && i < kn0) {
      const unsigned c = c0 + i * sz1;
      st32(S.phi, c, phi(i));
      st32(S.r, c, r[i]);
      st32(pout, c, p[i]);
    }
    if (i % GR == GR - 1) __builtin_amdgcn_sched_barrier(0);
  }
  if (g == 0 && t == 0) {
    st->rz1 = s;
    st->q = q;
    st->nan_flag = isnan(s) ? 1 : 0;
    /* (r, z) at the start of iteration q and, unless the sweep is over,
     * at that of the next */
    st->rzs[q & 1] = rzprev;
    if (stop) {
      if (MIXED) st->inner_done = 1;
      else st->done = 1;
    } else {
      st->rzs[(q + 1) & 1] = rz;
    }
  }
}

#endif
