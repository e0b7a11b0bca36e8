// k_vector.hip -- the passive vector of the reference (grid.cpp:616-715):
// a momentum-like field RV at the faces, transported by the gas velocity
// U = RU_int/Rho_face, diffused with eta, forced by V_Source (or by the gas's
// x velocity on its y component), and projected with its own pressure Q
// (a Poisson solve with the constant density Rho_forV).  Every product and sum
// in the order of the reference's whole-array passes (built with
// -ffp-contract=off), so the stencil parts round as the reference's do.
#include <math.h>

#include <algorithm>
#include <stdexcept>

#include "tpx_internal.h"

namespace tpx {

namespace {

struct RU3c { const double *__restrict__ a[3]; };
struct RU3w { double *__restrict__ a[3]; };

struct IxV {
  int mx, my, mz, nx;
  long nxy;
  __device__ __forceinline__ long operator()(int i, int j, int k) const {
    return (long)(k & mz) * nxy + (long)(j & my) * nx + (i & mx);
  }
};

__device__ __forceinline__ IxV ixv(const Geo &g) { return IxV{g.nx - 1, g.ny - 1, g.nz - 1, g.nx, g.nxy}; }

__device__ __forceinline__ bool cell(const Geo &g, int &i, int &j, int &k, long &c) {
  c = (long)xcd_block(blockIdx.x, gridDim.x) * block_dim_x() + threadIdx.x;
  if (c >= g.n) return false;
  i = (int)(c % g.nx);
  const long r = c / g.nx;
  j = (int)(r % g.ny);
  k = (int)(r / g.ny);
  return true;
}

__device__ __forceinline__ double bsum(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = block_dim_x() / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  return sh[0];
}

struct RvArgs {
  const double *rv_int[3], *rv_base[3];
  double *rv_np1[3], *rv_new[3];
  const double *ru_int[3], *rho_int;
  const double *filt;    // S2_type != 0: the filtered RU_int.x / Rho_face.x
  const double *scal;    // SC_RV_S2: the type-0 source summed over the cells
  double eta, rho_forv, c_post, c_pre, ncell;
  int s2_type, rk3;
};

// grid::Update_RV_WOQ (grid.cpp:646-692) as a z-marching tile.  Evaluated a
// thread a cell from global memory, every face reads up to 60 neighbours and
// forms V = RV_int/Rho_forV and U = RU_int/Rho_face anew at each (some 70
// divisions a cell): bound by address processing and divisions, 241 us at
// 128^3 against a floor of 70 us for its 19 field values a cell.  A block owns
// a TX x TY column and walks KC planes: RV_int, V and U of the planes k and
// k + 1 (one halo cell on each side; the divisions are done once, as a point is
// loaded) lie in LDS, the own column's values of plane k - 1 in registers, and
// the plane after next is loaded while this one is computed: 113 us.  49 KB of
// LDS a block of 256, three blocks a CU.  Same operands and order: the same
// bits.
struct RvTile { int TX, TY, KC; };

struct k_rv_woq {
  static constexpr int kBounds = 256;
  static __device__ __forceinline__ void run(const Geo &g, const RvArgs &a, const RvTile &tl) {
    extern __shared__ double sm[];
    const int TX = tl.TX, TY = tl.TY, KC = tl.KC;
    const int TW = TX + 2, TN = TW * (TY + 2);  // x from i0 - 1 to i0 + TX
    const IxV ix = ixv(g);
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int ntx = g.nx / TX, nty = g.ny / TY;
    const int i0 = (int)(b % ntx) * TX, j0 = (int)((b / ntx) % nty) * TY, k0 = (int)(b / (ntx * nty)) * KC;
    const int tid = (int)threadIdx.x, bd = (int)block_dim_x(), tx = tid % TX, ty = tid / TX;
    const int i = i0 + tx, j = j0 + ty;
    const double *__restrict__ rho = a.rho_int;
    // one point of a plane as loaded: RV_int, RU_int, Rho at the point and below it
    struct Raw { double rv[3], ru[3], r[4]; };
    auto load = [&](int kz, int e, Raw &w) {
      const int x = i0 + e % TW - 1, y = j0 + e / TW - 1;
      const long q = ix(x, y, kz);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        w.rv[d] = a.rv_int[d][q];
        w.ru[d] = a.ru_int[d][q];
      }
      w.r[0] = rho[q];
      w.r[1] = rho[ix(x - 1, y, kz)];
      w.r[2] = rho[ix(x, y - 1, kz)];
      w.r[3] = rho[ix(x, y, kz - 1)];
    };
    // V = RV_int/Rho_forV (tensor0.cpp:143-147), U.d = RU_int.d/Rho_face.d with
    // Rho_face = I_C2F(Rho_int) (grid.cpp:868)
    auto store = [&](const Raw &w, int slot, int e) {
      double *t = sm + slot * 9 * TN + e;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        t[d * TN] = w.rv[d];
        t[(3 + d) * TN] = w.rv[d] / a.rho_forv;
        t[(6 + d) * TN] = w.ru[d] / ((w.r[0] + w.r[1 + d]) * 0.5);
      }
    };
    // a plane is at most two points a thread: (TX + 2)(TY + 2) <= 2 TX TY
    auto load_plane = [&](int kz, Raw (&w)[2]) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (tid + u * bd < TN) load(kz, tid + u * bd, w[u]);
    };
    auto store_plane = [&](const Raw (&w)[2], int slot) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (tid + u * bd < TN) store(w[u], slot, tid + u * bd);
    };
    // quantity q (0-2 RV_int, 3-5 V, 6-8 U) of slot s at cell (i + dx, j + dy)
    auto T = [&](int s, int q, int dx, int dy) -> double {
      return sm[(s * 9 + q) * TN + (ty + 1 + dy) * TW + tx + 1 + dx];
    };
    // div_F2C(V) at (i + dx, j + dy) of plane `s`, the plane above in slot `n` (tensor0.cpp:249-256)
    auto divV = [&](int s, int n, int dx, int dy) {
      return (T(s, 3, dx + 1, dy) - T(s, 3, dx, dy)) * g.idx + (T(s, 4, dx, dy + 1) - T(s, 4, dx, dy)) * g.idy +
             (T(n, 5, dx, dy) - T(s, 5, dx, dy)) * g.idz;
    };
    Raw w[2];
    load_plane(k0 - 1, w);
    store_plane(w, 1);
    load_plane(k0, w);
    store_plane(w, 0);
    load_plane(k0 + 1, w);
    __syncthreads();
    // own-column values of the plane below
    double RVp[3], Vp[3], Uxp, Uxp1, Uyp, Uyp1, Uzp, dvp;
    auto carry = [&](int s, int n) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        RVp[d] = T(s, d, 0, 0);
        Vp[d] = T(s, 3 + d, 0, 0);
      }
      Uxp = T(s, 6, 0, 0);
      Uxp1 = T(s, 6, 1, 0);
      Uyp = T(s, 7, 0, 0);
      Uyp1 = T(s, 7, 0, 1);
      Uzp = T(s, 8, 0, 0);
      dvp = divV(s, n, 0, 0);
    };
    carry(1, 0);
    __syncthreads();
    store_plane(w, 1);
    __syncthreads();
    const double id[3] = {g.idx, g.idy, g.idz};
    int cur = 0;
    for (int kk = k0; kk < k0 + KC; ++kk) {
      const int nxt = cur ^ 1;
      const bool more = kk + 1 < k0 + KC;
      if (more) load_plane(kk + 2, w);
      const long c = (long)kk * g.nxy + (long)j * g.nx + i;
      const double div0 = divV(cur, nxt, 0, 0);
      double s2[3] = {0.0, 0.0, 0.0};
      if (a.s2_type == 0) {
        // V_Source (grid.cpp:616-641, vector_source.h): cos(X) on the y faces,
        // zero on the others, each minus its mean over the cells
        const double X = i * g.dx + g.dx / 2., A = 1., K = 1.;
        s2[1] = A * cos(K * X) - a.scal[SC_RV_S2] / a.ncell;
      } else {
        s2[1] = -1 * a.filt[c];
      }
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        const int ei = ax == 0, ej = ax == 1;
        const bool ez = ax == 2;
        const double dvm = ez ? dvp : divV(cur, nxt, -ei, -ej);
        const double g1 = (div0 - dvm) * id[ax];  // grad_C2F (tensor1.cpp:259-270)
        const double vc = T(cur, 3 + ax, 0, 0);
        // del2 (tensor0.cpp:258-266)
        double lap = (T(cur, 3 + ax, 1, 0) - 2 * vc + T(cur, 3 + ax, -1, 0)) * g.idx2;
        lap = lap + (T(cur, 3 + ax, 0, 1) - 2 * vc + T(cur, 3 + ax, 0, -1)) * g.idy2;
        lap = lap + (T(nxt, 3 + ax, 0, 0) - 2 * vc + Vp[ax]) * g.idz2;
        double rhs = a.eta / 3. * g1 + a.eta * lap;
        // convection: div_F2C of I_d(RV_int.ax) * I_ax(U.d) (grid.cpp:655-673)
        const double rc = T(cur, ax, 0, 0);
        const double ux0 = ((rc + T(cur, ax, -1, 0)) * 0.5) * ((T(cur, 6, 0, 0) + (ez ? Uxp : T(cur, 6, -ei, -ej))) * 0.5);
        const double ux1 =
            ((T(cur, ax, 1, 0) + rc) * 0.5) * ((T(cur, 6, 1, 0) + (ez ? Uxp1 : T(cur, 6, 1 - ei, -ej))) * 0.5);
        const double uy0 = ((rc + T(cur, ax, 0, -1)) * 0.5) * ((T(cur, 7, 0, 0) + (ez ? Uyp : T(cur, 7, -ei, -ej))) * 0.5);
        const double uy1 =
            ((T(cur, ax, 0, 1) + rc) * 0.5) * ((T(cur, 7, 0, 1) + (ez ? Uyp1 : T(cur, 7, -ei, 1 - ej))) * 0.5);
        const double uz0 = ((rc + RVp[ax]) * 0.5) * ((T(cur, 8, 0, 0) + (ez ? Uzp : T(cur, 8, -ei, -ej))) * 0.5);
        const double uz1 = ((T(nxt, ax, 0, 0) + rc) * 0.5) *
                           ((T(nxt, 8, 0, 0) + (ez ? T(cur, 8, 0, 0) : T(nxt, 8, -ei, -ej))) * 0.5);
        double conv = (ux1 - ux0) * g.idx;
        conv = conv + (uy1 - uy0) * g.idy;
        conv = conv + (uz1 - uz0) * g.idz;
        rhs -= conv;
        if (a.s2_type == 0 || ax == 1) rhs += s2[ax];
        const double np1 = a.rv_np1[ax][c] + a.c_post * rhs;
        a.rv_np1[ax][c] = np1;
        a.rv_new[ax][c] = a.rk3 ? np1 : 1 * a.rv_base[ax][c] + a.c_pre * rhs;
      }
      carry(cur, nxt);
      __syncthreads();
      if (more) store_plane(w, cur);
      cur = nxt;
      __syncthreads();
    }
  }
};

// The type-1 source's tensor0::Equal_Iy_C2F(dummy.x) on dummy.x itself
// (grid.cpp:683-685): the reference's loop (tensor0.cpp:308-315) runs j
// upwards and reads row j-1 after overwriting it, so along each (i, k) line
// f~_j = (f_j + f~_{j-1}) / 2, with f~_{-1} the old value of the last row (the
// periodic ghost).  f = RU_int.x / Rho_face.x.  One thread per line.
struct k_rv_filter {
  static constexpr int kBounds = 256;
  static __device__ __forceinline__ void run(const Geo &g, const double *__restrict__ rux,
                                             const double *__restrict__ rho, double *__restrict__ out) {
    const long line = (long)blockIdx.x * block_dim_x() + threadIdx.x;
    if (line >= (long)g.nx * g.nz) return;
    const int i = (int)(line % g.nx), k = (int)(line / g.nx);
    const IxV ix = ixv(g);
    auto f = [&](int j) {
      const long q = ix(i, j, k);
      return rux[q] / ((rho[q] + rho[ix(i - 1, j, k)]) * 0.5);
    };
    double prev = f(g.ny - 1);
    for (int j = 0; j < g.ny; ++j) {
      const double v = (f(j) + prev) * 0.5;
      out[ix(i, j, k)] = v;
      prev = v;
    }
  }
};

// grid::Compute_RHS_Pois_Q (grid.cpp:694-701) before its mean is removed:
// div_F2C(RV_new / Rho_forV) / (dt pre), with block sums for the mean (and
// for the statistics the sum of squares of V = RV_new / Rho_forV)
struct k_rhs_pois_q {
  static constexpr int kBounds = 256;
  static __device__ __forceinline__ void run(const Geo &g, RU3c rv, double rho_forv, double inv_dtpre,
                                             double *__restrict__ rhs, double *__restrict__ partials, long nb,
                                             int want_vv) {
    __shared__ double sh[256];
    int i, j, k;
    long c;
    double r = 0.0, vv = 0.0;
    if (cell(g, i, j, k, c)) {
      const IxV ix = ixv(g);
      const double v0 = rv.a[0][c] / rho_forv, v1 = rv.a[1][c] / rho_forv, v2 = rv.a[2][c] / rho_forv;
      r = (rv.a[0][ix(i + 1, j, k)] / rho_forv - v0) * g.idx + (rv.a[1][ix(i, j + 1, k)] / rho_forv - v1) * g.idy +
          (rv.a[2][ix(i, j, k + 1)] / rho_forv - v2) * g.idz;
      r = r * inv_dtpre;
      rhs[c] = r;
      vv = v0 * v0 + v1 * v1 + v2 * v2;
    }
    const double s = bsum(r, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
    if (want_vv) {
      __syncthreads();
      const double t = bsum(vv, sh);
      if (threadIdx.x == 0) partials[nb + blockIdx.x] = t;
    }
  }
};

// grid::Update_RV_WQ (grid.cpp:709-715)
struct k_rv_wq {
  static constexpr int kBounds = 256;
  static __device__ __forceinline__ void run(const Geo &g, const double *__restrict__ Q, RU3w np1, RU3w nw,
                                             double c_post, double c_pre, int rk3) {
    int i, j, k;
    long c;
    if (!cell(g, i, j, k, c)) return;
    const IxV ix = ixv(g);
    const double gq[3] = {(Q[c] - Q[ix(i - 1, j, k)]) * g.idx, (Q[c] - Q[ix(i, j - 1, k)]) * g.idy,
                          (Q[c] - Q[ix(i, j, k - 1)]) * g.idz};
    for (int d = 0; d < 3; ++d) {
      const double v = np1.a[d][c] + -(c_post)*gq[d];
      np1.a[d][c] = v;
      nw.a[d][c] = rk3 ? v : nw.a[d][c] + -(c_pre)*gq[d];
    }
  }
};

// block sums of the type-0 source's y component cos(X) over the cells
struct k_rv_source_sum {
  static constexpr int kBounds = 256;
  static __device__ __forceinline__ void run(const Geo &g, double *partials) {
    __shared__ double sh[256];
    int i, j, k;
    long c;
    double v = 0.0;
    if (cell(g, i, j, k, c)) {
      const double X = i * g.dx + g.dx / 2., A = 1., K = 1.;
      v = A * cos(K * X);
    }
    const double s = bsum(v, sh);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
  }
};

unsigned vgrid(const tpx_ctx *c) { return grid1d(c->g.n, 256); }

}  // namespace

void launch_rv_woq(tpx_ctx *c, const Coef &k, const double *const ru_int[3], const double *rho_int) {
  RvArgs a{};
  for (int d = 0; d < 3; ++d) {
    a.rv_int[d] = c->rv[c->rv_int][d];
    a.rv_base[d] = c->rv[c->rv_base][d];
    a.rv_np1[d] = c->rv[c->rv_np1][d];
    a.rv_new[d] = c->rv[c->rv_new][d];
    a.ru_int[d] = ru_int[d];
  }
  a.rho_int = rho_int;
  a.scal = c->scal;
  a.eta = c->p.eta;
  a.rho_forv = c->p.rho_forv;
  a.c_post = k.dt * k.post;
  a.c_pre = k.dt * k.pre;
  a.ncell = (double)c->g.n;
  a.s2_type = c->p.s2_type;
  a.rk3 = k.rk == 3;
  timing_begin(c, TPX_K_OTHER);
  if (a.s2_type != 0) {
    tpx_launch<k_rv_filter>(grid1d((long)c->g.nx * c->g.nz, 256), 256, 0, c->stream, c->g, ru_int[0], rho_int,
                            c->rv_filt);
    TPX_LAUNCH_CHECK();
    a.filt = c->rv_filt;
  }
  const Geo &g = c->g;
  RvTile tl;
  tl.TX = std::min(g.nx, 32);
  tl.TY = std::min(256 / tl.TX, g.ny);
  // a march of up to 16 planes, shorter while the launch has fewer than 1024
  // blocks (the two halo planes re-read by each block cost less than idle CUs)
  tl.KC = std::min(g.nz, 16);
  const int cols = (g.nx / tl.TX) * (g.ny / tl.TY);
  while (tl.KC > 2 && cols * (g.nz / tl.KC) < 1024) tl.KC /= 2;
  const int tile = (tl.TX + 2) * (tl.TY + 2);
  if (tile > 2 * tl.TX * tl.TY) throw std::logic_error("passive vector tile exceeds two points per thread");
  tpx_launch<k_rv_woq>((unsigned)(cols * (g.nz / tl.KC)), tl.TX * tl.TY, sizeof(double) * 18 * (size_t)tile, c->stream,
                       g, a, tl);
  TPX_LAUNCH_CHECK();
  timing_end(c, TPX_K_OTHER);
}

void launch_rhs_pois_q(tpx_ctx *c, const Coef &k, bool want_vv) {
  RU3c rv;
  for (int d = 0; d < 3; ++d) rv.a[d] = c->rv[c->rv_new][d];
  const unsigned nb = vgrid(c);
  timing_begin(c, TPX_K_OTHER);
  tpx_launch<k_rhs_pois_q>(nb, 256, 0, c->stream, c->g, rv, c->p.rho_forv, (1. / (k.dt * k.pre)), c->rhs_q,
                           c->partials, (long)nb, want_vv ? 1 : 0);
  TPX_LAUNCH_CHECK();
  launch_finish_sum(c, (int)nb, 0, SC_SUM_RHS_Q);
  if (want_vv) launch_finish_sum(c, (int)nb, (int)nb, SC_ST_VV);
  timing_end(c, TPX_K_OTHER);
}

void launch_rv_wq(tpx_ctx *c, const Coef &k) {
  RU3w np1, nw;
  for (int d = 0; d < 3; ++d) {
    np1.a[d] = c->rv[c->rv_np1][d];
    nw.a[d] = c->rv[c->rv_new][d];
  }
  timing_begin(c, TPX_K_OTHER);
  tpx_launch<k_rv_wq>(vgrid(c), 256, 0, c->stream, c->g, (const double *)c->Qv, np1, nw, k.dt * k.post,
                      k.dt * k.pre, k.rk == 3 ? 1 : 0);
  TPX_LAUNCH_CHECK();
  timing_end(c, TPX_K_OTHER);
}

void launch_rv_source_sum(tpx_ctx *c) {
  const unsigned nb = vgrid(c);
  tpx_launch<k_rv_source_sum>(nb, 256, 0, c->stream, c->g, c->partials);
  TPX_LAUNCH_CHECK();
  launch_finish_sum(c, (int)nb, 0, SC_RV_S2);
}

}  // namespace tpx
