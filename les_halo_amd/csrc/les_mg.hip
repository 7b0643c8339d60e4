// Multigrid preconditioner of the mixed-precision correction solve: one V-cycle per
// conjugate-gradient iteration, between the two halves of the symmetric red-black Gauss-Seidel
// pass that preconditioned it alone.
//
// The system couples strongly along k near the ground (2 m levels, 4 m columns) and along i and j
// aloft (60 m levels).  Coarsening i and j only, with whole columns solved at once (tridiagonal in
// k), handles both: the column solves remove any error along k, and the strong coupling aloft is
// along the directions that are coarsened.  A coarse grid's cells are pairs of the finer one's, or
// single ones where a direction has an odd cell left or its half would be an odd periodic row
// (red-black needs an even one); its operator is the same discretisation on those widths.
// Transfers are linear along i and j, the restriction the transpose of the prolongation in the cell
// volumes; they mirror at the i faces and wrap around in j.  With red-black column sweeps in
// mirrored order (red, black, coarse grid, black, red) the cycle is symmetric in the conjugate
// gradients' inner product.  The coarsest grid is one column: where levels are far apart
// (hundreds of metres), each level's mean is nearly free and only that column's solve settles it.
//
// A solve to a relative residual of 1e-7 takes 12 iterations in two passes at 300x300x90 and at
// 600x600x90 instead of about 1000, and a step 11.8 ms instead of 109 and 30.4 ms instead of 540.
// Bound: latency.  A V-cycle at 300x300x90 is 50 launches; the coarse column sweeps (8.7 us each on
// average, 42 % of the step) have a few hundred workgroups at most and wait for their loads, the
// finest grid's passes (14 to 32 us each) are the ones of les_mixed.hip.
#include <algorithm>
#include <cmath>

#include "les_mg.h"

namespace les {

namespace {

constexpr int MG_BX = 64;
constexpr int MG_SEG = 8;
constexpr int seg_levels(int kp) { return kp <= 8 * MG_SEG ? 8 : (kp <= 12 * MG_SEG ? 12 : 16); }

// One red-black half of the column sweeps: colour (i + j) & 1 == red of e solves
// D e - (k neighbours) = b + (i and j neighbours); FIRST: the other colour is zero.
template <bool FIRST>
__global__ __launch_bounds__(MG_BX) void k_mg_columns(MgLevel L, int kp, int red,
                                                      const float* __restrict__ c4s,
                                                      const float* __restrict__ b,
                                                      float* __restrict__ t, float* e,
                                                      const double* stopped) {
  if (*stopped != 0.0) return;
  const int hx = (L.nx + 1) >> 1;
  const int x = blockIdx.x * MG_BX + threadIdx.x;
  const int j = x / hx;
  if (j >= L.ny) return;
  const int i = 2 * (x - j * hx) + ((j + red) & 1);
  if (i >= L.nx) return;
  const float* inv = L.inv + L.kx[i] + L.ky[j];
  const float* up = L.up + L.kx[i] + L.ky[j];
  const int plane = L.nx * L.ny, o = i + L.nx * j;
  const int w = i > 0 ? -1 : 0, ea = i < L.nx - 1 ? 1 : 0;  // (an absent one's coupling is 0)
  const float2 cx = L.cx[i], cy = L.cy[j];
  const int s = j > 0 ? -L.nx : L.nx * (L.ny - 1), n = j < L.ny - 1 ? L.nx : -L.nx * (L.ny - 1);
  float last = 0.0f;
  constexpr int U = 6;  // levels whose loads are in flight together
  for (int k0 = 0; k0 < kp; k0 += U) {
    float r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u, kp - 1), q = o + plane * k;
      r[u] = b[q];
      if constexpr (!FIRST) r[u] += (cx.x * e[q + w] + cx.y * e[q + ea]) + (cy.x * e[q + s] + cy.y * e[q + n]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u;
      if (k >= kp) break;
      last = (r[u] + c4s[k] * last) * inv[k];
      t[o + plane * k] = last;
    }
  }
  last = 0.0f;
  for (int k0 = kp - 1; k0 >= 0; k0 -= U) {
    float r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = t[o + plane * max(k0 - u, 0)];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 - u;
      if (k < 0) break;
      last = r[u] + up[k] * last;
      e[o + plane * k] = last;
    }
  }
}

// The same for columns of at most MG_SEG * M levels, MG_SEG threads a column: each solves a segment
// of M levels in registers as if nothing came in from the segments before, and adds what does
// come in times the products of the recurrence's coefficients (L.gf forward, L.gb backward); all of
// a column's loads are in flight together and the serial chain is a segment and the segments'
// ends.  Mean over the coarse grids of 300x300x90: 8.7 us a launch against 29 with a thread per
// column.
template <int M, bool FIRST>
__global__ __launch_bounds__(32 * MG_SEG) void k_mg_segments(MgLevel L, int kp, int red,
                                                             const float* __restrict__ c4s,
                                                             const float* __restrict__ b, float* e,
                                                             const double* stopped) {
  __shared__ float endf[MG_SEG][32], endb[MG_SEG][32];
  if (*stopped != 0.0) return;
  const int hx = (L.nx + 1) >> 1, c = threadIdx.x, sg = threadIdx.y;
  const int x = blockIdx.x * 32 + c;
  const int j = min(x / hx, L.ny - 1);
  const int i0 = 2 * (x % hx) + ((j + red) & 1);
  const bool ok = x < hx * L.ny && i0 < L.nx;
  const int i = min(i0, L.nx - 1);
  const int tab = L.kx[i] + L.ky[j];
  const int plane = L.nx * L.ny, k0 = sg * M, o = i + L.nx * j;
  const int w = i > 0 ? -1 : 0, ea = i < L.nx - 1 ? 1 : 0;  // (an absent one's coupling is 0)
  const float2 cx = L.cx[i], cy = L.cy[j];
  const int s = j > 0 ? -L.nx : L.nx * (L.ny - 1), n = j < L.ny - 1 ? L.nx : -L.nx * (L.ny - 1);
  float r[M], up[M];
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int k = min(k0 + u, kp - 1), q = o + plane * k;
    r[u] = b[q];
    if constexpr (!FIRST) r[u] += (cx.x * e[q + w] + cx.y * e[q + ea]) + (cy.x * e[q + s] + cy.y * e[q + n]);
    up[u] = L.up[tab + k];
  }
  float last = 0.0f;
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int k = min(k0 + u, kp - 1);
    if (k0 + u < kp) last = (r[u] + (u > 0 ? c4s[k] * last : 0.0f)) * L.inv[tab + k];
    r[u] = last;
  }
  endf[sg][c] = last;
  __syncthreads();
  float in = 0.0f;  // the value below the segment
  for (int q = 0; q < sg; ++q) in = endf[q][c] + L.gf[tab + min(q * M + M, kp) - 1] * in;
#pragma unroll
  for (int u = 0; u < M; ++u) r[u] += L.gf[tab + min(k0 + u, kp - 1)] * in;
  last = 0.0f;
#pragma unroll
  for (int u = M - 1; u >= 0; --u) {
    if (k0 + u < kp) last = r[u] + up[u] * last;
    r[u] = last;
  }
  endb[sg][c] = last;
  __syncthreads();
  in = 0.0f;  // the value above the segment
  for (int q = MG_SEG - 1; q > sg; --q)
    if (q * M < kp) in = endb[q][c] + L.gb[tab + q * M] * in;
#pragma unroll
  for (int u = 0; u < M; ++u) {
    const int k = k0 + u;
    if (ok && k < kp) e[o + plane * k] = r[u] + L.gb[tab + k] * in;
  }
}

// b = R s from the finest grid: s in the split layout, colour 0 only
__global__ __launch_bounds__(256) void k_mg_restrict_split(Dims d, SplitSOR sp, MgLevel L,
                                                           const float* __restrict__ s0,
                                                           const double* stopped) {
  if (*stopped != 0.0) return;
  const int I = blockIdx.x * 64 + threadIdx.x, J = blockIdx.y * 4 + threadIdx.y, k = blockIdx.z;
  if (I >= L.nx || J >= L.ny) return;
  const int4 ri = L.ri[I], rj = L.rj[J];
  const float4 wi = L.wi[I], wj = L.wj[J];
  const int fi[4] = {ri.x, ri.y, ri.z, ri.w}, fj[4] = {rj.x, rj.y, rj.z, rj.w};
  const float ui[4] = {wi.x, wi.y, wi.z, wi.w}, uj[4] = {wj.x, wj.y, wj.z, wj.w};
  float a = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float r = 0.0f;
#pragma unroll
    for (int p = 0; p < 4; ++p)  // cell (fi + 1, fj + 1, k + 1) is of colour 0
      if (((fi[p] + fj[q] + k + 3) & 1) == 0)
        r += ui[p] * s0[(fi[p] >> 1) + sp.nr * (fj[q] + sp.nj * k)];
    a += uj[q] * r;
  }
  L.b[I + L.nx * (J + L.ny * k)] = a;
}

// z += P e on colour 0 of the finest grid
__global__ __launch_bounds__(256) void k_mg_prolong_split(Dims d, SplitSOR sp, MgLevel L,
                                                          float* __restrict__ z0,
                                                          const double* stopped) {
  if (*stopped != 0.0) return;
  const int ii = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, k = blockIdx.z;
  if (j >= d.jp) return;
  const int i = 2 * ii + ((j + k + 1) & 1);  // from 0: cell i + 1 of colour 0
  if (i >= d.ip) return;
  const int2 a = L.pi[i], c = L.pj[j];
  const float2 u = L.vi[i], v = L.vj[j];
  const float* e = L.e + L.nx * L.ny * k;
  const float lo = u.x * e[a.x + L.nx * c.x] + u.y * e[a.y + L.nx * c.x];
  const float hi = u.x * e[a.x + L.nx * c.y] + u.y * e[a.y + L.nx * c.y];
  z0[ii + sp.nr * (j + sp.nj * k)] += v.x * lo + v.y * hi;
}

// C.b = R (residual of F): after red and black sweeps from zero the black residual is zero and
// the red one is the coupling to the black columns
__global__ __launch_bounds__(256) void k_mg_restrict(MgLevel F, MgLevel C, const double* stopped) {
  if (*stopped != 0.0) return;
  const int I = blockIdx.x * 64 + threadIdx.x, J = blockIdx.y * 4 + threadIdx.y, k = blockIdx.z;
  if (I >= C.nx || J >= C.ny) return;
  const int4 ri = C.ri[I], rj = C.rj[J];
  const float4 wi = C.wi[I], wj = C.wj[J];
  const int fi[4] = {ri.x, ri.y, ri.z, ri.w}, fj[4] = {rj.x, rj.y, rj.z, rj.w};
  const float ui[4] = {wi.x, wi.y, wi.z, wi.w}, uj[4] = {wj.x, wj.y, wj.z, wj.w};
  const float* e = F.e + F.nx * F.ny * k;
  float a = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = fj[q];
    const int s = j > 0 ? j - 1 : F.ny - 1, n = j < F.ny - 1 ? j + 1 : 0;
    const float2 cy = F.cy[j];
    float r = 0.0f;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int i = fi[p];
      if ((i + j) & 1) continue;  // black
      const float ew = i > 0 ? e[i - 1 + F.nx * j] : 0.0f;
      const float ee = i < F.nx - 1 ? e[i + 1 + F.nx * j] : 0.0f;
      const float2 cx = F.cx[i];
      r += ui[p] * ((cx.x * ew + cx.y * ee) + (cy.x * e[i + F.nx * s] + cy.y * e[i + F.nx * n]));
    }
    a += uj[q] * r;
  }
  C.b[I + C.nx * (J + C.ny * k)] = a;
}

// F.e += P C.e on the red columns (the black ones are solved next)
__global__ __launch_bounds__(256) void k_mg_prolong(MgLevel F, MgLevel C, const double* stopped) {
  if (*stopped != 0.0) return;
  const int ii = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y, k = blockIdx.z;
  if (j >= F.ny) return;
  const int i = 2 * ii + (j & 1);
  if (i >= F.nx) return;
  const int2 a = C.pi[i], c = C.pj[j];
  const float2 u = C.vi[i], v = C.vj[j];
  const float* e = C.e + C.nx * C.ny * k;
  const float lo = u.x * e[a.x + C.nx * c.x] + u.y * e[a.y + C.nx * c.x];
  const float hi = u.x * e[a.x + C.nx * c.y] + u.y * e[a.y + C.nx * c.y];
  F.e[i + F.nx * (j + F.ny * k)] += v.x * lo + v.y * hi;
}

// One direction of a grid: cell widths in units of the finest spacing, and the pairing of its n
// cells into nc coarse ones (the first n - nc take two each, the rest one).
struct Axis {
  bool wrap;
  std::vector<double> h, x;  // widths and centres
  double len = 0.0;
  explicit Axis(const std::vector<double>& w, bool wr) : wrap(wr), h(w), x(w.size()) {
    for (size_t f = 0; f < h.size(); ++f) {
      x[f] = len + 0.5 * h[f];
      len += h[f];
    }
  }
  int n() const { return (int)h.size(); }
  double dist(int f) const {  // between the centres of f and f + 1 (around the end)
    return f + 1 < n() ? x[f + 1] - x[f] : x[0] + len - x[f];
  }
  int parent(int f, int nc) const { return f < 2 * (n() - nc) ? f >> 1 : f - (n() - nc); }
  Axis coarse(int nc) const {
    std::vector<double> w(nc, 0.0);
    for (int f = 0; f < n(); ++f) w[parent(f, nc)] += h[f];
    return Axis(w, wrap);
  }
  // coupling of the second difference to the neighbours f - 1 (lo) and f + 1
  double lo(int f, double c) const {
    if (n() == 1) return 0.0;
    if (f == 0) return wrap ? c / (h[0] * dist(n() - 1)) : 0.0;
    return c / (h[f] * dist(f - 1));
  }
  double hi(int f, double c) const {
    if (n() == 1 || (f == n() - 1 && !wrap)) return 0.0;
    return c / (h[f] * dist(f));
  }
  // fine cell f interpolates linearly from two cells of the coarse axis
  void from(const Axis& C, int f, int c[2], double w[2]) const {
    c[0] = c[1] = parent(f, C.n());
    w[0] = 1.0;
    w[1] = 0.0;
    const double off = x[f] - C.x[c[0]];
    if (off == 0.0) return;  // unpaired
    const int up = off > 0.0 ? 1 : 0, o = c[0] + (up ? 1 : -1), m = C.n();
    if (!wrap && (o < 0 || o >= m)) return;  // mirrored at the face: the cell itself
    w[1] = std::abs(off) / (up ? C.dist(c[0]) : C.dist((c[0] + m - 1) % m));
    w[0] = 1.0 - w[1];
    c[1] = (o + m) % m;
  }
};

int coarse_of(int n, bool wrap) {
  int nc = (n + 1) / 2;
  if (wrap && nc % 2 && nc > 1) ++nc;  // red-black columns need an even periodic row
  return nc < n ? nc : n;
}

}  // namespace

void mg_release(MgPlan& mg) {
  if (mg.mem) hipFree(mg.mem);
  mg = MgPlan{};
}

hipError_t mg_setup(Dims d, float c2, float c3, const std::vector<float>& cn4l,
                    const std::vector<float>& cn4s, MgPlan& mg) {
  mg_release(mg);
  const int kp = d.kp;
  struct Host {
    int nx, ny;
    size_t b, e, t, inv, up, gf, gb, ri, rj, wi, wj, pi, pj, vi, vj, cx, cy, kx, ky;
  };
  std::vector<Host> hs;
  std::vector<float> tab;  // the tables, uploaded together (int tables as their bits)
  auto put = [&](const void* p, size_t n) {
    const size_t at = (tab.size() + 3) / 4 * 4;  // 16-byte aligned
    tab.resize(at + n);
    std::copy((const float*)p, (const float*)p + n, tab.begin() + at);
    return at;
  };
  std::vector<float> up4(cn4l.begin(), cn4l.begin() + kp), dn4(cn4s.begin(), cn4s.begin() + kp);
  up4[kp - 1] = 0.0f;
  dn4[0] = 0.0f;
  const size_t o4l = put(up4.data(), kp), o4s = put(dn4.data(), kp);
  Axis fx(std::vector<double>(d.ip, 1.0), false), fy(std::vector<double>(d.jp, 1.0), true);
  size_t cells = 0;
  while ((int)hs.size() < MG_MAX) {
    int nx = coarse_of(fx.n(), false), ny = coarse_of(fy.n(), true);
    // One direction alone while its couplings are over four times the other's: the columns are
    // swept point by point in i and j, which leaves errors along a weak direction to the coarse grids
    // (61x34x64 of 1 m x 20 m: 9 iterations, 5.7 ms a step; both at once 200 and 62, the pass alone
    // 580 and 42).
    const double sx = c2 * fx.n() * fx.n() / (fx.len * fx.len), sy = c3 * fy.n() * fy.n() / (fy.len * fy.len);
    if (fy.n() > 1 && fx.n() > 1) {
      if (sx > 4.0 * sy) ny = fy.n();
      if (sy > 4.0 * sx) nx = fx.n();
    }
    if (nx == fx.n() && ny == fy.n()) break;  // one column
    const Axis ax = fx.coarse(nx), ay = fy.coarse(ny);
    Host H{};
    H.nx = nx;
    H.ny = ny;
    // transfers from and to the finer axis; the restriction is the prolongation's transpose in
    // the cell volumes
    auto transfers = [&](const Axis& F, const Axis& C, size_t& r, size_t& w, size_t& p, size_t& v) {
      const int nc = C.n(), nf = F.n();
      std::vector<int> ri(4 * nc, 0), pi(2 * nf), cnt(nc, 0);
      std::vector<float> wi(4 * nc, 0.0f), vi(2 * nf);
      for (int f = 0; f < nf; ++f) {
        int c[2];
        double x[2];
        F.from(C, f, c, x);
        for (int q = 0; q < 2; ++q) {
          pi[2 * f + q] = c[q];
          vi[2 * f + q] = (float)x[q];
          if (x[q] == 0.0) continue;
          int at = 0;
          while (at < cnt[c[q]] && ri[4 * c[q] + at] != f) ++at;
          if (at == cnt[c[q]]) ++cnt[c[q]];
          ri[4 * c[q] + at] = f;
          wi[4 * c[q] + at] += (float)(x[q] * F.h[f] / C.h[c[q]]);
        }
      }
      r = put(ri.data(), ri.size());
      w = put(wi.data(), wi.size());
      p = put(pi.data(), pi.size());
      v = put(vi.data(), vi.size());
    };
    transfers(fx, ax, H.ri, H.wi, H.pi, H.vi);
    transfers(fy, ay, H.rj, H.wj, H.pj, H.vj);
    // couplings, and the classes of cells with the same sum of them
    std::vector<float> sums[2];
    auto couplings = [&](const Axis& A, float c, size_t& at, std::vector<float>& sum, std::vector<int>& cls) {
      std::vector<float> v(2 * A.n());
      for (int f = 0; f < A.n(); ++f) {
        v[2 * f] = (float)A.lo(f, c);
        v[2 * f + 1] = (float)A.hi(f, c);
        const float t = v[2 * f] + v[2 * f + 1];
        int q = (int)(std::find(sum.begin(), sum.end(), t) - sum.begin());
        if (q == (int)sum.size()) sum.push_back(t);
        cls.push_back(q);
      }
      at = put(v.data(), v.size());
    };
    std::vector<int> kx, ky;
    couplings(ax, c2, H.cx, sums[0], kx);
    couplings(ay, c3, H.cy, sums[1], ky);
    const int ncl = (int)(sums[0].size() * sums[1].size());
    for (int& q : kx) q *= (int)sums[1].size() * kp;
    for (int& q : ky) q *= kp;
    H.kx = put(kx.data(), kx.size());
    H.ky = put(ky.data(), ky.size());
    const int M = seg_levels(kp);
    std::vector<float> inv((size_t)ncl * kp), up(inv.size()), gf(inv.size()), gb(inv.size());
    for (int m = 0; m < ncl; ++m) {
      const double dxy = (double)sums[0][m / sums[1].size()] + (double)sums[1][m % sums[1].size()];
      const size_t o = (size_t)m * kp;
      double last = 0.0, x = 1.0;
      for (int k = 0; k < kp; ++k) {
        const double dg = dxy + up4[k] + dn4[k], pv = dg - dn4[k] * last;
        // the last pivot of the one column left at the end: the constants, which are free
        const bool free = !(pv > 1e-9 * dg);
        last = free ? 0.0 : up4[k] / pv;
        inv[o + k] = free ? 0.0f : (float)(1.0 / pv);
        up[o + k] = (float)last;
        // products of the recurrences' coefficients from the start (end) of a segment
        x = (k % M ? x : 1.0) * (double)dn4[k] * inv[o + k];
        gf[o + k] = (float)x;
      }
      for (int k = kp - 1; k >= 0; --k) {
        x = (k % M == M - 1 || k == kp - 1 ? 1.0 : x) * (double)up[o + k];
        gb[o + k] = (float)x;
      }
    }
    H.inv = put(inv.data(), inv.size());
    H.up = put(up.data(), up.size());
    H.gf = put(gf.data(), gf.size());
    H.gb = put(gb.data(), gb.size());
    const size_t n = (size_t)H.nx * H.ny * kp;
    H.b = cells;
    H.e = cells + n;
    H.t = cells + 2 * n;
    cells += 3 * n;
    hs.push_back(H);
    fx = ax;
    fy = ay;
  }
  if (hs.empty()) return hipSuccess;
  const size_t nt = (tab.size() + 3) / 4 * 4;
  hipError_t err = hipMalloc(&mg.mem, (nt + cells) * sizeof(float));
  if (err == hipSuccess) err = hipMemcpy(mg.mem, tab.data(), tab.size() * sizeof(float), hipMemcpyHostToDevice);
  if (err == hipSuccess) err = hipMemset(mg.mem + nt, 0, cells * sizeof(float));
  if (err != hipSuccess) {
    mg_release(mg);
    return err;
  }
  float *T = mg.mem, *A = mg.mem + nt;
  mg.c4l = T + o4l;
  mg.c4s = T + o4s;
  for (const Host& H : hs) {
    MgLevel& L = mg.l[mg.nl++];
    L = MgLevel{H.nx, H.ny, (const float2*)(T + H.cx), (const float2*)(T + H.cy),
                (const int*)(T + H.kx), (const int*)(T + H.ky), A + H.b, A + H.e, A + H.t, T + H.inv, T + H.up,
                T + H.gf, T + H.gb,
                (const int4*)(T + H.ri), (const int4*)(T + H.rj), (const float4*)(T + H.wi),
                (const float4*)(T + H.wj), (const int2*)(T + H.pi), (const int2*)(T + H.pj),
                (const float2*)(T + H.vi), (const float2*)(T + H.vj)};
  }
  return hipSuccess;
}

void launch_mg_correct(hipStream_t st, Dims d, SplitSOR sp, Mixed mx, const MgPlan& mg) {
  const int kp = d.kp;
  const double* stopped = mx.cg + 4;
  auto columns = [&](const MgLevel& L, int red, bool first) {
    const int n = (L.nx + 1) / 2 * L.ny;
    if (kp > 16 * MG_SEG) {  // taller than the segments: a thread per column
      const dim3 grid((n + MG_BX - 1) / MG_BX), blk(MG_BX);
      if (first)
        hipLaunchKernelGGL(k_mg_columns<true>, grid, blk, 0, st, L, kp, red, mg.c4s, L.b, L.t, L.e, stopped);
      else
        hipLaunchKernelGGL(k_mg_columns<false>, grid, blk, 0, st, L, kp, red, mg.c4s, L.b, L.t, L.e, stopped);
      return;
    }
    const dim3 grid((n + 31) / 32), blk(32, MG_SEG);
    auto go = [&](auto f, auto m) {
      hipLaunchKernelGGL((k_mg_segments<decltype(m)::value, decltype(f)::value>), grid, blk, 0, st, L, kp,
                         red, mg.c4s, L.b, L.e, stopped);
    };
    auto pick = [&](auto f) {
      if (seg_levels(kp) == 8)
        go(f, std::integral_constant<int, 8>{});
      else if (seg_levels(kp) == 12)
        go(f, std::integral_constant<int, 12>{});
      else
        go(f, std::integral_constant<int, 16>{});
    };
    if (first)
      pick(std::true_type{});
    else
      pick(std::false_type{});
  };
  const dim3 blk(64, 4);
  auto grid_of_level = [&](int nx, int ny) { return dim3((nx + 63) / 64, (ny + 3) / 4, kp); };
  hipLaunchKernelGGL(k_mg_restrict_split, grid_of_level(mg.l[0].nx, mg.l[0].ny), blk, 0, st, d, sp, mg.l[0],
                     mx.q[0], stopped);
  for (int q = 0; q < mg.nl; ++q) {
    const MgLevel& L = mg.l[q];
    columns(L, 0, true);
    if (q + 1 == mg.nl) break;  // one column
    columns(L, 1, false);
    const MgLevel& C = mg.l[q + 1];
    hipLaunchKernelGGL(k_mg_restrict, grid_of_level(C.nx, C.ny), blk, 0, st, L, C, stopped);
  }
  for (int q = mg.nl - 2; q >= 0; --q) {
    const MgLevel& L = mg.l[q];
    hipLaunchKernelGGL(k_mg_prolong, grid_of_level((L.nx + 1) / 2, L.ny), blk, 0, st, L, mg.l[q + 1], stopped);
    columns(L, 1, false);
    columns(L, 0, false);
  }
  hipLaunchKernelGGL(k_mg_prolong_split, grid_of_level((d.ip + 1) / 2, d.jp), blk, 0, st, d, sp, mg.l[0],
                     mx.z[0], stopped);
}

}  // namespace les
