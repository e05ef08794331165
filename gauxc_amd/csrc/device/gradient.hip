// EXC nuclear gradient, RKS and UKS, FP64 (GauXC eval_exc_grad with
// include_weight_derivatives: reference_replicated_xc_host_integrator_
// exc_grad.hpp:106-600, weights.cxx:806-990; device counterparts
// increment_exc_grad.cu and cuda_ssf_1d.cu).
//
// GauXC contracts, per task, point and function mu on an atom other than the
// task's parent,
//   g_mu = w vrho X_mu grad B_mu
//        + 2 w vgamma [ X_mu (H_mu grad rho) + grad B_mu (grad rho . Xg_mu) ]
// with X = 2 P_sub B, Xg_j = 2 P_sub dB/dj and H_mu the Hessian of B_mu,
// and adds -2 g to the function's atom and +2 g to the parent (the grid
// moves with the parent).  Here the first and third terms are one product:
//   w vrho X + 2 w vgamma grad rho . Xg = 2 P_sub Za,
//   Za = w vrho B + 2 w vgamma grad rho . grad B,
// so a task needs two plane products (X = 2 P_sub B for the Hessian term of
// GGAs, Y = 2 P_sub Za) instead of four, and
//   g_mu = grad B_mu . Y_mu + X_mu (H_mu c),  c = 2 w vgamma grad rho.
// grad B and H c are evaluated where they are used (k_grad_contract), and so
// is grad B in the density stage and in Za, so of the chunk scratch's five
// planes collocation fills only B (0); X, stored by the density stage itself,
// goes to 1 (GGA), Za to 4, Y = 2 P_sub Za to 2.
// The grid-weight part contracts the SSF weight derivatives with w eps rho
// per point (k_ssf_grad).
//
// UKS (GauXC eval_exc_grad(Ps, Pz), the same driver with spin_dim 2): with
// X_N = P_s B, X_Z = P_z B (factor 1), rho_+- = (n +- m)/2 and the polarised
// functional,
//   g_mu = grad B_mu . Y_mu + X_N,mu (H_mu c_s) + X_Z,mu (H_mu c_z),
//   Y = P_s Za_s + P_z Za_z,
//   Za_s = w (vrho_a + vrho_b)/2 B + c_s . grad B,
//   Za_z = w (vrho_a - vrho_b)/2 B + c_z . grad B,
//   c_s = g1 grad n + g2 grad m,  c_z = g2 grad n + g3 grad m,
// g1 = (v_aa + v_ab + v_bb)/2, g2 = (v_aa - v_bb)/2, g3 = (v_aa - v_ab + v_bb)/2
// (w vsigma folded in), and f = w eps (rho_a + rho_b) for the weight part.
// Planes: X_N -> 2 and X_Z -> 3, Za_s and Za_z in turn -> 4, Y -> 1.
#include "internal.hpp"
#include "functional.hpp"
#include "shell_eval.hpp"
#include "ssf.hpp"

#include <type_traits>

namespace xcq {

// ---- per-point coefficients ------------------------------------------------
// From the raw sums of the P pass (factor 2: rho = sum B X, grad rho =
// 2 sum dB X): coef[block][4][64] = (w vrho, 2 w vsigma grad rho) -- the Za
// coefficients, whose gradient part is also the Hessian term's c -- and
// wf[block][64] = w eps rho; the block's (w eps rho, w rho) sums to red.
__global__ __launch_bounds__(64) void k_grad_points(const WorkItem* __restrict__ items,
                                                    const DevTask* __restrict__ tasks,
                                                    const double* __restrict__ weights,
                                                    int func, int gga,
                                                    const double* __restrict__ dp,
                                                    double* __restrict__ red,
                                                    double* __restrict__ coef,
                                                    double* __restrict__ wf) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  const int64_t b = t.red_off + wi.a;
  const int p = wi.a * kPtBlock + tid;
  double s[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) s[c] = dp[b * 256 + c * 64 + tid];
  double g[3], sig = 0.;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g[d] = 2.0 * s[1 + d];
    sig += g[d] * g[d];
  }
  double e = 0., n = 0., a = 0., cv[3] = {0., 0., 0.};
  if (p < t.npts) {
    const double w = weights[t.pt_off + p];
    const XCOut o = dev_eval_functional(func, s[0], sig);
    e = w * o.e;
    n = w * s[0];
    a = w * o.vr;
    if (gga) {
#pragma unroll
      for (int d = 0; d < 3; ++d) cv[d] = 2.0 * w * o.vs * g[d];
    }
  }
  coef[b * 256 + tid] = a;
#pragma unroll
  for (int d = 0; d < 3; ++d) coef[b * 256 + (1 + d) * 64 + tid] = cv[d];
  wf[b * 64 + tid] = e;
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * b] = e;
    red[2 * b + 1] = n;
  }
}

// UKS: from the raw sums of the P_s and P_z passes (factor 1) at block b,
// coef_s[b] = (w (vrho_a + vrho_b)/2, c_s), coef_z[b] = (w (vrho_a -
// vrho_b)/2, c_z) and wf[b] = w eps (rho_a + rho_b).  coef_s and coef_z may
// be the sum buffers themselves: each thread reads its own entries first.
__global__ __launch_bounds__(64) void k_grad_points_uks(const WorkItem* __restrict__ items,
                                                        const DevTask* __restrict__ tasks,
                                                        const double* __restrict__ weights,
                                                        int func, int gga, double* ds,
                                                        double* dz, double* __restrict__ red,
                                                        double* __restrict__ wf) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  const int64_t b = t.red_off + wi.a;
  const int p = wi.a * kPtBlock + tid;
  double sv[4], zv[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    sv[c] = ds[b * 256 + c * 64 + tid];
    zv[c] = dz[b * 256 + c * 64 + tid];
  }
  const double ra = 0.5 * (sv[0] + zv[0]), rb = 0.5 * (sv[0] - zv[0]);
  double gn[3], gm[3], nn = 0., mm = 0., nm = 0.;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    gn[d] = 2.0 * sv[1 + d];
    gm[d] = 2.0 * zv[1 + d];
    nn += gn[d] * gn[d];
    mm += gm[d] * gm[d];
    nm += gn[d] * gm[d];
  }
  double e = 0., n = 0., as = 0., az = 0., cs[3] = {0., 0., 0.}, cz[3] = {0., 0., 0.};
  if (p < t.npts) {
    const double w = weights[t.pt_off + p];
    const double saa = gga ? 0.25 * (nn + mm) + 0.5 * nm : 0.;
    const double sab = gga ? 0.25 * (nn - mm) : 0.;
    const double sbb = gga ? 0.25 * (nn + mm) - 0.5 * nm : 0.;
    const XCOutPol o = dev_eval_functional_pol(func, ra, rb, saa, sab, sbb);
    e = w * o.e;
    n = w * (ra + rb);
    as = 0.5 * w * (o.vra + o.vrb);
    az = 0.5 * w * (o.vra - o.vrb);
    if (gga) {
      const double vpp = w * o.vsaa, vpm = w * o.vsab, vmm = w * o.vsbb;
      const double g1 = 0.5 * (vpp + vpm + vmm), g2 = 0.5 * (vpp - vmm),
                   g3 = 0.5 * (vpp - vpm + vmm);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        cs[d] = g1 * gn[d] + g2 * gm[d];
        cz[d] = g2 * gn[d] + g3 * gm[d];
      }
    }
  }
  ds[b * 256 + tid] = as;
  dz[b * 256 + tid] = az;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    ds[b * 256 + (1 + d) * 64 + tid] = cs[d];
    dz[b * 256 + (1 + d) * 64 + tid] = cz[d];
  }
  wf[b * 64 + tid] = e;
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * b] = e;
    red[2 * b + 1] = n;
  }
}

// ---- basis-function part of the gradient -----------------------------------
// A shell's contribution at a point,
//   s_i = sum_f [ Y_f d_i B_f + sum_j c_j X_f d_i d_j B_f ],
// for B_f = R(r^2) m_f with R1 = -2 sum a c e^{-a r^2}, R2 = 4 sum a^2 c
// e^{-a r^2} (so d_i R = x_i R1, d_i d_j R = delta_ij R1 + x_i x_j R2).  The
// sums over f go into the polynomials y = sum_f Y_f m_f and p = sum_f X_f
// m_f, collected by Cartesian coefficient (7 functions of an f shell into 10
// coefficients, two terms each), which are then differentiated once per
// shell instead of each m_f by itself:
//   s_i = R d_i y + x_i R1 y
//       + R d_i (c . grad p) + R1 (d_i p (r . c) + x_i (c . grad p))
//       + p (c_i R1 + x_i (r . c) R2).
template <int L>
constexpr int kCart = (L + 1) * (L + 2) / 2;

// q[cart] = sum_f v_f C_f,cart; get(f) gives v_f.
template <int L, typename Get>
__device__ __forceinline__ void cart_coeffs(bool pure, double (&q)[kCart<L>], Get&& get) {
  if (!pure) {
#pragma unroll
    for (int ic = 0; ic < kCart<L>; ++ic) q[ic] = get(ic);
    return;
  }
#pragma unroll
  for (int ic = 0; ic < kCart<L>; ++ic) q[ic] = 0.;
#pragma unroll
  for (int m = 0; m < 2 * L + 1; ++m) {
    const double v = get(m);
#pragma unroll
    for (int ic = 0; ic < kCart<L>; ++ic)
      if (kSph.c[L][m][ic] != 0.) q[ic] = fma(kSph.c[L][m][ic], v, q[ic]);
  }
}

// Powers 0 .. L of a displacement; 0 where the exponent is negative.
template <int L>
struct Powers {
  double x[L + 1], y[L + 1], z[L + 1];
  __device__ __forceinline__ Powers(double px, double py, double pz) {
    x[0] = y[0] = z[0] = 1.;
#pragma unroll
    for (int k = 1; k <= L; ++k) {
      x[k] = x[k - 1] * px;
      y[k] = y[k - 1] * py;
      z[k] = z[k - 1] * pz;
    }
  }
  // d^i/dx^i d^j/dy^j d^k/dz^k of x^a y^b z^c, i + j + k <= 2.
  __device__ __forceinline__ double mono(int a, int b, int c, int i, int j, int k) const {
    auto f = [](int n, int d) { return d == 0 ? 1 : d == 1 ? n : n * (n - 1); };
    const int w = f(a, i) * f(b, j) * f(c, k);
    if (w == 0) return 0.;
    return (double)w * (x[a - i] * y[b - j] * z[c - k]);
  }
};

// s += R grad y + R1 r y for the polynomial y with coefficients q.
template <int L>
__device__ __forceinline__ void add_value(const Powers<L>& pw, const double (&q)[kCart<L>],
                                          double x, double y, double z, double R, double R1,
                                          double (&s)[3]) {
  double v = 0., g[3] = {0., 0., 0.};
  int ic = 0;
#pragma unroll
  for (int a = L; a >= 0; --a)
#pragma unroll
    for (int b = L - a; b >= 0; --b, ++ic) {
      const int c = L - a - b;
      v = fma(q[ic], pw.mono(a, b, c, 0, 0, 0), v);
      if (a) g[0] = fma(q[ic], pw.mono(a, b, c, 1, 0, 0), g[0]);
      if (b) g[1] = fma(q[ic], pw.mono(a, b, c, 0, 1, 0), g[1]);
      if (c) g[2] = fma(q[ic], pw.mono(a, b, c, 0, 0, 1), g[2]);
    }
  v *= R1;
  s[0] += R * g[0] + x * v;
  s[1] += R * g[1] + y * v;
  s[2] += R * g[2] + z * v;
}

// s += the Hessian of R p times (cx, cy, cz), p with coefficients q.
template <int L>
__device__ __forceinline__ void add_hessian(const Powers<L>& pw, const double (&q)[kCart<L>],
                                            double x, double y, double z, double R, double R1,
                                            double R2, double cx, double cy, double cz,
                                            double (&s)[3]) {
  double v = 0., g[3] = {0., 0., 0.}, h[6] = {0., 0., 0., 0., 0., 0.};  // xx xy xz yy yz zz
  int ic = 0;
#pragma unroll
  for (int a = L; a >= 0; --a)
#pragma unroll
    for (int b = L - a; b >= 0; --b, ++ic) {
      const int c = L - a - b;
      v = fma(q[ic], pw.mono(a, b, c, 0, 0, 0), v);
      if (a) g[0] = fma(q[ic], pw.mono(a, b, c, 1, 0, 0), g[0]);
      if (b) g[1] = fma(q[ic], pw.mono(a, b, c, 0, 1, 0), g[1]);
      if (c) g[2] = fma(q[ic], pw.mono(a, b, c, 0, 0, 1), g[2]);
      if (a > 1) h[0] = fma(q[ic], pw.mono(a, b, c, 2, 0, 0), h[0]);
      if (a && b) h[1] = fma(q[ic], pw.mono(a, b, c, 1, 1, 0), h[1]);
      if (a && c) h[2] = fma(q[ic], pw.mono(a, b, c, 1, 0, 1), h[2]);
      if (b > 1) h[3] = fma(q[ic], pw.mono(a, b, c, 0, 2, 0), h[3]);
      if (b && c) h[4] = fma(q[ic], pw.mono(a, b, c, 0, 1, 1), h[4]);
      if (c > 1) h[5] = fma(q[ic], pw.mono(a, b, c, 0, 0, 2), h[5]);
    }
  const double rc = x * cx + y * cy + z * cz;
  const double cg = cx * g[0] + cy * g[1] + cz * g[2];
  const double t = R1 * cg + v * rc * R2;  // along r
  const double u = v * R1;                 // along c
  s[0] += R * (cx * h[0] + cy * h[1] + cz * h[2]) + R1 * g[0] * rc + x * t + cx * u;
  s[1] += R * (cx * h[1] + cy * h[3] + cz * h[4]) + R1 * g[1] * rc + y * t + cy * u;
  s[2] += R * (cx * h[2] + cy * h[4] + cz * h[5]) + R1 * g[2] * rc + z * t + cz * u;
}

// One (task, 64-point block) per 256-thread workgroup; lane = point, wave w
// takes the task's shells w, w + 4, ..., their parameters staged in LDS 64
// at a time.  Per shell (with the weight derivatives: on an atom other than
// the parent) the sums above, reduced over the wave; runs of shells on one
// atom are added to that atom with one set of atomics, the parent's share
// (weight derivatives only) once per wave at the end.  NX = 1 (RKS): Y in
// plane y_pl, X in plane x_pl with the coefficients coef_s (GGA); NX = 2
// (UKS): X_N and X_Z in planes x_pl and x_pl + 1 with coef_s and coef_z.
// What bounds it: FP64 vector work and the reads of Y and X.  On 13 waters
// (883,000 points, PBE) it takes 0.85 ms.  4.1 ms of atomic additions to one
// gradient had hidden the arithmetic (kGradCopies).
__device__ __forceinline__ void reduce_lanes(double (&v)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d)
    for (int off = 32; off > 0; off >>= 1) v[d] += __shfl_xor(v[d], off);
}

struct GradShells {
  static constexpr int kMax = 64, kPrims = 4;
  double ox[kMax], oy[kMax], oz[kMax], a[kPrims][kMax], c[kPrims][kMax];
  int bf0[kMax], info[kMax], ish[kMax], atom[kMax];
};

template <bool GGA, int LMAX, int NX>
__global__ __launch_bounds__(256, LMAX > 3 || NX > 1 ? 2 : 3) void k_grad_contract(
    const WorkItem* __restrict__ items, const DevTask* __restrict__ tasks,
    const DevShell* __restrict__ shells, const int32_t* __restrict__ shell_list,
    const int32_t* __restrict__ lsh_first, const int32_t* __restrict__ shell_atom,
    const double* __restrict__ px, const double* __restrict__ py,
    const double* __restrict__ pz, const double* __restrict__ scratch,
    const double* __restrict__ coef_s, const double* __restrict__ coef_z, int weight_derivs,
    double* __restrict__ grad, int64_t gstride, int x_pl, int y_pl) {
  __shared__ GradShells st;
  grad += (int64_t)(blockIdx.x % kGradCopies) * gstride;
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = wi.a * kPtBlock + lane;
  const bool valid = p < t.npts;
  const int pc = min(p, t.npts - 1);
  const double gx = px[t.pt_off + pc], gy = py[t.pt_off + pc], gz = pz[t.pt_off + pc];
  const int64_t b = t.red_off + wi.a;
  double cs[3] = {0., 0., 0.}, cz[3] = {0., 0., 0.};
  if (GGA && valid) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      cs[d] = coef_s[b * 256 + (1 + d) * 64 + lane];
      if (NX > 1) cz[d] = coef_z[b * 256 + (1 + d) * 64 + lane];
    }
  }
  const int64_t ld = t.npts_pad;
  const int64_t plane = (int64_t)t.nbe * ld;
  const int64_t m0 = (int64_t)wi.a * kPtBlock + lane;
  const double* Yp = scratch + t.b_off + y_pl * plane + m0;
  const double* Xp = scratch + t.b_off + x_pl * plane + m0;
  int cur = -1;                            // atom of the running sum (uniform)
  double run[3] = {0., 0., 0.}, par[3] = {0., 0., 0.};
  auto add = [&](int at, double fac, double v0, double v1, double v2) {
    const double val = lane == 0 ? v0 : lane == 1 ? v1 : v2;
    if (lane < 3) atomicAdd(grad + 3 * (int64_t)at + lane, fac * val);
  };
  auto flush = [&]() {
    if (cur >= 0) add(cur, -2.0, run[0], run[1], run[2]);
  };
  for (int pass = 0; pass < t.nshells; pass += GradShells::kMax) {
    const int nsh = min(GradShells::kMax, t.nshells - pass);
    __syncthreads();  // the previous pass is done with the staged shells
    if (tid < nsh) {
      const int ish = shell_list[t.sh_off + pass + tid];
      const DevShell* sh = shells + ish;
      st.ish[tid] = ish;
      st.atom[tid] = shell_atom[ish];
      st.bf0[tid] = lsh_first[t.lsh_off + pass + tid];
      st.info[tid] = sh->l | (sh->pure ? 1 << 8 : 0) | (sh->nprim << 16);
      st.ox[tid] = sh->O[0];
      st.oy[tid] = sh->O[1];
      st.oz[tid] = sh->O[2];
      const int np = min(sh->nprim, GradShells::kPrims);
      for (int k = 0; k < np; ++k) {
        st.a[k][tid] = sh->alpha[k];
        st.c[k][tid] = sh->coeff[k];
      }
    }
    __syncthreads();
    for (int k = wave; k < nsh; k += 4) {
      const int at = __builtin_amdgcn_readfirstlane(st.atom[k]);
      if (at < 0 || (weight_derivs && at == t.iparent)) continue;
      const int bf0 = __builtin_amdgcn_readfirstlane(st.bf0[k]);
      const int info = __builtin_amdgcn_readfirstlane(st.info[k]);
      const int l = info & 0xff, nprim = info >> 16;
      const bool pure = (info >> 8) & 1;
      const double x = gx - st.ox[k], y = gy - st.oy[k], z = gz - st.oz[k];
      const double r2 = x * x + y * y + z * z;
      double R = 0., R1 = 0., R2 = 0.;
      auto prim = [&](double a, double c) {
        const double e = c * exp(-a * r2);
        R += e;
        R1 -= 2. * a * e;
        R2 += 4. * a * a * e;
      };
      for (int q = 0; q < min(nprim, GradShells::kPrims); ++q) prim(st.a[q][k], st.c[q][k]);
      if (nprim > GradShells::kPrims) {
        const DevShell* sh = shells + __builtin_amdgcn_readfirstlane(st.ish[k]);
        for (int q = GradShells::kPrims; q < nprim; ++q) prim(sh->alpha[q], sh->coeff[q]);
      }
      double s[3] = {0., 0., 0.};
      auto shell = [&](auto LC) {
        constexpr int L = decltype(LC)::value;
        const Powers<L> pw(x, y, z);
        double q[kCart<L>];
        const int64_t r0 = (int64_t)bf0 * ld;
        auto get = [&](const double* pl) {
          return [=](int f) { return valid ? pl[r0 + f * ld] : 0.; };
        };
        cart_coeffs<L>(pure, q, get(Yp));
        add_value<L>(pw, q, x, y, z, R, R1, s);
        if constexpr (GGA) {
          cart_coeffs<L>(pure, q, get(Xp));
          add_hessian<L>(pw, q, x, y, z, R, R1, R2, cs[0], cs[1], cs[2], s);
          if constexpr (NX > 1) {
            cart_coeffs<L>(pure, q, get(Xp + plane));
            add_hessian<L>(pw, q, x, y, z, R, R1, R2, cz[0], cz[1], cz[2], s);
          }
        }
      };
      if (l == 0) shell(std::integral_constant<int, 0>{});
      else if (l == 1) shell(std::integral_constant<int, 1>{});
      else if (l == 2) shell(std::integral_constant<int, 2>{});
      else if (l == 3 || LMAX == 3) shell(std::integral_constant<int, 3>{});
      else shell(std::integral_constant<int, LMAX>{});
      if (at != cur) {
        // The running sums are per lane; they are reduced when their atom's
        // run of shells ends.
        reduce_lanes(run);
        flush();
        cur = at;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          par[d] += run[d];
          run[d] = 0.;
        }
      }
#pragma unroll
      for (int d = 0; d < 3; ++d) run[d] += s[d];
    }
  }
  reduce_lanes(run);
  flush();
  if (weight_derivs && cur >= 0) {
#pragma unroll
    for (int d = 0; d < 3; ++d) par[d] += run[d];
    add(t.iparent, 2.0, par[0], par[1], par[2]);
  }
}

// ---- grid-weight part ---------------------------------------------------------
// Derivatives of the SSF weights w_i = w0_i P_A(r_i) / sum_C P_C(r_i)
// contracted with f_i = w_i eps_i rho_i, the points moving with their parent
// atom A (weights.cxx:806-990).  P_B = prod_{C != B} s(mu_BC), s(mu) = 1
// (mu <= -a), 0 (mu >= a), (1 - g(mu / a)) / 2 otherwise (g the Frisch
// polynomial, a = 0.64), formed here as that product; its logarithmic
// derivative t(mu) = s'(mu) / s(mu) in the factored form
//   1 - g(v) = (1 - v)^4 (5 v^3 + 20 v^2 + 29 v + 16) / 16,  g'(v) = 35 (1 - v^2)^3 / 16,
//   t(mu) = 35 (1 + v)^3 / ((mu - a)(5 v^3 + 20 v^2 + 29 v + 16)),  v = mu / a,
// which stays accurate up to the |mu| < a - 1e-4 bound the contraction uses.
// With neighbour lists (nbr_idx / nbr_i: row A holds every atom in order of
// increasing R_AB, A itself first, and 1 / (a R_AB)) the loops stop where the triangle
// inequality makes every remaining term vanish, as in the weights kernel: a
// factor s(mu_BC) differs from 1, and |mu_BC| can fall below a, only for
// R_BC < 2 d_B / (1 - a); P_B > 0 only for d_B <= (1 + a)/(1 - a) d_min; so
// the parent's list is read up to max(2 d_A / (1 - a), d_A + that bound) and
// each B's list up to 2 d_B / (1 - a), all widened by a relative 1e-10.  The
// terms skipped are exactly zero (factors exactly 1).  Without lists every
// loop runs over all atoms.
//
// One wave per 64-point block, lane = point.  All loops are uniform: they
// run as far as any lane needs, so indices and atoms are read by scalar
// loads and lanes that need less multiply by exact ones.  The first pass
// forms sum_B P_B and keeps the products of the first kSsfKeep atoms with
// P_B > kSsfTol in any lane; the second takes A (with P_A - sum in P_B's
// place, from dw/dR_C of w's numerator and denominator together) and those
// atoms, and forms for each neighbour C the derivative of s(mu_BC).  What
// falls on C is summed over the wave, four C at a time (a transposing
// reduction: 21 exchanges where 12 separate sums take 72); what falls on B
// and on A stays in registers and is summed once.
// What bounds it: FP64 vector work.  On 13 waters (883,000 points) 1.25 ms;
// with every thread's own loop bounds and one atomic addition per thread and
// term 6.4 ms.
constexpr double kSsfTol = 1e-13;

constexpr int kSsfKeep = 12;

template <bool LISTS>
__global__ __launch_bounds__(64) void k_ssf_grad(const WorkItem* __restrict__ items,
                                                 const DevTask* __restrict__ tasks,
                                                 const double* __restrict__ px,
                                                 const double* __restrict__ py,
                                                 const double* __restrict__ pz, int natoms,
                                                 const double* __restrict__ xyz,
                                                 const double* __restrict__ dnear,
                                                 const double* __restrict__ wf,
                                                 double* __restrict__ grad, int64_t gstride,
                                                 const int32_t* __restrict__ nbr_idx,
                                                 const double* __restrict__ nbr_i) {
  __shared__ double keep[kSsfKeep][64];
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int lane = threadIdx.x;
  const int p = wi.a * kPtBlock + lane;
  const int pc = min(p, t.npts - 1);
  const double f = wf[(t.red_off + wi.a) * 64 + lane];
  const double rx = px[t.pt_off + pc], ry = py[t.pt_off + pc], rz = pz[t.pt_off + pc];
  const int A = t.iparent;
  auto X = [&](int at, int d) { return xyz[3 * (int64_t)at + d]; };
  auto dist = [&](int at) {
    const double dx = rx - X(at, 0), dy = ry - X(at, 1), dz = rz - X(at, 2);
    return sqrt(dx * dx + dy * dy + dz * dz);
  };
  // Entry q of B's list: atom C and 1 / (a R_BC); lists start with B itself.
  auto nbr_at = [&](int B, int q) { return LISTS ? nbr_idx[(int64_t)B * natoms + q] : q; };
  auto nbr_inv = [&](int B, int q) {
    if (LISTS) return nbr_i[(int64_t)B * natoms + q];
    const double dx = X(B, 0) - X(q, 0), dy = X(B, 1) - X(q, 1), dz = X(B, 2) - X(q, 2);
    return 1. / (kSsfA * sqrt(dx * dx + dy * dy + dz * dz));
  };
  constexpr double kWiden = 1.0 + 1e-10;
  constexpr double bound = kSsfA - 1e-4;
  const double dA = dist(A);
  const bool on = p < t.npts && !(fabs(f) < 1e-12) && !(dA < 0.5 * (1. - kSsfA) * dnear[A]);
  if (!__any(on)) return;
  // Nearest atom (R_AB* <= 2 d_A) and the candidate bound.
  double cbound = INFINITY, imax = 0.;  // imax: 1 / (a R) at the list's end
  if (LISTS) {
    double dmin = dA;
    const double i2 = 1.0 / (kSsfA * 2.0 * dA * kWiden);
    for (int k = 1; k < natoms && __any(on && nbr_inv(A, k) >= i2); ++k)
      dmin = fmin(dmin, dist(nbr_at(A, k)));
    cbound = (1.0 + kSsfA) / (1.0 - kSsfA) * dmin * kWiden + 1e-12;
    imax = 1.0 / (kSsfA * fmax(2.0 * dA / (1.0 - kSsfA), dA + cbound) * kWiden);
  }
  // 1 / (a R) where B's list ends.
  auto reach = [&](double dB) { return (1.0 - kSsfA) / (kSsfA * 2.0 * dB * kWiden); };
  constexpr int q0 = LISTS ? 1 : 0;
  // P_B, 0 in lanes that are off or beyond the candidate bound.
  auto part = [&](int B, double dB) {
    double v = on && dB <= cbound ? 1. : 0.;
    if (!__any(v > 0.)) return v;
    const double rf = reach(dB);
    for (int q = q0; q < natoms; q += 4) {
      int C[4];
      double I[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int qj = min(q + j, natoms - 1);
        C[j] = nbr_at(B, qj);
        I[j] = nbr_inv(B, qj);
      }
      if (!__any(v > 0. && (!LISTS || I[0] > rf))) break;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (q + j < natoms && C[j] != B) v *= ssf_s((dB - dist(C[j])) * I[j]);
    }
    return v;
  };
  double sum = 0., pA = 0.;
  int nkeep = 0, kover = natoms, kept[kSsfKeep];
  for (int k = 0; k < natoms && (!LISTS || __any(on && nbr_inv(A, k) >= imax)); ++k) {
    const int B = nbr_at(A, k);
    const double pB = part(B, dist(B));
    sum += pB;
    if (B == A) pA = pB;
    else if (__any(pB > kSsfTol) && kover == natoms) {
      if (nkeep == kSsfKeep) kover = k;
      else {
        keep[nkeep][lane] = pB;
#pragma unroll
        for (int i = 0; i < kSsfKeep; ++i)
          if (i == nkeep) kept[i] = B;
        ++nkeep;
      }
    }
  }
  grad += (int64_t)(blockIdx.x % kGradCopies) * gstride;
  const double fs = on ? f / sum : 0.;
  double gA[3] = {0., 0., 0.};
  // The derivatives of B's factors, weighted by cf.
  auto derivs = [&](int B, double cf, bool act) {
    const double dB = dist(B), rf = reach(dB);
    const double iB = act && dB > 0. ? cf / dB : 0.;
    const double ub[3] = {(X(B, 0) - rx) * iB, (X(B, 1) - ry) * iB, (X(B, 2) - rz) * iB};
    double gb[3] = {0., 0., 0.};
    for (int q = q0; q < natoms; q += 4) {
      int C[4];
      double I[4], g[4][3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int qj = min(q + j, natoms - 1);
        C[j] = nbr_at(B, qj);
        I[j] = nbr_inv(B, qj);
      }
      if (LISTS && !__any(act && I[0] > rf)) break;
      bool any = false;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double dC = dist(C[j]);
        const double v = (dB - dC) * I[j], mu = kSsfA * v, iR = kSsfA * I[j];
        const bool in = q + j < natoms && C[j] != B && act && fabs(mu) < bound;
#pragma unroll
        for (int d = 0; d < 3; ++d) g[j][d] = 0.;
        if (!__any(in)) continue;
        const double v1 = 1. + v;
        const double tm = 35. * (v1 * v1 * v1) /
                          ((mu - kSsfA) * (((5. * v + 20.) * v + 29.) * v + 16.)) * iR;
        const double tt = in ? tm : 0.;
        const double e = cf * tt * mu * iR;
        const double iC = in ? cf * tt / dC : 0.;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const double s = e * (X(C[j], d) - X(B, d));
          gb[d] -= tt * ub[d] + s;
          const double r = d == 0 ? rx : d == 1 ? ry : rz;
          g[j][d] = C[j] == A ? 0. : iC * (X(C[j], d) - r) + s;
          gA[d] -= g[j][d];
        }
        any = any || C[j] != A;
      }
      if (!any) continue;
      // Sums over the wave: lanes of 16-lane group j end with those of C[j].
      double u[2][3], w[3];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          u[j][d] = (lane & 32 ? g[j + 2][d] : g[j][d]) +
                    __shfl_xor(lane & 32 ? g[j][d] : g[j + 2][d], 32);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        w[d] = (lane & 16 ? u[1][d] : u[0][d]) + __shfl_xor(lane & 16 ? u[0][d] : u[1][d], 16);
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) w[d] += __shfl_xor(w[d], off);
      }
      const int at = lane & 32 ? (lane & 16 ? C[3] : C[2]) : (lane & 16 ? C[1] : C[0]);
      const int d = lane & 15;
      const double val = d == 0 ? w[0] : d == 1 ? w[1] : w[2];
      if (d < 3 && val != 0.) atomicAdd(grad + 3 * (int64_t)at + d, val);
    }
    if (B == A) return;
#pragma unroll
    for (int d = 0; d < 3; ++d) gA[d] -= gb[d];
    reduce_lanes(gb);
    const double val = lane == 0 ? gb[0] : lane == 1 ? gb[1] : gb[2];
    if (lane < 3) atomicAdd(grad + 3 * (int64_t)B + lane, val);
  };
  derivs(A, (pA - sum) * fs, on);
  for (int i = 0; i < nkeep; ++i) {
    int B = 0;
#pragma unroll
    for (int q = 0; q < kSsfKeep; ++q)
      if (q == i) B = kept[q];
    const double pB = keep[i][lane];
    derivs(B, pB * fs, pB > kSsfTol);
  }
  // Atoms beyond the kept ones (many comparable distances): formed again.
  for (int k = kover; k < natoms && (!LISTS || __any(on && nbr_inv(A, k) >= imax)); ++k) {
    const int B = nbr_at(A, k);
    if (B == A) continue;
    const double pB = part(B, dist(B));
    if (__any(pB > kSsfTol)) derivs(B, pB * fs, pB > kSsfTol);
  }
  reduce_lanes(gA);
  const double val = lane == 0 ? gA[0] : lane == 1 ? gA[1] : gA[2];
  if (lane < 3) atomicAdd(grad + 3 * (int64_t)A + lane, val);
}

// The gradient's kGradCopies partial sums, added in order.
__global__ __launch_bounds__(256) void k_grad_sum(int n, int64_t gstride,
                                                  const double* __restrict__ part,
                                                  double* __restrict__ grad) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  double s = 0.;
#pragma unroll 16
  for (int c = 0; c < kGradCopies; ++c) s += part[c * gstride + i];
  grad[i] = s;
}

// ---- launchers ------------------------------------------------------------------
int launch_grad_points(const CtxView& v, const WorkRange& r, int func, int gga, const double* dp,
                       double* coef, double* wf) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_grad_points, dim3((unsigned)r.n), dim3(64), 0, v.stream, v.work + r.off,
                     v.tasks, v.w, func, gga, dp, v.red, coef, wf);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_grad_points_uks(const CtxView& v, const WorkRange& r, int func, int gga, double* ds,
                           double* dz, double* wf) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_grad_points_uks, dim3((unsigned)r.n), dim3(64), 0, v.stream,
                     v.work + r.off, v.tasks, v.w, func, gga, ds, dz, v.red, wf);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_grad_contract(const CtxView& v, const WorkRange& r, int gga,
                         const int32_t* shell_atom, const double* coef_s, const double* coef_z,
                         int weight_derivs, double* part, int64_t gstride, int x_pl, int y_pl,
                         int lmax) {
  if (r.n == 0) return XCQ_SUCCESS;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)r.n), dim3(256), 0, v.stream, v.work + r.off,
                       v.tasks, v.shells, v.shell_list, v.lsh, shell_atom, v.px, v.py, v.pz,
                       static_cast<const double*>(v.scratch), coef_s, coef_z, weight_derivs,
                       part, gstride, x_pl, y_pl);
  };
  auto pick = [&](auto LM) {
    constexpr int L = decltype(LM)::value;
    if (!coef_z) gga ? go(k_grad_contract<true, L, 1>) : go(k_grad_contract<false, L, 1>);
    else gga ? go(k_grad_contract<true, L, 2>) : go(k_grad_contract<false, L, 2>);
  };
  if (lmax <= 3) pick(std::integral_constant<int, 3>{});
  else pick(std::integral_constant<int, 4>{});
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_ssf_grad(const CtxView& v, const WorkRange& r, int natoms, const double* xyz,
                    const double* dnear, const double* wf, double* part, int64_t gstride,
                    const int32_t* nbr_idx, const double* nbr_i) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(nbr_idx ? k_ssf_grad<true> : k_ssf_grad<false>, dim3((unsigned)r.n),
                     dim3(64), 0, v.stream, v.work + r.off, v.tasks, v.px, v.py, v.pz, natoms,
                     xyz, dnear, wf, part, gstride, nbr_idx, nbr_i);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_grad_sum(hipStream_t s, int natoms, const double* part, int64_t gstride,
                    double* grad) {
  const int n = 3 * natoms;
  hipLaunchKernelGGL(k_grad_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, gstride,
                     part, grad);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

}  // namespace xcq
