// Density stage of the XC path: X = fac B P_sub, rho / grad rho, the
// functional with weight folding, the EXC/NEL block sums and the Z matrix.
//
// One 256-thread workgroup owns one (task, 64-point block) and walks every
// function tile of the task.  Per tile it forms the transposed product
// X^T = fac P_sub B^T (functions x 64 points) on the matrix cores and folds
//   rho_p = sum_j B_pj X_pj,   grad rho_p = 2 sum_j dB_pj X_pj
// (reference_local_host_work_driver.cxx:242-268) into per-point partials.
// After the last tile the block's 64 points are complete.  The sums go to
// memory (32 bytes per point), k_xc_points evaluates the functional
// (host_integrator_exc_vxc.hpp:445-502) and leaves the Z coefficients a = w
// vrho / 2, c = 2 w vsigma grad rho and the block's (w eps rho, w rho) sums,
// and a further launch forms
//   Z = a B + c . grad B        (reference_local_host_work_driver.cxx:678-713).
// X never reaches HBM.
//
// The K loop is software-pipelined, its LDS stages double buffered, one
// barrier per step.  A launch either runs one workgroup per (task, block)
// item or, in queued mode, one persistent workgroup per queue of items.
//
// Basis evaluation mode (template argument INSTAGE): 0 reads B and grad B
// from the planes the collocation stage stored, and so does the Z launch
// (k_z_from_coeffs); 3 and 4 evaluate them (up to that angular momentum) at
// the block's points from the shell parameters, as does k_z_in_stage
// (collocation.hip).  kProductOnly stops at the product, of any stored plane,
// for the EXC gradient.
#include "internal.hpp"
#include "functional.hpp"
#include "shell_eval.hpp"

#include <climits>
#include <type_traits>

namespace xcq {

using v4d = double __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ double bf16_val(unsigned short u) {
  return (double)__builtin_bit_cast(float, (unsigned)u << 16);
}

// Value plane of FP32 storage: FP32 value + bfloat16 residual (plane 5 of
// the task's scratch, 2 bytes per element).  nullptr for FP64 storage.
template <typename T>
__device__ __forceinline__ const unsigned short* lo_plane(const T* Bm, int plane) {
  if constexpr (sizeof(T) == 4)
    return reinterpret_cast<const unsigned short*>(Bm + 5 * (int64_t)plane);
  else
    return nullptr;
}

constexpr int kXLd = 66;  // LDS row stride of the X^T tile in doubles

// Four consecutive elements of a plane (16-byte aligned for FP32, 32 for FP64).
template <typename T>
using Vec4 = T __attribute__((ext_vector_type(4)));

// Z = a B + c . grad B for the block's 64 points, every function row.
// Thread (q = tid & 15, g = tid >> 4) owns points m0 + 4q .. 4q + 3 of rows
// g, g + 16, ...  Each pass loads kZRows rows with 4-wide vector loads
// before any of them is used, so every thread keeps up to 5 kZRows loads in
// flight instead of waiting on each row in turn (4 rows of FP32, 2 of FP64,
// which fit the register budget of the GEMM phase).  Row offsets are clamped
// to a valid row; rows past nbe are not stored.
// Also records, per granule of 32 functions, max |B| and max |Z| over the
// block's points (the FP32 part of B: its residual is covered by syr_mask's
// margin; float bits, so unsigned max orders them): LDS atomics into smax, then
// one device atomic per granule into the task's bound table (direct device
// atomics when the task has more granules than smax holds).  The B^T Z stage
// leaves out a block when npts * (max|B_i| max|Z_j| + max|Z_i| max|B_j|) is below
// the drop tolerance.
template <typename T, bool GGA, int kZRows = sizeof(T) == 4 ? 4 : 2>
__device__ __forceinline__ void write_z(const DevTask& t, int m0, int tid, double (*zc)[64],
                                        T* Bm, unsigned (*smax)[2], unsigned* tmax) {
  const int q = tid & 15, g = tid >> 4;
  const int ld = t.npts_pad, nbe = t.nbe, plane = nbe * ld;
  double a[4], cx[4], cy[4], cz[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    a[e] = zc[0][4 * q + e];
    cx[e] = zc[1][4 * q + e];
    cy[e] = zc[2][4 * q + e];
    cz[e] = zc[3][4 * q + e];
  }
  T* B = Bm + m0 + 4 * q;
  const unsigned short* lo = lo_plane(Bm, plane);
  if constexpr (sizeof(T) == 4) lo += m0 + 4 * q;
  for (int j0 = g; j0 < nbe; j0 += 16 * kZRows) {
    Vec4<T> b[kZRows], x[kZRows], y[kZRows], z[kZRows];
    uint2 l[kZRows];
#pragma unroll
    for (int u = 0; u < kZRows; ++u) {
      const int o = min(j0 + 16 * u, nbe - 1) * ld;
      b[u] = *reinterpret_cast<const Vec4<T>*>(B + o);
      if constexpr (sizeof(T) == 4) l[u] = *reinterpret_cast<const uint2*>(lo + o);
      if constexpr (GGA) {
        x[u] = *reinterpret_cast<const Vec4<T>*>(B + plane + o);
        y[u] = *reinterpret_cast<const Vec4<T>*>(B + 2 * plane + o);
        z[u] = *reinterpret_cast<const Vec4<T>*>(B + 3 * plane + o);
      }
    }
#pragma unroll
    for (int u = 0; u < kZRows; ++u) {
      const int j = j0 + 16 * u;
      if (j >= nbe) break;
      Vec4<T> out;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        double bv = (double)b[u][e];
        if constexpr (sizeof(T) == 4) {
          // bfloat16 residuals of points 2h, 2h + 1 are the low and high
          // halves of word h.
          const unsigned w = e < 2 ? l[u].x : l[u].y;
          bv += (double)__builtin_bit_cast(float, (e & 1) ? (w & 0xffff0000u) : (w << 16));
        }
        double zv = a[e] * bv;
        if constexpr (GGA) zv += cx[e] * (double)x[u][e] + cy[e] * (double)y[u][e] + cz[e] * (double)z[u][e];
        out[e] = (T)zv;
      }
      *reinterpret_cast<Vec4<T>*>(B + 4 * plane + j * ld) = out;
      if (tmax) {
        // A NaN counts as unbounded, so screening never hides it.
        float mb = 0.f, mz = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float fb = fabsf((float)b[u][e]), fz = fabsf((float)out[e]);
          mb = fmaxf(mb, fb != fb ? INFINITY : fb);
          mz = fmaxf(mz, fz != fz ? INFINITY : fz);
        }
        // The 16 lanes of this row (same g) hold its 64 points.
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
          mb = fmaxf(mb, __shfl_xor(mb, off));
          mz = fmaxf(mz, __shfl_xor(mz, off));
        }
        if (q == 0) {
          const int gr = j / kGran;
          if (gr < kGranLds) {
            atomicMax(&smax[gr][0], __float_as_uint(mb));
            atomicMax(&smax[gr][1], __float_as_uint(mz));
          } else {
            atomicMax(tmax + 2 * gr, __float_as_uint(mb));
            atomicMax(tmax + 2 * gr + 1, __float_as_uint(mz));
          }
        }
      }
    }
  }
  if (tmax) {
    __syncthreads();
    const int ng = min((nbe + kGran - 1) / kGran, kGranLds);
    if (tid < 2 * ng) atomicMax(tmax + tid, smax[tid >> 1][tid & 1]);
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// FP64 (v_mfma_f64_16x16x4_f64; accumulator register r of lane l holds row
// 4r + l/16).  Function tiles of up to 64 rows, a task's blocks of 16
// functions divided evenly over them; wave w owns 16 of the block's 64 points
// and every row of the tile, so
//  * rows are multiplied in steps of 16, not of a tile: the tile's number of
//    16-row blocks picks one of four K loops;
//  * a wave whose points all lie past npts skips its products (the point
//    group is rotated by the block index, so that this does not always idle
//    the same SIMD);
//  * the B^T operand, which no other wave needs, comes straight from memory
//    to registers, one K step of 16 ahead; only P_sub is staged in LDS.
// P_sub rows are gathered one K step ahead into registers as well: wave w
// fetches rows 4w .. 4w + 3 of the step, lane = function.  The rows' basis
// functions (64 of them per vector load, a whole chunk ahead) are broadcast
// by readlane, so no scalar load is waited for inside the K loop.
// INSTAGE > 0: the fold evaluates B and grad B itself, from X^T written over
// the stages and from the tile's shells, which were staged in LDS while the
// product ran; 0: it reads the planes the collocation stage stored.
//
// What bounds it: on gfx950 an FP64 MFMA and another wave's vector
// instructions do not overlap (measured: 0.45 ms of the one and 0.64 ms of
// the other take 1.06 ms together), so the products and the fold add up (4.7
// of the first version's 7.9 ms on 24 waters); the rest were chains of
// dependent loads, barriers and the functional on one wave of four, with two
// waves per SIMD to cover them.  The functional is now a launch of its own,
// the shells come from LDS, and four waves fit a SIMD (21 to 24 registers
// spill; three waves without spills: 6.7 ms).  24 waters: 8.9 (64-wide padded
// tiles, 1.4 times the products wanted) -> 6.1 ms; 150 waters: 152 -> 138 ms,
// there bound by L2 misses (890 GB, 6.5 TB/s); 84 functions: 52 -> 28 us.
//
// Mixed precision (T = float): FP32 operands on v_mfma_f32_16x16x4_f32 (lane l
// holds A[l%16][l/16] and B[l/16][l%16]; accumulator register r of lane l is
// row 4(l/16) + r), FP32 accumulation inside one 32-deep K block (eight
// chained MFMAs), FP64 across blocks.  The FP32 matrix cores round to
// nearest on every accumulation; the BF16 ones drop the low bits of the
// smaller products of a dot product, a bias towards zero that compounds into
// the integrated density (measured on gfx950: -0.6 ulp per 32-term BF16 dot
// product of positive terms spanning 20 binades, -0.004 ulp for the FP32
// MFMA on the same data).  The B^T operand is the FP32 part of the value
// plane; its bfloat16 residual enters the fold.  P is gathered from an FP32
// copy; fac (a power of two) scales the accumulated X, which is exact.  Three
// waves per SIMD (24 waters 4.7 ms, 150 waters 90; at four 40 registers
// spill: 4.9 and 96).  The kernel it replaces, with tiles of 32, 64 and 128
// functions padded to, a ring of direct-to-LDS dword loads and the
// functional inside, took 6.6 and 100 ms.
//
// INSTAGE = kProductOnly: X = fac P_sub B, with any stored plane for B, goes to
// plane x_plane (is added to it with accumulate) and nothing else is done (13
// waters: 1.35 ms; on 64-function padded tiles with both operands through LDS
// 2.0).
constexpr int kDensTile = 64;  // functions per tile
constexpr int kProductOnly = -1;

// Shells of one tile (at most one more than its functions, and one for each
// of the four waves' loops to end on), staged in LDS while the tile's
// product runs.
template <int NT>
struct FoldShells {
  static constexpr int kMax = NT + 5;
  double ox[kMax], oy[kMax], oz[kMax], a0[kMax], c0[kMax];
  int bf0[kMax], info[kMax], ish[kMax];
  int next;  // shell holding the function after the tile

  // Stages the shells from s_first on of task t's tile that ends at function
  // nhi (threads 0 .. kMax - 1); the first ones past it end the fold's loops.
  __device__ __forceinline__ void load(const DevTask& t, const ShellArgs& sa, int s_first, int nhi,
                                       int tid) {
    if (tid >= kMax) return;
    const int s = s_first + tid;
    int f0 = INT_MAX, f1 = INT_MAX, i = 0;
    if (s < t.nshells) {
      f0 = sa.lsh[t.lsh_off + s];
      i = sa.shell_list[t.sh_off + s];
      if (s + 1 < t.nshells) f1 = sa.lsh[t.lsh_off + s + 1];
    }
    const DevShellC c = sa.shc[i];
    bf0[tid] = f0;
    ish[tid] = i;
    info[tid] = c.info;
    ox[tid] = c.ox;
    oy[tid] = c.oy;
    oz[tid] = c.oz;
    a0[tid] = c.a0;
    c0[tid] = c.c0;
    if (f0 <= nhi && f1 > nhi) next = s;
  }
};

// Folds rows [nlo, nhi) of the X^T tile in LDS (row n - nlo, column =
// point) into this lane's partials r: rho += B X, grad rho / 2 += grad B X.
// The wave takes the tile's shells first, first + step, ... until one starts
// at or past nhi, leaving out those that end before nlo; lane = point, so a
// shell is wave-uniform; rows of X^T are LD doubles apart.  With B_f = R Y_f and grad
// B_f = R grad Y_f + dR r Y_f, a shell adds R sy to rho and R sg + dR r sy
// to grad rho / 2, where sy = sum Y_f X_f and sg = sum grad Y_f X_f over its
// functions in the range: the functions are formed from their angular
// factors alone.
// RES32: X was formed from the FP32 part B32 of B alone, so rho = B^T 2P B
// misses res^T X (res = B - B32, P symmetric), a first-order term that does
// not average out (it biased EXC by about -3e-10 relative): rho also takes
// sum res X.
template <bool GGA, bool RES32, int LD, int LMAX, int NT>
__device__ __forceinline__ void fold_staged(const ShellArgs& sa, const FoldShells<NT>& fs, int nlo,
                                            int nhi, int first, int step, const double* xt,
                                            double rx, double ry, double rz, double (&r)[4]) {
  for (int j = first;; j += step) {
    const int bf0 = uni(fs.bf0[j]);
    if (bf0 >= nhi) break;
    const int info = uni(fs.info[j]);
    const int l = info & 0xff, nprim = info >> 16;
    const bool pure = (info >> 8) & 1;
    if (NT > 64 && bf0 + (pure ? 2 * l + 1 : (l + 1) * (l + 2) / 2) <= nlo) continue;
    const double x = rx - fs.ox[j], y = ry - fs.oy[j], z = rz - fs.oz[j];
    const double a0 = fs.a0[j];
    const double r2 = x * x + y * y + z * z;
    double R = fs.c0[j] * exp(-a0 * r2), dR = -2. * a0 * R;
    if (nprim > 1) {
      const DevShell* sh = sa.shells + uni(fs.ish[j]);
      for (int k = 1; k < nprim; ++k) {
        const double a = sh->alpha[k], e = sh->coeff[k] * exp(-a * r2);
        R += e;
        dR += -2. * a * e;
      }
    }
    double sy = 0., sgx = 0., sgy = 0., sgz = 0., sres = 0.;
    shell_functions_l<LMAX, GGA, true, true>(
        l, x, y, z, R, dR, pure, [&](int f, double v, double gx, double gy, double gz) {
          const int n = bf0 + f;  // uniform
          if (n >= nlo && n < nhi) {
            const double xv = xt[(n - nlo) * LD];
            sy += v * xv;
            if constexpr (RES32) {
              const double b = R * v;
              sres += (b - (double)(float)b) * xv;
            }
            if constexpr (GGA) {
              sgx += gx * xv;
              sgy += gy * xv;
              sgz += gz * xv;
            }
          }
        });
    r[0] += R * sy;
    if constexpr (RES32) r[0] += sres;
    if constexpr (GGA) {
      const double d = dR * sy;
      r[1] += R * sgx + d * x;
      r[2] += R * sgy + d * y;
      r[3] += R * sgz + d * z;
    }
  }
}

template <typename T, bool GGA, int INSTAGE>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 4) void k_density(
    QueueArgs qa, const DevTask* __restrict__ tasks, const int32_t* __restrict__ bfmap,
    const T* __restrict__ Pall, T* __restrict__ scratch, double fac, ShellArgs sa,
    double* __restrict__ dens_out, int x_plane, int b_plane, int accumulate) {
  constexpr bool kF32 = sizeof(T) == 4;
  constexpr int kBI = kDensTile / 16;
  constexpr int kK = kF32 ? 32 : 16;      // K rows per stage
  constexpr int kKQ = kK / 4;             // MFMA steps, and rows per wave, of a stage
  constexpr int kLd = kDensTile + 16;     // stage row: four K rows hit distinct banks
  constexpr int kStage = kK * kLd;
  constexpr int kXtD = kDensTile * kXLd;  // X^T in doubles
  constexpr bool kFold = INSTAGE != kProductOnly, kEval = INSTAGE > 0;
  static_assert(2 * kStage * sizeof(T) <= kXtD * 8 && 4 * 64 * 4 <= kXtD, "LDS is shared");
  // P_sub stages [buf][k][function]; X^T and the per-point partials take
  // their place.
  __shared__ __attribute__((aligned(16))) double lds[kXtD];
  T* stage = reinterpret_cast<T*>(lds);
  double(*dens)[64][4] = reinterpret_cast<double(*)[64][4]>(lds);
  __shared__ FoldShells<kDensTile> fs;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int lf = lane & 15, lq = lane >> 4;
  auto arow = [&](int r) { return kF32 ? 4 * lq + r : 4 * r + lq; };  // accumulator rows

  XCQ_FOR_EACH_ITEM(qa, it) {
    const int64_t t0 = qa.tstamp ? wall_clock64() : 0;
    const WorkItem wi = qa.items[uniform64(it)];
    const DevTask t = tasks[wi.task];
    const int m0 = wi.a * kPtBlock;
    const int ld = t.npts_pad;
    const int nbe = t.nbe;
    const int plane = nbe * ld;
    const int64_t ldp = t.ldp;
    const T* P = Pall + t.p_off;
    T* Bm = scratch + (kF32 ? t.b_off_mx : t.b_off);
    const int32_t* bf = bfmap + t.bf_off;
    const int pg = (wave + wi.a) & 3;           // the wave's 16 points of the block
    const int pcol = m0 + 16 * pg + lf;         // this lane's point (column)
    const bool active = m0 + 16 * pg < t.npts;  // the wave has points
    const int nks = (nbe + kK - 1) / kK, nblk = (nbe + 15) / 16;
    // In-stage fold: lane = point (padded points take the task's last point:
    // finite values, which meet zero X) and this wave's density partials; on
    // stored planes the partials of the lane's column.
    double rx = 0., ry = 0., rz = 0.;
    if constexpr (kEval) {
      const int pl = min(m0 + lane, t.npts - 1);
      rx = sa.px[t.pt_off + pl];
      ry = sa.py[t.pt_off + pl];
      rz = sa.pz[t.pt_off + pl];
    }
    int s_cur = 0;
    double part[4] = {0., 0., 0., 0.};
    const auto rsB = __builtin_amdgcn_make_buffer_rsrc(
        Bm + (kFold ? 0 : (int64_t)b_plane * plane), 0, (int)((unsigned)plane * (unsigned)sizeof(T)), 0x00020000);
    auto ldB = [&](int vo, int so) -> T {  // element offsets: lane, scalar
      if constexpr (kF32)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rsB, vo * 4, so * 4, 0));
      else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rsB, vo * 8, so * 8, 0));
    };

    // Tiles of 16-row blocks [blk, blk + nbk).
    const int ntile = (nblk + kBI - 1) / kBI;
    for (int tile = 0; tile < ntile; ++tile) {
      const int blk = tile * nblk / ntile, nbk = (tile + 1) * nblk / ntile - blk;
      const int n0 = 16 * blk, nhi = min(n0 + 16 * nbk, nbe);
      // P is symmetric: P(n, k) is read as row bf[k], column bf[n], so that
      // neighbouring lanes touch neighbouring elements.  Rows of the tile
      // past nbe repeat the last function; their X is not used.
      const unsigned cn = (unsigned)sizeof(T) * (unsigned)bf[min(n0 + lane, nbe - 1)];
      int vrow = bf[min(lane, nbe - 1)];  // functions of the current 64 K rows
      int vnext = bf[min(64 + lane, nbe - 1)];
      T rp[kKQ], rb[kKQ];
      auto load = [&](int s) {
        if (s > 0 && s % (64 / kK) == 0) {
          vrow = vnext;
          vnext = bf[min(kK * s + 64 + lane, nbe - 1)];
        }
#pragma unroll
        for (int e = 0; e < kKQ; ++e) {
          const int row = __builtin_amdgcn_readlane(vrow, (kK * s + kKQ * wave + e) & 63);
          rp[e] = *reinterpret_cast<const T*>(
              reinterpret_cast<const char*>(P + (int64_t)row * ldp) + cn);
        }
        if (kK * (s + 1) <= nbe) {
#pragma unroll
          for (int ks = 0; ks < kKQ; ++ks) rb[ks] = ldB(lq * ld + pcol, (kK * s + 4 * ks) * ld);
        } else {
#pragma unroll
          for (int ks = 0; ks < kKQ; ++ks)
            rb[ks] = ldB(min(kK * s + 4 * ks + lq, nbe - 1) * ld + pcol, 0);
        }
      };
      load(0);
      if constexpr (kEval) {
        fs.load(t, sa, s_cur, nhi, tid);
      }
      v4d acc[kBI];
#pragma unroll
      for (int i = 0; i < kBI; ++i) acc[i] = v4d{0., 0., 0., 0.};
      auto contract = [&](auto NB) {
        constexpr int BI = decltype(NB)::value;
        for (int s = 0; s < nks; ++s) {
          T* st = stage + (s & 1) * kStage;
          T b[kKQ];
#pragma unroll
          for (int e = 0; e < kKQ; ++e) {
            // P rows past nbe are zero, B rows past it repeat the last one.
            const bool kok = kK * s + kKQ * wave + e < nbe;
            st[(kKQ * wave + e) * kLd + lane] = kok ? rp[e] : T(0);
            b[e] = rb[e];
          }
          __syncthreads();
          if (s + 1 < nks) load(s + 1);
          if (active) {
            v4f c[BI];
            if constexpr (kF32) {
#pragma unroll
              for (int i = 0; i < BI; ++i) c[i] = v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int ks = 0; ks < kKQ; ++ks) {
              T a[BI];
#pragma unroll
              for (int i = 0; i < BI; ++i) a[i] = st[(4 * ks + lq) * kLd + 16 * i + lf];
#pragma unroll
              for (int i = 0; i < BI; ++i) {
                if constexpr (kF32)
                  c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[ks], c[i], 0, 0, 0);
                else
                  acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[ks], acc[i], 0, 0, 0);
              }
            }
            if constexpr (kF32) {
#pragma unroll
              for (int i = 0; i < BI; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][r] += (double)c[i][r];
            }
          }
        }
      };
      switch (nbk) {
        case 1: contract(std::integral_constant<int, 1>{}); break;
        case 2: contract(std::integral_constant<int, 2>{}); break;
        case 3: contract(std::integral_constant<int, 3>{}); break;
        default: contract(std::integral_constant<int, 4>{}); break;
      }
#pragma unroll
      for (int i = 0; i < kBI; ++i) acc[i] *= fac;  // 1 or 2: exact
      if (x_plane >= 0) {
        // The X tile itself into plane x_plane (row = function, column =
        // point), for callers that contract it again (the EXC gradient).
        T* xo = Bm + (int64_t)x_plane * plane + pcol;
#pragma unroll
        for (int i = 0; i < kBI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = n0 + 16 * i + arow(r);
            if (row < nhi) {
              T* o = xo + (int64_t)row * ld;
              *o = !kFold && accumulate ? (T)(*o + acc[i][r]) : (T)acc[i][r];
            }
          }
      }
      if constexpr (kEval) {
        __syncthreads();  // every wave is done with the stages
#pragma unroll
        for (int i = 0; i < kBI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lds[(16 * i + arow(r)) * kXLd + 16 * pg + lf] = acc[i][r];
        __syncthreads();
        fold_staged<GGA, kF32, kXLd, INSTAGE>(sa, fs, n0, nhi, wave, 4, lds + lane, rx, ry, rz, part);
        s_cur = uni(fs.next);
      } else if constexpr (kFold) {
        const unsigned short* lo = lo_plane(Bm, plane);
#pragma unroll
        for (int i = 0; i < kBI; ++i) {
          if (16 * i >= nhi - n0) break;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = n0 + 16 * i + arow(r), o = min(j, nbe - 1) * ld + pcol;
            const double xv = j < nhi ? acc[i][r] : 0.;
            double b = (double)Bm[o];
            if constexpr (kF32) b += 2.0 * bf16_val(lo[o]);  // B32 + 2 res (see fold_staged)
            part[0] += b * xv;
            if constexpr (GGA) {
              part[1] += (double)Bm[plane + o] * xv;
              part[2] += (double)Bm[2 * plane + o] * xv;
              part[3] += (double)Bm[3 * plane + o] * xv;
            }
          }
        }
      }
      __syncthreads();  // the next tile's first stage write is safe
    }
    if constexpr (!kFold) continue;
    constexpr int ND = kEval ? 4 : 1;
    if constexpr (kEval) {
#pragma unroll
      for (int c = 0; c < 4; ++c) dens[wave][lane][c] = part[c];
    } else {
      // Sum over the four 16-lane groups (different functions, same point).
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        part[c] += __shfl_xor(part[c], 16);
        part[c] += __shfl_xor(part[c], 32);
        if (lane < 16) dens[0][16 * pg + lf][c] = part[c];
      }
    }
    __syncthreads();
    // The block's raw sums (sum B X, sum dB/dx X, ...) per point,
    // [block][4][64].
    if (tid < 64) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        double v = 0.;
#pragma unroll
        for (int d = 0; d < ND; ++d) v += dens[d][tid][c];
        dens_out[(t.red_off + wi.a) * 256 + c * 64 + tid] = v;
      }
    }
    stamp_item(qa, it, t0);
    __syncthreads();
  }
}

// The same in FP64 for tasks of many functions of large molecules: one
// workgroup per (task, pair of 64-point blocks), tiles of up to 128
// functions, each wave 32 points and every row of the tile.  On 150 waters
// the kernel above is bound by L2 misses (890 GB, 6.5 TB/s): P_sub of a task
// (2 MB and more) and the blocks' B panels do not stay in L2, P_sub is
// gathered once per point block and B read once per tile.  Twice the points
// and twice the functions per workgroup halve both, at two waves per SIMD
// (128 accumulator registers; 29 to 35 spill).  Density stage: 150 waters 137 -> 117 ms, 90
// waters 33.3 -> 30.0, 60 waters 18.6 -> 18.0, 40 waters 8.8 -> 9.1, 24 waters
// 6.1 -> 6.8; mixed precision (64-function tiles, half the bytes) lost at
// every size (150 waters 88 -> 95).  Lane (f, q) holds the adjacent points 2f,
// 2f + 1 of its wave's 32: one 16-byte load of B serves two MFMA columns.
template <bool GGA, int LMAX>
__global__ __launch_bounds__(256, 2) void k_density_wide(
    QueueArgs qa, const DevTask* __restrict__ tasks, const int32_t* __restrict__ bfmap,
    const double* __restrict__ Pall, double* __restrict__ scratch, double fac, ShellArgs sa,
    double* __restrict__ dens_out, int x_plane) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int NT = 128;
  constexpr int kBI = NT / 16;
  constexpr int kK = 16;
  constexpr int kKQ = kK / 4;
  constexpr int kLd = NT + 16;
  constexpr int kStage = kK * kLd;
  constexpr int kXL = 2 * kPtBlock + 2;  // X^T row (128 points) in doubles
  constexpr int kXtD = 64 * kXL;         // 64 rows at a time
  static_assert(2 * kStage <= kXtD, "LDS is shared");
  __shared__ __attribute__((aligned(16))) double lds[kXtD];
  double* stage = lds;
  double(*dens)[128][4] = reinterpret_cast<double(*)[128][4]>(lds);
  __shared__ FoldShells<NT> fs;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int lf = lane & 15, lq = lane >> 4;

  XCQ_FOR_EACH_ITEM(qa, it) {
    const int64_t t0 = qa.tstamp ? wall_clock64() : 0;
    const WorkItem wi = qa.items[uniform64(it)];
    const DevTask t = tasks[wi.task];
    const int m0 = 2 * wi.a * kPtBlock;
    const int ld = t.npts_pad;
    const int nbe = t.nbe;
    const int plane = nbe * ld;
    const int64_t ldp = t.ldp;
    const double* P = Pall + t.p_off;
    double* Bm = scratch + t.b_off;
    const int32_t* bf = bfmap + t.bf_off;
    const int pg = (wave + wi.a) & 3;           // the wave's 32 points of the pair
    const int pcol = m0 + 32 * pg + 2 * lf;     // this lane's first point (column)
    const bool active = m0 + 32 * pg < t.npts;  // the wave has points
    const int nks = (nbe + kK - 1) / kK, nblk = (nbe + 15) / 16;
    // Fold: waves 0, 2 take the first 64 points, waves 1, 3 the others.
    const int ph = wave & 1;
    const int pl = min(m0 + kPtBlock * ph + lane, t.npts - 1);
    const double rx = sa.px[t.pt_off + pl], ry = sa.py[t.pt_off + pl], rz = sa.pz[t.pt_off + pl];
    int s_cur = 0;
    double part[4] = {0., 0., 0., 0.};
    const auto rsB = __builtin_amdgcn_make_buffer_rsrc(
        Bm, 0, (int)((unsigned)plane * 8u), 0x00020000);
    auto ldB = [&](int vo, int so) {  // element offsets: lane, scalar
      return __builtin_bit_cast(v2d,
                                __builtin_amdgcn_raw_buffer_load_b128(rsB, vo * 8, so * 8, 0));
    };

    const int ntile = (nblk + kBI - 1) / kBI;
    for (int tile = 0; tile < ntile; ++tile) {
      const int blk = tile * nblk / ntile, nbk = (tile + 1) * nblk / ntile - blk;
      const int n0 = 16 * blk, nhi = min(n0 + 16 * nbk, nbe);
      const unsigned c0 = 8u * (unsigned)bf[min(n0 + lane, nbe - 1)];
      const unsigned c1 = 8u * (unsigned)bf[min(n0 + 64 + lane, nbe - 1)];
      int vrow = bf[min(lane, nbe - 1)];
      int vnext = bf[min(64 + lane, nbe - 1)];
      double rp[kKQ][2];
      v2d rb[kKQ];
#pragma unroll
      for (int ks = 0; ks < kKQ; ++ks) rb[ks] = v2d{0., 0.};
      auto load = [&](int s) {
        if (s > 0 && s % (64 / kK) == 0) {
          vrow = vnext;
          vnext = bf[min(kK * s + 64 + lane, nbe - 1)];
        }
#pragma unroll
        for (int e = 0; e < kKQ; ++e) {
          const int row = __builtin_amdgcn_readlane(vrow, (kK * s + kKQ * wave + e) & 63);
          const char* Pr = reinterpret_cast<const char*>(P + (int64_t)row * ldp);
          rp[e][0] = *reinterpret_cast<const double*>(Pr + c0);
          rp[e][1] = *reinterpret_cast<const double*>(Pr + c1);
        }
      };
      // Row block ks of the B rows of step s.
      auto loadB = [&](int s, int ks) {
        if (!active) return;
        if (kK * (s + 1) <= nbe) rb[ks] = ldB(lq * ld + pcol, (kK * s + 4 * ks) * ld);
        else rb[ks] = ldB(min(kK * s + 4 * ks + lq, nbe - 1) * ld + pcol, 0);
      };
      load(0);
#pragma unroll
      for (int ks = 0; ks < kKQ; ++ks) loadB(0, ks);
      fs.load(t, sa, s_cur, nhi, tid);
      v4d acc[kBI][2];
#pragma unroll
      for (int i = 0; i < kBI; ++i) acc[i][0] = acc[i][1] = v4d{0., 0., 0., 0.};
      auto contract = [&](auto NB) {
        constexpr int BI = decltype(NB)::value;
        for (int s = 0; s < nks; ++s) {
          double* st = stage + (s & 1) * kStage;
#pragma unroll
          for (int e = 0; e < kKQ; ++e) {
            // P rows past nbe are zero, B rows past it repeat the last one.
            const bool kok = kK * s + kKQ * wave + e < nbe;
            st[(kKQ * wave + e) * kLd + lane] = kok ? rp[e][0] : 0.;
            st[(kKQ * wave + e) * kLd + 64 + lane] = kok ? rp[e][1] : 0.;
          }
          __syncthreads();
          const bool more = s + 1 < nks;
          if (more) load(s + 1);
          if (active) {
#pragma unroll
            for (int ks = 0; ks < kKQ; ++ks) {
              double a[BI];
#pragma unroll
              for (int i = 0; i < BI; ++i) a[i] = st[(4 * ks + lq) * kLd + 16 * i + lf];
#pragma unroll
              for (int i = 0; i < BI; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                  acc[i][j] =
                      __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], rb[ks][j], acc[i][j], 0, 0, 0);
              if (more) loadB(s + 1, ks);
            }
          }
        }
      };
      // Tasks of this kernel have at least five blocks, so a tile has four.
      switch (nbk) {
        case 4: contract(std::integral_constant<int, 4>{}); break;
        case 5: contract(std::integral_constant<int, 5>{}); break;
        case 6: contract(std::integral_constant<int, 6>{}); break;
        case 7: contract(std::integral_constant<int, 7>{}); break;
        default: contract(std::integral_constant<int, 8>{}); break;
      }
#pragma unroll
      for (int i = 0; i < kBI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] *= fac;  // 1 or 2: exact
      if (x_plane >= 0 && active) {
        double* xo = Bm + (int64_t)x_plane * plane + pcol;
#pragma unroll
        for (int i = 0; i < kBI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = n0 + 16 * i + 4 * r + lq;
            if (row < nhi)
              *reinterpret_cast<v2d*>(xo + (int64_t)row * ld) = v2d{acc[i][0][r], acc[i][1][r]};
          }
      }
#pragma unroll
      for (int h = 0; h < NT / 64; ++h) {
        if (64 * h >= nhi - n0) break;
        __syncthreads();  // every wave is done with the stages (or the last rows)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            *reinterpret_cast<v2d*>(lds + (16 * i + 4 * r + lq) * kXL + 32 * pg + 2 * lf) =
                v2d{acc[4 * h + i][0][r], acc[4 * h + i][1][r]};
        __syncthreads();
        fold_staged<GGA, false, kXL, LMAX>(sa, fs, n0 + 64 * h, min(n0 + 64 * h + 64, nhi), wave >> 1, 2,
                                    lds + kPtBlock * ph + lane, rx, ry, rz, part);
      }
      s_cur = uni(fs.next);
      __syncthreads();  // the next tile's first stage write is safe
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) dens[wave >> 1][kPtBlock * ph + lane][c] = part[c];
    __syncthreads();
    if (tid < 128 && m0 + (tid & 64) < ld) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dens_out[(t.red_off + 2 * wi.a + (tid >> 6)) * 256 + c * 64 + (tid & 63)] =
            dens[0][tid][c] + dens[1][tid][c];
    }
    stamp_item(qa, it, t0);
    __syncthreads();
  }
}

// Functional from the density stage's raw sums, one wave
// per point block: the Z coefficients over the sums and the block's (EXC,
// NEL) partials.  A launch of its own: inside the density kernel it ran on
// one wave of four, for 3 of a workgroup's 50 us, and its registers alone
// kept that kernel at two waves per SIMD.
__global__ __launch_bounds__(64) void k_xc_points(const WorkItem* __restrict__ items,
                                                  const DevTask* __restrict__ tasks,
                                                  const double* __restrict__ weights, int func,
                                                  int gga, double* __restrict__ sums,
                                                  double* __restrict__ red) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  double* s = sums + (t.red_off + wi.a) * 256 + tid;
  const int p = wi.a * kPtBlock + tid;
  const double rho = s[0];
  const double gx = 2.0 * s[64], gy = 2.0 * s[128], gz = 2.0 * s[192];
  double e = 0., n = 0., za = 0., c = 0.;
  if (p < t.npts) {
    const double w = weights[t.pt_off + p];
    n = w * rho;
    if (func != 0) {
      const XCOut o =
          dev_eval_functional(func, rho, gga ? gx * gx + gy * gy + gz * gz : 0.);
      e = w * o.e;
      za = 0.5 * w * o.vr;
      c = gga ? 2.0 * w * o.vs : 0.;
    }
  }
  s[0] = za;
  s[64] = c * gx;
  s[128] = c * gy;
  s[192] = c * gz;
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * (t.red_off + wi.a)] = e;
    red[2 * (t.red_off + wi.a) + 1] = n;
  }
}

// ---------------------------------------------------------------------------
// UKS tail (GauXC's generic host driver with spin_dim 2,
// reference_replicated_xc_host_integrator_exc_vxc.hpp:387-547, and the
// device UKS kernels it mirrors, cuda/kernels/zmat_vxc.cu:62-96,197-274).
// Inputs per point block: the raw sums of the P_s and P_z density passes
// (sum B X, sum dB X; X = B P with factor 1).  One thread per point:
//   rho_+- = (rho_s +- rho_z) / 2, grad n = 2 sum dB X_s, grad m = 2 sum dB X_z,
//   sigma_{aa, ab, bb} = (|gn|^2 + |gm|^2)/4 +- gn.gm/2, (|gn|^2 - |gm|^2)/4
//   (eval_uvvar_gga_uks, reference_local_host_work_driver.cxx:270-330);
// the polarised functional; weight folding; the block's (w n eps, w n) sums;
// and the Z coefficients of eval_zmat_{lda,gga}_vxc_uks (:607-632, 715-770):
//   Z_s = (v_a + v_b)/4 B + c_s . grad B,  Z_z = (v_a - v_b)/4 B + c_z . grad B,
//   c_s = g1 gn + g2 gm, c_z = g3 gm + g2 gn, with g1 = (v_aa + v_ab + v_bb)/2,
//   g2 = (v_aa - v_bb)/2, g3 = (v_aa - v_ab + v_bb)/2 (weights folded in).
__global__ __launch_bounds__(64) void k_uks_points(const WorkItem* __restrict__ items,
                                                   const DevTask* __restrict__ tasks,
                                                   const double* __restrict__ weights, int func,
                                                   int gga, const double* __restrict__ ds,
                                                   const double* __restrict__ dz,
                                                   double* __restrict__ red,
                                                   double* __restrict__ zs,
                                                   double* __restrict__ zz) {
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
    n = w * (ra + rb);
    if (func != 0) {
      const double saa = gga ? 0.25 * (nn + mm) + 0.5 * nm : 0.;
      const double sab = gga ? 0.25 * (nn - mm) : 0.;
      const double sbb = gga ? 0.25 * (nn + mm) - 0.5 * nm : 0.;
      const XCOutPol o = dev_eval_functional_pol(func, ra, rb, saa, sab, sbb);
      e = w * o.e;
      const double fp = 0.5 * w * o.vra, fm = 0.5 * w * o.vrb;
      as = 0.5 * (fp + fm);
      az = 0.5 * (fp - fm);
      if (gga) {
        const double vpp = w * o.vsaa, vpm = w * o.vsab, vmm = w * o.vsbb;
        const double g1 = 0.5 * (vpp + vpm + vmm), g2 = 0.5 * (vpp - vmm),
                     g3 = 0.5 * (vpp - vpm + vmm);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          cs[d] = g1 * gn[d] + g2 * gm[d];
          cz[d] = g3 * gm[d] + g2 * gn[d];
        }
      }
    }
  }
  zs[b * 256 + tid] = as;
  zz[b * 256 + tid] = az;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    zs[b * 256 + (1 + d) * 64 + tid] = cs[d];
    zz[b * 256 + (1 + d) * 64 + tid] = cz[d];
  }
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * b] = e;
    red[2 * b + 1] = n;
  }
}

// ---------------------------------------------------------------------------
// FXC contraction tail, RKS (reference_replicated_xc_host_integrator_
// fxc_contraction.hpp:393-560 with spin_dim 1).  Inputs per point block: the
// raw sums of the P and trial-density passes with factor 2 (rho = sum B X,
// grad rho = 2 sum dB X; likewise trho, grad trho).  One thread per point:
//   tgamma = grad rho . grad trho,
//   A = v2rho2 trho + 2 v2rhogamma tgamma,
//   B = 2 (v2rhogamma trho + 2 v2gamma2 tgamma) grad rho + 2 vgamma grad trho
// (eval_tmat_{lda,gga}_vxc_rks, reference_local_host_work_driver.cxx:
// 1114-1143), weights folded in, and the Z coefficients of
// eval_zmat_gga_vxc_rks_ts (:1382-1408): a = A / 2, c = B.  The block's
// (w rho eps, w rho) sums of the ground-state density go to red.
__global__ __launch_bounds__(64) void k_fxc_points(const WorkItem* __restrict__ items,
                                                   const DevTask* __restrict__ tasks,
                                                   const double* __restrict__ weights, int func,
                                                   int gga, const double* __restrict__ dp,
                                                   const double* __restrict__ dt,
                                                   double* __restrict__ red,
                                                   double* __restrict__ zc) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  const int64_t b = t.red_off + wi.a;
  const int p = wi.a * kPtBlock + tid;
  double sv[4], tv[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    sv[c] = dp[b * 256 + c * 64 + tid];
    tv[c] = dt[b * 256 + c * 64 + tid];
  }
  double g[3], tg[3], sig = 0., tgam = 0.;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    g[d] = 2.0 * sv[1 + d];
    tg[d] = 2.0 * tv[1 + d];
    sig += g[d] * g[d];
    tgam += g[d] * tg[d];
  }
  double e = 0., n = 0., a = 0., cv[3] = {0., 0., 0.};
  if (p < t.npts) {
    const double w = weights[t.pt_off + p];
    n = w * sv[0];
    const XCOut o = dev_eval_functional(func, sv[0], sig);
    e = w * o.e;
    double vs, A, Bc;
    dev_fxc_point(func, sv[0], sig, tv[0], 2.0 * tgam, vs, A, Bc);
    a = 0.5 * w * A;
    if (gga) {
#pragma unroll
      for (int d = 0; d < 3; ++d) cv[d] = w * (2.0 * Bc * g[d] + 2.0 * vs * tg[d]);
    }
  }
  zc[b * 256 + tid] = a;
#pragma unroll
  for (int d = 0; d < 3; ++d) zc[b * 256 + (1 + d) * 64 + tid] = cv[d];
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * b] = e;
    red[2 * b + 1] = n;
  }
}

// UKS FXC contraction tail (reference_replicated_xc_host_integrator_
// fxc_contraction.hpp:94-600 with spin_dim 2; the trial kernels
// eval_tmat_{lda,gga}_vxc_uks and eval_zmat_*_uks_ts,
// reference_local_host_work_driver.cxx:1118-1124, 1149-1215, 1354-1367,
// 1441-1481).  FXC_s and FXC_z are the derivatives of VXC_s and VXC_z along
// the trial density, so this kernel writes the derivatives of k_uks_points'
// Z coefficients along (tP_s, tP_z): inputs are the raw sums of the four
// density passes (P_s, P_z, tP_s, tP_z; factor 1), the second derivatives
// come from dev_fxc_point_pol.  Padded points give zero coefficients.
__global__ __launch_bounds__(64) void k_fxc_points_uks(
    const WorkItem* __restrict__ items, const DevTask* __restrict__ tasks,
    const double* __restrict__ weights, int func, int gga, const double* __restrict__ ds,
    const double* __restrict__ dz, const double* __restrict__ dts,
    const double* __restrict__ dtz, double* __restrict__ red, double* __restrict__ zs,
    double* __restrict__ zz) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  const int64_t b = t.red_off + wi.a;
  const int p = wi.a * kPtBlock + tid;
  double sv[4], zv[4], tsv[4], tzv[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    sv[c] = ds[b * 256 + c * 64 + tid];
    zv[c] = dz[b * 256 + c * 64 + tid];
    tsv[c] = dts[b * 256 + c * 64 + tid];
    tzv[c] = dtz[b * 256 + c * 64 + tid];
  }
  double gn[3], gm[3], tgn[3], tgm[3];
  double nn = 0., mm = 0., nm = 0., dnn = 0., dmm = 0., dnm = 0.;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    gn[d] = 2.0 * sv[1 + d];
    gm[d] = 2.0 * zv[1 + d];
    tgn[d] = 2.0 * tsv[1 + d];
    tgm[d] = 2.0 * tzv[1 + d];
    nn += gn[d] * gn[d];
    mm += gm[d] * gm[d];
    nm += gn[d] * gm[d];
    dnn += 2.0 * gn[d] * tgn[d];
    dmm += 2.0 * gm[d] * tgm[d];
    dnm += tgn[d] * gm[d] + gn[d] * tgm[d];
  }
  double e = 0., n = 0., das = 0., daz = 0., dcs[3] = {0., 0., 0.}, dcz[3] = {0., 0., 0.};
  if (p < t.npts) {
    const double w = weights[t.pt_off + p];
    double x[5] = {fmax(0.5 * (sv[0] + zv[0]), 0.0), fmax(0.5 * (sv[0] - zv[0]), 0.0), 0., 0.,
                   0.};
    double dx[5] = {0.5 * (tsv[0] + tzv[0]), 0.5 * (tsv[0] - tzv[0]), 0., 0., 0.};
    if (gga) {
      const double stol2 = 2.1544346900318838e-43 * 2.1544346900318838e-43;
      x[2] = fmax(0.25 * (nn + mm) + 0.5 * nm, stol2);
      x[4] = fmax(0.25 * (nn + mm) - 0.5 * nm, stol2);
      const double hs = 0.5 * (x[2] + x[4]);
      x[3] = fmax(fmin(0.25 * (nn - mm), hs), -hs);
      dx[2] = 0.25 * (dnn + dmm) + 0.5 * dnm;
      dx[3] = 0.25 * (dnn - dmm);
      dx[4] = 0.25 * (dnn + dmm) - 0.5 * dnm;
    }
    n = w * sv[0];
    const XCOutPol o = dev_eval_functional_pol(func, x[0], x[1], x[2], x[3], x[4]);
    e = w * o.e;
    double out[10];
    dev_fxc_point_pol(func, x, dx, out);
    das = 0.25 * w * (out[5] + out[6]);
    daz = 0.25 * w * (out[5] - out[6]);
    if (gga) {
      const double g1 = 0.5 * w * (out[2] + out[3] + out[4]), g2 = 0.5 * w * (out[2] - out[4]),
                   g3 = 0.5 * w * (out[2] - out[3] + out[4]);
      const double dg1 = 0.5 * w * (out[7] + out[8] + out[9]), dg2 = 0.5 * w * (out[7] - out[9]),
                   dg3 = 0.5 * w * (out[7] - out[8] + out[9]);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        dcs[d] = dg1 * gn[d] + g1 * tgn[d] + dg2 * gm[d] + g2 * tgm[d];
        dcz[d] = dg3 * gm[d] + g3 * tgm[d] + dg2 * gn[d] + g2 * tgn[d];
      }
    }
  }
  zs[b * 256 + tid] = das;
  zz[b * 256 + tid] = daz;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    zs[b * 256 + (1 + d) * 64 + tid] = dcs[d];
    zz[b * 256 + (1 + d) * 64 + tid] = dcz[d];
  }
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    n += __shfl_xor(n, off);
  }
  if (tid == 0) {
    red[2 * b] = e;
    red[2 * b + 1] = n;
  }
}

// Z = a B + c . grad B of one point block from stored coefficients
// ([block][4][64]) and the stored planes, with the screening bounds when tmax
// is given.
template <typename T, bool GGA>
__global__ __launch_bounds__(256) void k_z_from_coeffs(const WorkItem* __restrict__ items,
                                                       const DevTask* __restrict__ tasks,
                                                       T* __restrict__ scratch,
                                                       const double* __restrict__ coef,
                                                       unsigned* __restrict__ tmax) {
  __shared__ double zc[4][64];
  __shared__ unsigned smax[kGranLds][2];
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x;
  (&zc[0][0])[tid] = coef[(t.red_off + wi.a) * 256 + tid];
  if (tid < 2 * kGranLds) (&smax[0][0])[tid] = 0u;
  __syncthreads();
  write_z<T, GGA>(t, wi.a * kPtBlock, tid, zc,
                  scratch + (sizeof(T) == 4 ? t.b_off_mx : t.b_off), smax,
                  tmax ? tmax + 2 * t.tmax_off : nullptr);
}

int launch_uks_points(const CtxView& v, const WorkRange& r, int func, int gga, const double* ds,
                      const double* dz, double* zs, double* zz) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_uks_points, dim3((unsigned)r.n), dim3(64), 0, v.stream, v.work + r.off,
                     v.tasks, v.w, func, gga, ds, dz, v.red, zs, zz);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_fxc_points(const CtxView& v, const WorkRange& r, int func, int gga, const double* dp,
                      const double* dt, double* zc) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_fxc_points, dim3((unsigned)r.n), dim3(64), 0, v.stream, v.work + r.off,
                     v.tasks, v.w, func, gga, dp, dt, v.red, zc);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_fxc_points_uks(const CtxView& v, const WorkRange& r, int func, int gga,
                          const double* ds, const double* dz, const double* dts,
                          const double* dtz, double* zs, double* zz) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_fxc_points_uks, dim3((unsigned)r.n), dim3(64), 0, v.stream,
                     v.work + r.off, v.tasks, v.w, func, gga, ds, dz, dts, dtz, v.red, zs, zz);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_z_from_coeffs(const CtxView& v, const WorkRange& r, int precision, int gga,
                         const double* coef, unsigned* tmax) {
  if (r.n == 0) return XCQ_SUCCESS;
  auto go = [&](auto kern, auto* scr) {
    hipLaunchKernelGGL(kern, dim3((unsigned)r.n), dim3(256), 0, v.stream, v.work + r.off, v.tasks,
                       scr, coef, tmax);
  };
  if (precision == XCQ_PREC_FP64) {
    auto* scr = static_cast<double*>(v.scratch);
    gga ? go(k_z_from_coeffs<double, true>, scr) : go(k_z_from_coeffs<double, false>, scr);
  } else {
    auto* scr = static_cast<float*>(v.scratch);
    gga ? go(k_z_from_coeffs<float, true>, scr) : go(k_z_from_coeffs<float, false>, scr);
  }
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_xc_points(const CtxView& v, const WorkRange& r, int func, int gga, double* sums) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_xc_points, dim3((unsigned)r.n), dim3(64), 0, v.stream, v.work + r.off,
                     v.tasks, v.w, func, gga, sums, v.red);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_density(const CtxView& v, const Chunk& c, int precision, int gga, double fac,
                   double* dens_out, const double* P_override, int x_plane) {
  XCQ_REQUIRE(x_plane < 5, XCQ_ERROR_INVALID_ARGUMENT, "the scratch has five planes");
  const ShellArgs sa{v.shells, v.shc, v.shell_list, v.lsh, v.px, v.py, v.pz};
  auto go = [&](auto kern, const WorkRange& r, const auto* P, auto* scr) {
    if (r.n)
      hipLaunchKernelGGL(kern, dim3(grid_of(r)), dim3(256), 0, v.stream, queue_args(v, r), v.tasks,
                         v.bfmap, P, scr, fac, sa, dens_out, x_plane, 0, 0);
  };
  auto go_wide = [&](auto kern, const auto* P, auto* scr) {
    if (c.dens_pair.n)
      hipLaunchKernelGGL(kern, dim3(grid_of(c.dens_pair)), dim3(256), 0, v.stream,
                         queue_args(v, c.dens_pair), v.tasks, v.bfmap, P, scr, fac, sa, dens_out,
                         x_plane);
  };
  // The blocks of all tasks, or without the wide ones: one launch, but for
  // queues, which each list has of its own.
  auto run = [&](auto kern, const auto* P, auto* scr, bool all) {
    if (c.dens[0].nq || c.dens[1].nq) {
      if (all) go(kern, c.dens[1], P, scr);
      go(kern, c.dens[0], P, scr);
    } else {
      go(kern, all ? c.coll : c.dens[0], P, scr);
    }
  };
  // In-stage, FP64 runs the wide tasks as pairs.
  auto pick = [&](const auto* P, auto* scr) {
    using T = std::remove_pointer_t<decltype(scr)>;
    if (v.in_stage == 0) {
      gga ? run(k_density<T, true, 0>, P, scr, true) : run(k_density<T, false, 0>, P, scr, true);
      return;
    }
    auto eval = [&](auto L) {
      constexpr int l = decltype(L)::value;
      if constexpr (sizeof(T) == 8)
        gga ? go_wide(k_density_wide<true, l>, P, scr) : go_wide(k_density_wide<false, l>, P, scr);
      constexpr bool all = sizeof(T) == 4;
      gga ? run(k_density<T, true, l>, P, scr, all) : run(k_density<T, false, l>, P, scr, all);
    };
    // Mixed precision evaluates up to f functions (effective_mode).
    if (sizeof(T) == 4 || v.max_l <= 3) eval(std::integral_constant<int, 3>{});
    else if constexpr (sizeof(T) == 8) eval(std::integral_constant<int, 4>{});
  };
  if (precision == XCQ_PREC_FP64)
    pick(P_override ? P_override : v.P, static_cast<double*>(v.scratch));
  else
    pick(v.Pf32, static_cast<float*>(v.scratch));
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_plane_product(const CtxView& v, const WorkRange& r, int in_pl, int out_pl,
                         const double* P, double fac, int accumulate) {
  if (r.n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL((k_density<double, false, kProductOnly>), dim3((unsigned)r.n), dim3(256), 0,
                     v.stream, queue_args(v, r), v.tasks, v.bfmap, P ? P : v.P,
                     static_cast<double*>(v.scratch), fac, ShellArgs{}, nullptr, out_pl, in_pl,
                     accumulate);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

}  // namespace xcq
