// FP64 contractions of the XC path on gfx950 matrix cores
// (v_mfma_f64_16x16x4_f64).
//
//  (X = fac B P_sub, the density reduction and Z live in density.hip.)
//  k_syr2k    : V = B^T Z + Z^T B, lower triangle, with the scatter-add
//               into VXC fused into the epilogue (GauXC: DSYR2K per task +
//               sym_inc_by_submat, scheme1_base.cxx:1712-1766).
//
// MFMA operand layout (16x16x4 f64, measured on gfx950): lane l holds
// A[l%16][l/16] and B[l/16][l%16]; accumulator register r of lane l is
// D[4*r + l/16][l%16] (rows interleave across the four 16-lane groups,
// unlike the FP32-output MFMAs whose register r holds row 4*(l/16) + r).
#include "syr2k.hpp"

#include <type_traits>

namespace xcq {

using v4d = double __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d mfma_f64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One 1 KiB fragment from memory into LDS: lane l's 16 bytes at base + off
// go to lds + 16 l.  Inline asm so that the compiler's wait insertion, which
// cannot tell the two stages apart, adds no wait for it before LDS reads; the K
// loop waits itself.
__device__ __forceinline__ void frag_to_lds(const double* base, unsigned off, const double* lds) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
  asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(m0) : "memory");
}

// ---------------------------------------------------------------------------
// One workgroup per region of up to 7 x 6 blocks of 16 x 16 functions (up to
// 8 x 8 when that is the whole task) and slice of the task's points.
//
// What bounds it: the matrix cores, once each operand is fetched few enough
// times.  Padding to 64-wide tiles and 64 points multiplied 1.8 to 2.3 times
// what is wanted (150 and 24 waters); a first version with one wave per 4 x
// 3 blocks, its operands straight from memory, multiplied 1.2 times but read
// 23 GB past L2 per 24-water call, with the matrix cores 41% busy.  So four
// waves share a region's fragments through LDS, and only blocks that hold
// wanted elements are multiplied: below nbe, on or below the diagonal, not
// negligible by the bound table.  The wanted blocks are dealt evenly to the
// waves, each block anywhere in the region; at 64 cycles per MFMA the four
// fragments a block reads for its four MFMAs take half of the LDS bandwidth.
//
// A fragment is 16 functions x 8 points of a plane in lane order: lane (f =
// l & 15, q = l >> 4) holds points k + 2q, k + 2q + 1 of function row f, the
// operands of two MFMAs whose K index q stands for the points k + 2q + j.
// (Any order of the points serves as long as both operands use it.)  It is
// one 16-byte load per lane from memory into LDS and one 16-byte LDS read.
// Two stages of up to 13 blocks (B and Z) fill a third of a CU's LDS: three
// workgroups per CU, one barrier per eight points.  Now 12.6 GB past L2 per
// 24-water call (98 M requests of 128 bytes; the planes hold 9.0 GB) beside 37 M
// atomic additions, 3.1 TB/s read, and the matrix cores 61% busy.
//
// Stage times, 64-wide padded tiles -> this: 24 waters 8.4 -> 4.4 ms, 150
// waters 94.6 -> 61 ms, 120 functions on 340,000 points 0.66 -> 0.10 ms, 84
// functions on 35,000 points 0.11 -> 0.03 ms.
//
// The points of a task with very many of them (20,000 after merging) are cut
// into slices, or that task would be one serial chain: on small molecules
// that chain was the whole stage.  A slice stores its blocks to part, and
// k_syr2k_reduce sums a task's slices in order.
__global__ __launch_bounds__(256, 3) void k_syr2k(QueueArgs qa, const DevTask* __restrict__ tasks,
                                                  const int32_t* __restrict__ bfmap,
                                                  const double* __restrict__ scratch,
                                                  double* __restrict__ vxc_all, double drop,
                                                  const unsigned* __restrict__ tmax,
                                                  double* __restrict__ part) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int kSyrSlots = kSyr<false>.slots, kSyrStaged = kSyr<false>.staged();
  constexpr int kStage = 2 * kSyrStaged * 128;  // doubles per stage
  __shared__ __attribute__((aligned(16))) double stage[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, lf = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  XCQ_FOR_EACH_ITEM(qa, it) {
    const int64_t t0 = qa.tstamp ? wall_clock64() : 0;
    const WorkItem wi = qa.items[uniform64(it)];
    const DevTask t = tasks[wi.task];
    const int nbe = t.nbe, ld = t.npts_pad;
    const SyrRegion rg = syr_region<false>(t, wi.a & 0xffff, wi.a >> 16);
    const int n8 = (t.npts + 7) / 8, sl = wi.b & 0xffff, ns = wi.b >> 16;
    const int s0 = (int)((int64_t)sl * n8 / ns), s1 = (int)((int64_t)(sl + 1) * n8 / ns);
    const uint64_t mask = syr_mask(t, rg, lane, tmax, drop);
    if (mask == 0) {
      stamp_item(qa, it, t0);
      continue;
    }
    const int count = __popcll(mask);
    // Staged blocks: the columns, then the rows that are not among them.
    // Staged block u is function block u + c0, or u + gap past the columns.
    const int nc = rg.c1 - rg.c0, gap = rg.r0 > rg.c1 ? rg.r0 - rg.c1 : 0;
    const int nst = rg.r1 - rg.c0 - gap;
    auto block_of = [&](int u) { return rg.c0 + u + (u < nc ? 0 : gap); };
    // The wave's blocks: ranks [w count / 4, (w + 1) count / 4) of the mask.
    int* slots = reinterpret_cast<int*>(stage);
    __syncthreads();  // the previous item is done with the stages
    if (wave == 0 && (mask >> lane & 1)) {
      const int rb = rg.r0 + lane / nc, cb = rg.c0 + lane % nc;
      const int ur = rb < rg.c1 ? rb - rg.c0 : rb - gap - rg.c0;
      slots[__popcll(mask & ((uint64_t(1) << lane) - 1))] = ur | (cb - rg.c0) << 8;
    }
    __syncthreads();
    const int b0 = wave * count / 4, n = (wave + 1) * count / 4 - b0;
    int ur[kSyrSlots], uc[kSyrSlots];  // staged row and column block per slot
#pragma unroll
    for (int k = 0; k < kSyrSlots; ++k) {
      const int v = __builtin_amdgcn_readfirstlane(slots[min(b0 + k, count - 1)]);
      ur[k] = v & 0xff;
      uc[k] = v >> 8;
    }
    __syncthreads();  // slots are read: the stages may be filled

    // Fragments wave, wave + 4, ... of the 2 nst of a stage (block u's B at
    // 2u, its Z at 2u + 1).  Rows past nbe are read at row nbe - 1; their
    // products are not stored.  Byte offsets in a task's planes end below
    // 4 GiB.
    constexpr int kLoads = (2 * kSyrStaged + 3) / 4;
    const double* Bm = scratch + t.b_off;
    const double* Zm = Bm + 4 * (int64_t)nbe * ld;
    const double* plane = wave & 1 ? Zm : Bm;  // c = wave + 4 e has wave's parity
    unsigned off[kLoads];
#pragma unroll
    for (int e = 0; e < kLoads; ++e)
      off[e] = (unsigned)(min(16 * block_of(min((wave + 4 * e) >> 1, nst - 1)) + lf, nbe - 1) * ld +
                          2 * lq) * 8u;
    auto issue = [&](int s, int buf) {
      const double* src = plane + 8 * s;
#pragma unroll
      for (int e = 0; e < kLoads; ++e)
        if (wave + 4 * e < 2 * nst)
          frag_to_lds(src, off[e], stage + buf * kStage + (wave + 4 * e) * 128);
    };
    v4d acc[kSyrSlots];
#pragma unroll
    for (int k = 0; k < kSyrSlots; ++k) acc[k] = v4d{0., 0., 0., 0.};
    auto contract = [&](auto N) {
      constexpr int kN = decltype(N)::value;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      issue(s0, 0);
      for (int s = s0; s < s1; ++s) {
        const int buf = (s - s0) & 1;
        // This wave's fragments of stage s have landed and its reads of the
        // other stage are done; past the barrier so are the others'.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + 1 < s1) issue(s + 1, buf ^ 1);
        const double* st = stage + buf * kStage + 2 * lane;
#pragma unroll
        for (int k = 0; k < kN; ++k) {
          const v2d bi = *reinterpret_cast<const v2d*>(st + ur[k] * 256);
          const v2d zi = *reinterpret_cast<const v2d*>(st + ur[k] * 256 + 128);
          const v2d bj = *reinterpret_cast<const v2d*>(st + uc[k] * 256);
          const v2d zj = *reinterpret_cast<const v2d*>(st + uc[k] * 256 + 128);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            acc[k] = mfma_f64(bi[j], zj[j], acc[k]);
            acc[k] = mfma_f64(zi[j], bj[j], acc[k]);
          }
        }
      }
    };
    switch (n) {
      case 0: contract(std::integral_constant<int, 0>{}); break;
      case 1: contract(std::integral_constant<int, 1>{}); break;
      case 2: contract(std::integral_constant<int, 2>{}); break;
      case 3: contract(std::integral_constant<int, 3>{}); break;
      case 4: contract(std::integral_constant<int, 4>{}); break;
      case 5: contract(std::integral_constant<int, 5>{}); break;
      case 6: contract(std::integral_constant<int, 6>{}); break;
      case 7: contract(std::integral_constant<int, 7>{}); break;
      case 8: contract(std::integral_constant<int, 8>{}); break;
      case 9: contract(std::integral_constant<int, 9>{}); break;
      case 10: contract(std::integral_constant<int, 10>{}); break;
      default: contract(std::integral_constant<int, 11>{}); break;
    }

    if (ns > 1) {
      double* dst = part + ((int64_t)wi.c * kSyrBlocks + b0) * 256 + lane;
#pragma unroll
      for (int k = 0; k < kSyrSlots; ++k)
        if (k < n) {
#pragma unroll
          for (int r = 0; r < 4; ++r) dst[(k * 4 + r) * 64] = acc[k][r];
        }
    } else {
      // Scatter-add, in transposed order: element (i, j) of the task (i >=
      // j) is added at (bf[j], bf[i]) of the column-major VXC, so that the 16
      // lanes of a lane group, 16 consecutive j, touch a few 128-byte column
      // segments instead of 16 columns.  The symmetrisation that follows
      // sums the two triangles, so which triangle an element lands in does
      // not matter.
      const int32_t* bf = bfmap + t.bf_off;
      double* vxc = vxc_all + t.p_off;
#pragma unroll
      for (int k = 0; k < kSyrSlots; ++k)
        if (k < n) {
          const int j = 16 * block_of(uc[k]) + lf, i0 = 16 * block_of(ur[k]) + lq;
          const int cj = bf[min(j, nbe - 1)];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = i0 + 4 * r;
            // Negligible contributions are not added (NaN still is).
            if (i < nbe && i >= j && !(fabs(acc[k][r]) < drop))
              atomicAdd(vxc + (int64_t)bf[i] * t.ldp + cj, acc[k][r]);
          }
        }
    }
    stamp_item(qa, it, t0);
  }
}

// Sums the slices of one block of a region in order and adds it to VXC.
// Item: task, region (as above), number of slices, first slice's place in
// part; blockIdx.y is the rank of the block among the region's wanted ones.
template <bool MX>
__global__ __launch_bounds__(256) void k_syr2k_reduce(const WorkItem* __restrict__ items,
                                                      const DevTask* __restrict__ tasks,
                                                      const int32_t* __restrict__ bfmap,
                                                      const double* __restrict__ part,
                                                      double* __restrict__ vxc_all, double drop,
                                                      const unsigned* __restrict__ tmax) {
  const WorkItem wi = items[blockIdx.x];
  const DevTask t = tasks[wi.task];
  const int tid = threadIdx.x, lane = tid & 63, rank = blockIdx.y;
  const SyrRegion rg = syr_region<MX>(t, wi.a & 0xffff, wi.a >> 16);
  uint64_t m = syr_mask(t, rg, lane, tmax, drop);
  if (rank >= __popcll(m)) return;
  for (int k = 0; k < rank; ++k) m &= m - 1;
  const int k = __ffsll((unsigned long long)m) - 1, nc = rg.c1 - rg.c0;  // the rank-th one
  const int rb = rg.r0 + k / nc, cb = rg.c0 + k % nc;
  const double* src = part + ((int64_t)wi.c * kSyrBlocks + rank) * 256 + tid;
  double v = 0.;
#pragma unroll 8
  for (int s = 0; s < wi.b; ++s) v += src[(int64_t)s * kSyrBlocks * 256];
  const int r = tid >> 6, lq = lane >> 4;
  const int i = 16 * rb + (MX ? 4 * lq + r : 4 * r + lq), j = 16 * cb + (lane & 15);
  const int32_t* bf = bfmap + t.bf_off;
  if (i < t.nbe && i >= j && !(fabs(v) < drop))
    atomicAdd(vxc_all + t.p_off + (int64_t)bf[i] * t.ldp + bf[j], v);
}

int launch_syr2k_mixed(const CtxView& v, const WorkRange& r, const unsigned* tm);

int launch_syr2k(const CtxView& v, const Chunk& c, int precision) {
  const int mx = precision != XCQ_PREC_FP64;
  const WorkRange &r = c.syr2k[mx], &sum = c.syr2k_sum[mx];
  if (r.n == 0) return XCQ_SUCCESS;
  const unsigned* tm = v.vxc_drop > 0.0 ? v.tmax : nullptr;
  if (mx) {
    if (int rc = launch_syr2k_mixed(v, r, tm)) return rc;
  } else {
    hipLaunchKernelGGL(k_syr2k, dim3(grid_of(r)), dim3(256), 0, v.stream, queue_args(v, r),
                       v.tasks, v.bfmap, static_cast<const double*>(v.scratch), v.vxc, v.vxc_drop,
                       tm, v.syr_part);
  }
  if (sum.n)
    hipLaunchKernelGGL(mx ? k_syr2k_reduce<true> : k_syr2k_reduce<false>,
                       dim3((unsigned)sum.n, mx ? kSyr<true>.blocks() : kSyr<false>.blocks()),
                       dim3(256), 0, v.stream, v.work + sum.off, v.tasks, v.bfmap, v.syr_part, v.vxc, v.vxc_drop, tm);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

}  // namespace xcq
