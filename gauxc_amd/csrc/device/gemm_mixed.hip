// Mixed-precision contractions of the XC path on gfx950
// (v_mfma_f32_16x16x32_bf16).
//
// Numerics (chosen from a CPU emulation against the FP64 path):
//  * dB/dx, dB/dy, dB/dz and Z are stored in FP32.  The value plane B is
//    stored as FP32 plus a bfloat16 residual (plane 5 of the task scratch),
//    about 32 significant bits: FP32 rounding of B was the largest error
//    term of the EXC/VXC budget.
//  * For B^T Z each FP32 operand element is split on the fly into three
//    bfloat16 slices (exact: 3 x 8 bits cover the FP32 significand); B's
//    residual is its fourth slice b3.
//  * A product is formed from the leading slice product (one MFMA, its own
//    FP32 accumulator, so the large partial sum is rounded once per K block)
//    and six correction products (b0 z1, b1 z0, b0 z2, b1 z1, b2 z0, b3 z0;
//    dropped terms are ~2^-24 relative) in a second FP32 accumulator, both
//    added to FP64 accumulators after every 32-deep K block, so FP32
//    rounding does not grow with the contraction length (npts can reach
//    2e4 in the B^T Z product).
//  * Densities, the functional, EXC/NEL and VXC accumulate in FP64.
//
// The regions of the B^T Z + Z^T B product are those of the FP64 kernel, with
// limits of their own (syr2k.hpp); the density stage is in density.hip.
// Operand layout of the MFMA (measured on gfx950): lane l holds
// A[l%16][8(l/16) .. 8(l/16)+7] and B[8(l/16) .. +7][l%16]; accumulator
// register r of lane l is D[4(l/16)+r][l%16].
#include "syr2k.hpp"

#include <type_traits>

namespace xcq {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kKB = 32;    // K block = MFMA depth

// Splits two FP32 values into three bfloat16 slices each (round to nearest
// even at every step, so x = a + b + c exactly); the slices of the pair come
// packed, one v_cvt_pk_bf16_f32 per slice.
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split3f_pair(f2v x, unsigned& a, unsigned& b, unsigned& c) {
  const bf2v h1 = __builtin_convertvector(x, bf2v);
  const f2v r1 = x - __builtin_convertvector(h1, f2v);
  const bf2v h2 = __builtin_convertvector(r1, bf2v);
  const f2v r2 = r1 - __builtin_convertvector(h2, f2v);
  const bf2v h3 = __builtin_convertvector(r2, bf2v);
  a = __builtin_bit_cast(unsigned, h1);
  b = __builtin_bit_cast(unsigned, h2);
  c = __builtin_bit_cast(unsigned, h3);
}

__device__ __forceinline__ v4f mfma_v(bf16x8 a, bf16x8 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Correction products (B slice, Z slice) after the leading b0 z0:
// (0,1) (1,0) (0,2) (1,1) (2,0) (3,0); slice 3 of B is the stored bfloat16
// residual of the value plane.
__device__ __forceinline__ constexpr int corr_b(int k) {
  return k == 1 ? 1 : k == 3 ? 1 : k == 4 ? 2 : k == 5 ? 3 : 0;
}
__device__ __forceinline__ constexpr int corr_z(int k) {
  return k == 0 ? 1 : k == 2 ? 2 : k == 3 ? 1 : 0;
}

// ---------------------------------------------------------------------------
// P (FP64, nbf x nbf) -> FP32 copy (the mixed density stage's P_sub source).
__global__ __launch_bounds__(256) void k_P_to_f32(int64_t n, const double* __restrict__ P,
                                                  float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)P[i];
}

// ---------------------------------------------------------------------------
// B^T Z + Z^T B with the VXC scatter-add.  One 256-thread workgroup per region
// (up to 6 x 5 blocks of 16 functions, or a whole task of up to 7) and slice
// of the task's points, K blocks of 32 points.
//
// Per K block the region's blocks are split into bfloat16 slices once (wave w
// takes blocks w, w + 4, ...; four lanes cover 128 bytes of a row) and staged
// in LDS as fragments, 1 KiB per block and slice; then each wave multiplies
// its share of the wanted blocks (below nbe, on or below the diagonal, not
// negligible; in row order, so that a row's seven fragments stay in registers
// while its columns pass).  Rows past nbe lie past the end of the plane and
// are read as zeros by the buffer loads.
// A fragment's 16 bytes of (function f, points 8q .. 8q + 7) are at unit 16 q +
// (f ^ 2q), which keeps the loader's writes (lane 4f + q) and the waves' reads
// (lane 16 q + f) free of bank conflicts.
//
// What bounds it: waiting.  24 waters read 7.3 GB past L2 (the planes hold 5.6,
// 10 bytes per function and point) beside 37 M atomic additions, 2.1 TB/s read,
// with the matrix cores 18% and the vector units 26% busy: no unit is near its
// limit, but a K block's split, its products and the barriers around them follow
// one another, with two workgroups per CU to overlap.  Tiles of 64 functions,
// padded and with both triangles of the diagonal ones, read and split twice
// as much: 24 waters 4.7 -> 3.5 ms, 150 waters 58 -> 51 ms.  Regions of 4 x 4
// blocks take 3.7 and 53 ms, of 4 x 3 at three workgroups per CU 3.9 and 55;
// blocks in row pairs that share a column's fragments, or fragments loaded a
// block ahead, spill registers in the K loop (6.5 and 3.9 ms).  The raw
// operands of the next K block wait in registers; they are local to the loop,
// so that they are not carried from item to item (17 registers spill, none
// in the K loops; carried 79).
// Slices and their order as in the FP64 kernel (k_syr2k).
__global__ __launch_bounds__(256, 2) void k_syr2k_mx(QueueArgs qa,
                                                     const DevTask* __restrict__ tasks,
                                                     const int32_t* __restrict__ bfmap,
                                                     const float* __restrict__ scratch,
                                                     double* __restrict__ vxc_all, double drop,
                                                     const unsigned* __restrict__ tmax,
                                                     double* __restrict__ part) {
  constexpr int kSlots = kSyr<true>.slots, kStaged = kSyr<true>.staged();
  constexpr int kLoads = (kStaged + 3) / 4;
  __shared__ v4u stage[kStaged * 7 * 64];  // [block][b0 b1 b2 b3 z0 z1 z2][16 q + (f ^ 2q)]
  const int tid = threadIdx.x, lane = tid & 63, lf = lane & 15, lq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wf = lane >> 2, wq = lane & 3;               // loader: function, point group
  const int wpos = 16 * wq + (wf ^ (wq << 1)), rpos = 16 * lq + (lf ^ (lq << 1));

  XCQ_FOR_EACH_ITEM(qa, it) {
    const int64_t t0 = qa.tstamp ? wall_clock64() : 0;
    const WorkItem wi = qa.items[uniform64(it)];
    const DevTask t = tasks[wi.task];
    const int nbe = t.nbe, ld = t.npts_pad;
    const SyrRegion rg = syr_region<true>(t, wi.a & 0xffff, wi.a >> 16);
    const int n32 = (t.npts + kKB - 1) / kKB, sl = wi.b & 0xffff, ns = wi.b >> 16;
    const int s0 = (int)((int64_t)sl * n32 / ns), s1 = (int)((int64_t)(sl + 1) * n32 / ns);
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
    __syncthreads();  // the previous item is done with the stage
    if (wave == 0 && (mask >> lane & 1)) {
      const int rb = rg.r0 + lane / nc, cb = rg.c0 + lane % nc;
      const int ur = rb < rg.c1 ? rb - rg.c0 : rb - gap - rg.c0;
      slots[__popcll(mask & ((uint64_t(1) << lane) - 1))] = ur | (cb - rg.c0) << 8;
    }
    __syncthreads();
    const int b0 = wave * count / 4, n = (wave + 1) * count / 4 - b0;
    int ur[kSlots], uc[kSlots];  // staged row and column block per slot
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
      const int v = __builtin_amdgcn_readfirstlane(slots[min(b0 + k, count - 1)]);
      ur[k] = v & 0xff;
      uc[k] = v >> 8;
    }

    const unsigned plane = (unsigned)nbe * (unsigned)ld;
    const float* Bm = scratch + t.b_off_mx;
    const auto rsB = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Bm), 0,
                                                       (int)(plane * 4u), 0x00020000);
    const auto rsZ = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(Bm + 4 * (int64_t)plane), 0, (int)(plane * 4u), 0x00020000);
    const auto rsL = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(Bm + 5 * (int64_t)plane), 0, (int)(plane * 2u), 0x00020000);
    unsigned off[kLoads];  // element of the loader's row and point group
#pragma unroll
    for (int e = 0; e < kLoads; ++e)
      off[e] = (unsigned)(16 * block_of(min(wave + 4 * e, nst - 1)) + wf) * (unsigned)ld + 8 * wq;
    struct Raw {
      v4u b[2], z[2], lo;
    };
    auto load = [&](Raw (&raw)[kLoads], int s) {
      const int so = s * kKB;
#pragma unroll
      for (int e = 0; e < kLoads; ++e) {
        if (wave + 4 * e >= nst) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          raw[e].b[h] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rsB, (int)(off[e] * 4u + 16u * h), so * 4, 0));
          raw[e].z[h] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rsZ, (int)(off[e] * 4u + 16u * h), so * 4, 0));
        }
        raw[e].lo = __builtin_bit_cast(
            v4u, __builtin_amdgcn_raw_buffer_load_b128(rsL, (int)(off[e] * 2u), so * 2, 0));
      }
    };
    auto split = [&](const v4u (&x)[2], v4u* dst) {
      v4u a, b, c;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // (Copies: a bit cast of a vector's element itself reads element 0.)
        const unsigned x0 = x[e >> 1][2 * (e & 1)], x1 = x[e >> 1][2 * (e & 1) + 1];
        const f2v v{__builtin_bit_cast(float, x0), __builtin_bit_cast(float, x1)};
        unsigned a1, b1, c1;
        split3f_pair(v, a1, b1, c1);
        a[e] = a1;
        b[e] = b1;
        c[e] = c1;
      }
      dst[0] = a;
      dst[64] = b;
      dst[128] = c;
    };
    double acc[kSlots][4];
#pragma unroll
    for (int k = 0; k < kSlots; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[k][r] = 0.;
    struct Frags {
      bf16x8 b[4], z[3];
    };
    auto frags = [&](Frags& f, int u) {
      const v4u* st = stage + u * 7 * 64 + rpos;
#pragma unroll
      for (int q = 0; q < 4; ++q) f.b[q] = __builtin_bit_cast(bf16x8, st[64 * q]);
#pragma unroll
      for (int q = 0; q < 3; ++q) f.z[q] = __builtin_bit_cast(bf16x8, st[64 * (4 + q)]);
    };
    auto contract = [&](auto N) {
      constexpr int kN = decltype(N)::value;
      Raw raw[kLoads];
      if (s0 < s1) load(raw, s0);
      for (int s = s0; s < s1; ++s) {
        __syncthreads();  // the stage's previous reads are done
#pragma unroll
        for (int e = 0; e < kLoads; ++e) {
          if (wave + 4 * e >= nst) break;
          v4u* dst = stage + (wave + 4 * e) * 7 * 64 + wpos;
          split(raw[e].b, dst);
          dst[3 * 64] = raw[e].lo;
          split(raw[e].z, dst + 4 * 64);
        }
        __syncthreads();
        if (s + 1 < s1) load(raw, s + 1);
        Frags row;
#pragma unroll
        for (int k = 0; k < kN; ++k) {
          Frags col;
          frags(col, uc[k]);
          if (k == 0 || ur[k] != ur[k - 1]) frags(row, ur[k]);
          // Leading products b0 z0 in one FP32 accumulator, the corrections
          // (b0 z1, b1 z0, b0 z2, b1 z1, b2 z0, b3 z0; b3 = stored residual)
          // in another, for B_i^T Z_j and Z_i^T B_j alike.
          v4f cm = mfma_v(row.b[0], col.z[0], v4f{0.f, 0.f, 0.f, 0.f});
          v4f cc = v4f{0.f, 0.f, 0.f, 0.f};
          cm = mfma_v(row.z[0], col.b[0], cm);
#pragma unroll
          for (int pr = 0; pr < 6; ++pr) {
            const int sb = corr_b(pr), sz = corr_z(pr);
            cc = mfma_v(row.b[sb], col.z[sz], cc);  // B_i^T Z_j
            cc = mfma_v(row.z[sz], col.b[sb], cc);  // Z_i^T B_j
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[k][r] += (double)cm[r] + (double)cc[r];
        }
      }
    };
    __syncthreads();  // slots are read: the stage may be filled
    switch (n) {
      case 0: contract(std::integral_constant<int, 0>{}); break;
      case 1: contract(std::integral_constant<int, 1>{}); break;
      case 2: contract(std::integral_constant<int, 2>{}); break;
      case 3: contract(std::integral_constant<int, 3>{}); break;
      case 4: contract(std::integral_constant<int, 4>{}); break;
      case 5: contract(std::integral_constant<int, 5>{}); break;
      case 6: contract(std::integral_constant<int, 6>{}); break;
      case 7: contract(std::integral_constant<int, 7>{}); break;
      default: contract(std::integral_constant<int, 8>{}); break;
    }

    if (ns > 1) {
      double* dst = part + ((int64_t)wi.c * kSyrBlocks + b0) * 256 + lane;
#pragma unroll
      for (int k = 0; k < kSlots; ++k)
        if (k < n) {
#pragma unroll
          for (int r = 0; r < 4; ++r) dst[(k * 4 + r) * 64] = acc[k][r];
        }
    } else {
      // Scatter-add into VXC in transposed order (see k_syr2k).
      const int32_t* bf = bfmap + t.bf_off;
      double* vxc = vxc_all + t.p_off;
#pragma unroll
      for (int k = 0; k < kSlots; ++k)
        if (k < n) {
          const int j = 16 * block_of(uc[k]) + lf, i0 = 16 * block_of(ur[k]) + 4 * lq;
          const int cj = bf[min(j, nbe - 1)];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = i0 + r;
            // Negligible contributions are not added (NaN still is).
            if (i < nbe && i >= j && !(fabs(acc[k][r]) < drop))
              atomicAdd(vxc + (int64_t)bf[i] * t.ldp + cj, acc[k][r]);
          }
        }
    }
    stamp_item(qa, it, t0);
  }
}

int launch_syr2k_mixed(const CtxView& v, const WorkRange& r, const unsigned* tm) {
  hipLaunchKernelGGL(k_syr2k_mx, dim3(grid_of(r)), dim3(256), 0, v.stream, queue_args(v, r),
                     v.tasks, v.bfmap, static_cast<const float*>(v.scratch), v.vxc, v.vxc_drop,
                     tm, v.syr_part);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

int launch_P_to_f32(hipStream_t s, int64_t n, const double* P, float* out) {
  if (n == 0) return XCQ_SUCCESS;
  hipLaunchKernelGGL(k_P_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, P, out);
  XCQ_HIP(hipGetLastError());
  return XCQ_SUCCESS;
}

}  // namespace xcq
