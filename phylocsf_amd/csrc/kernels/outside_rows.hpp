// outside_rows.hpp -- the pieces of an inside and outside pass over one tree with
// product rows split over the four waves of a workgroup, FP64 on
// v_mfma_f64_16x16x4f64 (adjoint_mfma.hip).
//
// A workgroup owns a tile of 16 columns; wave w owns rows 16 w .. 16 w + 15 of
// every message (lane (j, g): rows 16 w + 4 v + g of column j) and makes those
// rows of every product: 16 MFMAs, its A fragments read from memory straight
// into registers.  The other rows of a product's operand come from the other
// waves through LDS: value v of lane (j, g) of wave w is what K-step 4 w + v of
// the B operand wants in the same lane, so the exchange is 16-byte writes and
// reads without bank conflicts, and one barrier per product (two buffers
// alternate).  A wave reads back from memory only what it wrote itself.  The
// loads of the next product's A fragments (into the registers that the MFMAs
// have used up) and of the next node's operands are issued between the MFMAs:
// in one burst they would hold the wave up.
#pragma once
#include "fp64_tiles.hpp"
#include "prune_mfma.hpp"

namespace outside {

using fp64t::f64x4;
using pcsf_mfma::kNowhere;
using pcsf_mfma::Rsrc;

constexpr int kNT = 256;              // threads: four waves
constexpr int kSlot = 64 * 16;        // doubles of one 64 x 16 tile

struct Walk {
  double2* X;     // LDS: [2][4 waves][2][64]
  double* slots;  // this workgroup's tiles in memory
  const char* P;  // P of the current task's set
  Rsrc rs;        // the slots
  int lane, wave;
  int kx = 0;     // exchanges done

  // own rows into buffer kx & 1; the barrier makes them every wave's
  __device__ __forceinline__ void share(const f64x4& r) {
    double2* x = X + ((kx & 1) * 4 + wave) * 128 + lane;
    x[0] = make_double2(r[0], r[1]);
    x[64] = make_double2(r[2], r[3]);
    __syncthreads();
  }
  // all 64 rows as the B operand's 16 K-steps
  __device__ __forceinline__ void operand(double (&B)[16]) const {
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double2 v = X[((kx & 1) * 4 + w) * 128 + 64 * h + lane];
        B[4 * w + 2 * h] = v.x;
        B[4 * w + 2 * h + 1] = v.y;
      }
  }
  // this wave's 16 fragments of a 64 x 64 matrix in A-fragment order at byte
  // `so` of r
  __device__ __forceinline__ void fragments(double (&A)[16], Rsrc r, uint32_t so) const {
    so += wave * 8192u;
#pragma unroll
    for (int s = 0; s < 16; ++s)
      A[s] = pcsf_mfma::bload_f64(r, lane * 8u + (s & 7) * 512u, so + (s >> 3) * 4096u);
  }
  // A x B; A becomes the fragments at byte `so` of r
  __device__ __forceinline__ f64x4 product(double (&A)[16], const double (&B)[16], Rsrc r,
                                           uint32_t so) {
    so += wave * 8192u;
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], B[s], acc, 0, 0, 0);
      A[s] = pcsf_mfma::bload_f64(r, lane * 8u + (s & 7) * 512u, so + (s >> 3) * 4096u);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
    }
#pragma unroll
    for (int s = 4; s < 16; ++s) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
    ++kx;
    return acc;
  }
  // Four rows from this lane's part of the slot at byte `sso` of the slots, or
  // from byte `pso` of P.  (The pinned bases and mask keep the
  // choice a select: as a branch it would end the block in which loads and
  // MFMAs are interleaved.)
  // Of P, the pair of neighbouring lanes reads 32 bytes of its even column (lane
  // byte `even`, 16 to each), then of its odd one (`odd`): own() swaps the halves.
  __device__ __forceinline__ f64x4 read(bool slot, uint32_t sso, uint32_t pso, uint32_t even,
                                        uint32_t odd) const {
    typedef const __attribute__((address_space(1))) char* Global;
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    Global b0 = (Global)P + pso, b1 = (Global) reinterpret_cast<const char*>(slots) + (sso + wave * 2048u);
    asm volatile("" : "+s"(b0), "+s"(b1));
    const Global base = slot ? b1 : b0;
    uint32_t m = slot ? ~0u : 0u;
    asm volatile("" : "+v"(m));
    const uint32_t o0 = even ^ ((even ^ (lane * 16u)) & m);
    const uint32_t o1 = odd ^ ((odd ^ (lane * 16u + 1024u)) & m);
    const f64x2 a = *(const __attribute__((address_space(1))) f64x2*)(base + o0);
    const f64x2 b = *(const __attribute__((address_space(1))) f64x2*)(base + o1);
    return (f64x4){a.x, a.y, b.x, b.y};
  }
  // this lane's part of slot k (off: zeros)
  __device__ __forceinline__ f64x4 get(int k, bool on) const {
    uint32_t off = on ? lane * 16u : kNowhere;
    asm volatile("" : "+v"(off));
    const uint32_t so = k * (uint32_t)(kSlot * 8) + wave * 2048u;
    const double2 a = __builtin_bit_cast(double2, pcsf_mfma::bload4(rs, off, so));
    const double2 b = __builtin_bit_cast(double2, pcsf_mfma::bload4(rs, off, so + 1024u));
    return (f64x4){a.x, a.y, b.x, b.y};
  }
  // rows 0, 1 and rows 2, 3 of the lanes in two runs of 1 KB
  __device__ __forceinline__ void put(int k, const f64x4& r) {
    double2* d = reinterpret_cast<double2*>(reinterpret_cast<char*>(slots) +
                                            (size_t)(k * (uint32_t)(kSlot * 8)) + wave * 2048u) +
                 lane;
    d[0] = make_double2(r[0], r[1]);
    d[64] = make_double2(r[2], r[3]);
  }
};

// the value of the pair's other lane
__device__ __forceinline__ double other(double x) {
  constexpr int kFlip = 0xb1;  // quad_perm:[1,0,3,2]
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(x), kFlip, 0xf, 0xf, true),
      __builtin_amdgcn_update_dpp(0, __double2loint(x), kFlip, 0xf, 0xf, true));
}
// This lane's four rows of a message read by pairs (`pair`; else m is it).  The
// vector L1 looks up an address for every lane and 16 bytes unless neighbours
// share them: a pair halves the lookups of a gathered row (the outside pass over
// 60 regions on 100vertebrates 8.02 -> 7.63 ms).
__device__ __forceinline__ f64x4 own(const f64x4& m, bool pair, int lane) {
  // (every lane makes the moves: a select must not skip one)
  const double a0 = other(m[0]), a1 = other(m[1]), b0 = other(m[2]), b1 = other(m[3]);
  const bool odd = (lane & 1) && pair, even = !(lane & 1) && pair;
  return (f64x4){odd ? b0 : m[0], odd ? b1 : m[1], even ? a0 : m[2], even ? a1 : m[3]};
}

// The sum of v over the four lanes of a column (all of them end with it).
__device__ __forceinline__ double over_groups(double v) {
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// Every load is back.  In front of a loop whose loads wait one turn: the
// compiler counts the loads in flight at a loop's head over both ways in, so
// what the way in leaves pending would be waited for in every turn.
__device__ __forceinline__ void settle() { __builtin_amdgcn_s_waitcnt(0x0f70); }

}  // namespace outside
