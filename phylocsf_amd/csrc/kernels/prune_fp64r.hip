// prune_fp64r.hip -- the FP64 matrix-core forward (precision PCSF_FP64M) with
// each product's rows split over the waves of a workgroup: short chains for
// few columns, and one kernel for every tree without a generated program.
//
// prune_fp64m.hpp gives a wave 16 columns and all 64 rows of every message: a
// product is 64 v_mfma_f64_16x16x4f64 of 64 cycles (1.7 us), so a tree of g
// internal branches takes at least 1.7 g us however few columns there are.
// Here the four waves of a workgroup share CT tiles of 16 columns: wave w
// makes rows 16 w .. 16 w + 15 of each message, 16 MFMAs per tile (they chain
// at full rate, 64 cycles each), and owns those rows of every live tile.
// Between products the waves exchange alpha through LDS: lane (j, g) of wave
// w holds rows 16 w + 4 v + g of column j, and K-step 4 w + v of the next
// product's B operand wants exactly that value in the same lane, so the
// exchange is 16-byte reads and writes without bank conflicts, one barrier
// per product (two with CT = 2, whose single buffer saves LDS).  A wave's
// part of P (16 A fragments) goes from memory to registers a product ahead
// (two at CT = 1, where a product is shorter than the memory latency) and the
// next nodes' leaf messages with it, one load after each MFMA: in one burst
// the loads hold the wave up until the memory pipeline has taken them (29
// mammals, 14 blocks: 42 us in bursts, 33 us interleaved).  Live tiles below
// the top of the program's stack wait in LDS, private to their lane, so the
// depth needs no registers: 226 VGPRs (190 with two tiles) and two workgroups per
// CU whatever the tree, where the interpreter over prune_fp64m.hpp's layout kept every slot
// live through its dispatch (one workgroup per CU above three slots).
//
// Measured (us per forward over both models, against the column-per-wave
// kernel of the time): 29mammals, 37 columns 32 (74); 12flies, 100 columns 18 (34);
// 53birds, which has no generated program, 8182 blocks 4310 (5069).  What bounds
// it at size is the traffic of P from L2 (32 KB per product for 16 CT columns
// where the other kernel stages it once for 64): a tree's generated program takes
// over where these workgroups no longer all fit (prune_fp64m.hip has the figures).
//
// Every element is the same sum in the same order as in prune_fp64m.hpp
// (K-steps ascending from zero, leaf factors and siblings multiplied in the
// program's order, the root's dot over the 16 rows of a lane before the
// lanes), so the results are the same bits and a dispatch between the two
// kernels is free of rounding.  Paths are relative to the mlin/PhyloCSF tree.
#include <algorithm>
#include <type_traits>

#include "fp64_tiles.hpp"
#include "prune_mfma.hpp"

using pcsf_mfma::MfmaParams;

namespace {

using fp64t::f64x4;

constexpr int kNT = 256;  // four waves

struct RTask {
  int q, set;
  int64_t g;
};

// Tasks are (model, tile of 16 CT columns) as in prune_mfma.hpp's task_at;
// tiles without a column of their region, padding blocks and inactive sets
// are passed over.
template <int CT>
__device__ __forceinline__ bool next_rtask(const MfmaParams& p, int64_t& j, RTask* t) {
  constexpr int GC = 16 * CT;
  for (;; ++j) {
    pcsf_mfma::Task u;
    if (!pcsf_mfma::task_at(p, j, &u)) return false;
    const int64_t c0 = (p.g0 + u.g) * GC;
    const int r = p.block_region[c0 / kAlignCols];
    if (r < 0 || c0 - p.astart[r] >= p.off[r + 1] - p.off[r]) continue;
    t->q = u.q;
    t->g = u.g;
    t->set = p.shared_sets ? u.q : (r - p.r0) * p.nm + u.q;
    if (p.active[t->set]) return true;
  }
}

template <int CT>
struct RWalk {
  static constexpr int GC = 16 * CT;
  const MfmaParams& p;
  static constexpr int NX = CT == 1 ? 2 : 1;  // exchange buffers
  static constexpr int NA = CT == 1 ? 3 : 2;  // steps whose tiles are in flight or in use
  static constexpr int NL = CT == 1 ? 3 : 1;  // leaf messages of a step kept
  double2* X;      // LDS: alpha exchange, [NX][CT][4 waves][2][64]
  double2* stk;    // LDS: waiting tiles, [slots - 1][CT][2][256]
  const uint8_t* codes_s;
  int tid, lane, wave, j, g;
  int q = 0, set = 0;

  // The message of leaf `leaf` (PSets::d_P64F's leaf layout: rows 16 mo + 4 v + g
  // at 16 mo + 4 g + v); nothing is read unless `on` (an offset past the buffer's
  // end).  A lane's four rows are 32 bytes; read one lane's own column at a time
  // the vector L1 looks up an address for every lane and 16 bytes, so a pair of
  // neighbouring lanes reads 32 bytes of its even column, then of its odd one,
  // and own() swaps the halves (252,344 columns on 53birds 4.55 -> 4.42 ms, a
  // gene's fit 2.52 -> 2.35).
  __device__ __forceinline__ void leaf(f64x4 (&m)[CT], int leaf, bool on) const {
    constexpr uint32_t kBranchBytes = kTile64 * 8;
    const pcsf_mfma::Rsrc r =
        pcsf_mfma::make_rsrc(p.P64F + (size_t)set * p.nbr * kTile64, p.nbr * kBranchBytes);
    const uint32_t part = on ? g * 32u + (j & 1) * 16u : 0x80000000u;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const uint32_t two =
          *reinterpret_cast<const uint16_t*>(codes_s + leaf * GC + 16 * c + (j & ~1));
      const uint32_t even = min(two & 0xffu, 64u), odd = min(two >> 8, 64u);  // 255: `Marginalize
      const uint32_t so = leaf * kBranchBytes + wave * 128u;
      const double2 a = __builtin_bit_cast(double2, pcsf_mfma::bload4(r, even * 512u + part, so));
      const double2 b = __builtin_bit_cast(double2, pcsf_mfma::bload4(r, odd * 512u + part, so));
      m[c] = (f64x4){a.x, a.y, b.x, b.y};
    }
  }
  // the value of the pair's other lane
  __device__ __forceinline__ static double other(double x) {
    constexpr int kFlip = 0xb1;  // quad_perm:[1,0,3,2]
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(x), kFlip, 0xf, 0xf, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(x), kFlip, 0xf, 0xf, true));
  }
  // this lane's four rows of a message that leaf() loaded
  __device__ __forceinline__ f64x4 own(const f64x4& m) const {
    // (every lane makes the moves: a select must not skip one)
    const double a0 = other(m[0]), a1 = other(m[1]), b0 = other(m[2]), b1 = other(m[3]);
    const bool odd = j & 1;
    return (f64x4){odd ? b0 : m[0], odd ? b1 : m[1], odd ? m[2] : a0, odd ? m[3] : a1};
  }
  // this wave's A fragments of branch `br`
  __device__ __forceinline__ void tile(double (&A)[16], int br) const {
    constexpr uint32_t kBranchBytes = kTile64 * 8;
    const pcsf_mfma::Rsrc r =
        pcsf_mfma::make_rsrc(p.P64F + (size_t)set * p.nbr * kTile64, p.nbr * kBranchBytes);
    const uint32_t so = br * kBranchBytes + wave * 8192u;
#pragma unroll
    for (int s = 0; s < 16; ++s)
      A[s] = pcsf_mfma::bload_f64(r, lane * 8u + (s & 7) * 512u, so + (s >> 3) * 4096u);
  }
  __device__ __forceinline__ void share(const f64x4 (&cur)[CT], int buf) const {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      double2* x = X + ((buf * CT + c) * 4 + wave) * 128 + lane;
      x[0] = make_double2(cur[c][0], cur[c][1]);
      x[64] = make_double2(cur[c][2], cur[c][3]);
    }
  }
  __device__ __forceinline__ void shared_rows(double (&B)[16], int buf, int c) const {
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double2 v = X[((buf * CT + c) * 4 + w) * 128 + 64 * h + lane];
        B[4 * w + 2 * h] = v.x;
        B[4 * w + 2 * h + 1] = v.y;
      }
  }
  __device__ __forceinline__ void push(const f64x4 (&cur)[CT], int d) const {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      double2* s = stk + (size_t)(d * CT + c) * 512 + tid;
      s[0] = make_double2(cur[c][0], cur[c][1]);
      s[256] = make_double2(cur[c][2], cur[c][3]);
    }
  }
  __device__ __forceinline__ void pop_mul(f64x4 (&cur)[CT], int d) const {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const double2* s = stk + (size_t)(d * CT + c) * 512 + tid;
      const double2 a = s[0], b = s[256];
      cur[c] *= (f64x4){a.x, a.y, b.x, b.y};
    }
  }
  // ln z and the root posterior's expected ln pi: wave c takes tile c (the
  // arithmetic of prune_fp64m.hpp's root)
  __device__ __forceinline__ void root(int buf, int64_t col0) const {
    if (wave >= CT) return;
    const int pq = p.prior_per_set ? set : q;
    const double2* x = X + ((buf * CT + wave) * 4) * 128 + lane;
    double z = 0.0, e = 0.0;
#pragma unroll 1
    for (int k = 0; k < 8; ++k) {  // rows 16 mo + 4 v + g, v = 2 h, 2 h + 1, of k = 2 mo + h
      const double2 a = x[64 * k];
      const int row = pq * 64 + 8 * k + g;
      const double w0 = a.x * p.pi[row], w1 = a.y * p.pi[row + 4];
      z += w0;
      z += w1;
      e = fma(w0, p.lnpi[row], e);
      e = fma(w1, p.lnpi[row + 4], e);
    }
    z += __shfl_xor(z, 16);
    z += __shfl_xor(z, 32);
    e += __shfl_xor(e, 16);
    e += __shfl_xor(e, 32);
    const int64_t col = col0 + 16 * wave + j;
    if (g == 0) {
      p.logz[(size_t)q * p.ld + col] = log(z);
      p.colelpr[(size_t)q * p.ld + col] = (z != 0.0) ? e / z : 0.0;
    }
  }
};

// One step of the program: the gather or sibling op that completes a node's
// alpha, then the product of the branch above it (or the root).
struct Step {
  int e0, e1;  // the op's first two words
  int g0, g1;  // the product's
};
__device__ __forceinline__ Step uniform(const int4& e, const int4& g) {
  return Step{__builtin_amdgcn_readfirstlane(e.x), __builtin_amdgcn_readfirstlane(e.y),
              __builtin_amdgcn_readfirstlane(g.x), __builtin_amdgcn_readfirstlane(g.y)};
}

template <int CT>
__global__ __launch_bounds__(kNT, 2) void prune_fp64r_kernel(MfmaParams p, int slots, int nsteps) {
  extern __shared__ __attribute__((aligned(16))) double2 lds[];
  constexpr int GC = 16 * CT;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  double2* stk = lds + RWalk<CT>::NX * CT * 512;
  uint8_t* codes_s = reinterpret_cast<uint8_t*>(stk + (slots - 1) * CT * 512);
  RWalk<CT> w{p, lds, stk, codes_s, tid, lane, wave, lane & 15, lane >> 4};
  // the program in LDS: its words must not wait behind the loads in flight
  int4* prog = reinterpret_cast<int4*>(codes_s + (p.nl * GC + 15) / 16 * 16);
  for (int e = tid; e < 2 * nsteps; e += kNT) prog[e] = reinterpret_cast<const int4*>(p.prog)[e];
  __syncthreads();
  RTask t;
  for (int64_t jt = 0; next_rtask<CT>(p, jt, &t); ++jt) {
    const int64_t col0 = (p.g0 + t.g) * GC;
    __syncthreads();  // the previous task's gathers and root are done
    {
      const uint32_t* src = reinterpret_cast<const uint32_t*>(p.codes);
      uint32_t* dst = reinterpret_cast<uint32_t*>(codes_s);
      constexpr int words = GC / 4;
      for (int e = tid; e < p.nl * words; e += kNT) {
        const int l = e / words, wd = e - l * words;
        dst[e] = src[((size_t)l * p.ld + (size_t)col0) / 4 + wd];
      }
    }
    __syncthreads();
    w.q = t.q;
    w.set = t.set;
    constexpr int NA = RWalk<CT>::NA, NL = RWalk<CT>::NL;
    f64x4 cur[CT];  // the top of the stack
    // step k's words and tile sit in slot k % NA, its leaf messages in k % NL
    Step S[NA];
    f64x4 L0[NL][CT], L1[NL][CT];
    double A[NA][16];
    const int last = 2 * (nsteps - 1);
    auto words = [&](int k) {
      const int e = min(2 * k, last);
      return uniform(prog[e], prog[e + 1]);
    };
    // step s's leaf messages and product's tile.  Operands that the op does
    // not have are loads that read nothing (the root's tile is branch 0's): a
    // branch around the loads would move registers at its join
    auto fetch = [&](const Step& s, f64x4 (&l0)[CT], f64x4 (&l1)[CT], double (&a)[16]) {
      const int op = s.e0 & 0xff;
      w.leaf(l0, s.e1 & 0xffff, op != OP_MULPOP);
      w.leaf(l1, (s.e1 >> 16) & 0xffff, op == OP_CHERRY);
      w.tile(a, step_branch(s.g0, s.g1));
    };
#pragma unroll
    for (int i = 0; i < NA - 1; ++i) {
      S[i] = words(i);
      fetch(S[i], L0[i % NL], L1[i % NL], A[i]);
    }
    int k = 0;
    auto node = [&](const Step& s, const f64x4 (&l0)[CT], const f64x4 (&l1)[CT]) {  // alpha
      const int op = s.e0 & 0xff, d = (s.e0 >> 8) & 0xff;
      if (op == OP_MULPOP) {
        w.pop_mul(cur, d);
      } else if (op == OP_LEAFMUL) {
#pragma unroll
        for (int c = 0; c < CT; ++c) cur[c] *= w.own(l0[c]);
      } else {  // OP_CHERRY: a new top of the stack
        if (d > 0) w.push(cur, d - 1);
#pragma unroll
        for (int c = 0; c < CT; ++c) cur[c] = w.own(l0[c]) * w.own(l1[c]);
      }
    };
    // step k in slot I: its node, then its product; true at the root
    auto step = [&](auto slot) -> bool {
      constexpr int I = decltype(slot)::value, N = (I + NA - 1) % NA;
      constexpr int IL = I % NL, LN = N % NL;
      const int buf = RWalk<CT>::NX == 2 ? k & 1 : 0;
      node(S[I], L0[IL], L1[IL]);
      w.share(cur, buf);
      __syncthreads();  // alpha complete (and with two buffers the other is free again)
      if ((S[I].g0 & 0xff) == OP_ROOT) return true;
      double B[CT][16];
      w.shared_rows(B[0], buf, 0);
      S[N] = words(k + NA - 1);
      fetch(S[N], L0[LN], L1[LN], A[N]);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (c + 1 < CT) w.shared_rows(B[c + 1], buf, c + 1);
        f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 16; ++s)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[I][s], B[c][s], acc, 0, 0, 0);
        cur[c] = acc;
      }
      // LDS reads first, then one load after each product: loads issued in one
      // burst hold the wave up until the memory pipeline has taken them all
      if constexpr (CT == 1) {  // 4 leaf loads and 16 of the tile over 16 products
        __builtin_amdgcn_sched_group_barrier(0x100, 11, 0);
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
      } else {
        __builtin_amdgcn_sched_group_barrier(0x100, 8 + 2 * CT + 1, 0);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
#pragma unroll
          for (int s = 0; s < 8; ++s) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
        }
      }
      if (RWalk<CT>::NX == 1) __syncthreads();  // every wave has read this alpha
      ++k;
      return false;
    };
    for (;;) {
      if (step(std::integral_constant<int, 0>())) break;
      if (step(std::integral_constant<int, 1>())) break;
      if constexpr (NA == 3)
        if (step(std::integral_constant<int, 2>())) break;
    }
    w.root(RWalk<CT>::NX == 2 ? k & 1 : 0, col0);
  }
}

template <int CT>
size_t lds_bytes(int nl, int slots, int nsteps) {
  return (size_t)(RWalk<CT>::NX + slots - 1) * CT * 8192 + ((size_t)nl * 16 * CT + 15) / 16 * 16 +
         (size_t)nsteps * 32;
}

template <int CT>
hipError_t launch(MfmaParams p, int slots, int nsteps, int cus, hipStream_t s) {
  p.g0 *= kAlignCols / (16 * CT);
  p.ngroups *= kAlignCols / (16 * CT);
  const size_t lds = lds_bytes<CT>(p.nl, slots, nsteps);
  auto kern = prune_fp64r_kernel<CT>;
  int per_cu = 0;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kNT, lds);
  if (e != hipSuccess) return e;
  if (per_cu < 1) return hipErrorInvalidValue;
  const int64_t tasks = p.ngroups * p.nm;
  const int grid = (int)std::min<int64_t>((int64_t)per_cu * cus, tasks);
  hipLaunchKernelGGL(kern, dim3((grid + 7) / 8 * 8), dim3(kNT), lds, s, p, slots, nsteps);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fp64_rows(const MfmaParams& p, int64_t blocks, int slots, int nsteps, int cus,
                            hipStream_t s) {
  // one tile per workgroup while that leaves every workgroup resident (two
  // per CU): the shortest chain; two tiles share each load of P above.  A
  // tree of thousands of leaves fits LDS at one tile only.
  constexpr size_t kLds = 160 << 10;  // per CU
  const bool two = 4 * blocks > 2 * (int64_t)cus && lds_bytes<2>(p.nl, slots, nsteps) <= kLds;
  return two ? launch<2>(p, slots, nsteps, cus, s) : launch<1>(p, slots, nsteps, cus, s);
}
