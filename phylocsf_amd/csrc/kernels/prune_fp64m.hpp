// prune_fp64m.hpp -- the FP64 forward on matrix cores (precision
// PCSF_FP64M), driven by a tree's straight-line op program (generated per
// shipped tree); prune_fp64r.hip takes the other trees and the small calls.
//
// Same result as PhyloLik.ensure_alpha and the root posterior
// (lib/CamlPaml/PhyloLik.ml:73-93,127-138), per column ln z and the root's
// expected ln pi (the elpr_anc term of src/PhyloCSF.ml), in FP64 throughout
// with no rescaling, as the reference.  Organised like the fused MFMA kernel
// (prune_mfma.hpp): a wave owns 16 columns; the four waves of a workgroup
// walk the host's op program (post-order, fewest live tiles) in lock step;
// partials never leave registers -- a 64 x 16 FP64 tile is 32 VGPRs in the
// accumulator layout of v_mfma_f64_16x16x4f64 (fp64_tiles.hpp), which is
// also the next product's B operand -- and each internal-child message
// m = P alpha is a 64 x 64 by 64 x 16 product on those MFMAs with P staged in
// LDS.  The P tiles are double-buffered: every product issues the next
// tile's loads straight from memory into the idle buffer (the sets' P64F
// holds P in the MFMA's A-fragment order, so the copy is a plain one), and
// the barrier opening the next product is the only wait.  Leaf messages are
// the columns of P (in the leaf-branch layout of P64F the four lanes of a
// column read one 128-byte line per 16 rows), all ones for `Marginalize.  Paths are
// relative to the mlin/PhyloCSF tree.
#pragma once
#include "fp64_tiles.hpp"
#include "prune_mfma.hpp"

namespace pcsf_mfma {

namespace f64m {

using Tile64 = fp64t::Tile;
using fp64t::f64x4;

constexpr int kWaves = fp64t::kWaves;
constexpr int kNT = 64 * kWaves;     // threads per workgroup
constexpr int kGC = fp64t::kCols;    // columns per workgroup
constexpr int kTileBytes = 4096 * 8; // one P tile

struct NoMask {};  // FP64 needs no constant-column masks (no rescaling)

struct Walk64 {
  typedef __attribute__((address_space(3))) double L3;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  const MfmaParams& p;
  const double (*Pbuf)[4096];  // LDS: double-buffered P tile
  L3 (*Pbuf3)[4096];           // the same, as LDS addresses
  const uint8_t* codes_s;      // LDS: the group's leaf codes, nl x kGC
  int tid, lane, grp, wave_s, ccol;
  int q = 0, set = 0;
  int64_t col = 0;
  bool has_next = false;
  int next_set = 0;
  int kg = 0;  // products done (selects the LDS buffer)
  Tile64 pf;   // the next op's (first) leaf message, issued during a product

  __device__ __forceinline__ int oset() const {
    int s = set;
    asm volatile("" : "+s"(s));
    return s;
  }
  // the message of leaf `leaf` for this lane's codon (message 64: ones), in
  // eight pieces of two rows
  struct LeafAt {
    Rsrc r;
    uint32_t off, so;
  };
  __device__ __forceinline__ LeafAt leaf_at(int leaf) const {
    const int code = codes_s[leaf * kGC + ccol];
    const uint32_t c = code == PCSF_MARGINALIZE ? 64u : (uint32_t)code;
    constexpr uint32_t kBranchBytes = kTile64 * 8;
    return {make_rsrc(p.P64F + (size_t)oset() * p.nbr * kTile64, p.nbr * kBranchBytes),
            c * 512u + (uint32_t)grp * 32u, leaf * kBranchBytes};
  }
  __device__ __forceinline__ static void leaf_piece(Tile64& t, const LeafAt& at, int k) {
    const int mo = k >> 1, h = k & 1;
    const double2 d =
        __builtin_bit_cast(double2, bload4(at.r, at.off + 128u * mo + 16u * h, at.so));
    t.r[mo][2 * h] = d.x;
    t.r[mo][2 * h + 1] = d.y;
  }
  __device__ __forceinline__ Tile64 leaf(int leaf) const {
    const LeafAt at = leaf_at(leaf);
    Tile64 t;
#pragma unroll
    for (int k = 0; k < 8; ++k) leaf_piece(t, at, k);
    return t;
  }
  __device__ __forceinline__ static void mul(Tile64& s, const Tile64& o) {
#pragma unroll
    for (int mo = 0; mo < 4; ++mo) s.r[mo] *= o.r[mo];
  }
  // s = leaf a0 o leaf a1
  __device__ __forceinline__ void cherry(Tile64& s, NoMask&, int a0, int a1, bool use_pf) {
    const Tile64 o = leaf(a1);
    s = use_pf ? pf : leaf(a0);
    mul(s, o);
  }
  // the no-table programs have no table reads
  __device__ __forceinline__ void cherryt(Tile64&, NoMask&, int, int, int, bool) {}
  // s = s o leaf a0
  __device__ __forceinline__ void leafmul(Tile64& s, NoMask&, int a0, bool use_pf) {
    mul(s, use_pf ? pf : leaf(a0));
  }
  // s = s o o
  __device__ __forceinline__ void mulpop(Tile64& s, NoMask&, const Tile64& o, const NoMask&) {
    mul(s, o);
  }
  // s = P s for the tile staged in LDS; the next product's tile (branch
  // next_br of this set, or the next task's first) is loaded meanwhile into
  // the idle buffer, 16 bytes per lane at the wave's base + 16 lane: the
  // layout the tile has in memory; and the next leaf op's message into pf.
  // The loads stand between the MFMAs (in one burst in front of them each
  // would keep the wave from its first for some 50 clocks), and the fragments
  // are read from LDS kAhead steps before their MFMA (the compiler left two
  // MFMAs between a read and its use).  100vertebrates, 120 regions of 100 to
  // 3000 columns at a scale of their own: 7.49 -> 6.51 ms with the three.
  __device__ __forceinline__ void gemm(Tile64& s, const NoMask&, int next_br, int pf_leaf,
                                       uint32_t) {
    constexpr int kAhead = 6;
    __syncthreads();  // Pbuf[kg&1] complete; Pbuf[(kg&1)^1] no longer read
    __builtin_amdgcn_sched_barrier(0);  // a product is a scheduling region of its own
    L3* dst = Pbuf3[(kg & 1) ^ 1];
    constexpr int kPer = kTileBytes / 16 / kNT;  // 16-byte pieces per thread
    if (next_br == kNoBranch && has_next) {
      typedef const __attribute__((address_space(1))) void* GPtr;
      const double* nsrc = p.P64F + ((size_t)next_set * p.nbr + p.first_gemm_br) * kTile64;
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        __builtin_amdgcn_global_load_lds((GPtr)(nsrc + (tid + kNT * k) * 2),
                                         (LdsPtr)(dst + (64 * wave_s + kNT * k) * 2), 16, 0, 0);
    }
    const Rsrc rt = make_rsrc(p.P64F + (size_t)oset() * p.nbr * kTile64, p.nbr * kTile64 * 8u);
    const uint32_t so = next_br * (kTile64 * 8u);
    const bool ahead = pf_leaf != kNoBranch;
    const LeafAt at = leaf_at(ahead ? pf_leaf : 0);
    const double* frag = Pbuf[kg & 1] + lane;
    double a[kAhead];
#pragma unroll
    for (int t = 0; t < kAhead; ++t) a[t] = frag[t * 64];
    Tile64 m;
#pragma unroll
    for (int t = 0; t < 64; ++t) {
      const int mo = t >> 4, k = t & 15, i = t >> 2;
      f64x4 c = k == 0 ? (f64x4){0.0, 0.0, 0.0, 0.0} : m.r[mo];
      m.r[mo] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t % kAhead], s.r[k >> 2][k & 3], c, 0, 0, 0);
      if (t + kAhead < 64) a[t % kAhead] = frag[(t + kAhead) * 64];
      if ((t & 3) == 0 && i < 8 && next_br != kNoBranch)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (LdsPtr)(dst + (64 * wave_s + kNT * i) * 2),
                                                 16, (uint32_t)tid * 16u, so + 16u * kNT * i, 0, 0);
      if ((t & 3) == 2 && i < 8 && ahead) leaf_piece(pf, at, i);
      if (t & 1) __builtin_amdgcn_sched_barrier(0);  // the order stays as written
    }
    s = m;
    __builtin_amdgcn_sched_barrier(0);
    ++kg;
  }
  // ln z and the root posterior's expected ln pi of this lane's column
  __device__ __forceinline__ void root(const Tile64& s) {
    const int pq = p.prior_per_set ? set : q;
    Tile64 pr, w;
#pragma unroll
    for (int mo = 0; mo < 4; ++mo)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * mo + 4 * v + grp;
        pr.r[mo][v] = p.pi[pq * 64 + row];
        w.r[mo][v] = s.r[mo][v] * pr.r[mo][v];
        pr.r[mo][v] = p.lnpi[pq * 64 + row];
      }
    Tile64 one;
#pragma unroll
    for (int mo = 0; mo < 4; ++mo) one.r[mo] = (f64x4){1.0, 1.0, 1.0, 1.0};
    const double z = fp64t::column_dot(w, one);
    const double e = fp64t::column_dot(w, pr);  // sum_x alpha_x pi_x ln pi_x
    if (grp == 0) {
      p.logz[(size_t)q * p.ld + col] = log(z);
      p.colelpr[(size_t)q * p.ld + col] = (z != 0.0) ? e / z : 0.0;
    }
  }
};

// two workgroups per CU: a generated program keeps only its live tiles in
// registers
template <int NS, class PROG>
__global__ __launch_bounds__(kNT, 2) void prune_fp64m_kernel(MfmaParams p) {
  __shared__ __attribute__((aligned(16))) double Pbuf[2][4096];
  extern __shared__ __attribute__((aligned(16))) uint8_t codes_s[];  // nl x kGC
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int grp = lane >> 4, lcol = lane & 15;
  Tile64 S[NS];
  NoMask K[NS];
#pragma unroll
  for (int d = 0; d < NS; ++d)
#pragma unroll
    for (int mo = 0; mo < 4; ++mo) S[d].r[mo] = (f64x4){0.0, 0.0, 0.0, 0.0};

  Task cur;
  int64_t jc = 0;
  if (!next_task<kGC>(p, jc, &cur)) return;
  if (p.first_gemm_br != kNoBranch) {
    const double* src = p.P64F + ((size_t)cur.set * p.nbr + p.first_gemm_br) * kTile64;
#pragma unroll
    for (int k = 0; k < 4096 / 2 / kNT; ++k)
      reinterpret_cast<double2*>(Pbuf[0])[tid + kNT * k] =
          reinterpret_cast<const double2*>(src)[tid + kNT * k];
  }
  Walk64 w{p, Pbuf, (Walk64::L3 (*)[4096])Pbuf, codes_s, tid, lane, grp, wave,
           wave * 16 + lcol};
  for (;;) {
    Task nxt;
    int64_t jn = jc + 1;
    const bool has_next = next_task<kGC>(p, jn, &nxt);
    const int64_t gabs = p.g0 + cur.g;
    __syncthreads();  // the previous task's gathers are done with codes_s
    {
      const uint32_t* src = reinterpret_cast<const uint32_t*>(p.codes);
      uint32_t* dst = reinterpret_cast<uint32_t*>(codes_s);
      constexpr int words = kGC / 4;
      for (int e = tid; e < p.nl * words; e += kNT) {
        const int l = e / words, wd = e - l * words;
        dst[e] = src[((size_t)l * p.ld + (size_t)gabs * kGC) / 4 + wd];
      }
    }
    __syncthreads();
    w.q = cur.q;
    w.set = cur.set;
    w.has_next = has_next;
    w.next_set = has_next ? nxt.set : 0;
    w.col = gabs * kGC + w.ccol;
    PROG::run(w, S, K);
    if (!has_next) break;
    cur = nxt;
    jc = jn;
  }
}

template <int NS, class PROG>
hipError_t launch_ns(const MfmaParams& prm, int cus, hipStream_t s) {
  auto kern = prune_fp64m_kernel<NS, PROG>;
  const size_t dyn = ((size_t)prm.nl * kGC + 15) / 16 * 16;
  int per_cu = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kNT, dyn);
  if (e != hipSuccess) return e;
  const int grid = (std::max(per_cu, 1) * cus + 7) / 8 * 8;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kNT), dyn, s, prm);
  return hipGetLastError();
}

}  // namespace f64m

// the forward of a tree's generated program PROG (TreeLaunch signature;
// precision and launch shape do not apply)
template <class PROG>
hipError_t launch_fp64m_tree(const MfmaParams& prm, int, int, int cus, hipStream_t s) {
  return f64m::launch_ns<PROG::NS, PROG>(prm, cus, s);
}

}  // namespace pcsf_mfma
