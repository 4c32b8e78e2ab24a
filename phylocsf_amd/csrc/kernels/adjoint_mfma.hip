// adjoint_mfma.hip -- the outside (preorder) pass on FP64 matrix cores:
// d ln z / d t_br per region and branch, and d ln z / d rho per column.
//
// The gradient the reference's PhyloEM defines (lib/CamlPaml/PhyloEM.ml:
// 140-182): d ELL / d t_br = sum_ab xi_br[a,b] (dP/dt)_ab / P_ab with the
// branch posteriors xi of PhyloLik.add_branch_posteriors (PhyloLik.ml:
// 140-174) and dP/dt = Q P(t) (Q.ml:260-275); by the Fisher identity it is
// d ln z / d t_br, and with every branch scaled by rho, d ln z / d rho =
// sum_br b_br d ln z / d t_br (PhyloEM.ml:162-182).  For the branch into
// child c of node p with sibling s, with messages m_c = P_c alpha_c:
//   w_c = beta_p o m_s,   d ln z / d t_c = w_c . (Q m_c) / z,
//   beta_c = P_c^T w_c    (PhyloLik.ensure_beta, PhyloLik.ml:96-120),
// beta_root = pi (PhyloLik.ml:62), alpha_p = m_l o m_r (:78-90).
//
// Layout (outside_rows.hpp): a workgroup owns 16 columns of one region's block,
// its four waves 16 rows each of every product.  Inside, each internal node's
// message goes to the workgroup's slots in memory.  Outside, w_c is exchanged
// once and serves two products, P_c^T w_c (beta_c) and Q^T w_c, whose dot with
// m_c is w_c . (Q m_c): Q's fragments stay in 32 registers for the whole task.
// A leaf child needs no product: Q m_c is the column of Q P_c of its codon,
// which the P builder writes beside P^T (zeros for `Marginalize: Q 1 = 0).  So
// there are three products per internal branch and none per leaf branch (300
// per 16 columns and model on 100vertebrates; 394 with Q m_c as a product).
// A node's two messages are read once, a turn ahead; its beta stays in
// registers, and so do w_c and m_c of the child that comes next in index order
// (every node has one in a post-order tree, but for cherries): only a second
// internal child's w_c waits in memory.
// Per-branch sums run over the wave's lanes in row rotations and lane swaps,
// over the waves in LDS, and go to the region's total with one FP64 atomic per
// (workgroup, branch).  No rescaling, as the reference (FP64 range).
// Against one column tile per wave and P staged in LDS (64 columns per
// workgroup, the same products): forward and gradient of one region of 300
// columns 278 -> 165 us on 12flies, 926 -> 347 on 58mammals, 1536 -> 526 on
// 100vertebrates; 12 such regions 1973 -> 1081 there; 60 regions of 800 10787
// -> 9991.  The small calls are a chain of products a quarter as long; the
// large ones wait for memory (26 GB of messages and w at 3.2 TB/s with the
// matrix cores 46% busy), where reloading P's fragments cost 2.0 of 8.0 ms,
// the leaf gathers 1.1 and the inside pass's stores 1.2; with the gathers by
// pairs of lanes it is 7.6.
#include "outside_rows.hpp"

namespace {

using namespace outside;

// sum over the 64 lanes (every lane ends with it)
__device__ __forceinline__ double wave_sum(double v) {
#define PCSF_ROR_ADD(N)                                                                        \
  v += __hiloint2double(                                                                       \
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + N, 0xf, 0xf, false),           \
      __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + N, 0xf, 0xf, false));
  PCSF_ROR_ADD(8)
  PCSF_ROR_ADD(4)
  PCSF_ROR_ADD(2)
  PCSF_ROR_ADD(1)
#undef PCSF_ROR_ADD
  {
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false,
                                                    false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false,
                                                    false);
    v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
  }
  {
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false,
                                                    false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false,
                                                    false);
    v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
  }
  return v;
}

// This workgroup's place when the grid is numbered XCD by XCD (workgroup b
// runs on XCD b % 8; the grid is a multiple of 8).
__device__ __forceinline__ int xcd_rank() {
  return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
}

__device__ __forceinline__ double dot4(const f64x4& a, const f64x4& b) {
  return fma(a[0], b[0], fma(a[1], b[1], fma(a[2], b[2], a[3] * b[3])));
}

// BIG: a tree whose arrays would take more LDS than two workgroups per CU
// have; children, branch lengths and per-branch sums are then in memory.
template <bool BIG>
__global__ __launch_bounds__(kNT, 2) void adjoint_rows_kernel(AdjointArgs p) {
  __shared__ __attribute__((aligned(16))) double2 X[2 * 512];
  __shared__ double part[4][16];
  extern __shared__ __attribute__((aligned(16))) double dyn[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, g = lane >> 4;
  const int n = p.n, nl = p.nl, nm = p.nm, nbr = p.nbr, nin = n - nl;
  uint8_t* codes_s = reinterpret_cast<uint8_t*>(dyn);  // nl x 16
  double* gsum = dyn + 2 * nl;                         // [4 waves][nbr] sums of the task
  double* branch = gsum + 4 * nbr;
  int2* node = reinterpret_cast<int2*>(branch + nbr);  // children of node nl + k
  if constexpr (!BIG) {
    for (int k = tid; k < nbr; k += kNT) branch[k] = p.branch[k];
    for (int k = tid; k < nin; k += kNT) node[k] = make_int2(p.lc[nl + k], p.rc[nl + k]);
  }
  Walk w{X, p.scratch + (size_t)blockIdx.x * 2 * nin * kSlot, nullptr, Rsrc(), lane, wave};
  w.rs = pcsf_mfma::make_rsrc(w.slots, 2u * nin * (kSlot * 8u));
  const int64_t ntile = p.nblocks * (kAlignCols / 16), ntask = ntile * nm;
  for (int64_t i0 = 0; i0 < ntask; i0 += gridDim.x) {
    const int64_t task = i0 + xcd_rank();
    if (task >= ntask) continue;
    const int q = (int)(task / ntile);
    const int64_t b0 = p.c0 + (task - q * ntile) * 16;
    const int r = p.block_region[b0 / kAlignCols];
    if (r < 0) continue;  // padding block (uniform over the workgroup)
    const int64_t len = p.off[r + 1] - p.off[r];
    if (b0 - p.astart[r] >= len) continue;  // no column of the region in this tile
    const int set = (r - p.r0) * nm + q;
    if (!p.active[set]) continue;
    const int64_t col = b0 + j;
    const bool valid = col - p.astart[r] < len;
    w.P = reinterpret_cast<const char*>(p.P64F + (size_t)set * nbr * kTile64);
    const Rsrc rP = pcsf_mfma::make_rsrc(w.P, nbr * (kTile64 * 8u));
    const Rsrc rT = pcsf_mfma::make_rsrc(p.P64FT + (size_t)set * nbr * 4096, nbr * 32768u);
    __syncthreads();  // the previous task is done with X, part, gsum and codes_s
    for (int e = tid; e < nl * 4; e += kNT)
      reinterpret_cast<uint32_t*>(codes_s)[e] = *reinterpret_cast<const uint32_t*>(
          p.codes + (size_t)(e >> 2) * p.ld + b0 + 4 * (e & 3));
    double A[16], Qf[16], B[16];
    if (nin > 1) w.fragments(A, rP, nl * (kTile64 * 8u));
    // Q^T in A-fragment order: QT[k * 64 + a] = Q[a][k], row k of Q^T
#pragma unroll
    for (int s = 0; s < 16; ++s)
      Qf[s] = p.QT[(size_t)q * 4096 + (16 * wave + j) * 64 + 4 * s + g];
    f64x4 prior;
#pragma unroll
    for (int v = 0; v < 4; ++v) prior[v] = p.pi[q * 64 + 16 * wave + 4 * v + g];
    __syncthreads();
    // the message of node c, a leaf's from P's columns (by pairs of lanes: own()
    // when it is used), an internal node's own rows from its slot (an absent one:
    // something in range)
    const uint32_t piece = g * 32u + (j & 1) * 16u;
    auto two = [&](int lf) -> uint32_t {  // the codes of this pair's columns
      return *reinterpret_cast<const uint16_t*>(codes_s + lf * 16 + (j & ~1));
    };
    auto message = [&](int c, bool on) -> f64x4 {
      const bool slot = on && c >= nl;
      const int lf = on && !slot ? c : 0;
      uint32_t w2 = two(lf);
      if (!on) w2 = 64u << 8 | 64u;
      asm volatile("" : "+v"(w2));
      const uint32_t even = min(w2 & 0xffu, 64u), odd = min(w2 >> 8, 64u);  // 255: `Marginalize
      return w.read(slot, (slot ? c - nl : 0) * (kSlot * 8u), lf * (kTile64 * 8u) + wave * 128u,
                    even * 512u + piece, odd * 512u + piece);
    };
    auto leaf_q = [&](int c) -> f64x4 {  // Q m_c for a leaf c, by pairs (zeros otherwise)
      const int lf = c < nl ? c : 0;
      const uint32_t w2 = two(lf), e = w2 & 0xffu, o = w2 >> 8;
      uint32_t even = e == PCSF_MARGINALIZE || c >= nl ? kNowhere : e * 512u + piece;
      uint32_t odd = o == PCSF_MARGINALIZE || c >= nl ? kNowhere : o * 512u + piece;
      asm volatile("" : "+v"(even), "+v"(odd));
      const uint32_t so = lf * 32768u + wave * 128u;
      const double2 x = __builtin_bit_cast(double2, pcsf_mfma::bload4(rT, even, so));
      const double2 y = __builtin_bit_cast(double2, pcsf_mfma::bload4(rT, odd, so));
      return (f64x4){x.x, x.y, y.x, y.y};
    };
    auto kids = [&](int k) {
      const int2 v = BIG ? make_int2(p.lc[nl + k], p.rc[nl + k]) : node[k];
      return make_int2(__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y));
    };
    // ---- inside (PhyloLik.ml:78-92)
    f64x4 last = {0.0, 0.0, 0.0, 0.0};  // the message of node i - 1
    int2 kd = kids(0);
    f64x4 ml = message(kd.x, true), mr = message(kd.y, true);
    bool lastl = false, lastr = false;
    settle();
#pragma unroll 1
    for (int k = 0; k < nin - 1; ++k) {
      w.share((lastl ? last : own(ml, kd.x < nl, lane)) * (lastr ? last : own(mr, kd.y < nl, lane)));
      w.operand(B);
      kd = kids(k + 1);
      lastl = kd.x == nl + k;
      lastr = kd.y == nl + k;
      ml = message(kd.x, !lastl);
      mr = message(kd.y, !lastr);
      // the next product's fragments replace these as they are used up; after
      // the last inside product the first outside one's, P^T of node n - 2
      const bool in = k + 1 < nin - 1;
      last = w.product(A, B, in ? rP : rT,
                             in ? (nl + k + 1) * (kTile64 * 8u) : (uint32_t)(n - 2) * 32768u);
      w.put(k, last);
    }
    ml = lastl ? last : own(ml, kd.x < nl, lane);
    mr = lastr ? last : own(mr, kd.y < nl, lane);
    const double zp = over_groups(dot4(ml * mr, prior));
    if (g == 0) part[wave][j] = zp;
    __syncthreads();
    const double z = (part[0][j] + part[1][j]) + (part[2][j] + part[3][j]);
    const double zinv = (z != 0.0) ? 1.0 / z : 0.0;
    const double scale = valid ? zinv : 0.0;
    double* gb = p.grad_branch ? p.grad_branch + ((size_t)(r - p.r0) * nm + q) * nbr : nullptr;
    // ---- outside (PhyloLik.ml:96-120), parents before children
    double dr = 0.0;  // own rows' part of d z / d rho
    auto branch_done = [&](int c, double v) {  // v: own rows' part of w_c . (Q m_c)
      dr = fma(BIG ? p.branch[c] : branch[c], v, dr);
      if (p.grad_branch) {
        const double t = wave_sum(v * scale);
        if (lane == 0) {
          if constexpr (BIG)
            atomicAdd(gb + c, t);
          else
            gsum[wave * nbr + c] = t;
        }
      }
    };
    f64x4 wk, mk;  // of the node the next product is for: w and message
    // node nl + k with its beta, its children's messages and (leaf children) Q m:
    // a leaf branch is done, w of an internal child kept for the next product
    // or put away until its turn comes
    auto descend = [&](int k, int2 c, f64x4 b, f64x4 ml, f64x4 mr, f64x4 d0, f64x4 d1) {
      const f64x4 w0 = b * mr, w1 = b * ml;
      if (c.x < nl)
        branch_done(c.x, dot4(w0, d0));
      else if (c.x != nl + k - 1)
        w.put(nin + c.x - nl, w0);
      if (c.y < nl)
        branch_done(c.y, dot4(w1, d1));
      else if (c.y != nl + k - 1)
        w.put(nin + c.y - nl, w1);
      const bool right = c.y == nl + k - 1;
      wk = right ? w1 : w0;
      mk = right ? mr : ml;
    };
    kd = kids(nin - 1);
    descend(nin - 1, kd, prior, ml, mr, own(leaf_q(kd.x), true, lane), own(leaf_q(kd.y), true, lane));
    kd = kids(max(nin - 2, 0));
    ml = message(kd.x, true);
    mr = message(kd.y, true);
    f64x4 wf = wk, mf = mk;
    bool far = false;
    // node nl + k, its children's messages in ml and mr; the next node's go to
    // ln and rn (two turns alternate: a copy would wait for the loads)
    auto turn = [&](int k, f64x4 ml, f64x4 mr, f64x4& ln, f64x4& rn) {
      if (far) {
        wk = wf;
        mk = mf;
      }
      w.share(wk);
      w.operand(B);
      const f64x4 d0 = leaf_q(kd.x), d1 = leaf_q(kd.y);
      const int2 c = kd;
      const int kn = max(k - 1, 0);
      kd = kids(kn);
      far = c.x != nl + k - 1 && c.y != nl + k - 1;
      f64x4 acc = {0.0, 0.0, 0.0, 0.0}, qa = {0.0, 0.0, 0.0, 0.0};
      const uint32_t so = (uint32_t)(nl + kn) * 32768u + wave * 8192u;
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], B[s], acc, 0, 0, 0);
        qa = __builtin_amdgcn_mfma_f64_16x16x4f64(Qf[s], B[s], qa, 0, 0, 0);
        A[s] = pcsf_mfma::bload_f64(rT, lane * 8u + (s & 7) * 512u, so + (s >> 3) * 4096u);
      }
      wf = w.get(nin + kn, far);
      mf = w.get(kn, far);
      ln = message(kd.x, true);
      rn = message(kd.y, true);
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
      }
      ++w.kx;
      branch_done(nl + k, dot4(mk, qa));
      descend(k, c, acc, own(ml, c.x < nl, lane), own(mr, c.y < nl, lane), own(d0, true, lane),
              own(d1, true, lane));
    };
    settle();
    f64x4 ln, rn;
#pragma unroll 1
    for (int k = nin - 2; k >= 0; k -= 2) {
      turn(k, ml, mr, ln, rn);
      if (k == 0) break;
      turn(k - 1, ln, rn, ml, mr);
    }
    dr = over_groups(dr);
    __syncthreads();  // z's partial sums have been read
    if (g == 0) part[wave][j] = dr;
    __syncthreads();
    if (tid < 16) {
      p.logz[(size_t)q * p.ald + col] = log(z);
      p.coldrho[(size_t)q * p.ald + col] =
          ((part[0][j] + part[1][j]) + (part[2][j] + part[3][j])) * scale;
    }
    if (!BIG && p.grad_branch) {
      for (int br = tid; br < nbr; br += kNT)
        atomicAdd(gb + br, (gsum[br] + gsum[nbr + br]) + (gsum[2 * nbr + br] + gsum[3 * nbr + br]));
    }
  }
}

}  // namespace

// Two workgroups per CU (registers), in a grid of a multiple of 8 (xcd_rank).
AdjointPlan adjoint_plan(const pcsf_model* m, int64_t nblocks) {
  const int64_t tasks = nblocks * m->nm * (kAlignCols / 16);
  AdjointPlan p;
  p.grid = (int)std::min<int64_t>((tasks + 7) / 8 * 8, m->ctx->num_cus / 4 * 8);
  p.scratch = (size_t)p.grid * 2 * (m->n - m->nl) * kSlot;
  return p;
}

namespace {

AdjointArgs make_args(const pcsf_model* m, const pcsf_batch* b, const RegionChunk& ch,
                      double* scratch) {
  AdjointArgs a;
  a.codes = b->al.d_codes;
  a.ld = b->al.ld;
  a.ald = b->al.ld;
  a.c0 = ch.block0 * kAlignCols;
  a.nblocks = ch.nblocks;
  a.n = m->n;
  a.nl = m->nl;
  a.nm = m->nm;
  a.nbr = m->nbr;
  a.lc = m->d_lc;
  a.rc = m->d_rc;
  a.P64F = ch.sets->d_P64F;
  a.P64FT = ch.sets->d_P64FT;
  a.QT = m->d_QT;
  a.pi = m->d_pi;
  a.branch = m->d_branch;
  a.block_region = b->al.d_block_region;
  a.astart = b->al.d_astart;
  a.off = b->d_offsets;
  a.active = ch.sets->d_active;
  a.r0 = ch.r0;
  a.logz = b->d_alogz;
  a.coldrho = b->d_acolelpr;
  a.grad_branch = nullptr;
  a.scratch = scratch;
  return a;
}

}  // namespace

hipError_t launch_adjoint_mfma(const pcsf_model* m, const pcsf_batch* b, const RegionChunk& ch,
                               const AdjointPlan& plan, double* grad_branch, double* scratch,
                               hipStream_t s) {
  if (ch.sets->d_epi) return hipErrorInvalidValue;  // Q is per model
  AdjointArgs a = make_args(m, b, ch, scratch);
  a.grad_branch = grad_branch;
  if (ch.nblocks <= 0 || m->nm <= 0) return hipSuccess;
  const size_t codes = (size_t)m->nl * 16;
  const size_t lds = codes + (size_t)m->nbr * 40 + (size_t)(m->n - m->nl) * 8;
  if (lds <= 60 * 1024) {  // two workgroups per CU
    hipLaunchKernelGGL(adjoint_rows_kernel<false>, dim3(plan.grid), dim3(kNT), lds, s, a);
  } else {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(adjoint_rows_kernel<true>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)codes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(adjoint_rows_kernel<true>, dim3(plan.grid), dim3(kNT), codes, s, a);
  }
  return hipGetLastError();
}
