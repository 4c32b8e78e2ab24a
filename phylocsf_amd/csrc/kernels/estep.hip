// estep.hip -- PhyloEM's expected substitution counts on FP64 matrix cores
// (collect_sufficient_statistics, lib/CamlPaml/PhyloEM.ml:14-20, over
// PhyloLik.add_branch_posteriors, lib/CamlPaml/PhyloLik.ml:140-174) for the
// 64-codon alphabet with `Certain and `Marginalize leaves (and states >= 64,
// the reference's vector of zeros).  Paths are relative to the mlin/PhyloCSF
// tree.
//
// estep_passes_kernel: per 64-column block (four waves of 16 columns, the
//   tiles of fp64_tiles.hpp), the inside pass (ensure_alpha, PhyloLik.ml:
//   73-93) keeps every internal node's message to its parent, m_c = P_c
//   alpha_c, then the outside pass (ensure_beta, :96-120) keeps beta_c =
//   P_c^T (beta_p o m_s) for the branch into internal child c of p with sibling
//   s; both as tiles in the accumulator layout, the nodes of 16 columns side by side.
// estep_counts_kernel: per branch, S = sum_col u v^T as a 64 x 64 product
//   over the chunk's columns on v_mfma_f64_16x16x4f64 (K = columns) with
//     u_c = w beta_p o m_s / z   (zero where beta_p <= 0 or z <= 0, the
//                                 entries the reference skips)
//     v_c = alpha_c = m_l o m_r  (a leaf's v is its leaf vector),
//   made from the tiles on the way into LDS, then ecounts_br += P_br o S -- the
//   branch posteriors xi = diag(u) P diag(v) summed over columns (:140-174)
//   without k^2 updates per column.
// Messages and betas are 58 KB a column on 58mammals and are written once, in
// runs of 512 bytes (u and v of every branch, which the passes used to write for
// the counts in 8-byte pieces, were 87 KB beside the messages' own 58): a chunk
// of 32,768 columns takes 1.03 ms in the passes (1.98 before; bound by memory
// and by the wait for each node's two messages) and 0.93 in the counts (1.0),
// whose workgroups wait for a tile's loads (2.5 TB/s, matrix cores 45% busy).
// Leaf messages come from a table per leaf branch (a column of P, its row sums
// for `Marginalize, zeros) in the order in which a lane reads them, states as
// bytes by leaf: both made once per call or chunk on the GPU.
#include "fp64_tiles.hpp"

namespace {

using namespace fp64t;

constexpr int kLeafMsgs = 66;             // per leaf branch: 64 codons, 64 `Marginalize, 65 zeros
constexpr int kLeafTable = kLeafMsgs * 64;

// the message of a leaf from its branch's table (row 16 mo + 4 v + g of message
// c at c * 64 + 16 mo + 4 g + v)
__device__ __forceinline__ Tile leaf_message(const double* __restrict__ L, int c, int grp) {
  const double2* src = reinterpret_cast<const double2*>(L + c * 64 + 4 * grp);
  Tile t;
#pragma unroll
  for (int mo = 0; mo < 4; ++mo)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const double2 d = src[8 * mo + h];
      t.r[mo][2 * h] = d.x;
      t.r[mo][2 * h + 1] = d.y;
    }
  return t;
}

__global__ __launch_bounds__(64 * kWaves, 2) void estep_passes_kernel(EstepArgs p) {
  // P_c or P_c^T in A-fragment order, double-buffered: product k of a block
  // (p.seq[k]) reads buffer k & 1 while product k + 1's tile is copied into
  // the other
  __shared__ __attribute__((aligned(16))) double Af[2][4096];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63,
            grp = lane >> 4;
  const int j = lane & 15;
  const int n = p.n, nl = p.nl;
  const int64_t nblocks = (p.ncols + kCols - 1) / kCols;
  auto issue = [&](int k) {  // product k's tile into buffer k & 1
    if (k >= p.nseq) return;
    const int code = p.seq[k];
    const double* src = (code >= 0) ? p.Pf + (size_t)code * 4096 : p.PTf + (size_t)(-1 - code) * 4096;
    copy_tile((L3*)&Af[k & 1][0], src, wave, tid);
  };
  for (int64_t blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
    __syncthreads();  // the previous block is done with both buffers
    issue(0);
    int kp = 0;  // products done in this block
    const int64_t tile = blk * kWaves + wave, col = tile * 16 + j;
    const bool valid = col < p.ncols;
    double* M = p.M + (size_t)tile * (n - nl) * kTileDoubles;
    double* B = p.B + (size_t)tile * (n - nl) * kTileDoubles;
    auto msg = [&](int c) -> Tile {
      return (c < nl) ? leaf_message(p.Lm + (size_t)c * kLeafTable,
                                     p.codes[(size_t)c * p.ldu + col], grp)
                      : load(M + (size_t)(c - nl) * kTileDoubles, lane);
    };
    // ---- inside pass (PhyloLik.ml:73-93)
    double z = 0.0;
    for (int i = nl; i < n; ++i) {
      Tile a = msg(p.lc[i]);
      const Tile mr = msg(p.rc[i]);
#pragma unroll
      for (int mo = 0; mo < 4; ++mo) a.r[mo] *= mr.r[mo];  // alpha_i
      if (i == n - 1) {
        Tile pr;
#pragma unroll
        for (int mo = 0; mo < 4; ++mo)
#pragma unroll
          for (int v = 0; v < 4; ++v) pr.r[mo][v] = p.prior[16 * mo + 4 * v + grp];
        z = column_dot(a, pr);
        break;
      }
      __syncthreads();  // P_i landed; the other buffer is no longer read
      issue(kp + 1);
      store(M + (size_t)(i - nl) * kTileDoubles, gemm(Af[kp & 1], a, lane), lane);
      ++kp;
    }
    if (grp == 0) {
      const double w = valid ? (p.weights ? p.weights[col] : 1.0) : 0.0;
      p.scale[col] = (valid && z > 0.0) ? w / z : 0.0;
      if (valid) p.z[col] = z;
    }
    // ---- outside pass (PhyloLik.ml:96-120), parents before children
    for (int pn = n - 1; pn >= nl; --pn) {
      const int kid[2] = {p.lc[pn], p.rc[pn]};
      if (kid[0] < nl && kid[1] < nl) continue;
      Tile bp;
      if (pn == n - 1) {
#pragma unroll
        for (int mo = 0; mo < 4; ++mo)
#pragma unroll
          for (int v = 0; v < 4; ++v) bp.r[mo][v] = p.prior[16 * mo + 4 * v + grp];
      } else {
        bp = load(B + (size_t)(pn - nl) * kTileDoubles, lane);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int c = kid[s];
        if (c < nl) continue;
        Tile wt = msg(kid[1 - s]);  // beta_p o m_sibling
#pragma unroll
        for (int mo = 0; mo < 4; ++mo) wt.r[mo] *= bp.r[mo];
        __syncthreads();  // P_c^T landed; the other buffer is no longer read
        issue(kp + 1);
        store(B + (size_t)(c - nl) * kTileDoubles, gemm(Af[kp & 1], wt, lane), lane);
        ++kp;
      }
    }
  }
}

// ecounts_br += P_br o sum_col u v^T over the chunk's column tiles.  Workgroup
// (branch, split) takes the split's share of the tiles.  Of a tile, wave w makes
// rows 16 w .. 16 w + 15 of u and v (lane (j, g), element v: row 16 w + 4 v + g
// of column j, as the tiles lie in memory) while the tile before it is
// multiplied; they go through LDS (rows of 16 columns, 18 doubles apart), where
// lane (i, k) reads columns 2 k, 2 k + 1 (+ 8) of a row: two K-steps in 16 bytes.
// Wave w multiplies its own rows of u with all of v (four 16 x 16 accumulators)
// and adds P o its sums with FP64 atomics (P o S is linear in S).
constexpr int kRow = 18;  // doubles between rows in LDS
__global__ __launch_bounds__(256, 3) void estep_counts_kernel(EstepArgs p, double* ecounts) {
  __shared__ __attribute__((aligned(16))) double X[2][2][64 * kRow];  // [buffer][u, v][row]
  const int c = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, g = lane >> 4;
  const int nl = p.nl, up = p.parent[c], sib = p.lc[up] == c ? p.rc[up] : p.lc[up];
  const int64_t nin = p.n - nl, used = (p.ncols + 15) / 16;
  const int64_t per = (used + gridDim.y - 1) / gridDim.y;
  const int64_t tb = per * blockIdx.y, te = std::min<int64_t>(used, tb + per);
  if (tb >= te) return;
  f64x4 prior;
#pragma unroll
  for (int v = 0; v < 4; ++v) prior[v] = p.prior[16 * w + 4 * v + g];
  const int a0 = c >= nl ? p.lc[c] : 0, a1 = c >= nl ? p.rc[c] : 0;  // below c
  // this lane's rows of the message of node b (code: a leaf's)
  auto msg = [&](int b, int code, int64_t t) -> f64x4 {
    f64x4 m;
    if (b < nl) {
      const double2* src = reinterpret_cast<const double2*>(p.Lm + (size_t)b * kLeafTable +
                                                            code * 64 + 16 * w + 4 * g);
      const double2 x = src[0], y = src[1];
      m = (f64x4){x.x, x.y, y.x, y.y};
    } else {
      const double* src = p.M + (t * nin + (b - nl)) * kTileDoubles + w * 256 + lane;
#pragma unroll
      for (int v = 0; v < 4; ++v) m[v] = src[64 * v];
    }
    return m;
  };
  // Leaf codes are read a tile before the messages that they select: in one
  // fetch the wave would wait for a code, and for all loads before it, in front
  // of its products.
  int ks = 0, k0 = 0, k1 = 0, kc = 0;
  auto codes = [&](int64_t t) {
    auto of = [&](int b) { return p.codes[(size_t)b * p.ldu + t * 16 + j]; };
    if (sib < nl) ks = of(sib);
    if (c < nl) {
      kc = of(c);
    } else {
      if (a0 < nl) k0 = of(a0);
      if (a1 < nl) k1 = of(a1);
    }
  };
  f64x4 bp = prior, ms, x0, x1;
  double sc = 0.0;
  int code = 0;
  auto fetch = [&](int64_t t) {  // with the codes of tile t; then those of t + 1
    if (up != p.n - 1) {
      const double* src = p.B + (t * nin + (up - nl)) * kTileDoubles + w * 256 + lane;
#pragma unroll
      for (int v = 0; v < 4; ++v) bp[v] = src[64 * v];
    }
    ms = msg(sib, ks, t);
    sc = p.scale[t * 16 + j];
    if (c >= nl) {
      x0 = msg(a0, k0, t);
      x1 = msg(a1, k1, t);
    } else {
      code = kc;
    }
    if (t + 1 < te) codes(t + 1);
  };
  f64x4 acc[4];
#pragma unroll
  for (int no = 0; no < 4; ++no) acc[no] = (f64x4){0.0, 0.0, 0.0, 0.0};
  codes(tb);
  fetch(tb);
  for (int64_t t = tb; t < te; ++t) {
    double(*buf)[64 * kRow] = X[(t - tb) & 1];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * w + 4 * v + g;
      buf[0][row * kRow + j] = bp[v] > 0.0 ? bp[v] * ms[v] * sc : 0.0;
      // a column without a scale (past the last, or z <= 0) adds nothing
      buf[1][row * kRow + j] = c >= nl ? x0[v] * x1[v] : (code == row || code == 64) ? 1.0 : 0.0;
    }
    if (t + 1 < te) fetch(t + 1);
    // rows of the other waves are in; a wave is at most one tile ahead, in the
    // other buffer
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = (lane & 15) * kRow + 8 * h + 2 * g;
      const double2 a = *reinterpret_cast<const double2*>(&buf[0][16 * w * kRow + at]);
#pragma unroll
      for (int no = 0; no < 4; ++no) {
        const double2 b = *reinterpret_cast<const double2*>(&buf[1][16 * no * kRow + at]);
        acc[no] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, acc[no], 0, 0, 0);
        acc[no] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, acc[no], 0, 0, 0);
      }
    }
  }
  // acc[no][v] of lane i + 16 g: S[16 w + 4 v + g][16 no + i]
  const double* Pb = p.P + (size_t)c * 4096;
  double* E = ecounts + (size_t)c * 4096;
#pragma unroll
  for (int no = 0; no < 4; ++no)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int a = 16 * w + 4 * v + g, b = 16 * no + j;
      atomicAdd(E + a * 64 + b, Pb[a * 64 + b] * acc[no][v]);
    }
}

// P and P^T of every branch into the A-fragment order of fp64_tiles.hpp:
// M[row][col] at ((row / 16) * 16 + col / 4) * 64 + row % 16 + 16 (col % 4);
// of a leaf branch its table of messages.
__global__ __launch_bounds__(256) void estep_frags_kernel(const double* __restrict__ P, int nl,
                                                          double* __restrict__ Pf,
                                                          double* __restrict__ PTf,
                                                          double* __restrict__ Lm) {
  __shared__ double sums[64];
  const int br = blockIdx.x, tid = threadIdx.x;
  const double* src = P + (size_t)br * 4096;
  if (br >= nl) {
    for (int e = tid; e < 4096; e += 256) {
      const int row = e >> 6, col = e & 63;
      const int f = ((row >> 4) * 16 + (col >> 2)) * 64 + (row & 15) + 16 * (col & 3);
      Pf[(size_t)br * 4096 + f] = src[row * 64 + col];   // M = P
      PTf[(size_t)br * 4096 + f] = src[col * 64 + row];  // M = P^T
    }
    return;
  }
  if (tid < 64) {
    double t = 0.0;
    for (int b = 0; b < 64; ++b) t += src[tid * 64 + b];
    sums[tid] = t;
  }
  __syncthreads();
  double* out = Lm + (size_t)br * kLeafTable;
  for (int e = tid; e < kLeafTable; e += 256) {
    const int c = e >> 6, k = e & 63, row = (k & 48) + 4 * (k & 3) + ((k >> 2) & 3);
    out[e] = c < 64 ? src[row * 64 + c] : c == 64 ? sums[row] : 0.0;
  }
}

// States of a chunk's columns (ncols x nl) as bytes by leaf (nl x ldu): the
// message to read of the leaf's table; zeros past the last column.
__global__ __launch_bounds__(256) void estep_codes_kernel(const int32_t* __restrict__ leaves,
                                                          int nl, int64_t ncols, int64_t ldu,
                                                          uint8_t* __restrict__ codes) {
  const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;  // (four columns, leaf)
  if (e >= (int64_t)nl * (ldu / 4)) return;
  const int64_t c0 = e / nl * 4;
  const int l = (int)(e - c0 / 4 * nl);
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int32_t x = c0 + i < ncols ? leaves[(size_t)(c0 + i) * nl + l] : 64;
    word |= (x < 0 ? 64u : x < 64 ? (uint32_t)x : 65u) << (8 * i);
  }
  *reinterpret_cast<uint32_t*>(codes + (size_t)l * ldu + c0) = word;
}

}  // namespace

size_t estep_leaf_table_doubles() { return kLeafTable; }

hipError_t launch_estep_frags(const double* P, int nl, int nbr, double* Pf, double* PTf,
                              double* Lm, hipStream_t s) {
  if (nbr <= 0) return hipSuccess;
  hipLaunchKernelGGL(estep_frags_kernel, dim3(nbr), dim3(256), 0, s, P, nl, Pf, PTf, Lm);
  return hipGetLastError();
}

std::vector<int32_t> estep_sequence(int n, const std::vector<int32_t>& lc,
                                    const std::vector<int32_t>& rc) {
  const int nl = (n + 1) / 2;
  std::vector<int32_t> seq;
  for (int i = nl; i < n - 1; ++i) seq.push_back(i);  // inside: P_i, nodes in order
  for (int pn = n - 1; pn >= nl; --pn)                // outside: P_c^T, internal children
    for (int c : {lc[pn], rc[pn]})
      if (c >= nl) seq.push_back(-1 - c);
  return seq;
}

hipError_t launch_estep(const EstepArgs& a, const int32_t* leaves, double* ecounts, int num_cus,
                        hipStream_t s) {
  if (a.ncols <= 0) return hipSuccess;
  const int64_t nblocks = (a.ncols + kCols - 1) / kCols;
  if (nblocks * kCols > a.ldu || a.ldu % kCols) return hipErrorInvalidValue;
  const int64_t words = a.nl * (a.ldu / 4);
  hipLaunchKernelGGL(estep_codes_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s,
                     leaves, a.nl, a.ncols, a.ldu, a.codes);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // two workgroups per CU (LDS)
  const int g = (int)std::min<int64_t>(nblocks, 2 * num_cus);
  hipLaunchKernelGGL(estep_passes_kernel, dim3(g), dim3(64 * kWaves), 0, s, a);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  // splits of the columns per branch: enough workgroups to fill the device (three
  // per CU) eight times over, so that the last round is a small part (16 splits,
  // two and a half rounds on 58mammals: 1.04 ms against 0.93)
  const int splits = (int)std::max<int64_t>(
      1, std::min<int64_t>({64, nblocks, (24 * num_cus + a.n - 2) / (a.n - 1)}));
  hipLaunchKernelGGL(estep_counts_kernel, dim3(a.n - 1, splits), dim3(256), 0, s, a, ecounts);
  return hipGetLastError();
}
