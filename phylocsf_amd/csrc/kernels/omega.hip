// omega.hip -- the omega test's rate models on the GPU, one per set (region,
// hypothesis) of a chunk, rebuilt at every lock-step evaluation from the
// set's twelve settings (kappa, omega, sigma, nine F3x4 frequency ratios):
//
//   pi   codon frequencies, the stops' share scaled by sigma
//        (src/OmegaModel.ml:24-40)
//   S    exchangeabilities: one nucleotide apart, kappa on transitions, omega
//        on nonsynonymous changes between sense codons (:42-74)
//   Q    q_ij = s_ij pi_j / scale, scale = -sum_i pi_i q_ii (the mean-rate
//        normalisation of P14n.instantiate_q, lib/CamlPaml/P14n.ml)
//   eigensystem of Q through the symmetric A = Pi^1/2 Q Pi^-1/2 by cyclic
//        Jacobi rotations in parallel order (Golub & Van Loan, Matrix
//        Computations, sec. 8.5: the round-robin ordering applies 32 disjoint
//        rotations at once, 63 rounds per sweep), until the off-diagonal mass
//        is below 1e-30 of the total or stops falling (it converges
//        quadratically to a rounding floor near 1e-31: eight sweeps for the
//        omega models), at most 64 sweeps; V = Pi^-1/2 U and V^-1 = U^T Pi^1/2.
//        A cold build also stores U as the set's reference basis U0; a later
//        build of the same set with the same pi (kappa or omega changed)
//        starts from it: A' = U0^T A U0 is near-diagonal, the rotations go on
//        from U = U0, and the stopping rule is unchanged (a few sweeps instead
//        of eight; Golub & Van Loan on Jacobi for nearby matrices).  Starting
//        from the fixed U0, not from the previous build, keeps the result a
//        function of the settings and U0's (the fit's starting point), not of
//        the path between them.  A set whose settings did not change keeps its
//        eigensystem.
//
// One 512-thread workgroup per set, A and U in LDS (rows padded to 65
// doubles).  A round is a serial chain (32 rotations from A, their update of
// A, the next 32 rotations), so what bounds the kernel is that chain's latency:
// * A <- J^T (A J) in one step: the 2 x 2 block of rows (p, q) and columns
//   (p', q') of two pairs is read, rotated by columns, then by rows, and
//   written by one thread (columns first, as two separate passes did);
// * U <- U J, which the chain does not wait for, runs on waves 1-7 while wave
//   0 makes the next round's rotations (two divisions, two square roots and a
//   reciprocal, about half of the chain);
// so a round has two barriers and one trip of A through LDS (three barriers,
// two trips and 256 threads before).  The multiply-adds are spelled out: the
// rounding of a rotation is part of the fit's path.
// Outputs in the sets' own-model layout: V transposed, V^-1, the eigenvalues,
// the normalised root prior and its log.  Paths are relative to the
// mlin/PhyloCSF tree.
#include "../internal.hpp"

namespace {

constexpr int kLd = 65;  // LDS row stride of A and U (doubles)
constexpr int kNT = 512;
typedef double f64x4 __attribute__((ext_vector_type(4)));

// Code.Codon64 amino acids (lib/CamlPaml/Code.ml:153-173); stops TAA, TAG, TGA
__constant__ char kAmino[65] = "KNKNTTTTRSRSIIMIQHQHPPPPRRRRLLLLEDEDAAAAGGGGVVVV*Y*YSSSS*CWCLFLF";
constexpr int kTAA = 48, kTAG = 50, kTGA = 56;

__device__ __forceinline__ bool stop_codon(int c) { return c == kTAA || c == kTAG || c == kTGA; }

// s_ij of the omega model (0 unless i, j are one nucleotide apart)
__device__ __forceinline__ double exchangeability(const double* qs, int i, int j) {
  const int d = i ^ j;
  int field = -1;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    if (d == (d & (3 << (2 * p)))) field = p;
  if (d == 0 || field < 0) return 0.0;
  const int x = (i >> (2 * field)) & 3, y = (j >> (2 * field)) & 3;
  const double kp = ((x ^ y) == 2) ? qs[0] : 1.0;  // A <-> G, C <-> T
  const double op = (!stop_codon(i) && !stop_codon(j) && kAmino[i] != kAmino[j]) ? qs[1] : 1.0;
  return kp * op;
}

// (x, y) <- (c x - s y, s x + c y)
__device__ __forceinline__ void rotate(double c, double s, double& x, double& y) {
  const double a = fma(c, x, -(s * y));
  y = fma(s, x, c * y);
  x = a;
}

// sum over 256 partials (thread t < 256 holds part), the tree t + (t + 128),
// ..., t + (t + 1): the same in every thread
__device__ __forceinline__ double sum256(double part, double* red, double* out, int tid) {
  if (tid < 256) red[tid] = part;
  __syncthreads();
  if (tid < 64) {
    double v = (red[tid] + red[tid + 128]) + (red[tid + 64] + red[tid + 192]);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w);
    if (tid == 0) *out = v;
  }
  __syncthreads();
  return *out;
}

// One 64 x 64 product of LDS matrices on the matrix cores into registers: wave
// w makes tiles 2 w and 2 w + 1 of the 4 x 4 tiles of 16 x 16; left(i, l) and
// right(l, j) address the operands.
template <class L, class R>
__device__ __forceinline__ void product(f64x4 (&t)[2], int tid, L left, R right) {
  const int lane = tid & 63, w = tid >> 6, i = lane & 15, k = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int mo = (2 * w + h) >> 2, no = (2 * w + h) & 3;
    t[h] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int s = 0; s < 16; ++s)
      t[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(left(16 * mo + i, 4 * s + k),
                                                  right(4 * s + k, 16 * no + i), t[h], 0, 0, 0);
  }
}
__device__ __forceinline__ void put(double* A, const f64x4 (&t)[2], int tid) {
  const int lane = tid & 63, w = tid >> 6, i = lane & 15, k = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int mo = (2 * w + h) >> 2, no = (2 * w + h) & 3;
#pragma unroll
    for (int v = 0; v < 4; ++v) A[(16 * mo + 4 * v + k) * kLd + 16 * no + i] = t[h][v];
  }
}

// mode per set: kEigCold builds from scratch and stores U in ref (64 x 64
// per set), kEigWarm starts from ref, kEigKeep leaves the outputs (unchanged
// settings, or an inactive set)
__global__ __launch_bounds__(kNT, 4) void omega_eigen_kernel(
    const double* __restrict__ qs_all, const uint8_t* __restrict__ mode, double* __restrict__ ref,
    double* __restrict__ VT, double* __restrict__ Vinv, double* __restrict__ lam,
    double* __restrict__ pi_out, double* __restrict__ lnpi_out) {
  __shared__ double A[64 * kLd], U[64 * kLd];
  __shared__ double pi[64], sq[64], diag[64];
  __shared__ double cs[2][32], sn[2][32];  // a round's rotations and the next one's
  __shared__ int pp[2][32], qq[2][32];
  __shared__ double red[256];
  __shared__ double sum_s, scale_s;
  const int set = blockIdx.x, tid = threadIdx.x;
  const int md = mode[set];
  if (md == kEigKeep) return;  // uniform over the workgroup
  const double* qs = qs_all + (size_t)set * 12;
  // codon frequencies (OmegaModel.ml:24-40)
  if (tid < 64) {
    double f[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const double* r = qs + 3 + 3 * p;
      const double tot = r[0] + (r[1] + (r[2] + 1.0));
      const int n = (tid >> (2 * (2 - p))) & 3;
      f[p] = (n == 3 ? 1.0 : r[n]) / tot;
    }
    pi[tid] = f[0] * (f[1] * f[2]);  // sc[c], divided by the stop factor below
  }
  __syncthreads();
  if (tid == 0) {
    const double denom = 1.0 - (1.0 - qs[2]) * (pi[kTAA] + (pi[kTAG] + pi[kTGA]));
    red[0] = denom;
  }
  __syncthreads();
  if (tid < 64) {
    pi[tid] = pi[tid] / red[0];
    sq[tid] = sqrt(pi[tid]);
  }
  __syncthreads();
  // Q's off-diagonal into A (row i: s_ij pi_j), its diagonal -sum_j q_ij in
  // the host's order, then the mean-rate scale
  for (int e = tid; e < 4096; e += kNT) {
    const int i = e >> 6, j = e & 63;
    A[i * kLd + j] = (i == j) ? 0.0 : exchangeability(qs, i, j) * pi[j];
  }
  __syncthreads();
  if (tid < 64) {
    double off = 0.0;
    for (int j = 0; j < 64; ++j)
      if (j != tid) off = A[tid * kLd + j] + off;
    diag[tid] = 0.0 - off;
  }
  __syncthreads();
  if (tid == 0) {
    double scale = 0.0;
    for (int i = 0; i < 64; ++i)
      if (diag[i] != 0.0) scale = scale - pi[i] * diag[i];
    scale_s = scale;
  }
  __syncthreads();
  const double scale = scale_s;
  // A = Pi^1/2 Q Pi^-1/2 symmetrised (the host's formula), U = I; the total
  // squared mass for the stopping rule
  for (int e = tid; e < 4096; e += kNT) {
    const int i = e >> 6, j = e & 63;
    const double qij = ((i == j) ? diag[i] : A[i * kLd + j]) / scale;
    const double qji = ((i == j) ? diag[i] : A[j * kLd + i]) / scale;
    U[i * kLd + j] = 0.5 * (sq[i] * qij / sq[j] + sq[j] * qji / sq[i]);
  }
  __syncthreads();
  double* vt = VT + (size_t)set * 4096;
  double* vi = Vinv + (size_t)set * 4096;
  double* u0 = ref + (size_t)set * 4096;
  double part = 0.0;
  if (tid < 256)
    for (int e = tid; e < 4096; e += 256) {
      const double x = U[(e >> 6) * kLd + (e & 63)];
      part = fma(x, x, part);
    }
  const double total = sum256(part, red, &sum_s, tid);
  for (int e = tid; e < 4096; e += kNT) {
    const int i = e >> 6, j = e & 63;
    A[i * kLd + j] = U[i * kLd + j];
    U[i * kLd + j] = (md == kEigWarm) ? u0[e] : (i == j) ? 1.0 : 0.0;
  }
  if (md == kEigWarm) {
    // A <- U0^T (A U0), each product through registers so that no third LDS
    // matrix is needed
    f64x4 t[2];
    __syncthreads();
    product(t, tid, [&](int i, int l) { return A[i * kLd + l]; },
            [&](int l, int j) { return U[l * kLd + j]; });
    __syncthreads();
    put(A, t, tid);
    __syncthreads();
    product(t, tid, [&](int i, int l) { return U[l * kLd + i]; },
            [&](int l, int j) { return A[l * kLd + j]; });
    __syncthreads();
    put(A, t, tid);
    __syncthreads();
    for (int e = tid; e < 4096; e += kNT) {  // symmetric up to rounding: the mean
      const int i = e >> 6, j = e & 63;
      if (i >= j) continue;
      const double m = 0.5 * (A[i * kLd + j] + A[j * kLd + i]);
      A[i * kLd + j] = m;
      A[j * kLd + i] = m;
    }
  }
  __syncthreads();
  // the 32 rotations of a round into buffer b (round-robin pairing: 63 fixed,
  // the others on a circle)
  auto rotations = [&](int round, int b) {
    int i, j;
    if (tid == 0) {
      i = 63;
      j = round;
    } else {
      i = round + tid;
      j = round - tid;
      i = i >= 63 ? i - 63 : i;
      j = j < 0 ? j + 63 : j;
    }
    const int p = min(i, j), q = max(i, j);
    const double apq = A[p * kLd + q];
    double c = 1.0, s = 0.0;
    if (fabs(apq) >= 1e-300) {
      const double tau = (A[q * kLd + q] - A[p * kLd + p]) / (2.0 * apq);
      const double t = copysign(1.0, tau) / (fabs(tau) + hypot(1.0, tau));
      c = 1.0 / hypot(1.0, t);
      s = t * c;
    }
    pp[b][tid] = p;
    qq[b][tid] = q;
    cs[b][tid] = c;
    sn[b][tid] = s;
  };
  double prev = INFINITY;
  for (int sweep = 0; sweep < 64; ++sweep) {
    // off-diagonal mass
    double o = 0.0;
    if (tid < 256)
      for (int e = tid; e < 4096; e += 256) {
        const int i = e >> 6, j = e & 63;
        if (i != j) o = fma(A[i * kLd + j], A[i * kLd + j], o);
      }
    const double off = sum256(o, red, &sum_s, tid);
    const bool converged = !(off > 1e-30 * total) || !(off < prev);
    prev = off;
    if (converged) break;
    if (tid < 32) rotations(0, 0);
    __syncthreads();
    for (int round = 0; round < 63; ++round) {
      const int b = round & 1;
      // A <- J^T (A J): two 2 x 2 blocks per thread
      {
        const int k2 = tid & 31, p2 = pp[b][k2], q2 = qq[b][k2];
        const double c2 = cs[b][k2], s2 = sn[b][k2];
        double x[2], y[2], u[2], v[2];
        int p1[2], q1[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k1 = (tid >> 5) + 16 * h;
          p1[h] = pp[b][k1] * kLd;
          q1[h] = qq[b][k1] * kLd;
          x[h] = A[p1[h] + p2];
          y[h] = A[p1[h] + q2];
          u[h] = A[q1[h] + p2];
          v[h] = A[q1[h] + q2];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k1 = (tid >> 5) + 16 * h;
          const double c1 = cs[b][k1], s1 = sn[b][k1];
          rotate(c2, s2, x[h], y[h]);
          rotate(c2, s2, u[h], v[h]);
          rotate(c1, s1, x[h], u[h]);
          rotate(c1, s1, y[h], v[h]);
          A[p1[h] + p2] = x[h];
          A[p1[h] + q2] = y[h];
          A[q1[h] + p2] = u[h];
          A[q1[h] + q2] = v[h];
        }
      }
      __syncthreads();
      if (tid < 64) {
        if (tid < 32 && round + 1 < 63) rotations(round + 1, b ^ 1);
      } else {  // U <- U J (columns p, q of every pair), row = lane
        double* row = U + (tid & 63) * kLd;
        const int k0 = (tid >> 6) - 1;
        double x[5], y[5];
#pragma unroll
        for (int h = 0; h < 5; ++h) {
          const int k = min(k0 + 7 * h, 31);
          x[h] = row[pp[b][k]];
          y[h] = row[qq[b][k]];
        }
#pragma unroll
        for (int h = 0; h < 5; ++h) {
          const int k = k0 + 7 * h;
          if (k < 32) {  // (uniform over the wave)
            rotate(cs[b][k], sn[b][k], x[h], y[h]);
            row[pp[b][k]] = x[h];
            row[qq[b][k]] = y[h];
          }
        }
      }
      __syncthreads();
    }
  }
  // outputs: V^T[m][i] = U[i][m] / sq[i], V^-1[m][i] = U[i][m] sq[i]; a
  // cold build's U is the set's reference basis
  __syncthreads();
  for (int e = tid; e < 4096; e += kNT) {
    const int m = e >> 6, i = e & 63;
    const double u = U[i * kLd + m];
    vt[e] = u / sq[i];
    vi[e] = u * sq[i];
    if (md == kEigCold) u0[e] = U[(e >> 6) * kLd + (e & 63)];
  }
  if (tid < 64) lam[(size_t)set * 64 + tid] = A[tid * kLd + tid];
  if (tid == 0) {
    double tot = 0.0;
    for (int i = 0; i < 64; ++i) tot += pi[i];
    red[0] = tot;
  }
  __syncthreads();
  if (tid < 64) {
    const double pn = pi[tid] / red[0];
    pi_out[(size_t)set * 64 + tid] = pn;
    lnpi_out[(size_t)set * 64 + tid] = log(pn);
  }
}

}  // namespace

hipError_t launch_omega_eigen(int nsets, const PSets& sets, hipStream_t s) {
  if (nsets <= 0) return hipSuccess;
  hipLaunchKernelGGL(omega_eigen_kernel, dim3(nsets), dim3(kNT), 0, s, sets.d_qs, sets.d_mode, sets.d_eref,
                     sets.d_eVT, sets.d_eVinv, sets.d_elam, sets.d_epi, sets.d_elnpi);
  return hipGetLastError();
}
