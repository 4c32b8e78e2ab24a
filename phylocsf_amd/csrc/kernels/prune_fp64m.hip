// prune_fp64m.hip -- launcher of the FP64 forward on matrix cores: the
// tree's generated program (prune_fp64m.hpp) where it has one and the columns
// fill the device, the row-split kernel (prune_fp64r.hip) otherwise.
#include "prune_tree.hpp"

using pcsf_mfma::MfmaParams;

hipError_t launch_forward_fp64m(const pcsf_model* m, const pcsf_batch* b, const RegionChunk& ch,
                                hipStream_t s) {
  if (!ch.sets->d_P64F) return hipErrorInvalidValue;
  MfmaParams prm{};
  prm.codes = b->al.d_codes;
  prm.ld = b->al.ld;
  prm.g0 = ch.block0;  // one group of kGC = kAlignCols columns per block
  prm.ngroups = ch.nblocks;
  prm.nl = m->nl;
  prm.nm = m->nm;
  prm.nbr = m->nbr;
  prm.first_gemm_br = m->first_gemm_br;
  prm.prog = m->d_prog;
  prm.pi = ch.sets->d_epi ? ch.sets->d_epi : m->d_pi;
  prm.lnpi = ch.sets->d_epi ? ch.sets->d_elnpi : m->d_lnpi;
  prm.prior_per_set = ch.sets->d_epi ? 1 : 0;
  prm.logz = b->d_alogz;
  prm.colelpr = b->d_acolelpr;
  prm.block_region = b->al.d_block_region;
  prm.active = ch.sets->d_active;
  prm.r0 = ch.r0;
  prm.shared_sets = ch.sets == &m->fixed ? 1 : 0;
  prm.P64F = ch.sets->d_P64F;
  prm.astart = b->al.d_astart;
  prm.off = b->d_offsets;
  if (prm.ngroups == 0) return hipSuccess;
  const int cus = m->ctx->num_cus;
  // 64-column blocks of work.  Up to four per CU the row-split kernel is the
  // faster one (58mammals: 251 against 285 us at 366 blocks, 529 against 556
  // at 772), above it the generated program, which reads P once per 64
  // columns (898 against 850 us at 1520 blocks, 3619 against 3207 at 6214).
  const int64_t blocks = ch.work > 0 ? ch.work : ch.nblocks * m->nm;
  if (m->specialized && m->tree_p && blocks > 4 * (int64_t)cus) {
    const auto* t = static_cast<const pcsf_mfma::TreeProgram*>(m->tree_p);
    if (t->fp64m) return t->fp64m(prm, 0, 0, cus, s);
  }
  return launch_fp64_rows(prm, blocks, m->slots, (int)(m->prog.size() / kOpWords / 2), cus, s);
}
