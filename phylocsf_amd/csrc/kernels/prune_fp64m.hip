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
  // 64-column blocks of work.  While the row-split kernel finds a place for every
  // 16 columns at once (two workgroups per CU: half a block per CU) it is the
  // faster one; beyond, the generated program, which reads P once per 64 columns.
  // us a forward at 64 / 128 / 160 / 256 / 512 / 1000 blocks on 256 CUs, row-split against
  // generated: 12flies 39 / 47 / 57 / 60 / 91 / 164 against 51 / 53 / 53 / 55 / 78 / 139,
  // 58mammals 82 / 122 / 182 / 193 / 349 / 663 against 154 / 161 / 163 / 173 / 292 / 562,
  // 120mammals 142 / 217 / 409 / 423 / 800 / 1507 against 303 / 310 / 318 / 335 / 577 / 1100.
  // With a set per region and many short regions, bound by the sets, the two are
  // within 5% of each other from 100 blocks on.
  const int64_t blocks = ch.work > 0 ? ch.work : ch.nblocks * m->nm;
  if (m->specialized && m->tree_p && blocks > cus / 2) {
    const auto* t = static_cast<const pcsf_mfma::TreeProgram*>(m->tree_p);
    if (t->fp64m) return t->fp64m(prm, 0, 0, cus, s);
  }
  return launch_fp64_rows(prm, blocks, m->slots, (int)(m->prog.size() / kOpWords / 2), cus, s);
}
