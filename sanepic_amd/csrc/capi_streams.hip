// capi_streams.hip -- detectors that share a line of sight.
//
// Detectors with the same focal-plane offsets cross the same pixels at the
// same times, and their polarisation angles differ by constants.  The
// operator of the reference filters every detector (write_tfAS and do_PtNd,
// sanepic.cc:2390-2637); P x of such a set is a combination of three streams
// with constant coefficients, and the noise filter is linear, so the set
// needs three forward and three inverse transforms, one gather and one set of
// run records however many detectors it holds (kernels.h SkyStream).  The
// products are the same sums in another order.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <map>
#include <vector>

#include "ctx.h"

using namespace sctx;

namespace sctx {

bool use_streams(const sanepic_ctx *c) {
  // the gather runs in the column pass, without gains; whole launches only
  // (use_runs is false otherwise)
  return c->nstream > 0 && use_runs(c);
}

static void free_streams(sanepic_ctx *c) {
  dfree(c, c->line_pix, (int64_t)c->nline * c->nseg * c->ns);
  dfree(c, c->d_streams, c->nstream);
  dfree(c, c->d_sdet, c->nsdet);
  dfree(c, c->d_sbeg, c->nset + 1);
  dfree(c, c->mix, 6 * (int64_t)c->nset * c->ns);
  dfree(c, c->mix32, 6 * (int64_t)c->nset * c->ns);
  c->nstream = c->nset = c->nline = 0;
}

// Finds the sets (equal offsets, and the same pixels sample by sample: a
// sample without pointing takes the pixel before it, which may be another
// detector's) at pixelisation, while c->pix holds compressed pixels.  Only
// orientations of at most 64 rad and no half-wave plate: the reference
// evaluates psi + psidet, and -psi + 2 Omega t (763-765) with t in samples,
// in FP64 per detector, so two detectors' angles differ by a constant only to
// the rounding of those sums (2e-12 in A x at 2^19 samples of a plate at
// 0.048 rad a sample, growing with t; below 1e-14 for the bounded angles).
// Sets of four or more detectors become three streams; every other detector
// stays a stream of its own, which costs it more than the usual passes: its
// records hold two idle sums (40 instead of 24 bytes a run in FP64) and its
// record pass batches its loads less, 1.3 to 1.4 times a detector's share of an
// FP64 iteration (10 sharing + 25, 4 x 2^17: 725 us with one stream each, 791
// shared; 16 + 48, 2 x 2^18: 1590 and 1645).  In FP64 a set pays where own
// detectors times 3/2 and its three streams stay below the number of detectors
// (16 + 25: 837 and 761; 8 + 9: 366 and 308).  Half the width of records and
// angles halves that surcharge: a mixed context shares when that leaves at most
// four streams for every five detectors (16 + 48: 1141 and 1082; 10 + 25: 526
// and 530).
int find_streams(sanepic_ctx *c) {
  if (!c->share || !c->runs || c->pin_owner || !c->sub.empty() || c->single || c->zsorted || c->nc != 3 || c->g.M != 1 ||
      c->pregather || c->recal || c->chunk != 0 || !c->ang64 || c->ndet < 4 || c->ndet > 65535 || c->ns % 16 != 0 ||
      c->cfg.hwp)
    return 0;
  std::map<std::pair<uint64_t, uint64_t>, std::vector<int32_t>> sight;
  std::vector<int32_t> lead((size_t)c->ndet);
  size_t largest = 0;
  for (int32_t d = 0; d < (int32_t)c->ndet; d++) {
    lead[(size_t)d] = d;
    uint64_t k[2];
    std::memcpy(&k[0], &c->offx[(size_t)d], 8);
    std::memcpy(&k[1], &c->offy[(size_t)d], 8);
    if (!(std::fabs(c->detc[(size_t)d].psidet) <= 64.0)) continue;
    auto &v = sight[{k[0], k[1]}];
    v.push_back(d);
    lead[(size_t)d] = v[0];
    largest = std::max(largest, v.size());
  }
  if (largest < 4) return 0;
  std::vector<int32_t> flag((size_t)c->ndet, 0);
  {
    int32_t *dl = nullptr, *df = nullptr;
    ACHK(c, dalloc(c, dl, c->ndet));
    ACHK(c, dalloc(c, df, c->ndet));
    HIPCHK(c, hipMemcpyAsync(dl, lead.data(), c->ndet * 4, hipMemcpyHostToDevice, c->st));
    HIPCHK(c, hipMemsetAsync(df, 0, c->ndet * 4, c->st));
    LCHK(c, launch_same_pixels(c->pix, c->nseg * c->ns, dl, c->ndet, df, c->st));
    ACHK(c, d2h(c, flag.data(), df, c->ndet * 4));
    dfree_later(c, dl, c->ndet);
    dfree_later(c, df, c->ndet);
  }
  std::vector<SkyStream> vs;
  std::vector<SkyDet> sdet;
  std::vector<int32_t> sbeg(1, 0);
  std::vector<char> taken((size_t)c->ndet, 0);
  int32_t line = 0;
  for (auto &e : sight) {
    std::vector<int32_t> dets;
    for (int32_t d : e.second)
      if (!flag[(size_t)d]) dets.push_back(d);
    if (dets.size() < 4) continue;
    for (int32_t d : dets) {
      const double delta = 2.0 * (c->detc[(size_t)d].psidet - c->detc[(size_t)dets[0]].psidet);
      sdet.push_back(SkyDet{d, 0, std::cos(delta), std::sin(delta)});
      taken[(size_t)d] = 1;
    }
    sbeg.push_back((int32_t)sdet.size());
    vs.push_back(SkyStream{dets[0], line, 1, 0, 0});
    vs.push_back(SkyStream{dets[0], line, 2, 1, 0});
    vs.push_back(SkyStream{dets[0], line, 2, 3, (uint64_t)1 << 62});
    line++;
  }
  const int32_t nset = line;
  for (int32_t d = 0; d < (int32_t)c->ndet; d++)
    if (!taken[(size_t)d]) vs.push_back(SkyStream{d, line++, 3, 0, 0});
  const int64_t nvs = (int64_t)vs.size(), nown = nvs - 3 * nset;
  if (nset == 0 || 5 * nvs > 4 * c->ndet) return 0;
  if (c->cfg.precision == SANEPIC_FP64 && 6 * nset + 3 * nown >= 2 * c->ndet) return 0;
  c->nstream = (int)vs.size();
  c->nset = nset;
  c->nline = line;
  c->nsdet = (int64_t)sdet.size();
  // line_pix: the lines' pixels [nline][nseg ns], from which the run layout is built
  if (dalloc(c, c->d_streams, c->nstream) || dalloc(c, c->d_sdet, c->nsdet) || dalloc(c, c->d_sbeg, nset + 1) ||
      dalloc(c, c->line_pix, (int64_t)line * c->nseg * c->ns)) {
    free_streams(c);  // no room for them: one stream per detector
    return 0;
  }
  HIPCHK(c, hipMemcpy(c->d_streams, vs.data(), vs.size() * sizeof(SkyStream), hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(c->d_sdet, sdet.data(), sdet.size() * sizeof(SkyDet), hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(c->d_sbeg, sbeg.data(), sbeg.size() * 4, hipMemcpyHostToDevice));
  std::vector<int32_t> first((size_t)line);
  for (const SkyStream &v : vs) first[(size_t)v.set] = v.det;
  const int64_t spd = c->nseg * c->ns;
  for (int32_t l = 0; l < line; l++)
    LCHK(c, launch_copy_i32(c->pix + first[(size_t)l] * spd, c->line_pix + l * spd, spd, c->st));
  return 0;
}

// Back to one stream per detector: relative calibration chosen after the
// pixelisation (its gains differ between the detectors of a set), or no room for
// the mixing weights.
int drop_streams(sanepic_ctx *c) {
  if (!c->nstream) return 0;
  HIPCHK(c, hipStreamSynchronize(c->st));
  const int64_t nl = (int64_t)c->nline * c->nseg * c->ns;
  dfree(c, c->rmeta, nl / 16);
  dfree(c, c->rperm, c->nrec);
  dfree(c, c->rec64, 5 * c->nrec);
  dfree(c, c->rec32, 5 * c->nrec);
  ItemSet &r = c->ritems;
  dfree(c, r.pix, r.items.n);
  dfree(c, r.beg, r.items.n);
  dfree(c, r.len, r.items.n);
  dfree(c, r.slot, r.items.n);
  dfree(c, r.sp_pix, r.items.nsplit);
  dfree(c, r.sp_first, r.items.nsplit);
  dfree(c, r.sp_count, r.items.nsplit);
  dfree(c, r.partial, 8 * std::max<int64_t>(1, r.nslots));
  c->ritems = ItemSet();
  c->nrec = 0;
  free_streams(c);
  ACHK(c, build_runs(c));
  return c->split_chosen ? 0 : set_split(c, default_split(c));
}

template <typename T>
int run_streams(sanepic_ctx *c, OpArgs<T> a, bool chi2, int64_t *nb) {
  a.vs = c->d_streams;
  a.nvs = c->nstream;
  a.nset = c->nset;
  a.sdet = c->d_sdet;
  a.sbeg = c->d_sbeg;
  if constexpr (sizeof(T) == 8) a.mix = c->mix;
  else a.mix = c->mix32;
  a.mode = ROW_FWD | ROW_FILTER | ROW_INV | (chi2 ? ROW_CHI2 : 0);
  a.rowdet = 1;
  {
    ProfScope ps(c, 0);
    LCHK(c, launch_col_fwd_streams<T>(a, c->st));
  }
  {
    ProfScope ps(c, 1);
    LCHK(c, launch_row_streams<T>(a, c->st, nb));
  }
  ProfScope ps(c, 2);
  LCHK(c, launch_col_inv_streams<T>(a, c->st));
  return 0;
}
template int run_streams<double>(sanepic_ctx *, OpArgs<double>, bool, int64_t *);
template int run_streams<float>(sanepic_ctx *, OpArgs<float>, bool, int64_t *);

}  // namespace sctx

int sanepic_streams(sanepic_ctx *c, int32_t *streams, int32_t *lines) {
  ACHK(c, check_ready(c, false));
  if (!streams || !lines) return fail(c, SANEPIC_EINVAL, "null output");
  const bool on = use_streams(c);
  *streams = on ? c->nstream : (int32_t)c->ndet;
  *lines = on ? c->nline : (int32_t)c->ndet;
  return SANEPIC_OK;
}
