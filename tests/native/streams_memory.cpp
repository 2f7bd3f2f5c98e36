// Shared lines of sight on a device without room for them: the context keeps
// one stream per detector instead of failing.
#include "fake_hip.h"

static void fill(sanepic_ctx &c) {
  c.ndet = 4;
  c.nseg = 2;
  c.ns = 8192;
  c.ntot = c.ndet * c.nseg * c.ns;
  c.nc = 3;
  c.g.M = 1;
  c.g.log2N = 13;
  c.g.log2N1 = 9;
  c.g.log2N2 = 4;
  c.g.N = c.ns;
  c.g.N1 = 512;
  c.g.N2 = 16;
  c.g.ppd = 1;
  c.g.npairs = 4;
  c.g.nseg = 2;
  c.gauto = c.g;
  c.gauto.nseg = 1;
  c.offx.assign(4, 0.1);
  c.offy.assign(4, 0.2);
  c.detc.resize(4);
  for (int d = 0; d < 4; d++) c.detc[(size_t)d].psidet = 0.3 * d;
  c.spn.assign((size_t)(4 * (c.ns / 2 + 1)), 1.0);
  c.pix = (int32_t *)((uintptr_t)1 << 43);  // never read: launches do nothing here
  c.ang64 = (uint64_t *)((uintptr_t)1 << 43);
  c.pixelized = true;
}

int main() {
  using namespace sctx;
  const size_t line_pix = 2 * 8192 * 4, mix = 6 * 8192 * 8;
  fake::room = int64_t(1) << 32;
  {  // found where there is room
    sanepic_ctx c;
    fill(c);
    CHECK(find_streams(&c) == 0 && c.nstream == 3 && c.nset == 1 && c.nline == 1);
    c.nrec = 1;  // as built
    CHECK(use_streams(&c));
    CHECK(setup_pointing(&c) == 0 && c.mix && c.nstream == 3);
  }
  {  // no room for the line's pixels
    sanepic_ctx c;
    fill(c);
    fake::refuse = line_pix;
    CHECK(find_streams(&c) == 0 && c.nstream == 0 && c.nset == 0 && !c.line_pix && !c.d_streams && !c.d_sdet &&
          !c.d_sbeg);
    fake::refuse = 0;
  }
  {  // no room for the mixing weights
    sanepic_ctx c;
    fill(c);
    CHECK(find_streams(&c) == 0 && c.nstream == 3);
    c.nrec = 1;
    fake::refuse = mix;
    CHECK(setup_pointing(&c) == 0 && c.nstream == 0 && !c.mix && c.wt && !use_streams(&c));
    fake::refuse = 0;
  }
  std::puts("ok");
  return 0;
}
