// The state that a failed sanepic_set_recalib leaves, on a device that has no
// memory left (the HIP calls below stand in for the runtime's).
#include "fake_hip.h"

int main() {
  sanepic_ctx c;
  c.ndet = 5;
  c.nseg = 2;
  c.ns = 8192;
  c.ntot = c.ndet * c.nseg * c.ns;
  c.nc = 3;
  c.g.M = 1;
  c.g.log2N1 = 9;
  c.g.log2N2 = 4;
  c.npix = 100;
  c.pixelized = true;
  c.nrec = 1000;
  CHECK(sctx::use_runs(&c) && !sctx::use_streams(&c));
  c.nstream = 3;  // records of a shared line of sight
  c.nset = c.nline = 1;
  CHECK(sctx::use_runs(&c) && sctx::use_streams(&c));
  // a layout for streams never reaches the passes of one stream per detector
  for (int k = 0; k < 3; k++) {
    c.recal = k == 0;
    c.pregather = k == 1;
    c.chunk = k == 2;
    CHECK(!sctx::use_runs(&c) && !sctx::use_streams(&c));
  }
  c.recal = c.pregather = false;
  c.chunk = 0;
  fake::room = 0;
  CHECK(sanepic_set_recalib(&c, 1) == SANEPIC_ENOMEM);
  CHECK(!c.recal && sctx::use_streams(&c));
  // with memory for the gains only: the streams are gone, and so is their layout
  fake::room = 4096;
  CHECK(sanepic_set_recalib(&c, 1) == SANEPIC_ENOMEM);
  CHECK(!c.recal && c.nstream == 0 && !sctx::use_runs(&c) && !sctx::use_streams(&c));
  std::puts("ok");
  return 0;
}
