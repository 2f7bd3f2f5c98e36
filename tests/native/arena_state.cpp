// What a context's slabs keep from the device: a detector group's buffers after
// their release, and requests that only fit once idle slabs are given back.
#include "fake_hip.h"

constexpr int64_t MB = int64_t(1) << 20;

struct Groups {
  sanepic_ctx parent, group;
  Groups() {
    parent.ntot = group.ntot = int64_t(1) << 24;
    group.pin_owner = &parent;
    parent.sub.push_back(&group);
  }
  ~Groups() { parent.arena.free_all(); }
};

int main() {
  using namespace sctx;
  fake::room = 4096 * MB;
  {  // a group's TOD goes back to the device, also when small buffers came after its release
    Groups g;
    char *tod = nullptr, *small = nullptr;
    CHECK(dalloc(&g.group, tod, 1024 * MB) == 0);
    dfree(&g.group, tod, 1024 * MB);
    int64_t n = 0;
    CHECK(sanepic_device_bytes(&g.parent, &n) == SANEPIC_OK && n == 1024 * MB && n == fake::held());
    CHECK(dalloc(&g.group, small, MB) == 0);
    g.parent.arena.trim();
    CHECK(fake::held() <= 256 * MB);
    CHECK(sanepic_device_bytes(&g.parent, &n) == SANEPIC_OK && n == MB);
    dfree(&g.group, small, MB);
    g.parent.arena.trim();
    CHECK(fake::held() == 0);
  }
  {  // the groups' temporaries serve the parent's large buffers
    Groups g;
    char *tmp = nullptr, *buf = nullptr;
    CHECK(dalloc(&g.group, tmp, 400 * MB) == 0);
    dfree_later(&g.group, tmp, 400 * MB);
    flush_frees(&g.group);
    const int64_t room = fake::room;
    fake::room = 0;
    CHECK(dalloc(&g.parent, buf, 300 * MB) == 0);
    fake::room = room;
    dfree(&g.parent, buf, 300 * MB);
  }
  {  // a request that fits only after idle slabs are given back
    Groups g;
    char *a = nullptr, *b = nullptr, *c = nullptr, *d = nullptr;
    CHECK(dalloc(&g.group, a, 300 * MB) == 0 && dalloc(&g.group, b, 300 * MB) == 0);
    dfree(&g.group, a, 300 * MB);
    dfree(&g.group, b, 300 * MB);
    const int64_t room = fake::room;
    fake::room = 0;
    CHECK(dalloc(&g.parent, c, 500 * MB) == 0);
    dfree(&g.parent, c, 500 * MB);
    CHECK(dalloc(&g.group, d, 590 * MB) == 0);
    dfree(&g.group, d, 590 * MB);
    char *e = nullptr;
    CHECK(dalloc(&g.parent, e, 700 * MB) == SANEPIC_ENOMEM && e == nullptr);
    g.parent.arena.trim();
    CHECK(fake::room == 600 * MB);
    fake::room = room + 600 * MB;
  }
  {  // temporaries kept past a set-up too
    sanepic_ctx c;
    c.ntot = int64_t(1) << 22;
    char *tmp = nullptr, *buf = nullptr;
    CHECK(dalloc(&c, tmp, 100 * MB) == 0);
    dfree_later(&c, tmp, 100 * MB);
    const int64_t room = fake::room;
    fake::room = 0;
    CHECK(dalloc(&c, buf, 120 * MB) == 0);
    fake::room = room;
    dfree(&c, buf, 120 * MB);
    c.arena.free_all();
  }
  CHECK(fake::held() == 0);
  std::puts("ok");
  return 0;
}
