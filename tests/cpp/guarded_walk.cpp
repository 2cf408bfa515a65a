// The kernels that follow a decomposition whose guard is up, on pairs that lead
// in a circle: they do nothing, and they end.  (An iteration enqueued behind one
// whose decomposition was too deep has such pairs: new ones mixed with half made
// ones of another tree.)  Linked with the kernels compiled for the CPU.
#include <cstdio>
#include <vector>

#include "fl_kernels.h"

static int fail(const char* what) {
  std::printf("%s\n", what);
  return 1;
}

int main() {
  for (const uint32_t n : {1u, 2u, 3000u}) {
    std::vector<uint64_t> cp(n), rt(n), mask(n, 0);
    std::vector<uint32_t> row(n + 1, 0), next(n), hc(n, 0xffffffffu), base(n, 0);
    std::vector<uint32_t> buckets[7], order(n), pcnt(n), pdest(n, 7), ppos(n), spos(n, 7), root(n, 7), sub(n + 1);
    for (auto& b : buckets) b.assign(n + FL_BUCKET_PAD, 0);
    std::vector<uint8_t> act(n, 1u | 4u), outlet(n, 1);  // active, every site its chain's tail
    std::vector<double> area(n, 1.0), h(n, 0.5), h2(n, -1.0), rest(n, 1.0);
    std::vector<double> cval((size_t)FL_LIST * n);
    std::vector<uint2> cmeta(n);
    std::vector<uint32_t> ctrl(FL_CTRL_WORDS, 0);
    for (uint32_t v = 0; v < n; v++) {
      next[v] = (v + 1) % n;
      cp[v] = rt[v] = (1ull << 32) | ((v + 1) % n);  // unmarked: one further, without an end
    }
    if (n == 1) cp[0] = rt[0] = 1ull << 63;  // (a pair of itself ends)
    fl_dev_terrain t;
    t.n = n;
    t.row_ptr = row.data();
    t.col = nullptr;
    t.is_outlet = outlet.data();
    t.area = area.data();
    t.erod = t.uplift = t.tan_ms = rest.data();
    fl_dev_work w;
    w.h = h.data();
    w.h2 = h2.data();
    w.A = w.tau = w.dnext = w.parea = w.pK = w.pdn = rest.data();
    w.cval = cval.data();
    w.next = next.data();
    w.cmask = mask.data();
    w.hc = hc.data();
    w.cp = cp.data();
    w.rt = rt.data();
    w.sub = sub.data();
    w.bcnt = buckets[0].data();
    w.bnodes = buckets[1].data();
    w.boff = buckets[2].data();
    w.bnoff = buckets[3].data();
    w.bcur = buckets[4].data();
    w.bncur = buckets[5].data();
    w.ucum = buckets[6].data();
    w.cmeta = cmeta.data();
    w.head_base = base.data();
    w.perm = order.data();
    w.pcnt = pcnt.data();
    w.pdest = pdest.data();
    w.ppos = ppos.data();
    w.spos = spos.data();
    w.root = root.data();
    w.act = act.data();
    w.ctrl = ctrl.data();
    w.flags = (int*)ctrl.data();
    w.counters = ctrl.data() + FL_NUM_FLAGS;
    w.guard = ctrl.data() + FL_FLAG_DEEP;
    *w.guard = 1;
    for (const bool lakes : {false, true})
      for (const bool scan : {false, true}) {
        fl_launch_chain_count(nullptr, t, w, lakes);
        fl_launch_chain_layout(nullptr, t, w, lakes, scan);
        for (const auto& b : {buckets[0], buckets[1], buckets[4], buckets[5]})
          for (uint32_t x : b)
            if (x) return fail("a bucket was counted");
        for (uint32_t v = 0; v < n; v++)
          if (root[v] != 7 || spos[v] != 7 || pdest[v] != 7 || h2[v] != -1.0) return fail("a site was placed");
        if (*w.guard != 1) return fail("the guard came down");
      }
  }
  std::printf("ok\n");
  return 0;
}
