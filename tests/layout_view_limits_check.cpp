// Host check of the views that calls keep in place (morello_amd/csrc/layout_factor.h, MoveView): layouts of as many physical dims as there
// can be, most of them two digits, against each other. Built with the address sanitizer: nothing is written past the arrays.
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <vector>

#include "../morello_amd/csrc/layout_factor.h"

using namespace mrl;

static uint32_t state = 2718281;
static uint32_t rnd(uint32_t n) { return state = state * 1664525u + 1013904223u, (state >> 8) % n; }

// Physical dims of up to MRL_MAX_PHYS over `shape`: a Dynamic dim for each logical one, then Packed and OddEven ones of 2 and 4.
static mrl_layout draw(uint32_t rank) {
  mrl_layout l{};
  uint32_t order[MRL_MAX_RANK];
  for (uint32_t d = 0; d < rank; d++) order[d] = d;
  for (uint32_t d = rank; d > 1; d--) std::swap(order[d - 1], order[rnd(d)]);
  for (uint32_t d = 0; d < rank; d++) l.dims[l.ndims].logical_dim = decltype(l.dims[0].logical_dim)(order[d]), l.dims[l.ndims++].kind = MRL_DYNAMIC;
  const uint32_t extra = rnd(3) == 0 ? rnd(MRL_MAX_PHYS - rank + 1) : MRL_MAX_PHYS - rank;
  for (uint32_t e = 0; e < extra; e++) {
    mrl_physdim &p = l.dims[l.ndims++];
    p.logical_dim = decltype(p.logical_dim)(rnd(rank)), p.kind = decltype(p.kind)(rnd(3) ? MRL_PACKED : MRL_ODDEVEN), p.size = rnd(2) ? 2 : 4;
  }
  return l;
}

int main() {
  int views = 0, most = 0, full = 0;
  for (int t = 0; t < 200000; t++) {
    const uint32_t rank = 1 + rnd(MRL_MAX_RANK);
    uint32_t shape[MRL_MAX_RANK];
    for (uint32_t d = 0; d < rank; d++) shape[d] = rnd(8) == 0 ? 1 : 1u << (1 + rnd(rank <= 2 ? 16 : 24 / rank));
    const mrl_layout a = draw(rank), b = draw(rank);
    LayoutEval ea, eb;
    if (!make_layout_eval(a, shape, rank, &ea) || !make_layout_eval(b, shape, rank, &eb)) continue;
    auto view = std::make_unique<MoveView>();   // (on the heap by itself, so that a write past it is seen)
    std::vector<MoveDim> same;
    const bool has = common_view(a, b, shape, rank, view.get());
    if (has != common_view(a, b, shape, rank, &same)) return std::printf("a view in place and none in a vector, or the other way\n"), 1;
    if (view->size() > VIEW_MAX_DIGITS) return std::printf("%u digits\n", view->size()), 1;
    most = int(std::max<uint32_t>(most, view->size()));
    full += a.ndims == MRL_MAX_PHYS && b.ndims == MRL_MAX_PHYS;
    if (!has) continue;
    views++;
    if (view->size() != same.size() || same_order(*view) != same_order(same)) return std::printf("sizes differ\n"), 1;
    uint64_t count = 1;
    for (uint32_t d = 0; d < view->size(); d++) {
      if ((*view)[d].size != same[d].size || (*view)[d].ss != same[d].ss || (*view)[d].ds != same[d].ds) return std::printf("digits differ\n"), 1;
      count *= same[d].size;
    }
    for (uint32_t d = 0; d < rank; d++) {
      if (count % shape[d] != 0) return std::printf("the view misses elements\n"), 1;
      count /= shape[d];
    }
    // some of the elements, where the layouts' index expressions send them
    for (int e = 0; e < 8; e++) {
      uint32_t at[MRL_MAX_RANK];
      for (uint32_t d = 0; d < rank; d++) at[d] = rnd(shape[d]);
      const int64_t from = layout_offset(ea, at), to = layout_offset(eb, at);
      int64_t rest = from, got = 0;   // the digits of the source offset, largest strides first
      std::vector<MoveDim> by_source(same);
      std::sort(by_source.begin(), by_source.end(), [](const MoveDim &x, const MoveDim &y) { return x.ss > y.ss; });
      for (const MoveDim &m : by_source) got += rest / m.ss * m.ds, rest %= m.ss;
      if (rest != 0 || got != to) return std::printf("element %lld goes to %lld, expected %lld\n", (long long)from, (long long)got, (long long)to), 1;
    }
  }
  std::printf("views %d, of up to %d digits, both layouts full %d\n", views, most, full);
  if (views < 1000 || full < 1000 || most <= int(MOVE_MAX_RANK)) return std::printf("too few\n"), 1;
  std::printf("layout view limits ok\n");
  return 0;
}
