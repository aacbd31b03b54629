// Two layouts of one logical shape as a common strided view (host code).
//
// A Packed(n) physical dim splits its logical dim into "which group of n" and "which of the n";
// an OddEven(n) dim splits a strip of n into "which pair" and "odd or even" and stores the
// parity outermost (morello/src/layout.rs:221-272).  Either way a layout is a mixed-radix
// decomposition of each logical index, one stride per digit.  Two layouts of the same shape can
// be given the same digits whenever their radices refine each other (8 and 16 do, 6 and 4 do
// not); the Move between them is then a plain permutation of a higher-rank tensor, which the
// strided Move kernels take.  Where they do not, the caller falls back to index arithmetic per
// element.
#pragma once
#include <algorithm>

#include "layout_math.h"

namespace mrl {

constexpr uint32_t MOVE_MAX_RANK = 12;

// One digit of the common view: `size` values, `ss` / `ds` elements apart on the two sides.
struct MoveDim {
  uint32_t size;
  int64_t ss, ds;
};

// Digits of a layout at the most (an OddEven dim has two), and of a common view: every one ends a digit of one of the two sides.
constexpr uint32_t LAYOUT_MAX_DIGITS = 2 * MRL_MAX_PHYS, VIEW_MAX_DIGITS = 2 * LAYOUT_MAX_DIGITS;

// A common view, kept in place: every call of a Compose forms four or five of them, and vectors' allocations and a stable sort's buffer
// took more of such a call than the launch's own arguments.
struct MoveView {
  MoveDim dims[VIEW_MAX_DIGITS];
  uint32_t n = 0;
  const MoveDim *data() const { return dims; }
  uint32_t size() const { return n; }
  bool empty() const { return n == 0; }
  void clear() { n = 0; }
  void push_back(const MoveDim &d) { dims[n++] = d; }
  MoveDim &back() { return dims[n - 1]; }
  const MoveDim &operator[](uint32_t i) const { return dims[i]; }
};

namespace detail {

struct Digit {
  uint32_t size;
  int64_t stride;
};

struct Digits {
  Digit of[MRL_MAX_RANK][LAYOUT_MAX_DIGITS];
  uint32_t n[MRL_MAX_RANK];
  void add(uint32_t dim, uint32_t size, int64_t stride) { of[dim][n[dim]++] = {size, stride}; }
};

// Digits of each logical dim, most significant first.  False for a layout this view cannot
// express (an OddEven dim that is not the innermost dim of its logical dim).
inline bool digits_of(const mrl_layout &l, const uint32_t *shape, uint32_t rank, Digits *out) {
  uint32_t phys[MRL_MAX_PHYS];
  if (!physical_shape(l, shape, rank, phys)) return false;
  int64_t stride[MRL_MAX_PHYS], running = 1;
  for (int i = int(l.ndims) - 1; i >= 0; i--) stride[i] = running, running *= phys[i];
  uint32_t remaining[MRL_MAX_RANK];
  for (uint32_t d = 0; d < rank; d++) remaining[d] = shape[d], out->n[d] = 0;
  for (uint32_t i = 0; i < l.ndims; i++) {
    const uint32_t ld = l.dims[i].logical_dim;
    remaining[ld] /= phys[i];
    if (phys[i] == 1) continue;
    if (l.dims[i].kind == MRL_ODDEVEN) {
      if (remaining[ld] != 1 || phys[i] != l.dims[i].size) return false;
      // index within the strip e = 2 * pair + parity lives at parity * (n / 2) + pair
      out->add(ld, phys[i] / 2, stride[i]);
      out->add(ld, 2, stride[i] * (phys[i] / 2));
    } else {
      out->add(ld, phys[i], stride[i]);
    }
  }
  for (uint32_t d = 0; d < rank; d++)
    if (remaining[d] != 1) return false;
  return true;
}

}  // namespace detail

// The common view of `src` and `dst` layouts over `shape`, digits with contiguous neighbours
// on both sides merged, size-one digits dropped.  False when there is none (or it has more
// than MOVE_MAX_RANK digits).
template <class View>   // MoveView, or a vector
bool common_view(const mrl_layout &src, const mrl_layout &dst, const uint32_t *shape, uint32_t rank, View *view) {
  detail::Digits a, b;
  if (!detail::digits_of(src, shape, rank, &a) || !detail::digits_of(dst, shape, rank, &b)) return false;
  MoveDim dims[VIEW_MAX_DIGITS];
  uint32_t n = 0;
  for (uint32_t d = 0; d < rank; d++) {
    // Least significant digits first; the larger of the two current digits is split.
    int ia = int(a.n[d]) - 1, ib = int(b.n[d]) - 1;
    detail::Digit ra{1, 0}, rb{1, 0};
    if (ia >= 0) ra = a.of[d][ia];
    if (ib >= 0) rb = b.of[d][ib];
    while (ia >= 0 && ib >= 0) {
      const uint32_t take = std::min(ra.size, rb.size);
      if (ra.size % take != 0 || rb.size % take != 0) return false;
      // Slowest to fastest on the destination side, those of one stride in the order in which they came.
      uint32_t at = n++;
      for (; at > 0 && dims[at - 1].ds < rb.stride; at--) dims[at] = dims[at - 1];
      dims[at] = {take, ra.stride, rb.stride};
      ra.size /= take, ra.stride *= take;
      rb.size /= take, rb.stride *= take;
      if (ra.size == 1 && --ia >= 0) ra = a.of[d][ia];
      if (rb.size == 1 && --ib >= 0) rb = b.of[d][ib];
    }
    if (ia >= 0 || ib >= 0) return false;  // the two products differ: not the same shape
  }
  // Digits that continue each other are merged.
  view->clear();
  for (uint32_t i = 0; i < n; i++) {
    const MoveDim &m = dims[i];
    if (m.size == 1) continue;
    if (!view->empty()) {
      MoveDim &last = view->back();
      if (last.ss == m.ss * int64_t(m.size) && last.ds == m.ds * int64_t(m.size)) {
        last.size *= m.size, last.ss = m.ss, last.ds = m.ds;
        continue;
      }
    }
    view->push_back(m);
  }
  return view->size() <= MOVE_MAX_RANK;
}

// Whether a common view says that both sides store the elements in the same order.
template <class View>
bool same_order(const View &view) {
  return view.empty() || (view.size() == 1 && view[0].ss == 1 && view[0].ds == 1);
}

}  // namespace mrl
