// How many workgroups walk the columns of a volume: the launch rule of the kernels that step along depth and keep the
// planes they have fetched (conv_ring.hip, wgrad_ring.hip).
#pragma once
#include <cstdint>

namespace sfh {

// Columns are cut into `segs` segments of `seg_steps` steps (the last one shorter); of the `items` = columns x segments each
// of `wgs` workgroups takes `items_per_wg` consecutive ones. cost: the busiest workgroup's time in steps.
struct ColumnCut {
  int segs, seg_steps, items, items_per_wg, wgs;
  int64_t cost;
};

// The cut by which the busiest of at most `wgs` workgroups ends soonest, `ncols` columns of `steps` steps. Its time is its
// steps (3.6 us each forward where the launch is short of the power limit, 2.1 in the weight gradient) and one step per item: the
// item's first planes come from memory with nothing beside them (1.5 to 2 us measured), and what short items lose otherwise.
// items < 0: too many.
//
// us, against cutting until every workgroup has an item, which leaves up to half of them idle behind two items of the others:
// forward (and data gradient; of a forward only where nobody takes its sums, cut_batch) 32 -> 32 at 54x105x99 53.5 -> 37.7, 36x101x119 39.1 -> 28.8, 96x80x112 59.4 -> 44.5, two samples of 57x87x77 67.1 -> 47.7,
// 32 -> 64 at 75x107x122 111 -> 92; weight gradient with its sum 32 -> 32 at 96x80x112 63.9 -> 54.3, 54x105x99 53.2 -> 47.0, two
// samples of 57x87x77 72.5 -> 58.5, 64 -> 32 at 110x48x111 91.2 -> 69.9, 128 -> 64 at 60x35x45 76.4 -> 60.8.
template <typename I>
inline ColumnCut cut_columns_in(I ncols, I steps, I wgs) {
  auto parts = [](I a, I b) { return (a + b - 1) / b; };
  ColumnCut best{};
  best.items = -1;
  const I most = parts(4 * wgs, ncols);  // more than four items to a workgroup even nothing out any more
  // one count of segments for each length there is, the smallest: `segs` segments are `len` steps long and no fewer are
  I len = 0;
  for (I segs = 1; segs <= most && segs <= steps; segs = len > 1 ? parts(steps, len - 1) : steps + 1) {
    len = parts(steps, segs);
    const I items = ncols * segs;
    if (items > 0x7fffffff) break;
    const I per_wg = parts(items, wgs);
    const int64_t cost = (int64_t)per_wg * (int64_t)(len + 1);
    if (best.items < 0 || cost < best.cost) best = ColumnCut{(int)segs, (int)len, (int)items, (int)per_wg, 0, cost};
  }
  if (best.items > 0) best.wgs = (int)parts((I)best.items, (I)best.items_per_wg);
  return best;
}
// (32-bit divisions wherever they do: launches and their queries ask for the cut on the host)
inline ColumnCut cut_columns(int64_t ncols, int64_t steps, int64_t wgs) {
  if (ncols < 1 << 20 && steps < 1 << 10 && wgs < 1 << 20) return cut_columns_in<uint32_t>((uint32_t)ncols, (uint32_t)steps, (uint32_t)wgs);
  return cut_columns_in<int64_t>(ncols, steps, wgs);
}

// The cut until every workgroup has an item, and no further: the order of sums that were taken before the busiest workgroup's time decided. For
// launches whose sums are read: statistics move with their order, and with them all that a network computes behind them (its
// logits by 4e-3, as by any other rounding).
inline ColumnCut cut_until_busy(int64_t ncols, int64_t steps, int64_t wgs) {
  auto parts = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  int64_t segs = ncols >= wgs ? 1 : parts(wgs, ncols);
  if (segs > steps) segs = steps;
  const int64_t len = parts(steps, segs);
  segs = parts(steps, len);
  ColumnCut c{(int)segs, (int)len, -1, 0, 0, 0};
  if (ncols * segs > 0x7fffffff) return c;
  c.items = (int)(ncols * segs);
  c.items_per_wg = (int)parts(c.items, wgs);
  c.wgs = (int)parts(c.items, c.items_per_wg);
  c.cost = c.items_per_wg * (len + 1);
  return c;
}

// The cut of `n` samples of `cols` columns: one line of columns (parts 1), or every sample by workgroups of its own (parts n; the cut is that of
// one), whose sums are then those of one sample, so that the normalisation behind the convolution needs no statistics pass. That is worth an
// end up to an eighth later where somebody takes the sums (`records`), and only there: three samples of 51x126x40 end 27 steps against 24 (32 -> 64
// channels). Samples of a few columns stay in one line (the statistics pass of a smaller one is the same launch whatever it reads). One sample
// whose sums are taken keeps their order.
struct BatchCut {
  int parts;
  ColumnCut cut;
};
inline BatchCut cut_batch(int64_t n, int64_t cols, int64_t steps, int64_t wgs, bool records) {
  if (records && n == 1) return BatchCut{1, cut_until_busy(cols, steps, wgs)};
  const BatchCut line{1, cut_columns(cols * n, steps, wgs)};
  if (!records || line.cut.items < 0 || n == 1 || wgs / n < 8) return line;
  const BatchCut apart{(int)n, cut_columns(cols, steps, wgs / n)};
  return apart.cut.items > 0 && 8 * apart.cut.cost <= 9 * line.cut.cost && apart.cut.wgs >= 8 ? apart : line;
}

}  // namespace sfh
