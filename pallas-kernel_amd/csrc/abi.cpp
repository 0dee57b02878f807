// Error plumbing and small host helpers of the tops-hip C ABI.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <functional>
#include <vector>

#include "tops_hip.h"

static thread_local char g_err[512] = "";

extern "C" const char* tops_last_error(void) { return g_err; }

extern "C" const char* tops_version(void) { return "tops-hip 0.1.0 (gfx950)"; }

extern "C" int tops_set_error(int code, const char* msg) {
  snprintf(g_err, sizeof(g_err), "%s", msg ? msg : "");
  return code;
}

extern "C" int64_t tops_gla_state_bytes(int total_chunks, int H, int K, int V) {
  return (int64_t)total_chunks * H * K * V * 4;
}

// Host-side varlen chunk map (replaces tops/utils.py:71-90 prepare_chunk_indices and the
// per-sequence chunk counts of tops/cpu/ops/gla/chunk.py:206-212).
//   cu_seqlens [N+1] (host), chunk_size C.
//   chunk_offsets [N+1] (out): first global chunk of each sequence; chunk_offsets[N] = total.
//   chunk_indices [total][2] (out, optional): (sequence id, chunk id within sequence).
// Returns the total number of chunks, or a negative error code.
extern "C" int tops_prepare_chunk_indices(const int32_t* cu_seqlens, int N, int C,
                                          int32_t* chunk_offsets, int32_t* chunk_indices,
                                          int capacity) {
  if (!cu_seqlens || !chunk_offsets || N <= 0 || C <= 0)
    return tops_set_error(TOPS_ERR_NULL, "prepare_chunk_indices: bad arguments");
  int total = 0;
  chunk_offsets[0] = 0;
  for (int n = 0; n < N; ++n) {
    const int len = cu_seqlens[n + 1] - cu_seqlens[n];
    // an empty sequence has no chunk (tops/utils.py:71-90 gives it none); its state
    // passes through unchanged
    if (len < 0) return tops_set_error(TOPS_ERR_SHAPE, "prepare_chunk_indices: negative segment length");
    const int nc = (len + C - 1) / C;
    if (chunk_indices) {
      if (total + nc > capacity) return tops_set_error(TOPS_ERR_SHAPE, "prepare_chunk_indices: capacity");
      for (int c = 0; c < nc; ++c) {
        chunk_indices[2 * (total + c)] = n;
        chunk_indices[2 * (total + c) + 1] = c;
      }
    }
    total += nc;
    chunk_offsets[n + 1] = total;
  }
  return total;
}

// ---- sequence-parallel split: the search of SegPlan (tops/utils.py) over segment counts and
// piece lengths.  A call with boundaries not seen before runs it between its arguments and its
// first launch, up to nine candidates with a sort each: in Python it took 32 us for five
// sequences on 8 slots and 2.2 ms for 200 on 128, more than the sweep time it saves (20 us at
// five packed sequences, T8191 H16); here 6 and 28 us, of a plan of 0.12 and 0.62 ms.
namespace {

// Longest first.  Sizes are chunks of near-equal parts, so a histogram sorts them; a single
// sequence of millions of tokens may exceed it.
void sort_descending(std::vector<int32_t>& sizes, std::vector<int32_t>& hist, int32_t top) {
  if (top > (1 << 16)) {
    std::sort(sizes.begin(), sizes.end(), std::greater<int32_t>());
    return;
  }
  hist.assign(top + 1, 0);
  for (int32_t x : sizes) ++hist[x];
  size_t i = 0;
  for (int32_t x = top; x >= 0; --x)
    for (int32_t k = hist[x]; k > 0; --k) sizes[i++] = x;
}

struct Scratch {
  std::vector<int32_t> hist;
  std::vector<int64_t> load;
};
constexpr int64_t kAbove = INT64_MAX;

// Chunks until the last of `slots` workers is done, the longest item first, or kAbove as soon as
// that is known to exceed `limit`.  Sorts `sizes`.
int64_t lpt_span(std::vector<int32_t>& sizes, int slots, Scratch& w, double limit) {
  if (sizes.empty()) return 0;
  int32_t top = 0;
  int64_t sum = 0;
  for (int32_t x : sizes) {
    top = std::max(top, x);
    sum += x;
  }
  if (sizes.size() <= (size_t)slots) return top;
  int64_t span = std::max<int64_t>(top, (sum + slots - 1) / slots);   // a lower bound
  if ((double)span > limit) return kAbove;
  sort_descending(sizes, w.hist, top);
  w.load.assign(sizes.rend() - slots, sizes.rend());    // ascending: a min-heap as it stands
  int64_t* h = w.load.data();
  for (size_t i = slots; i < sizes.size(); ++i) {
    const int64_t x = h[0] + sizes[i];                  // the least loaded worker takes it
    if (x > span) {
      span = x;
      if ((double)span > limit) return kAbove;
    }
    int at = 0;
    for (int c = 1; c < slots; c = 2 * at + 1) {
      if (c + 1 < slots && h[c + 1] < h[c]) ++c;
      if (h[c] >= x) break;
      h[at] = h[c];
      at = c;
    }
    h[at] = x;
  }
  return *std::max_element(w.load.begin(), w.load.end());
}

// n chunks in k near-equal parts
void add_parts(std::vector<int32_t>& out, int n, int k) {
  const int base = n / k, rem = n % k;
  for (int i = 0; i < k; ++i) out.push_back(base + (i < rem));
}

// Span of the state pass with pieces of at most about x chunks (`parts`: their sizes).
int64_t pieces_span(const int32_t* handing, int n, int x, int slots, std::vector<int32_t>& parts,
                    Scratch& w, double limit) {
  parts.clear();
  for (int i = 0; i < n; ++i) add_parts(parts, handing[i], (handing[i] + x - 1) / x);
  return lpt_span(parts, slots, w, limit);
}

}  // namespace

extern "C" int tops_balance_rounds(const int32_t* sizes, int n, int slots) {
  if (!sizes || n <= 0 || slots <= 0)
    return tops_set_error(TOPS_ERR_NULL, "balance_rounds: bad arguments");
  try {
    std::vector<int32_t> s(sizes, sizes + n);
    for (int32_t x : s)
      if (x < 0) return tops_set_error(TOPS_ERR_SHAPE, "balance_rounds: negative size");
    Scratch w;
    return (int)lpt_span(s, slots, w, (double)kAbove);
  } catch (...) {
    return tops_set_error(TOPS_ERR_SHAPE, "balance_rounds: out of memory");
  }
}

extern "C" int tops_piece_balance(const int32_t* handing, int n, int sub, int slots) {
  if (!handing || n <= 0 || sub <= 0 || slots <= 0)
    return tops_set_error(TOPS_ERR_NULL, "piece_balance: bad arguments");
  for (int i = 0; i < n; ++i)
    if (handing[i] <= 0) return tops_set_error(TOPS_ERR_SHAPE, "piece_balance: empty segment");
  try {
    std::vector<int32_t> parts;
    Scratch w;
    int best = sub;
    int64_t low = kAbove;
    for (int x = sub; x <= 2 * sub; x += std::max(sub / 4, 1)) {
      const int64_t span = pieces_span(handing, n, x, slots, parts, w, (double)low);
      if (span < low) { low = span; best = x; }
      if (parts.size() <= (size_t)slots) break;   // one round: longer pieces only take longer
    }
    return best;
  } catch (...) {
    return tops_set_error(TOPS_ERR_SHAPE, "piece_balance: out of memory");
  }
}

extern "C" int tops_segment_balance(const int32_t* chunks, int32_t* counts, int N, int slots,
                                    int min_seg, int min_piece) {
  if (!chunks || !counts || N <= 0 || slots <= 0 || min_seg <= 0 || min_piece <= 0)
    return tops_set_error(TOPS_ERR_NULL, "segment_balance: bad arguments");
  int64_t total = 0;
  for (int i = 0; i < N; ++i) {
    if (chunks[i] < 0 || counts[i] <= 0)
      return tops_set_error(TOPS_ERR_SHAPE, "segment_balance: negative length or no segment");
    total += chunks[i];
  }
  try {
    std::vector<int32_t> flat, best(counts, counts + N), c(N);
    Scratch w;
    std::vector<std::vector<int32_t>> seen{best};
    int64_t span = 0;
    auto cost = [&](const std::vector<int32_t>& m, double low) {
      flat.clear();
      int64_t hand = 0;
      for (int i = 0; i < N; ++i) {
        add_parts(flat, chunks[i], m[i]);
        hand += chunks[i] - chunks[i] / m[i];     // all parts but the last, a shortest one
      }
      const int64_t sub = hand ? std::max<int64_t>((hand + slots - 1) / slots, min_piece) : 0;
      const int64_t states = (int64_t)flat.size() + (hand ? (hand + sub - 1) / sub : 0);
      // (the sum in the order below, so that the choice does not hang on the rounding)
      const double a = 2.0 / 3.0 * (double)sub, b = 4.0 / 3.0 * (double)states / slots;
      span = lpt_span(flat, slots, w, low - a - b + 1.0);
      return (double)span + a + b;
    };
    double low = cost(best, (double)kAbove);
    const int64_t t0 = std::max<int64_t>((total + slots - 1) / slots, min_seg);
    if ((double)span > 1.1 * (double)t0) {
      for (int64_t t = t0; t <= 2 * t0; t += std::max<int64_t>(t0 / 8, 1)) {
        for (int i = 0; i < N; ++i) c[i] = (int32_t)std::max<int64_t>((chunks[i] + t - 1) / t, 1);
        if (*std::max_element(c.begin(), c.end()) <= 1 ||
            std::find(seen.begin(), seen.end(), c) != seen.end())
          continue;
        seen.push_back(c);
        const double e = cost(c, low);
        if (e < low) { low = e; best = c; }
      }
    }
    std::copy(best.begin(), best.end(), counts);
    return TOPS_OK;
  } catch (...) {
    return tops_set_error(TOPS_ERR_SHAPE, "segment_balance: out of memory");
  }
}
