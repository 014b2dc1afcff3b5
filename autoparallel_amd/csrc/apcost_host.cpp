// Host side of the table build (plain C++, no device code): what a planner does with the
// flattened tables between the encoding and the launches.  Identical edges, tilings, packed tile
// records and the checks in front of the kernels are passes over arrays of up to a few million
// rows; on a graph of 15 000 edges the interpreter's share of them was forty times the device's
// work.
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <vector>

#include "apcost.h"
#include "apcost_error.h"
#include "apcost_parallel.h"

using apc_internal::check_params;
using apc_internal::fail;
using apc_internal::in_parallel;
using apc_internal::threads_for;
using apc_internal::thrown;

int apc_internal::thrown(const char *who) {
  try {
    throw;
  } catch (const std::exception &e) {
    return fail(-4, "%s: %s", who, e.what());
  } catch (...) {
    return fail(-4, "%s: an exception", who);
  }
}

namespace {

// ------------------------------------------------------------------------------------------
// A 128-bit hash of byte runs: two independent chains of multiply-and-fold steps over 8-byte words.
// It only proposes equal edges; equality is decided by comparing the bytes.  (Its constants: the first 64
// bits behind the point of the square roots of 101, 103, 107 and 109, made odd.)
// ------------------------------------------------------------------------------------------
struct Hash128 {
  uint64_t a = 0x0CC4A61194F81761ull, b = 0x261DC1F2B8A998C9ull;
  static uint64_t fold(uint64_t x, uint64_t y) {
    const unsigned __int128 p = (unsigned __int128)x * y;
    return (uint64_t)p ^ (uint64_t)(p >> 64);
  }
  void word(uint64_t w) {
    a = fold(a ^ w, 0x5815A7BE0543C11Dull);
    b = fold(b + w, 0x70B7ED67FC9B5C43ull) + w;
  }
  void run(const void *data, size_t bytes) {
    const unsigned char *p = static_cast<const unsigned char *>(data);
    for (; bytes >= 8; p += 8, bytes -= 8) {
      uint64_t w;
      memcpy(&w, p, 8);
      word(w);
    }
    if (bytes) {
      uint64_t w = 0;
      memcpy(&w, p, bytes);
      word(w ^ ((uint64_t)bytes << 56));
    }
  }
};

// Everything an edge's matrix depends on: both spec lists, flags, the consumer strategies' rows of
// the strategy table, the pass-through values.
struct EdgeContent {
  const int32_t *src_begin, *n_src, *tgt_begin, *n_tgt, *flags;
  const int64_t *pt_begin;
  const int32_t *strat_begin;
  int64_t n_specs;
  const uint32_t *codes;
  const int32_t *tensor;
  int64_t n_strategies;
  const int64_t *flops, *rw_bytes;
  const int8_t *dtype;
  const uint8_t *zero_cost;
  const int32_t *num_args;
  int64_t n_pt;
  const double *pt_values;

  // Calls f(pointer, bytes) for every run of edge e; false when a range leaves its table.
  template <typename F>
  bool runs(int64_t e, F &&f) const {
    const int64_t ns = n_src[e], nt = n_tgt[e], sb = src_begin[e], tb = tgt_begin[e], st = strat_begin[e];
    if (ns < 0 || nt < 0 || sb < 0 || tb < 0 || st < 0 || sb + ns > n_specs || tb + nt > n_specs || st + nt > n_strategies) return false;
    const bool pt = pt_begin[e] >= 0;
    if (pt && (ns * nt > n_pt || pt_begin[e] > n_pt - ns * nt)) return false;
    f(codes + sb, 4 * (size_t)ns);
    f(tensor + sb, 4 * (size_t)ns);
    f(codes + tb, 4 * (size_t)nt);
    f(tensor + tb, 4 * (size_t)nt);
    f(flops + st, 8 * (size_t)nt);
    f(rw_bytes + st, 8 * (size_t)nt);
    f(dtype + st, (size_t)nt);
    f(zero_cost + st, (size_t)nt);
    f(num_args + st, 4 * (size_t)nt);
    if (pt) f(pt_values + pt_begin[e], 8 * (size_t)(ns * nt));
    return true;
  }
  bool same_shape(int64_t x, int64_t y) const {
    return n_src[x] == n_src[y] && n_tgt[x] == n_tgt[y] && flags[x] == flags[y] && (pt_begin[x] >= 0) == (pt_begin[y] >= 0);
  }
  bool equal(int64_t x, int64_t y) const {
    if (!same_shape(x, y)) return false;
    const void *px[10];
    int n = 0;
    runs(x, [&](const void *p, size_t) { px[n++] = p; });
    int k = 0;
    bool eq = true;
    runs(y, [&](const void *p, size_t bytes) {
      eq = eq && memcmp(px[k], p, bytes) == 0;
      ++k;
    });
    return eq;
  }
};

}  // namespace

extern "C" {

int apc_edge_classes_host(int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t n_strategies,
                          const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype_code, const uint8_t *zero_cost,
                          const int32_t *num_args, int64_t n_edges, const int32_t *edge_src_begin, const int32_t *edge_n_src,
                          const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt, const int32_t *edge_flags,
                          const int64_t *edge_pt_begin, const int32_t *edge_strat_begin, int64_t n_pt, const double *pt_values,
                          int64_t *first_same) try {
  if (n_specs < 0 || n_strategies < 0 || n_edges < 0 || n_pt < 0) return fail(-1, "apc_edge_classes_host: negative count");
  if (n_edges == 0) return 0;
  if (!edge_src_begin || !edge_n_src || !edge_tgt_begin || !edge_n_tgt || !edge_flags || !edge_pt_begin || !edge_strat_begin ||
      !first_same || (n_specs > 0 && (!spec_codes || !spec_tensor)) || (n_pt > 0 && !pt_values) ||
      (n_strategies > 0 && (!flops || !rw_bytes || !dtype_code || !zero_cost || !num_args)))
    return fail(-1, "apc_edge_classes_host: NULL array");
  const EdgeContent c{edge_src_begin, edge_n_src, edge_tgt_begin, edge_n_tgt, edge_flags, edge_pt_begin, edge_strat_begin, n_specs,
                      spec_codes, spec_tensor, n_strategies, flops, rw_bytes, dtype_code, zero_cost, num_args, n_pt, pt_values};
  struct Key {
    uint64_t a, b;
  };
  std::vector<Key> key(n_edges);
  std::vector<uint8_t> known(n_edges);
  int64_t bytes = 0;
  for (int64_t e = 0; e < n_edges; ++e) bytes += 8 * (int64_t)std::max(edge_n_src[e], 0) + 30 * (int64_t)std::max(edge_n_tgt[e], 0);
  const int threads = threads_for(bytes);
  in_parallel(n_edges, threads, [&](int64_t b, int64_t end) {
    for (int64_t e = b; e < end; ++e) {
      Hash128 h;
      h.word(((uint64_t)(uint32_t)edge_n_src[e] << 32) | (uint32_t)edge_n_tgt[e]);
      h.word((uint64_t)(uint32_t)edge_flags[e] * 2 + (edge_pt_begin[e] >= 0));
      known[e] = c.runs(e, [&](const void *p, size_t n) { h.run(p, n); });
      key[e] = Key{h.a, h.b};
    }
  });
  // open addressing over the hashes, edges in order: the first edge of a hash stands for it.  (An edge
  // whose ranges leave the tables stands for itself; the validator reports it.)
  int64_t slots = 16;
  while (slots < 2 * n_edges) slots *= 2;
  std::vector<int64_t> table(slots, -1);
  for (int64_t e = 0; e < n_edges; ++e) {
    first_same[e] = e;
    if (!known[e]) continue;
    int64_t at = (int64_t)(key[e].a & (uint64_t)(slots - 1));
    for (;; at = (at + 1) & (slots - 1)) {
      const int64_t f = table[at];
      if (f < 0) {
        table[at] = e;
        break;
      }
      if (key[f].a == key[e].a && key[f].b == key[e].b) {
        first_same[e] = f;
        break;
      }
    }
  }
  // the proposals, compared byte by byte: an edge that only shares a hash stands for itself
  in_parallel(n_edges, threads, [&](int64_t b, int64_t end) {
    for (int64_t e = b; e < end; ++e)
      if (first_same[e] != e && !c.equal(first_same[e], e)) first_same[e] = e;
  });
  return 0;
} catch (...) {
  return thrown("apc_edge_classes_host");
}

// ------------------------------------------------------------------------------------------
// Tilings.
// ------------------------------------------------------------------------------------------
namespace {

struct EdgeTiling {  // how one edge's matrix is cut
  int64_t col_chunks, chunk_width, row_tiles, rows_per_tile;
};

EdgeTiling cut(int64_t ns, int64_t nt, int64_t tile_entries, int64_t rows_per_wavefront_pass) {
  EdgeTiling t;
  t.col_chunks = (ns + APC_TILE_MAX_COLS - 1) / APC_TILE_MAX_COLS;
  t.chunk_width = (ns + t.col_chunks - 1) / t.col_chunks;
  int64_t rows = std::min<int64_t>(std::max<int64_t>(tile_entries / t.chunk_width, 1), APC_TILE_MAX_ROWS);
  if (rows_per_wavefront_pass > 0 && t.col_chunks == 1)
    rows = std::min(rows, rows_per_wavefront_pass * std::max<int64_t>(64 / t.chunk_width, 1));
  t.row_tiles = (nt + rows - 1) / rows;
  t.rows_per_tile = (nt + t.row_tiles - 1) / t.row_tiles;  // balanced
  return t;
}

}  // namespace

int apc_count_tiles_host(int64_t n_edges, const int32_t *edge_n_src, const int32_t *edge_n_tgt, const int64_t *first_same,
                         int64_t tile_entries, int64_t max_copies, int64_t rows_per_wavefront_pass, int64_t *edge_canonical,
                         int64_t *n_tiles, int64_t *n_duplicates) try {
  if (n_edges < 0 || tile_entries < 1) return fail(-1, "apc_count_tiles_host: n_edges >= 0 and tile_entries >= 1");
  if (!n_tiles || !n_duplicates || (n_edges > 0 && (!edge_n_src || !edge_n_tgt || !edge_canonical)))
    return fail(-1, "apc_count_tiles_host: NULL array");
  *n_tiles = *n_duplicates = 0;
  // per class of identical edges: the tiled edge that takes the next copy, and how many it has taken
  const int64_t room = std::min<int64_t>(APC_TILE_MAX_DUPS, std::max<int64_t>(max_copies - 1, 0));
  std::vector<int64_t> tiled, taken;
  if (first_same) {
    tiled.assign(n_edges, -1);
    taken.assign(n_edges, 0);
  }
  for (int64_t e = 0; e < n_edges; ++e) {
    edge_canonical[e] = e;
    if (first_same) {
      const int64_t f = first_same[e];
      if (f < 0 || f > e) return fail(-2, "edge %lld: first_same %lld is no earlier edge", (long long)e, (long long)f);
      if (tiled[f] < 0 || taken[f] >= room) {
        tiled[f] = e;  // (also when the previous one is full)
        taken[f] = 0;
      } else {
        edge_canonical[e] = tiled[f];
        ++taken[f];
        ++*n_duplicates;
        continue;
      }
    }
    if (edge_n_src[e] > 0 && edge_n_tgt[e] > 0) {
      const EdgeTiling t = cut(edge_n_src[e], edge_n_tgt[e], tile_entries, rows_per_wavefront_pass);
      *n_tiles += t.col_chunks * t.row_tiles;
    }
  }
  return 0;
} catch (...) {
  return thrown("apc_count_tiles_host");
}

int apc_fill_tiles_host(int64_t n_edges, const int32_t *edge_n_src, const int32_t *edge_n_tgt, const int64_t *edge_entry_begin,
                        const int64_t *edge_canonical, int64_t tile_entries, int64_t rows_per_wavefront_pass, int64_t n_tiles,
                        int64_t n_duplicates, int64_t *edge_dup_begin, int64_t *edge_dup_count, int64_t *dup_entry_begin,
                        int64_t *dup_row_begin, int32_t *tile_edge, int32_t *tile_row_begin, int32_t *tile_row_count,
                        int32_t *tile_col_begin, int32_t *tile_col_count) try {
  if (n_edges < 0 || n_tiles < 0 || n_duplicates < 0 || tile_entries < 1) return fail(-1, "apc_fill_tiles_host: negative count");
  if (n_edges > 0 && (!edge_n_src || !edge_n_tgt || !edge_entry_begin || !edge_canonical || !edge_dup_begin || !edge_dup_count))
    return fail(-1, "apc_fill_tiles_host: NULL edge array");
  if ((n_duplicates > 0 && (!dup_entry_begin || !dup_row_begin)) ||
      (n_tiles > 0 && (!tile_edge || !tile_row_begin || !tile_row_count || !tile_col_begin || !tile_col_count)))
    return fail(-1, "apc_fill_tiles_host: NULL output");
  // duplicates grouped by the edge that is tiled for them, in edge order inside a group
  std::fill(edge_dup_count, edge_dup_count + n_edges, 0);
  int64_t dups = 0;
  for (int64_t e = 0; e < n_edges; ++e) {
    const int64_t c = edge_canonical[e];
    if (c < 0 || c > e) return fail(-2, "edge %lld: canonical edge %lld is no earlier edge", (long long)e, (long long)c);
    if (c != e) {
      ++edge_dup_count[c];
      ++dups;
    }
  }
  if (dups != n_duplicates) return fail(-2, "%lld duplicate edges, the arrays hold %lld", (long long)dups, (long long)n_duplicates);
  int64_t at = 0;
  for (int64_t e = 0; e < n_edges; ++e) {
    edge_dup_begin[e] = at;
    at += edge_dup_count[e];
  }
  std::vector<int64_t> next(edge_dup_begin, edge_dup_begin + n_edges);
  int64_t row = 0, t = 0;
  for (int64_t e = 0; e < n_edges; ++e) {
    const int64_t c = edge_canonical[e], ns = edge_n_src[e], nt = edge_n_tgt[e];
    if (c != e) {
      dup_entry_begin[next[c]] = edge_entry_begin[e];
      dup_row_begin[next[c]++] = row;
    } else if (ns > 0 && nt > 0) {
      const EdgeTiling k = cut(ns, nt, tile_entries, rows_per_wavefront_pass);
      if (t + k.col_chunks * k.row_tiles > n_tiles) return fail(-2, "more tiles than the arrays hold (%lld)", (long long)n_tiles);
      for (int64_t ri = 0; ri < k.row_tiles; ++ri)
        for (int64_t ci = 0; ci < k.col_chunks; ++ci, ++t) {
          const int64_t rb = ri * k.rows_per_tile, cb = ci * k.chunk_width;
          tile_edge[t] = (int32_t)e;
          tile_row_begin[t] = (int32_t)rb;
          tile_row_count[t] = (int32_t)std::min(k.rows_per_tile, nt - rb);
          tile_col_begin[t] = (int32_t)cb;
          tile_col_count[t] = (int32_t)std::min(k.chunk_width, ns - cb);
        }
    }
    row += nt;
  }
  if (t != n_tiles) return fail(-2, "%lld tiles, the arrays hold %lld", (long long)t, (long long)n_tiles);
  return 0;
} catch (...) {
  return thrown("apc_fill_tiles_host");
}

int apc_order_tiles_host(int64_t n_tiles, const apc_tile *records, apc_tile *ordered) try {
  if (n_tiles < 0) return fail(-1, "apc_order_tiles_host: negative count");
  if (n_tiles > 0 && (!records || !ordered)) return fail(-1, "apc_order_tiles_host: NULL array");
  // by counting: first the rank of the first tile of every size (a record that the validator would refuse counts as the largest)
  constexpr int kMost = APC_TILE_MAX_ROWS * APC_TILE_MAX_COLS;
  const auto size = [](const apc_tile &t) {
    const uint32_t n = (uint32_t)(t.counts & 0xFFFF) * (uint32_t)(t.counts >> 16);
    return n <= (uint32_t)kMost ? (int)n : kMost;
  };
  std::vector<uint64_t> next(kMost + 2, 0);
  for (int64_t t = 0; t < n_tiles; ++t) ++next[kMost - size(records[t]) + 1];
  for (int s = 0; s <= kMost; ++s) next[s + 1] += next[s];
  // rank k is tile k / 8 of die k mod 8: where that one is in the launch's order (tile_of_block in apcost.hip)
  constexpr uint64_t kDies = 8, kRound = kDies * APC_TILE_RUN;
  const uint64_t full = (uint64_t)n_tiles / kRound * kRound, rest = (uint64_t)n_tiles - full, per = (rest + kDies - 1) / kDies;
  // (the last, incomplete round: `whole` dies take `per` tiles each, one the `left` others)
  const uint64_t whole = per > 0 ? rest / per : 0, left = rest - whole * per, dies = whole + (left > 0 ? 1 : 0);
  for (int64_t t = 0; t < n_tiles; ++t) {
    const uint64_t k = next[kMost - size(records[t])]++;
    const uint64_t within = k < full ? k % kRound : k - full;
    uint64_t at;
    if (k < full) at = k - within + within % kDies * APC_TILE_RUN + within / kDies;
    else if (within < left * dies) at = full + within % dies * per + within / dies;
    else at = full + (within - left * dies) % whole * per + left + (within - left * dies) / whole;
    ordered[at] = records[t];
  }
  return 0;
} catch (...) {
  return thrown("apc_order_tiles_host");
}

int apc_tile_records_host(int64_t n_specs, const int32_t *spec_tensor, int64_t n_edges, const int32_t *edge_src_begin,
                          const int32_t *edge_n_src, const int32_t *edge_tgt_begin, const int32_t *edge_flags,
                          const int64_t *edge_pt_begin, const int64_t *edge_entry_begin, const int32_t *edge_strat_begin,
                          const int64_t *edge_dup_begin, const int64_t *edge_dup_count, int64_t n_tiles, const int32_t *tile_edge,
                          const int32_t *tile_row_begin, const int32_t *tile_row_count, const int32_t *tile_col_begin,
                          const int32_t *tile_col_count, apc_tile *records) {
  if (n_specs < 0 || n_edges < 0 || n_tiles < 0) return fail(-1, "apc_tile_records_host: negative count");
  if (n_tiles == 0) return 0;
  if (!tile_edge || !tile_row_begin || !tile_row_count || !tile_col_begin || !tile_col_count || !records ||
      (n_specs > 0 && !spec_tensor) ||
      (n_edges > 0 && (!edge_src_begin || !edge_n_src || !edge_tgt_begin || !edge_flags || !edge_pt_begin || !edge_entry_begin ||
                       !edge_strat_begin || !edge_dup_begin || !edge_dup_count)))
    return fail(-1, "apc_tile_records_host: NULL array");
  for (int64_t t = 0; t < n_tiles; ++t) {
    apc_tile r;
    memset(&r, 0, sizeof(r));
    r.edge = tile_edge[t];
    r.row_begin = tile_row_begin[t];
    r.col_begin = tile_col_begin[t];
    r.counts = (tile_row_count[t] & 0xFFFF) | ((tile_col_count[t] & 0x7FFF) << 16);
    if (n_edges > 0) {
      // (an edge or spec outside its table takes the nearest row: the validator reports it)
      const int64_t e = r.edge >= 0 && r.edge < n_edges ? r.edge : 0;
      r.src_begin = edge_src_begin[e];
      r.n_src = edge_n_src[e];
      r.tgt_begin = edge_tgt_begin[e];
      r.flags = edge_flags[e];
      r.strat_begin = edge_strat_begin[e];
      r.entry_begin = edge_entry_begin[e];
      r.pt_begin = edge_pt_begin[e];
      r.dup_begin = (int32_t)edge_dup_begin[e];
      r.dup_count = (int32_t)edge_dup_count[e];
      if (n_specs > 0)
        r.tensor = spec_tensor[std::min(std::max((int64_t)edge_src_begin[e] + tile_col_begin[t], (int64_t)0), n_specs - 1)];
    }
    records[t] = r;
  }
  return 0;
}

int apc_validate_tiling_host(int64_t n_tensors, const int32_t *tensor_rank, const int32_t *tensor_itemsize, const int64_t *tensor_shape,
                             int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int32_t *num_args,
                             int64_t n_edges, const int32_t *edge_n_src, const int32_t *edge_n_tgt, const int64_t *edge_canonical,
                             const int64_t *edge_dup_count, int64_t n_duplicates, int64_t n_tiles, const int32_t *tile_edge,
                             const int32_t *tile_row_count, const int32_t *tile_col_count) try {
  if (n_tensors < 0 || n_strategies < 0 || n_edges < 0 || n_tiles < 0) return fail(-1, "apc_validate_tiling_host: negative count");
  if ((n_tensors > 0 && (!tensor_rank || !tensor_itemsize || !tensor_shape)) || (n_strategies > 0 && (!flops || !rw_bytes || !num_args)) ||
      (n_edges > 0 && (!edge_n_src || !edge_n_tgt || !edge_canonical || !edge_dup_count)) ||
      (n_tiles > 0 && (!tile_edge || !tile_row_count || !tile_col_count)))
    return fail(-1, "apc_validate_tiling_host: NULL array");
  constexpr int64_t kExact = (int64_t)1 << 53;  // integers below convert to fp64 exactly
  int32_t fewest = 1;
  bool large = false;
  for (int64_t s = 0; s < n_strategies; ++s) {
    fewest = std::min(fewest, num_args[s]);
    large |= flops[s] >= kExact || rw_bytes[s] >= kExact;
  }
  if (fewest < 1) return fail(-2, "strat_num_args must be >= 1");
  if (large) return fail(-2, "flop / byte counts must stay below 2**53 to convert to fp64 exactly");
  // every edge is either tiled completely or a duplicate of an edge that is
  std::vector<int64_t> area(n_edges, 0);
  for (int64_t t = 0; t < n_tiles; ++t) {
    if (tile_edge[t] < 0 || tile_edge[t] >= n_edges) return fail(-2, "tile %lld: edge %d out of range", (long long)t, tile_edge[t]);
    area[tile_edge[t]] += (int64_t)tile_row_count[t] * tile_col_count[t];
  }
  int64_t untiled = 0, dups = 0;
  for (int64_t e = 0; e < n_edges; ++e) {
    const bool tiled = edge_canonical[e] == e;
    if (area[e] != (tiled ? (int64_t)edge_n_src[e] * edge_n_tgt[e] : 0))
      return fail(-2, "tiles do not cover every (non-duplicate) edge matrix exactly once");
    untiled += !tiled;
    dups += edge_dup_count[e];
  }
  if (dups != untiled || n_duplicates != untiled) return fail(-2, "duplicate-edge lists do not account for every de-duplicated edge");
  for (int64_t t = 0; t < n_tensors; ++t) {
    const int64_t *shape = tensor_shape + t * APC_MAX_RANK;
    const int rank = std::min(tensor_rank[t], APC_MAX_RANK);
    bool zero = tensor_itemsize[t] == 0;
    for (int d = 0; d < rank; ++d) {
      if (shape[d] < 0) return fail(-2, "tensor sizes must not be negative");
      zero |= shape[d] == 0;
    }
    // (the product of the exact sizes, stopped where it passes the bound)
    unsigned __int128 n = zero ? 0 : (unsigned __int128)(tensor_itemsize[t] < 0 ? 0 : tensor_itemsize[t]);
    for (int d = 0; d < rank && n > 0 && n < (unsigned __int128)kExact; ++d) n *= (uint64_t)shape[d];
    if (n >= (unsigned __int128)kExact) return fail(-2, "tensor byte counts must stay below 2**53");
  }
  return 0;
} catch (...) {
  return thrown("apc_validate_tiling_host");
}

int apc_pack_tiles_host(int64_t n_tensors, const int32_t *tensor_rank, const int32_t *tensor_itemsize, const int64_t *tensor_shape,
                        const int64_t *tensor_stride, int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor,
                        int64_t n_strategies, const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype_code,
                        const uint8_t *zero_cost, const int32_t *num_args, int64_t n_edges, const int64_t *edge_row_begin,
                        int64_t n_tiles, const apc_tile *tiles, int64_t n_dups, const int64_t *dup_entry_begin,
                        const int64_t *dup_row_begin, apc_packed_tile *packed) try {
  if (n_tensors < 0 || n_specs < 0 || n_strategies < 0 || n_edges < 0 || n_tiles < 0 || n_dups < 0)
    return fail(-1, "apc_pack_tiles_host: negative count");
  if (n_tiles == 0) return 0;
  if (!tiles || !packed || !spec_codes || !spec_tensor || !edge_row_begin || !flops || !rw_bytes || !dtype_code || !zero_cost ||
      !num_args || (n_dups > 0 && (!dup_entry_begin || !dup_row_begin)) ||
      (n_tensors > 0 && (!tensor_rank || !tensor_itemsize || !tensor_shape || !tensor_stride)))
    return fail(-1, "apc_pack_tiles_host: NULL array");
  std::atomic<int64_t> bad{n_tiles};  // the first tile that cannot be packed
  in_parallel(n_tiles, threads_for(n_tiles * (int64_t)sizeof(apc_packed_tile)), [&](int64_t begin, int64_t end) {
    for (int64_t t = begin; t < end; ++t) {
      const apc_tile &tl = tiles[t];
      apc_packed_tile &pk = packed[t];
      memset(&pk, 0, sizeof(pk));
      const int64_t rows = tl.counts & 0xFFFF, cols = tl.counts >> 16, rb = tl.row_begin, first = rb * cols;
      const int64_t sb = tl.src_begin, tb = (int64_t)tl.tgt_begin + rb, st = (int64_t)tl.strat_begin + rb;
      bool holds = tl.edge >= 0 && tl.edge < n_edges && rows >= 1 && rows <= APC_TILE_MAX_ROWS && cols >= 1 && cols <= APC_TILE_MAX_COLS &&
                   tl.col_begin == 0 && cols == tl.n_src && rb >= 0 && sb >= 0 && sb + cols <= n_specs && tb >= 0 && tb + rows <= n_specs &&
                   st >= 0 && st + rows <= n_strategies && tl.tensor < n_tensors && tl.dup_count >= 0 &&
                   tl.dup_count <= APC_PACKED_MAX_DUPS && tl.dup_begin >= 0 && (int64_t)tl.dup_begin + tl.dup_count <= n_dups;
      for (int64_t j = 0; holds && j < rows; ++j) holds = num_args[st + j] >= 1 && num_args[st + j] <= 0x7FFF;
      if (!holds) {
        int64_t seen = bad.load();
        while (t < seen && !bad.compare_exchange_weak(seen, t)) {
        }
        continue;
      }
      pk.rows = (int32_t)rows;
      pk.cols = (int32_t)cols;
      pk.dup_count = tl.dup_count;
      pk.tensor = tl.tensor;
      pk.edge = tl.edge;
      pk.entry_begin = tl.entry_begin + first;
      pk.row_begin = edge_row_begin[tl.edge] + rb;
      pk.pt_begin = tl.pt_begin < 0 ? -1 : tl.pt_begin + first;
      if (tl.tensor >= 0) {
        pk.tensor_rank = tensor_rank[tl.tensor];
        pk.tensor_itemsize = tensor_itemsize[tl.tensor];
        memcpy(pk.tensor_shape, tensor_shape + (int64_t)tl.tensor * APC_MAX_RANK, sizeof(pk.tensor_shape));
        memcpy(pk.tensor_stride, tensor_stride + (int64_t)tl.tensor * APC_MAX_RANK, sizeof(pk.tensor_stride));
      }
      memcpy(pk.col_codes, spec_codes + sb, 4 * (size_t)cols);
      memcpy(pk.col_tensor, spec_tensor + sb, 4 * (size_t)cols);
      memcpy(pk.row_codes, spec_codes + tb, 4 * (size_t)rows);
      memcpy(pk.row_tensor, spec_tensor + tb, 4 * (size_t)rows);
      memcpy(pk.row_flops, flops + st, 8 * (size_t)rows);
      memcpy(pk.row_rw_bytes, rw_bytes + st, 8 * (size_t)rows);
      bool mixed = false;
      for (int64_t j = 0; j < cols; ++j) mixed |= spec_tensor[sb + j] < 0 || spec_tensor[sb + j] != tl.tensor;
      for (int64_t j = 0; j < rows; ++j) {
        mixed |= spec_tensor[tb + j] < 0;
        pk.row_meta[j] = (int32_t)((uint32_t)(uint8_t)dtype_code[st + j] | ((uint32_t)(zero_cost[st + j] != 0) << 8) |
                                   ((uint32_t)num_args[st + j] << 16));
      }
      pk.flags = tl.flags | (mixed ? APC_PACKED_MIXED : 0);
      for (int d = 0; d < tl.dup_count; ++d) {
        pk.dup_entry_begin[d] = dup_entry_begin[tl.dup_begin + d] + first;
        pk.dup_row_begin[d] = dup_row_begin[tl.dup_begin + d] + rb;
      }
    }
  });
  if (bad.load() < n_tiles)
    return fail(-2, "tile %lld: rows outside the tables, not whole rows, or num_args outside 1 .. %d", (long long)bad.load(), 0x7FFF);
  return 0;
} catch (...) {
  return thrown("apc_pack_tiles_host");
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// Checks in front of the kernels, which trust their indices.
// ------------------------------------------------------------------------------------------
// The first malformed row, named: one row after the other, in order.
static int explain_rows(const apc_params *params, int64_t n_tensors, const int32_t *tensor_rank,
                        int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor,
                        int64_t n_edges, const int32_t *edge_src_begin, const int32_t *edge_n_src,
                        const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt,
                        const int32_t *edge_flags, const int64_t *edge_pt_begin,
                        const int64_t *edge_entry_begin, const int32_t *edge_strat_begin, int64_t n_pt,
                        int64_t n_strategies) {
  const int M = params->mesh_ndim;
  for (int64_t t = 0; t < n_tensors; ++t)
    if (tensor_rank[t] < 0 || tensor_rank[t] > APC_MAX_RANK)
      return fail(-2, "tensor %lld: rank %d outside [0, %d]", (long long)t, tensor_rank[t], APC_MAX_RANK);
  for (int64_t s = 0; s < n_specs; ++s) {
    const int t = spec_tensor[s];
    if (t < -1 || t >= n_tensors)
      return fail(-2, "spec %lld: tensor row %d out of range [-1, %lld)", (long long)s, t, (long long)n_tensors);
    if (M < 4 && (spec_codes[s] >> (8 * M)) != 0)
      return fail(-2, "spec %lld: placement bytes beyond mesh ndim %d are set (0x%08x)", (long long)s, M,
                  spec_codes[s]);
    for (int i = 0; i < M; ++i) {
      const uint32_t c = (spec_codes[s] >> (8 * i)) & 0xFF;
      if ((c >> 6) == 3) return fail(-2, "spec %lld: placement code 0x%02x has no meaning", (long long)s, c);
      if ((c >> 6) == 0 && c != 0) return fail(-2, "spec %lld: placement code 0x%02x has no meaning", (long long)s, c);
      if ((c >> 6) == 2 && t >= 0 && (int)(c & 0x0F) >= tensor_rank[t])
        return fail(-2, "spec %lld: Shard(%d) on a rank-%d tensor", (long long)s, (int)(c & 0x0F), tensor_rank[t]);
    }
  }
  int64_t expect = 0;
  for (int64_t e = 0; e < n_edges; ++e) {
    if (edge_entry_begin[e] != expect)
      return fail(-2, "edge %lld: entry_begin %lld, expected %lld (offsets must be the running sum of n_tgt*n_src)",
                  (long long)e, (long long)edge_entry_begin[e], (long long)expect);
    const int64_t ns = edge_n_src[e], nt = edge_n_tgt[e];
    if (ns < 0 || nt < 0) return fail(-2, "edge %lld: negative strategy count", (long long)e);
    if (ns > APC_MAX_STRATEGIES || nt > APC_MAX_STRATEGIES)
      return fail(-2, "edge %lld: %lld x %lld strategies, at most %d a side", (long long)e, (long long)nt,
                  (long long)ns, APC_MAX_STRATEGIES);
    if (edge_src_begin[e] < 0 || edge_src_begin[e] + ns > n_specs)
      return fail(-2, "edge %lld: producer spec range [%d, +%lld) outside the spec table", (long long)e,
                  edge_src_begin[e], (long long)ns);
    if (edge_tgt_begin[e] < 0 || edge_tgt_begin[e] + nt > n_specs)
      return fail(-2, "edge %lld: consumer spec range [%d, +%lld) outside the spec table", (long long)e,
                  edge_tgt_begin[e], (long long)nt);
    if (edge_strat_begin[e] < 0 || edge_strat_begin[e] + nt > n_strategies)
      return fail(-2, "edge %lld: strategy rows [%d, +%lld) outside the strategy table", (long long)e,
                  edge_strat_begin[e], (long long)nt);
    bool needs_pt = (edge_flags[e] & APC_EDGE_NO_PRODUCER) != 0;
    if (!needs_pt) {
      for (int64_t j = 0; j < ns && !needs_pt; ++j) needs_pt = spec_tensor[edge_src_begin[e] + j] < 0;
      for (int64_t j = 0; j < nt && !needs_pt; ++j) needs_pt = spec_tensor[edge_tgt_begin[e] + j] < 0;
    }
    if (needs_pt && (edge_pt_begin[e] < 0 || edge_pt_begin[e] + ns * nt > n_pt))
      return fail(-2, "edge %lld: pass-through values [%lld, +%lld) outside pt_values", (long long)e,
                  (long long)edge_pt_begin[e], (long long)(ns * nt));
    expect += ns * nt;
  }
  if (edge_entry_begin[n_edges] != expect)
    return fail(-2, "entry_begin[n_edges] = %lld, expected %lld", (long long)edge_entry_begin[n_edges],
                (long long)expect);
  return 0;
}

static int check_tiles(const int32_t *spec_tensor, int64_t n_edges, const int32_t *edge_src_begin, const int32_t *edge_n_src,
                       const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt, const int32_t *edge_flags,
                       const int64_t *edge_pt_begin, const int64_t *edge_entry_begin, const int32_t *edge_strat_begin,
                       int64_t n_tiles, const apc_tile *tiles, int64_t n_dups, const int64_t *dup_entry_begin) {
  for (int64_t t = 0; t < n_tiles; ++t) {
    const apc_tile &tl = tiles[t];
    const int e = tl.edge;
    const int row_count = tl.counts & 0xFFFF, col_count = tl.counts >> 16;
    if (e < 0 || e >= n_edges) return fail(-2, "tile %lld: edge %d out of range", (long long)t, e);
    if (row_count < 1 || row_count > APC_TILE_MAX_ROWS || tl.row_begin < 0 ||
        tl.row_begin + row_count > edge_n_tgt[e])
      return fail(-2, "tile %lld: rows [%d, +%d) outside edge %d (n_tgt %d, max %d per tile)", (long long)t,
                  tl.row_begin, row_count, e, edge_n_tgt[e], APC_TILE_MAX_ROWS);
    if (col_count < 1 || col_count > APC_TILE_MAX_COLS || tl.col_begin < 0 ||
        tl.col_begin + col_count > edge_n_src[e])
      return fail(-2, "tile %lld: cols [%d, +%d) outside edge %d (n_src %d, max %d per tile)", (long long)t,
                  tl.col_begin, col_count, e, edge_n_src[e], APC_TILE_MAX_COLS);
    if (tl.src_begin != edge_src_begin[e] || tl.n_src != edge_n_src[e] || tl.tgt_begin != edge_tgt_begin[e] ||
        tl.flags != edge_flags[e] || tl.strat_begin != edge_strat_begin[e] ||
        tl.entry_begin != edge_entry_begin[e] || tl.pt_begin != edge_pt_begin[e])
      return fail(-2, "tile %lld: record does not repeat the fields of edge %d", (long long)t, e);
    if (tl.tensor != spec_tensor[edge_src_begin[e] + tl.col_begin])
      return fail(-2, "tile %lld: tensor %d is not the tensor of its first producer spec", (long long)t, tl.tensor);
    if (tl.dup_count < 0 || tl.dup_count > APC_TILE_MAX_DUPS || tl.dup_begin < 0 ||
        (int64_t)tl.dup_begin + tl.dup_count > n_dups)
      return fail(-2, "tile %lld: duplicate list [%d, +%d) outside dup_entry_begin", (long long)t, tl.dup_begin,
                  tl.dup_count);
    for (int d = 0; d < tl.dup_count; ++d) {
      // the offset must be the start of another edge with the same matrix shape
      const int64_t off = dup_entry_begin[tl.dup_begin + d];
      int64_t lo = 0, hi = n_edges;  // first edge whose entry_begin >= off, then skip empty edges
      while (lo < hi) {
        const int64_t mid = (lo + hi) / 2;
        if (edge_entry_begin[mid] < off) lo = mid + 1; else hi = mid;
      }
      while (lo < n_edges && (int64_t)edge_n_src[lo] * edge_n_tgt[lo] == 0) ++lo;
      if (lo >= n_edges || edge_entry_begin[lo] != off || lo == e || edge_n_src[lo] != edge_n_src[e] ||
          edge_n_tgt[lo] != edge_n_tgt[e])
        return fail(-2, "tile %lld: duplicate offset %lld is not the start of an edge shaped like edge %d",
                    (long long)t, (long long)off, e);
    }
  }
  return 0;
}

// Whether every row is well formed, without saying which is not: the rows of each table side by
// side, on several threads.  (explain_rows above walks them in order; on the 430 000 specs of a
// 20 000-edge graph that took 8 ms, this 0.5 ms.)
static bool tables_hold(const apc_params *params, int64_t n_tensors, const int32_t *tensor_rank, int64_t n_specs,
                        const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t n_edges, const int32_t *edge_src_begin,
                        const int32_t *edge_n_src, const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt,
                        const int32_t *edge_flags, const int64_t *edge_pt_begin, const int64_t *edge_entry_begin,
                        const int32_t *edge_strat_begin, int64_t n_pt, int64_t n_strategies) {
  const int M = params->mesh_ndim;
  for (int64_t t = 0; t < n_tensors; ++t)
    if (tensor_rank[t] < 0 || tensor_rank[t] > APC_MAX_RANK) return false;
  // per placement byte: the smallest tensor rank it is valid on (0 for a placement that is no Shard), 99: never valid
  uint8_t least_rank[256];
  for (int c = 0; c < 256; ++c) least_rank[c] = (c >> 6) == 3 || ((c >> 6) == 0 && c != 0) ? 99 : (c >> 6) == 2 ? (c & 0x0F) + 1 : 0;
  const uint32_t beyond = M < 4 ? ~0u << (8 * M) : 0u;
  std::atomic<bool> ok{true};
  in_parallel(n_specs, threads_for(8 * n_specs), [&](int64_t b, int64_t e) {
    bool good = true;
    for (int64_t s = b; s < e; ++s) {
      const uint32_t c = spec_codes[s];
      const int t = spec_tensor[s];
      if (t < -1 || t >= n_tensors) {
        good = false;
        break;
      }
      // (no DTensorSpec: a Shard of any dim passes)
      const int rank = t >= 0 ? tensor_rank[t] : 98;
      const int need = std::max(std::max(least_rank[c & 0xFF], least_rank[(c >> 8) & 0xFF]),
                                std::max(least_rank[(c >> 16) & 0xFF], least_rank[c >> 24]));
      good &= (c & beyond) == 0 && need <= rank;
    }
    if (!good) ok.store(false, std::memory_order_relaxed);
  });
  if (!ok.load() || edge_entry_begin[0] != 0) return false;
  in_parallel(n_edges, threads_for(64 * n_edges + 8 * n_specs), [&](int64_t b, int64_t end) {
    bool good = true;
    for (int64_t e = b; e < end && good; ++e) {
      const int64_t ns = edge_n_src[e], nt = edge_n_tgt[e], sb = edge_src_begin[e], tb = edge_tgt_begin[e], st = edge_strat_begin[e];
      good = ns >= 0 && nt >= 0 && ns <= APC_MAX_STRATEGIES && nt <= APC_MAX_STRATEGIES && sb >= 0 && sb + ns <= n_specs && tb >= 0 &&
             tb + nt <= n_specs && st >= 0 && st + nt <= n_strategies && edge_entry_begin[e + 1] - edge_entry_begin[e] == ns * nt;
      if (!good || (edge_pt_begin[e] >= 0 && edge_pt_begin[e] + ns * nt <= n_pt)) continue;
      // without pass-through values: a producer and a tensor behind every spec
      bool needs_pt = (edge_flags[e] & APC_EDGE_NO_PRODUCER) != 0;
      for (int64_t j = 0; j < ns; ++j) needs_pt |= spec_tensor[sb + j] < 0;
      for (int64_t j = 0; j < nt; ++j) needs_pt |= spec_tensor[tb + j] < 0;
      good = !needs_pt;
    }
    if (!good) ok.store(false, std::memory_order_relaxed);
  });
  return ok.load();
}

extern "C" {

int apc_validate_tables_host(const apc_params *params, int64_t n_tensors, const int32_t *tensor_rank,
                             int64_t n_specs, const uint32_t *spec_codes, const int32_t *spec_tensor,
                             int64_t n_edges, const int32_t *edge_src_begin, const int32_t *edge_n_src,
                             const int32_t *edge_tgt_begin, const int32_t *edge_n_tgt,
                             const int32_t *edge_flags, const int64_t *edge_pt_begin,
                             const int64_t *edge_entry_begin, const int32_t *edge_strat_begin, int64_t n_pt,
                             int64_t n_strategies, int64_t n_tiles, const apc_tile *tiles, int64_t n_dups,
                             const int64_t *dup_entry_begin) try {
  if (int rc = check_params(params)) return rc;
  if (!tables_hold(params, n_tensors, tensor_rank, n_specs, spec_codes, spec_tensor, n_edges, edge_src_begin, edge_n_src,
                   edge_tgt_begin, edge_n_tgt, edge_flags, edge_pt_begin, edge_entry_begin, edge_strat_begin, n_pt, n_strategies))
    if (int rc = explain_rows(params, n_tensors, tensor_rank, n_specs, spec_codes, spec_tensor, n_edges, edge_src_begin, edge_n_src,
                              edge_tgt_begin, edge_n_tgt, edge_flags, edge_pt_begin, edge_entry_begin, edge_strat_begin, n_pt, n_strategies))
      return rc;
  return check_tiles(spec_tensor, n_edges, edge_src_begin, edge_n_src, edge_tgt_begin, edge_n_tgt, edge_flags, edge_pt_begin,
                     edge_entry_begin, edge_strat_begin, n_tiles, tiles, n_dups, dup_entry_begin);
} catch (...) {
  return thrown("apc_validate_tables_host");
}

int apc_validate_row_minima_host(int64_t n_edges, const int32_t *edge_n_src, const int32_t *edge_n_tgt, int64_t n_tiles,
                                 const apc_tile *tiles) {
  if (n_edges < 0 || n_tiles < 0) return fail(-1, "apc_validate_row_minima_host: negative count");
  if ((n_edges > 0 && (!edge_n_src || !edge_n_tgt)) || (n_tiles > 0 && !tiles))
    return fail(-1, "apc_validate_row_minima_host: NULL array");
  for (int64_t e = 0; e < n_edges; ++e)
    if (edge_n_tgt[e] > 0 && (edge_n_src[e] < 1 || edge_n_src[e] > APC_TILE_MAX_COLS))
      return fail(-2, "edge %lld: %d producer strategies; row minima inside the table launch need 1 .. %d", (long long)e,
                  edge_n_src[e], APC_TILE_MAX_COLS);
  for (int64_t t = 0; t < n_tiles; ++t) {
    const apc_tile &tl = tiles[t];
    if (tl.edge < 0 || tl.edge >= n_edges) return fail(-2, "tile %lld: edge %d out of range", (long long)t, tl.edge);
    if (tl.col_begin != 0 || (tl.counts >> 16) != edge_n_src[tl.edge])
      return fail(-2, "tile %lld: columns [%d, +%d) are not the whole rows of edge %d (%d columns)", (long long)t,
                  tl.col_begin, tl.counts >> 16, tl.edge, edge_n_src[tl.edge]);
  }
  return 0;
}

int apc_validate_packed_tiles_host(int64_t n_tensors, const int32_t *tensor_rank, const int32_t *tensor_itemsize,
                                   const int64_t *tensor_shape, const int64_t *tensor_stride, int64_t n_specs,
                                   const uint32_t *spec_codes, const int32_t *spec_tensor, int64_t n_strategies,
                                   const int64_t *flops, const int64_t *rw_bytes, const int8_t *dtype_code,
                                   const uint8_t *zero_cost, const int32_t *num_args, int64_t n_edges,
                                   const int64_t *edge_row_begin, int64_t n_tiles, const apc_tile *tiles, int64_t n_dups,
                                   const int64_t *dup_entry_begin, const int64_t *dup_row_begin,
                                   const apc_packed_tile *packed) {
  if (n_tiles < 0 || n_tensors < 0 || n_specs < 0 || n_strategies < 0 || n_edges < 0 || n_dups < 0)
    return fail(-1, "apc_validate_packed_tiles_host: negative count");
  if (n_tiles == 0) return 0;
  if (!tiles || !packed || !spec_codes || !spec_tensor || !edge_row_begin || !flops || !rw_bytes || !dtype_code || !zero_cost ||
      !num_args || (n_dups > 0 && (!dup_entry_begin || !dup_row_begin)) ||
      (n_tensors > 0 && (!tensor_rank || !tensor_itemsize || !tensor_shape || !tensor_stride)))
    return fail(-1, "apc_validate_packed_tiles_host: NULL array");
  for (int64_t t = 0; t < n_tiles; ++t) {
    const apc_tile &tl = tiles[t];
    const apc_packed_tile &pk = packed[t];
    const int rows = tl.counts & 0xFFFF, cols = tl.counts >> 16;
    if (tl.edge < 0 || tl.edge >= n_edges) return fail(-2, "tile %lld: edge %d out of range", (long long)t, tl.edge);
    if (tl.col_begin != 0 || cols != tl.n_src || cols < 1 || cols > APC_TILE_MAX_COLS || rows < 1 || rows > APC_TILE_MAX_ROWS)
      return fail(-2, "tile %lld: a packed tile holds 1 .. %d whole rows of at most %d columns (%d rows, columns [%d, +%d) of %d)",
                  (long long)t, APC_TILE_MAX_ROWS, APC_TILE_MAX_COLS, rows, tl.col_begin, cols, tl.n_src);
    if (tl.dup_count < 0 || tl.dup_count > APC_PACKED_MAX_DUPS || tl.dup_begin < 0 || (int64_t)tl.dup_begin + tl.dup_count > n_dups)
      return fail(-2, "tile %lld: %d identical edges, a packed tile serves at most %d", (long long)t, tl.dup_count,
                  APC_PACKED_MAX_DUPS);
    if (tl.src_begin < 0 || (int64_t)tl.src_begin + cols > n_specs || tl.tgt_begin < 0 ||
        (int64_t)tl.tgt_begin + tl.row_begin + rows > n_specs || tl.strat_begin < 0 ||
        (int64_t)tl.strat_begin + tl.row_begin + rows > n_strategies)
      return fail(-2, "tile %lld: spec or strategy rows outside their tables", (long long)t);
    const int64_t first = (int64_t)tl.row_begin * cols;
    bool mixed = false;
    for (int j = 0; j < cols; ++j) {
      const int64_t sp = (int64_t)tl.src_begin + j;
      if (pk.col_codes[j] != spec_codes[sp] || pk.col_tensor[j] != spec_tensor[sp])
        return fail(-2, "packed tile %lld: producer spec %d differs from the spec table", (long long)t, j);
      mixed |= spec_tensor[sp] < 0 || spec_tensor[sp] != tl.tensor;
    }
    for (int j = 0; j < rows; ++j) {
      const int64_t ts = (int64_t)tl.tgt_begin + tl.row_begin + j, sr = (int64_t)tl.strat_begin + tl.row_begin + j;
      if (pk.row_codes[j] != spec_codes[ts] || pk.row_tensor[j] != spec_tensor[ts])
        return fail(-2, "packed tile %lld: consumer spec %d differs from the spec table", (long long)t, j);
      mixed |= spec_tensor[ts] < 0;
      if (num_args[sr] < 1 || num_args[sr] > 0x7FFF)
        return fail(-2, "packed tile %lld: num_args %d of consumer strategy %d does not fit its 15 bits", (long long)t,
                    num_args[sr], j);
      const int32_t meta = (int32_t)(uint8_t)dtype_code[sr] | ((int32_t)(zero_cost[sr] != 0) << 8) | (num_args[sr] << 16);
      if (pk.row_flops[j] != flops[sr] || pk.row_rw_bytes[j] != rw_bytes[sr] || pk.row_meta[j] != meta)
        return fail(-2, "packed tile %lld: consumer strategy %d differs from the strategy table", (long long)t, j);
    }
    if (pk.rows != rows || pk.cols != cols || pk.dup_count != tl.dup_count || pk.tensor != tl.tensor || pk.edge != tl.edge ||
        pk.flags != (tl.flags | (mixed ? APC_PACKED_MIXED : 0)) || pk.entry_begin != tl.entry_begin + first ||
        pk.row_begin != edge_row_begin[tl.edge] + tl.row_begin || pk.pt_begin != (tl.pt_begin < 0 ? -1 : tl.pt_begin + first))
      return fail(-2, "packed tile %lld: header does not repeat the fields of tile record %lld", (long long)t, (long long)t);
    if (tl.tensor >= 0) {
      if (tl.tensor >= n_tensors) return fail(-2, "tile %lld: tensor %d out of range", (long long)t, tl.tensor);
      if (pk.tensor_rank != tensor_rank[tl.tensor] || pk.tensor_itemsize != tensor_itemsize[tl.tensor] ||
          memcmp(pk.tensor_shape, tensor_shape + (int64_t)tl.tensor * APC_MAX_RANK, sizeof(pk.tensor_shape)) != 0 ||
          memcmp(pk.tensor_stride, tensor_stride + (int64_t)tl.tensor * APC_MAX_RANK, sizeof(pk.tensor_stride)) != 0)
        return fail(-2, "packed tile %lld: tensor row differs from the tensor table", (long long)t);
    }
    for (int d = 0; d < tl.dup_count; ++d)
      if (pk.dup_entry_begin[d] != dup_entry_begin[tl.dup_begin + d] + first ||
          pk.dup_row_begin[d] != dup_row_begin[tl.dup_begin + d] + tl.row_begin)
        return fail(-2, "packed tile %lld: identical edge %d differs from the duplicate lists", (long long)t, d);
  }
  return 0;
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// Rounding and pruning of a labelling problem (apc_diffusion_sweeps states its arrays): the host's
// part between two calls of the sweeps.  Sums in incidence order, one rounding per addition.
// ------------------------------------------------------------------------------------------
namespace {

// As numpy takes minima: of values with a NaN among them a NaN.  The running minima pass one over; whether there may be
// one is read off the values' sum, a NaN for any (and where infinities cancel), at one addition a value.
inline double with_nan(const double *v, int64_t n, int64_t stride = 1) {
  double d = __builtin_inf();
  for (int64_t i = 0; i < n; ++i) {
    const double x = v[i * stride];
    d = x < d || x != x ? x : d;
  }
  return d;
}

// (a loop of its own: in one with the comparisons neither becomes vector instructions)
inline void add_up(const double *v, int64_t n, double (&s)[8]) {
  int64_t i = 0;
  for (; i + 8 <= n; i += 8)
    for (int j = 0; j < 8; ++j) s[j] += v[i + j];
  for (; i < n; ++i) s[0] += v[i];
}

inline bool may_hold_nan(const double (&s)[8]) {
  const double t = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
  return t != t;
}

// The smallest of n values, +inf of none (eight running minima: the order of the comparisons is free), NaN passed over.
inline double least_number(const double *v, int64_t n) {
  double d[8];
  for (double &x : d) x = __builtin_inf();
  int64_t i = 0;
  for (; i + 8 <= n; i += 8)
    for (int j = 0; j < 8; ++j) d[j] = v[i + j] < d[j] ? v[i + j] : d[j];
  for (; i < n; ++i) d[0] = v[i] < d[0] ? v[i] : d[0];
  for (int j = 1; j < 8; ++j) d[0] = d[j] < d[0] ? d[j] : d[0];
  return d[0];
}

double least(const double *v, int64_t n) {
  double d = __builtin_inf(), s[8] = {};
  for (int64_t i = 0; i < n; i += 1024) {  // (runs that stay in the first cache between the two loops)
    const int64_t run = std::min<int64_t>(1024, n - i);
    const double x = least_number(v + i, run);
    d = x < d ? x : d;
    add_up(v + i, run, s);
  }
  return may_hold_nan(s) ? with_nan(v, n) : d;
}

struct LabelProblem {
  int64_t n_classes, n_edges;
  const int64_t *label_begin, *inc_begin;
  const int32_t *inc_edge;
  const uint8_t *inc_side;
  const int64_t *edge_begin;
  const int32_t *edge_i, *edge_j;
  const double *theta, *unary;
  bool theta_may_hold_nan = false;  // (where minima() is used: look_for_nan() first)

  void look_for_nan() {
    std::atomic<bool> found{false};
    const int64_t n = edge_begin[n_edges], runs = (n + 4095) / 4096;
    in_parallel(runs, threads_for(4 * n), [&](int64_t b, int64_t e) {
      double s[8] = {};
      add_up(theta + b * 4096, std::min(n, e * 4096) - b * 4096, s);
      if (may_hold_nan(s)) found.store(true, std::memory_order_relaxed);
    });
    theta_may_hold_nan = found.load();
  }
  int64_t labels(int64_t c) const { return label_begin[c + 1] - label_begin[c]; }
  int64_t other(int64_t k, int side) const { return side == 0 ? edge_j[k] : edge_i[k]; }
  // every index the walks below use lies inside its array, and every matrix has its classes' shape
  bool holds() const {
    if (n_classes < 0 || n_edges < 0 || !label_begin || !inc_begin || !edge_begin || label_begin[0] != 0 || inc_begin[0] != 0 || edge_begin[0] != 0)
      return false;
    for (int64_t c = 0; c < n_classes; ++c)
      if (label_begin[c + 1] < label_begin[c] || inc_begin[c + 1] < inc_begin[c]) return false;
    for (int64_t k = 0; k < n_edges; ++k) {
      if (edge_i[k] < 0 || edge_i[k] >= n_classes || edge_j[k] < 0 || edge_j[k] >= n_classes) return false;
      if (edge_begin[k + 1] - edge_begin[k] != labels(edge_i[k]) * labels(edge_j[k])) return false;
    }
    for (int64_t c = 0; c < n_classes; ++c)
      for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
        const int64_t k = inc_edge[t];
        if (k < 0 || k >= n_edges || inc_side[t] > 1 || (inc_side[t] == 0 ? edge_i[k] : edge_j[k]) != c) return false;
      }
    return true;
  }
  bool has_empty_matrix() const {
    for (int64_t k = 0; k < n_edges; ++k)
      if (edge_begin[k + 1] == edge_begin[k]) return true;
    return false;
  }
  // out[x] = min over the other end's labels of the matrix of edge k, x a label of the class on side `side`
  void minima(int64_t k, int side, double *out) const {
    const double *m = theta + edge_begin[k];
    const int64_t ni = labels(edge_i[k]), nj = labels(edge_j[k]);
    if (theta_may_hold_nan) {
      for (int64_t x = 0; x < (side == 0 ? ni : nj); ++x) out[x] = side == 0 ? with_nan(m + x * nj, nj) : with_nan(m + x, ni, nj);
    } else if (side == 0) {
      for (int64_t x = 0; x < ni; ++x) out[x] = least_number(m + x * nj, nj);
    } else {
      for (int64_t y = 0; y < nj; ++y) out[y] = __builtin_inf();
      for (int64_t x = 0; x < ni; ++x)
        for (int64_t y = 0; y < nj; ++y) out[y] = m[x * nj + y] < out[y] ? m[x * nj + y] : out[y];
    }
  }
  // score[x] += the matrix of edge k at (x, label of the other end)
  void add_fixed(int64_t k, int side, int64_t label, double *score) const {
    const double *m = theta + edge_begin[k];
    const int64_t ni = labels(edge_i[k]), nj = labels(edge_j[k]);
    if (side == 0)
      for (int64_t x = 0; x < ni; ++x) score[x] += m[x * nj + label];
    else
      for (int64_t y = 0; y < nj; ++y) score[y] += m[label * nj + y];
  }
};

int64_t first_minimum(const double *v, int64_t n) {
  int64_t at = 0;
  double sum = n > 0 ? v[0] : 0.0;
  for (int64_t i = 1; i < n; ++i) {
    if (v[i] < v[at]) at = i;
    sum += v[i];
  }
  if (sum != sum)  // (the first NaN, if there is one)
    for (int64_t i = 0; i < n; ++i)
      if (v[i] != v[i]) return i;
  return at;
}

}  // namespace

extern "C" {

int apc_label_incidence_host(int64_t n_classes, int64_t n_edges, const int32_t *edge_i, const int32_t *edge_j, int64_t *inc_begin,
                             int32_t *inc_edge, uint8_t *inc_side, int64_t *color) try {
  if (n_classes < 0 || n_edges < 0 || !inc_begin || (n_classes > 0 && !color) || (n_edges > 0 && (!edge_i || !edge_j || !inc_edge || !inc_side)))
    return fail(-1, "apc_label_incidence_host: NULL array or negative count");
  for (int64_t k = 0; k < n_edges; ++k)
    if (edge_i[k] < 0 || edge_i[k] >= n_classes || edge_j[k] < 0 || edge_j[k] >= n_classes)
      return fail(-2, "edge %lld: classes %d, %d outside [0, %lld)", (long long)k, edge_i[k], edge_j[k], (long long)n_classes);
  std::fill(inc_begin, inc_begin + n_classes + 1, 0);
  for (int64_t k = 0; k < n_edges; ++k) ++inc_begin[edge_i[k] + 1], ++inc_begin[edge_j[k] + 1];
  for (int64_t c = 0; c < n_classes; ++c) inc_begin[c + 1] += inc_begin[c];
  std::vector<int64_t> next(inc_begin, inc_begin + n_classes);
  for (int64_t k = 0; k < n_edges; ++k)
    for (int side = 0; side < 2; ++side) {
      const int64_t at = next[side == 0 ? edge_i[k] : edge_j[k]]++;
      inc_edge[at] = (int32_t)k;
      inc_side[at] = (uint8_t)side;
    }
  std::vector<int64_t> used_by;  // colour -> the last class that saw it on a neighbour
  for (int64_t c = 0; c < n_classes; ++c) color[c] = -1;
  for (int64_t c = 0; c < n_classes; ++c) {
    for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
      const int64_t k = inc_edge[t], col = color[inc_side[t] == 0 ? edge_j[k] : edge_i[k]];
      if (col >= 0) used_by[col] = c;
    }
    int64_t col = 0;
    while (col < (int64_t)used_by.size() && used_by[col] == c) ++col;
    if (col == (int64_t)used_by.size()) used_by.push_back(-1);
    color[c] = col;
  }
  return 0;
} catch (...) {
  return thrown("apc_label_incidence_host");
}

#define APC_LABEL_PROBLEM                                                                                                     \
  int64_t n_classes, const int64_t *label_begin, const int64_t *inc_begin, const int32_t *inc_edge, const uint8_t *inc_side,  \
      int64_t n_edges, const int64_t *edge_begin, const int32_t *edge_i, const int32_t *edge_j, const double *theta,          \
      const double *unary
#define APC_LABEL_PROBLEM_OF(who)                                                                                             \
  LabelProblem g{n_classes, n_edges, label_begin, inc_begin, inc_edge, inc_side, edge_begin, edge_i, edge_j, theta, unary};      \
  if (!g.holds()) return fail(-2, who ": the index arrays do not describe a labelling problem");                               \
  if (g.has_empty_matrix()) return fail(-2, who ": a matrix of a class without labels has no minimum")

int apc_label_minima_host(APC_LABEL_PROBLEM, double *class_min, double *edge_min) try {
  APC_LABEL_PROBLEM_OF("apc_label_minima_host");
  for (int64_t c = 0; c < n_classes; ++c) {
    const int64_t b = label_begin[c], e = label_begin[c + 1];
    class_min[c] = e > b ? unary[b + first_minimum(unary + b, e - b)] : 0.0;
  }
  in_parallel(n_edges, threads_for(4 * edge_begin[n_edges]), [&](int64_t b, int64_t e) {
    for (int64_t k = b; k < e; ++k) edge_min[k] = least(theta + edge_begin[k], edge_begin[k + 1] - edge_begin[k]);
  });
  return 0;
} catch (...) {
  return thrown("apc_label_minima_host");
}

int apc_round_labels_host(APC_LABEL_PROBLEM, int64_t *labels) try {
  APC_LABEL_PROBLEM_OF("apc_round_labels_host");
  g.look_for_nan();
  std::vector<double> score, d;
  for (int64_t c = 0; c < n_classes; ++c) labels[c] = -1;
  for (int64_t c = 0; c < n_classes; ++c) {
    const int64_t n = g.labels(c);
    score.assign(unary + label_begin[c], unary + label_begin[c + 1]);
    d.resize(n);
    for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
      const int64_t k = inc_edge[t];
      const int side = inc_side[t];
      const int64_t fixed = labels[g.other(k, side)];
      if (fixed >= 0) {
        g.add_fixed(k, side, fixed, score.data());
      } else {
        g.minima(k, side, d.data());
        for (int64_t x = 0; x < n; ++x) score[x] += d[x];
      }
    }
    if (n > 0) labels[c] = first_minimum(score.data(), n);
  }
  return 0;
} catch (...) {
  return thrown("apc_round_labels_host");
}

int apc_refine_labels_host(APC_LABEL_PROBLEM, int64_t max_rounds, int64_t *labels) try {
  APC_LABEL_PROBLEM_OF("apc_refine_labels_host");
  for (int64_t c = 0; c < n_classes; ++c)
    if (labels[c] < -1 || labels[c] >= g.labels(c)) return fail(-2, "apc_refine_labels_host: label %lld of class %lld", (long long)labels[c], (long long)c);
  std::vector<uint8_t> todo(n_classes, 1), again(n_classes);
  std::vector<double> score;
  for (int64_t round = 0; round < max_rounds; ++round) {
    std::fill(again.begin(), again.end(), 0);
    bool any = false;
    for (int64_t c = 0; c < n_classes; ++c) {
      if (!todo[c] || labels[c] < 0) continue;
      score.assign(unary + label_begin[c], unary + label_begin[c + 1]);
      for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
        const int64_t k = inc_edge[t], o = g.other(k, inc_side[t]);
        // (a neighbour without labels has nothing to fix)
        if (labels[o] >= 0) g.add_fixed(k, inc_side[t], labels[o], score.data());
      }
      const int64_t best = first_minimum(score.data(), g.labels(c));
      if (score[best] < score[labels[c]]) {
        labels[c] = best;
        for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) again[g.other(inc_edge[t], inc_side[t])] = 1, any = true;
      }
    }
    if (!any) break;
    todo.swap(again);
  }
  return 0;
} catch (...) {
  return thrown("apc_refine_labels_host");
}

int apc_prune_masks_host(APC_LABEL_PROBLEM, const double *class_min, const double *edge_min, double bound, double limit,
                         uint8_t *dead_label, uint8_t *dead_pair) try {
  APC_LABEL_PROBLEM_OF("apc_prune_masks_host");
  g.look_for_nan();
  const int threads = threads_for(8 * edge_begin[n_edges]);
  in_parallel(n_classes, threads, [&](int64_t begin, int64_t end) {
    std::vector<double> b, d;
    for (int64_t c = begin; c < end; ++c) {
      const int64_t n = g.labels(c), l0 = label_begin[c];
      b.resize(n);
      d.resize(n);
      for (int64_t x = 0; x < n; ++x) b[x] = (bound - class_min[c]) + unary[l0 + x];
      for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
        const int64_t k = inc_edge[t];
        g.minima(k, inc_side[t], d.data());
        for (int64_t x = 0; x < n; ++x) b[x] = (b[x] - edge_min[k]) + d[x];
      }
      for (int64_t x = 0; x < n; ++x) dead_label[l0 + x] = !(b[x] <= limit);  // (NaN: dead)
    }
  });
  in_parallel(n_edges, threads, [&](int64_t begin, int64_t end) {
    for (int64_t k = begin; k < end; ++k) {
      const int64_t ni = g.labels(edge_i[k]), nj = g.labels(edge_j[k]);
      const uint8_t *di = dead_label + label_begin[edge_i[k]], *dj = dead_label + label_begin[edge_j[k]];
      const double *m = theta + edge_begin[k], rest = bound - edge_min[k];
      uint8_t *out = dead_pair + edge_begin[k];
      for (int64_t x = 0; x < ni; ++x)
        for (int64_t y = 0; y < nj; ++y) out[x * nj + y] = (uint8_t)(!(rest + m[x * nj + y] <= limit)) | di[x] | dj[y];
    }
  });
  return 0;
} catch (...) {
  return thrown("apc_prune_masks_host");
}

// ------------------------------------------------------------------------------------------
// Which workgroup of apc_diffusion_sweeps_resident holds which matrices, and what it needs to know
// about them: the layout is stated at the kernel (ResidentPlan in apcost.hip).
// ------------------------------------------------------------------------------------------
int apc_sweep_plan_host(int64_t n_classes, const int64_t *label_begin, const int64_t *inc_begin, const int32_t *inc_edge,
                        const uint8_t *inc_side, int64_t n_edges, const int64_t *edge_begin, const int32_t *edge_i,
                        const int32_t *edge_j, int64_t n_colors, const int64_t *color_begin, const int32_t *color_nodes,
                        int64_t max_workgroups, int64_t capacity_words, int32_t *plan, int64_t *plan_begin, int64_t *sizes) try {
  const LabelProblem g{n_classes, n_edges, label_begin, inc_begin, inc_edge, inc_side, edge_begin, edge_i, edge_j, nullptr, nullptr};
  if (!g.holds()) return fail(-2, "apc_sweep_plan_host: the index arrays do not describe a labelling problem");
  if (!plan || !plan_begin || !sizes || !color_begin || max_workgroups < 1 || n_colors < 0) return fail(-1, "apc_sweep_plan_host: NULL array or no workgroup");
  std::fill(sizes, sizes + 5, 0);
  if (color_begin[0] != 0 || color_begin[n_colors] != n_classes) return fail(-2, "apc_sweep_plan_host: the colours must partition the classes");
  std::vector<int32_t> color(n_classes, -1);
  for (int64_t c = 0; c < n_colors; ++c)
    for (int64_t k = color_begin[c]; k < color_begin[c + 1]; ++k) {
      if (k < 0 || k >= n_classes || color_nodes[k] < 0 || color_nodes[k] >= n_classes) return fail(-2, "apc_sweep_plan_host: class out of range");
      color[color_nodes[k]] = (int32_t)c;
    }
  for (int64_t k = 0; k < n_edges; ++k)
    if (color[edge_i[k]] < 0 || color[edge_j[k]] < 0 || color[edge_i[k]] == color[edge_j[k]])
      return fail(-2, "apc_sweep_plan_host: edge %lld joins two classes of one colour", (long long)k);
  for (int64_t k = 0; k < n_edges; ++k)
    if (edge_begin[k + 1] == edge_begin[k]) return 0;  // (an empty matrix: left to the launches)
  if (n_edges == 0) return 0;  // (no plan: sizes[0] stays 0)
  const int64_t total = edge_begin[n_edges];
  std::vector<int32_t> owner(n_edges);
  int64_t lds = 0, n_wg = 0, threads = 0;
  auto deep = [&](int64_t c) { return inc_begin[c + 1] - inc_begin[c] > 4; };
  // By teams: a matrix has wavefronts of its own, as many as leave one `per_wave` elements and a lane a row; the workgroups
  // take them in order.
  struct Team {
    int64_t first_wave, waves;
  };
  std::vector<Team> teams(n_edges);
  auto team_bytes = [&](int64_t el, int64_t r, int64_t in) { return 32 * r + 8 * el + 4 * (in + APC_SWEEP_MAX_WAVES + 1); };
  auto by_teams = [&](int64_t per_wave, int64_t most_waves) {
    std::vector<int64_t> seen(n_classes, -1);  // the last workgroup that met the class
    int64_t elements = 0, rows = 0, incs = 0, waves = 0, words = 0;
    n_wg = lds = 0;
    for (int64_t k = 0; k < n_edges; ++k) {
      const int64_t size = edge_begin[k + 1] - edge_begin[k], ni = g.labels(edge_i[k]), nj = g.labels(edge_j[k]);
      int64_t w = 1;
      while (w < most_waves && (std::max(ni, nj) > 64 * w || size > per_wave * w)) w *= 2;
      if (std::max(ni, nj) > 64 * w || (w < APC_SWEEP_MAX_WAVES && size > 2 * per_wave * w)) return false;
      for (int attempt = 0;; ++attempt) {
        int64_t in = incs;
        for (int64_t c : {edge_i[k], edge_j[k]})
          if (seen[c] != n_wg && deep(c)) in += inc_begin[c + 1] - inc_begin[c];
        if (waves + w <= most_waves && team_bytes(elements + size, rows + ni + nj, in) <= APC_SWEEP_LDS_BYTES && elements + size <= 0x10000 && in <= 0xFFFF) {
          teams[k] = {waves, w};
          elements += size, rows += ni + nj, incs = in, waves += w;
          seen[edge_i[k]] = seen[edge_j[k]] = n_wg;
          lds = std::max(lds, team_bytes(elements, rows, incs));
          owner[k] = (int32_t)n_wg;
          break;
        }
        if (attempt == 1) return false;
        words += 8 + 9 * rows + incs + 4 * APC_SWEEP_MAX_WAVES + 3;
        if (++n_wg >= max_workgroups) return false;
        elements = rows = incs = waves = 0;
      }
    }
    words += 8 + 9 * rows + incs + 4 * APC_SWEEP_MAX_WAVES + 3;
    ++n_wg;
    return words <= capacity_words;
  };
  // Edges in order, workgroup by workgroup, until its share of the elements, its threads (one per row of a step)
  // or its memory is full.  (Neighbouring edges of a planning program share classes: kept together, most
  // exchanges stay inside a workgroup.)  256 threads, one wavefront per SIMD, unless that takes too many workgroups.
  int64_t share = std::max<int64_t>(APC_SWEEP_MIN_ELEMENTS, (total + APC_SWEEP_AIM_WORKGROUPS - 1) / APC_SWEEP_AIM_WORKGROUPS);
  auto bytes = [&](int64_t el, int64_t r, int64_t in) { return 8 * (el + 1) + (32 + 8 + 8) * r + 8 * 64 + 4 * in + 4 * (n_colors + 1) + 16; };
  auto assign = [&](int64_t threads) {
    std::vector<int64_t> seen(n_classes, -1);  // the last workgroup that met the class
    std::vector<int64_t> step_rows(n_colors, 0);
    int64_t elements = 0, rows = 0, incs = 0;
    n_wg = lds = 0;
    for (int64_t k = 0; k < n_edges; ++k) {
      const int64_t size = edge_begin[k + 1] - edge_begin[k], ni = g.labels(edge_i[k]), nj = g.labels(edge_j[k]);
      for (int attempt = 0;; ++attempt) {
        int64_t in = incs;
        for (int64_t c : {edge_i[k], edge_j[k]})
          if (seen[c] != n_wg) in += inc_begin[c + 1] - inc_begin[c];
        int64_t &ri = step_rows[color[edge_i[k]]], &rj = step_rows[color[edge_j[k]]];
        const bool fits = bytes(elements + size, rows + ni + nj, in) <= APC_SWEEP_LDS_BYTES && elements + size <= 0x10000 && in <= 0xFFFF &&
                          ri + ni <= threads && rj + nj <= threads;
        if (fits && (rows == 0 || elements + size <= share)) {
          elements += size, rows += ni + nj, incs = in, ri += ni, rj += nj;
          seen[edge_i[k]] = seen[edge_j[k]] = n_wg;
          lds = std::max(lds, bytes(elements, rows, incs));
          owner[k] = (int32_t)n_wg;
          break;
        }
        if (attempt == 1 || rows == 0) return false;  // one matrix alone does not fit
        ++n_wg;
        elements = rows = incs = 0;
        std::fill(step_rows.begin(), step_rows.end(), 0);
      }
    }
    return ++n_wg <= max_workgroups;
  };
  // One workgroup that exchanges nothing, else teams (four wavefronts a SIMD where two make too many workgroups, and then more elements a
  // wavefront), else runs.  (Figures at the kernels.  Eight wavefronts a workgroup against sixteen, us a sweep: 358 matrices of at
  // most 24 labels 3.5 / 4.4, 794 of 40 9.3 / 11.0; 512 elements a wavefront against 1 024: 1 428 matrices of at most 64 labels 8.1 /
  // 8.5, 358 of 124 6.7 / 7.4.)
  //   With two colours a sweep of the runs is two steps, and small matrices are little work between them.  us a sweep, runs / teams, of at most
  //   so many labels with so many elements a matrix: 300 of 3 (4) 2.4 / 2.9, 200 of 5 (8) 3.0 / 3.4, 40 of 5 (9) 2.8 / 3.5; then 500 of 6 (13) 3.7 / 3.3, 60
  //   of 7 (14) 2.9 / 2.4, 300 of 8 (20) 2.9 / 2.7, though 80 of 6 (13) 3.1 / 3.7 and 30 of 7 (13) 3.2 / 4.1.  With sixteen wavefronts a workgroup 1 900 of 4 (6)
  //   3.6 / 5.2, 2 600 of 10 (30) 4.4 / 6.7, 1 900 of 12 (42) 4.3 / 4.9; then 2 600 of 14 (56) 4.1 / 3.3, 1 900 of 16 (72) 4.6 / 3.5.  With three colours and more a
  //   step more a sweep decides for the teams (315 of 3 (2) 3.7 / 2.8, 659 of 5 (5) 4.7 / 3.7), short of 64 matrices of 5 labels 3.2 / 3.8.
  bool of_teams = false;
  if (total > APC_SWEEP_MIN_ELEMENTS || !assign(threads = 256) || n_wg > 1) {
    constexpr struct {
      int64_t waves, per_wave, elements_of_two_colours;
    } kForms[] = {{APC_SWEEP_MAX_WAVES / 2, 512, 10}, {APC_SWEEP_MAX_WAVES, 512, 48}, {APC_SWEEP_MAX_WAVES, 1024, 48}, {APC_SWEEP_MAX_WAVES, 2048, 48}, {APC_SWEEP_MAX_WAVES, 4096, 48}};
    auto teams_hold = [&](bool small_too) {
      for (const auto &form : kForms)
        if ((small_too || n_colors > 2 || total >= form.elements_of_two_colours * n_edges) && by_teams(form.per_wave, form.waves)) {
          threads = 64 * form.waves;
          return true;
        }
      return false;
    };
    of_teams = teams_hold(false);
    // (the matrices do not fill the shares exactly: larger ones until the workgroups are few enough)
    for (int attempt = 0; !of_teams; ++attempt, share += share / 4) {
      threads = share > APC_SWEEP_WIDE_ELEMENTS ? 1024 : 256;
      if (assign(threads) || assign(threads = 1024)) break;
      if (attempt == 12 && !(of_teams = teams_hold(true))) return 0;
    }
  }
  // classes whose matrices lie in several workgroups exchange their minima through memory: a slot per (incidence, label)
  std::vector<int64_t> slot(inc_begin[n_classes], -1);
  int64_t n_slots = 0;
  for (int64_t c = 0; c < n_classes; ++c) {
    bool shared = false;
    for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) shared |= owner[inc_edge[t]] != owner[inc_edge[inc_begin[c]]];
    if (!shared) continue;
    for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) {
      slot[t] = n_slots;
      n_slots += g.labels(c);
    }
  }
  if (n_slots > (of_teams ? 0x3FFFFFF : 0x3FFFFFFF) || total > INT32_MAX) return 0;
  std::vector<int64_t> inc_of(2 * n_edges);  // (edge, side) -> incidence
  for (int64_t t = 0; t < inc_begin[n_classes]; ++t) inc_of[2 * (int64_t)inc_edge[t] + inc_side[t]] = t;
  int64_t at = 0;
  std::vector<int64_t> row_of(2 * n_edges, 0), inc_at(n_classes, 0), met(n_classes, -1);
  for (int64_t w = 0, first = 0; w < n_wg; ++w) {
    int64_t last = first;
    while (last < n_edges && owner[last] == w) ++last;
    struct Side {  // one side of an edge: the rows of its class
      int64_t k;
      int side;
      int64_t c;
    };
    std::vector<Side> sides;
    for (int64_t k = first; k < last; ++k) sides.push_back({k, 0, edge_i[k]}), sides.push_back({k, 1, edge_j[k]});
    std::stable_sort(sides.begin(), sides.end(), [&](const Side &x, const Side &y) {
      return of_teams && x.k != y.k ? x.k < y.k : color[x.c] < color[y.c];
    });
    int64_t n_rows = 0, n_inc = 0, n_el = 0;
    std::vector<int64_t> classes;
    std::vector<int64_t> steps;  // first rows of the colours that have any
    int32_t last_color = -1;
    for (const Side &x : sides) {
      if (color[x.c] != last_color) {
        steps.push_back(n_rows);
        last_color = color[x.c];
      }
      row_of[2 * x.k + x.side] = n_rows;
      n_rows += g.labels(x.c);
      if (met[x.c] != w && (!of_teams || deep(x.c))) {
        met[x.c] = w;
        classes.push_back(x.c);
        inc_at[x.c] = n_inc;
        n_inc += inc_begin[x.c + 1] - inc_begin[x.c];
      }
    }
    steps.push_back(n_rows);
    std::vector<int64_t> el_of(last - first);
    for (int64_t k = first; k < last; ++k) {
      el_of[k - first] = n_el;
      n_el += edge_begin[k + 1] - edge_begin[k];
    }
    const int64_t words = (8 + 9 * n_rows + n_inc + (of_teams ? 4 * APC_SWEEP_MAX_WAVES : (int64_t)steps.size()) + 3) / 4 * 4;
    if (at + words > capacity_words) return fail(-1, "apc_sweep_plan_host: the plan does not fit %lld words", (long long)capacity_words);
    plan_begin[w] = at;
    int32_t *p = plan + at;
    std::fill(p, p + words, 0);
    p[0] = (int32_t)edge_begin[first];  // (a workgroup's edges are consecutive: one run of theta)
    p[1] = (int32_t)n_el;
    p[2] = (int32_t)n_rows;
    p[3] = (int32_t)n_inc;
    p[4] = of_teams ? 0 : (int32_t)steps.size() - 1;
    p[5] = of_teams ? APC_SWEEP_TEAMS : 0;
    int32_t *q = p + 8, *label = p + 8 + 8 * n_rows;
    // where the minima of incidence t at label 0 are: a row here, or a slot
    auto place = [&](int64_t t) {
      return owner[inc_edge[t]] == w ? row_of[2 * (int64_t)inc_edge[t] + inc_side[t]] : slot[t] | 0x40000000;
    };
    for (const Side &x : sides) {  // in the order of row_of
      const int64_t nj = g.labels(edge_j[x.k]), ni = g.labels(edge_i[x.k]), n = g.labels(x.c), t = inc_of[2 * x.k + x.side];
      const int64_t degree = inc_begin[x.c + 1] - inc_begin[x.c];
      for (int64_t y = 0; y < n; ++y, q += 8) {
        q[0] = (int32_t)(uint32_t)((el_of[x.k - first] + (x.side == 0 ? y * nj : y)) | ((x.side == 0 ? nj : ni) << 16));
        q[1] = (int32_t)(uint32_t)((x.side == 0 ? 1 : nj) | (y << 16));
        q[2] = slot[t] >= 0 ? (int32_t)(slot[t] + y) : -1;
        q[3] = (int32_t)(uint32_t)(inc_at[x.c] | (degree << 16));
        for (int64_t u = 0; u < 4; ++u) q[4 + u] = u < degree ? (int32_t)(place(inc_begin[x.c] + u) + y) : (int32_t)n_rows;
        *label++ = (int32_t)((uint32_t)(label_begin[x.c] + y) | (t == inc_begin[x.c] ? 0x80000000u : 0u));  // (its first matrix stores a class)
      }
    }
    q = label;
    for (int64_t c : classes)
      for (int64_t t = inc_begin[c]; t < inc_begin[c + 1]; ++t) *q++ = (int32_t)place(t);
    if (of_teams) {
      for (size_t i = 0; i < sides.size(); i += 2) {  // (the two sides of an edge stand together)
        const int64_t k = sides[i].k;
        for (int64_t of_team = 0; of_team < teams[k].waves; ++of_team) {
          int32_t *wave = q + 4 * (teams[k].first_wave + of_team);
          wave[0] = (int32_t)row_of[2 * k + sides[i].side];
          wave[1] = (int32_t)(uint32_t)(g.labels(sides[i].c) | g.labels(sides[i + 1].c) << 16);
          wave[2] = (int32_t)((k - first) | of_team << 8 | teams[k].waves << 16);
        }
      }
    } else {
      for (int64_t r : steps) *q++ = (int32_t)r;
    }
    at += words;
    first = last;
  }
  plan_begin[n_wg] = at;
  sizes[0] = n_wg;
  sizes[1] = at;
  sizes[2] = n_slots;
  sizes[3] = lds;
  sizes[4] = threads;
  return 0;
} catch (...) {
  return thrown("apc_sweep_plan_host");
}

#undef APC_LABEL_PROBLEM
#undef APC_LABEL_PROBLEM_OF

}  // extern "C"
