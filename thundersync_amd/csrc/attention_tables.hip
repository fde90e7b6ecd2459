// Host code: the integer tables of an attention layout and one call's run
// table, built in one pass each (a streamed chunk builds both on every call).
#include <algorithm>
#include <cmath>
#include <exception>
#include <vector>

#include "attention_impl.h"

// the host mirrors (thundersync_amd/_abi.py) assume these sizes
static_assert(sizeof(ts_attn_layout) == 72 && sizeof(ts_attn_layout_sizes) == 128, "ts_attn layout ABI");

namespace ts {
namespace attn {

// work-group slots of one launch (256 CUs, one attention work-group each), the
// last-level cache the 8 XCDs share, and the relative width of a cost band of
// the launch order (thundersync_amd/attention.py gives the reasons)
constexpr int64_t kLaunchSlots = 256;
constexpr int64_t kSharedCacheBytes = 256ll << 20;
constexpr double kOrderBand = 0.05;

int cost_band(int64_t cost) {
  static const double width = std::log(1.0 + kOrderBand);
  return (int)std::floor(std::log((double)std::max<int64_t>(cost, 1)) / width);
}

// An ordered work list: (index, first row or key) pairs in descending cost
// bands, in the given order within a band, with the items' costs in list order.
struct WorkList {
  std::vector<int32_t> item;   // 2 per entry
  std::vector<int64_t> cost;
  int64_t sum = 0, most = 0;
  void add(int32_t index, int32_t first, int64_t c) {
    item.push_back(index);
    item.push_back(first);
    cost.push_back(c);
    sum += c;
    most = std::max(most, c);
  }
  void order() {
    const size_t n = cost.size();
    if (n < 2) return;
    std::vector<int> band(n);
    const int top = cost_band(most);
    std::vector<size_t> at(top + 2, 0);
    for (size_t i = 0; i < n; ++i) {
      band[i] = top - cost_band(cost[i]);
      ++at[band[i] + 1];
    }
    for (int b = 0; b <= top; ++b) at[b + 1] += at[b];
    std::vector<int32_t> it(2 * n);
    std::vector<int64_t> co(n);
    for (size_t i = 0; i < n; ++i) {
      const size_t j = at[band[i]]++;
      it[2 * j] = item[2 * i];
      it[2 * j + 1] = item[2 * i + 1];
      co[j] = cost[i];
    }
    item.swap(it);
    cost.swap(co);
  }
  // items that run item-major at the head of the launch: all of them when the
  // rows the work-groups re-read fit half the shared cache, else those of a
  // quarter or more of a slot's average share
  int64_t long_items(int64_t heads, int64_t reread_bytes) const {
    if (reread_bytes <= kSharedCacheBytes / 2) return (int64_t)cost.size();
    const double total = (double)sum * (double)heads;
    if (cost.empty() || total == 0.0) return 0;
    const double threshold = 0.25 * total / (double)kLaunchSlots;
    size_t n = 0;
    while (n < cost.size() && (double)cost[n] >= threshold) ++n;
    return (int64_t)n;
  }
};

int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

int layout_tables(const ts_attn_layout* layout, void* blob, int64_t blob_bytes, int32_t* run_visits,
                  ts_attn_layout_sizes* sizes, const char* what) {
  TS_CHECK_ARG(layout && sizes, "%s: null argument", what);
  const ts_attn_layout& L = *layout;
  TS_CHECK_ARG(L.hq > 0 && L.hkv > 0 && L.hq % L.hkv == 0 && L.kv_block > 0 && L.n_segs >= 0 && L.n_runs >= 0 &&
                   L.n_spans >= 0 && (L.n_segs == 0 || (L.seg_q && L.seg_span0)) && (L.n_spans == 0 || L.spans) &&
                   (L.n_runs == 0 || L.run_len),
               "%s: bad description", what);
  const int group = L.hq / L.hkv, qb = q_block_rows(group), kvb = L.kv_block;
  constexpr int kDqBlock = 64;  // rows per item of the dS route's dQ pass (groups that are a multiple of 4)

  // sizes
  int64_t n_q = 0, n_dq = 0, n_kv = 0;
  std::vector<int32_t> nvisit(L.n_runs, 0);
  for (int32_t s = 0; s < L.n_segs; ++s) {
    const int64_t len = L.seg_q[2 * s + 1];
    TS_CHECK_ARG(len >= 0 && L.seg_span0[s] >= 0 && L.seg_span0[s] <= L.seg_span0[s + 1] &&
                     L.seg_span0[s + 1] <= L.n_spans, "%s: segment %d", what, s);
    n_q += (len + qb - 1) / qb;
    if (group % 4 == 0) n_dq += (len + kDqBlock - 1) / kDqBlock;
    for (int64_t i = L.seg_span0[s]; i < L.seg_span0[s + 1]; ++i) {
      const int32_t r = L.spans[2 * i];
      TS_CHECK_ARG(r >= 0 && r < L.n_runs, "%s: segment %d names run %d of %d", what, s, r, L.n_runs);
      ++nvisit[r];
    }
  }
  for (int32_t r = 0; r < L.n_runs; ++r)
    if (nvisit[r]) n_kv += (L.run_len[r] + kvb - 1) / kvb;
  TS_CHECK_ARG(n_q < (1ll << 31) && n_kv < (1ll << 31) && n_dq < (1ll << 31), "%s: too many work items", what);
  const int64_t n_sp = L.n_segs ? L.seg_span0[L.n_segs] : 0;
  ts_attn_layout_sizes z;
  memset(&z, 0, sizeof z);
  z.n_q_work = n_q;
  z.n_kv_work = n_kv;
  z.n_dq_work = n_dq;
  int64_t at = 0;
  auto part = [&](int64_t bytes) {
    const int64_t o = at;
    at += align256(bytes);
    return o;
  };
  z.segs = part(L.n_segs * (int64_t)sizeof(ts_attn_segment));
  z.spans = part(n_sp * (int64_t)sizeof(ts_attn_ref));
  z.visits = part(n_sp * (int64_t)sizeof(ts_attn_ref));
  z.q_work = part(n_q * 8);
  z.kv_work = part(n_kv * 8);
  z.dq_work = part(n_dq * 8);
  z.span_ds = part(std::max<int64_t>(n_sp, 1) * 8);
  z.visit_ds = part(std::max<int64_t>(n_sp, 1) * 8);
  z.bytes = std::max<int64_t>(at, 256);
  if (!blob) {
    *sizes = z;
    return TS_OK;
  }
  TS_CHECK_ARG(blob_bytes >= z.bytes && (uintptr_t)blob % 8 == 0 && (L.n_runs == 0 || run_visits),
               "%s: tables of %lld bytes, need %lld", what, (long long)blob_bytes, (long long)z.bytes);

  char* b = (char*)blob;
  ts_attn_segment* segs = (ts_attn_segment*)(b + z.segs);
  ts_attn_ref* spans = (ts_attn_ref*)(b + z.spans);
  ts_attn_ref* visits = (ts_attn_ref*)(b + z.visits);
  int64_t* span_ds = (int64_t*)(b + z.span_ds);
  int64_t* visit_ds = (int64_t*)(b + z.visit_ds);
  span_ds[0] = visit_ds[0] = 0;
  int32_t first = 0;
  for (int32_t r = 0; r < L.n_runs; ++r) {
    run_visits[2 * r] = first;
    run_visits[2 * r + 1] = nvisit[r];
    first += nvisit[r];
  }

  WorkList q, dq, kv;
  q.item.reserve(2 * n_q);
  q.cost.reserve(n_q);
  std::vector<int32_t> filled(L.n_runs, 0);
  int64_t ds = 0;
  for (int32_t s = 0; s < L.n_segs; ++s) {
    const int64_t row0 = L.seg_q[2 * s], len = L.seg_q[2 * s + 1], s0 = L.seg_span0[s], s1 = L.seg_span0[s + 1];
    int64_t keys = 0;
    for (int64_t i = s0; i < s1; ++i) keys += L.run_len[L.spans[2 * i]];
    TS_CHECK_ARG(keys < (1ll << 31) && len < (1ll << 31), "%s: segment %d too long", what, s);
    segs[s].q_row0 = row0;
    segs[s].q_len = (int32_t)len;
    segs[s].kv_len = (int32_t)keys;
    segs[s].span0 = (int32_t)s0;
    segs[s].nspan = (int32_t)(s1 - s0);
    for (int64_t i = s0; i < s1; ++i) {
      const int32_t r = L.spans[2 * i], kpos = L.spans[2 * i + 1];
      const int32_t v = run_visits[2 * r] + filled[r]++;
      spans[i].index = r;
      spans[i].kpos = kpos;
      visits[v].index = s;
      visits[v].kpos = kpos;
      // the span's dS rectangle (ts_attn_ds_layout)
      span_ds[i] = visit_ds[v] = ds;
      ds += ds_rect_blocks(DsRect{(int)(keys - len - kpos), (L.run_len[r] + 15) >> 4, (int)len}) * kDsBlock;
    }
    // an item costs the keys its last row sees
    for (int64_t q0 = 0; q0 < len; q0 += qb) q.add(s, (int32_t)q0, keys - len + std::min(q0 + qb, len));
    if (group % 4 == 0)
      for (int64_t q0 = 0; q0 < len; q0 += kDqBlock)
        dq.add(s, (int32_t)q0, keys - len + std::min(q0 + kDqBlock, len));
  }
  // a dK/dV item costs the rows of its visits that see its first key
  kv.item.reserve(2 * n_kv);
  kv.cost.reserve(n_kv);
  int64_t key_rows = 0;
  for (int32_t r = 0; r < L.n_runs; ++r) {
    key_rows += L.run_len[r];
    if (!nvisit[r]) continue;
    for (int64_t k0 = 0; k0 < L.run_len[r]; k0 += kvb) {
      int64_t cost = 0;
      for (int32_t i = 0; i < nvisit[r]; ++i) {
        const ts_attn_ref& v = visits[run_visits[2 * r] + i];
        const ts_attn_segment& g = segs[v.index];
        const int64_t row = std::max<int64_t>(0, v.kpos + k0 - (g.kv_len - g.q_len));
        cost += std::max<int64_t>(0, g.q_len - row);
      }
      kv.add(r, (int32_t)k0, cost);
    }
  }
  q.order();
  dq.order();
  kv.order();
  if (n_q) memcpy(b + z.q_work, q.item.data(), n_q * 8);
  if (n_dq) memcpy(b + z.dq_work, dq.item.data(), n_dq * 8);
  if (n_kv) memcpy(b + z.kv_work, kv.item.data(), n_kv * 8);
  // rows the forward / dQ work-groups re-read: K and V of every run; the dK/dV
  // work-groups: Q and dO of every row (2-byte elements of head dim 128, all heads)
  const int64_t kv_bytes = key_rows * L.hkv * D * 4, q_bytes = L.q_rows * L.hq * D * 4;
  z.n_q_long = q.long_items(L.hkv * (group / heads_per_block(group)), kv_bytes);
  z.n_kv_long = kv.long_items(L.hkv, q_bytes);
  z.n_dq_long = dq.long_items(L.hkv * (group / 4), kv_bytes);
  z.ds_head = ds;
  *sizes = z;
  return TS_OK;
}

}  // namespace attn
}  // namespace ts

extern "C" int ts_attn_layout_tables(const ts_attn_layout* layout, void* blob, int64_t blob_bytes, int32_t* run_visits,
                                     ts_attn_layout_sizes* sizes) {
  const char* what = "ts_attn_layout_tables";
  try {
    return ts::attn::layout_tables(layout, blob, blob_bytes, run_visits, sizes, what);
  } catch (const std::exception& e) {  // host memory
    ts::set_error("%s: %s", what, e.what());
    return TS_ERR_INVALID;
  }
}

extern "C" int ts_attn_run_table(int32_t n_runs, const int32_t* run_len, const int32_t* run_source,
                                 const int64_t* run_offset, const int32_t* run_visits, int32_t n_sources,
                                 const int64_t* sources, ts_attn_run* runs) {
  const char* what = "ts_attn_run_table";
  TS_CHECK_ARG(n_runs >= 0 && n_sources >= 0 &&
                   (n_runs == 0 || (run_len && run_source && run_offset && run_visits && sources && runs)),
               "%s: null argument", what);
  for (int32_t r = 0; r < n_runs; ++r) {
    TS_CHECK_ARG(run_source[r] >= 0 && run_source[r] < n_sources, "%s: run %d names source %d of %d", what, r,
                 run_source[r], n_sources);
    const int64_t* x = sources + 12 * (int64_t)run_source[r];  // k, v, dk, dv: address, row stride, head stride
    ts_attn_run u;
    memset(&u, 0, sizeof u);
    auto row = [&](const int64_t* t) { return t[0] ? (uint64_t)t[0] + 2 * (uint64_t)(run_offset[r] * t[1]) : 0; };
    u.k = row(x);
    u.k_row_stride = x[1];
    u.k_head_stride = x[2];
    u.v = row(x + 3);
    u.v_row_stride = x[4];
    u.v_head_stride = x[5];
    u.dk = row(x + 6);
    u.dk_row_stride = x[7];
    u.dk_head_stride = x[8];
    u.dv = row(x + 9);
    u.dv_row_stride = x[10];
    u.dv_head_stride = x[11];
    u.len = run_len[r];
    u.visit0 = run_visits[2 * r];
    u.nvisit = run_visits[2 * r + 1];
    runs[r] = u;
  }
  return TS_OK;
}
