// Randomised check of the host-only planners of libkvc (kvc_decode_plan,
// kvc_prefill_plan, kvc_prefill_plan_split), built with AddressSanitizer / UndefinedBehaviorSanitizer
// on the host side by tests/test_plan_fuzz_asan.py.  Every plan of a valid
// batch must succeed after at most one capacity retry and satisfy the
// invariants the kernels rely on:
//   decode, segment mode: segments tile the flattened page list in order,
//     each within one page of the others and at most 128 pages; pieces tile
//     every request's pages exactly once, partial indices 0..n-1 (or -1 for a
//     single piece); workspace sized for max_partitions;
//   decode, small-batch mode: one segment and one piece per request, at most
//     16 pages each, no partials;
//   prefill: every query of every request in exactly one work unit per KV
//     head; the workgroup table covers the units once, no workgroup empty,
//     and within each XCD's workgroups the loads (key tiles + 2 per unit)
//     differ by at most one unit's cost;
//   split prefill (few units over long histories): every key tile of every unit
//     in exactly one piece, the records moved to the piece's first key, partials
//     numbered once and in order per unit, one merge record per cut unit, the
//     image of whole units behind it, and all of it within the capacity that
//     the wrapper reserves.
// Prints "ok <iterations>" and exits 0, or the first violation and exits 1.
#include <algorithm>
#include <array>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <vector>

#include "kvc.h"

namespace {

int fail(const char* what, int it) {
  std::printf("violation at iteration %d: %s (%s)\n", it, what, kvc_last_error());
  return 1;
}

#define CHECK(cond, what) \
  do {                    \
    if (!(cond)) return fail(what, it); \
  } while (0)

int check_decode(const std::vector<int32_t>& indptr, const std::vector<int32_t>& lpl,
                 const kvc_decode_schedule& s, const std::vector<int32_t>& img, int it) {
  const int B = s.batch;
  const int64_t total = B ? indptr[B] : 0;
  CHECK(s.total_pages == total, "total_pages");
  CHECK(s.plan_ints == kvc_decode_plan_ints(B, s.num_segments), "plan_ints");
  const int32_t* seg = img.data();
  const int32_t* pc = img.data() + s.pieces_offset;
  const int32_t* np = img.data() + s.nparts_offset;
  CHECK(int64_t(s.nparts_offset) + B <= int64_t(img.size()), "nparts inside the image");
  if (s.small_batch) {
    CHECK(s.num_segments == B && s.num_pieces == B && s.max_partitions == 1, "small shape");
    CHECK(s.workspace_bytes == 0 && s.heads_per_group == 1, "small workspace");
    for (int b = 0; b < B; ++b) {
      CHECK(indptr[b + 1] - indptr[b] <= 16, "small request within 16 pages");
      CHECK(pc[8 * b] == b && pc[8 * b + 1] == indptr[b] && pc[8 * b + 2] == indptr[b + 1],
            "small piece = request");
      CHECK(pc[8 * b + 3] == -1 && pc[8 * b + 4] == indptr[b + 1] - 1 &&
                pc[8 * b + 5] == lpl[b], "small piece tail");
      CHECK(np[b] == (indptr[b + 1] > indptr[b] ? 1 : 0), "small nparts");
    }
    return 0;
  }
  const int S = s.num_segments;
  CHECK((total == 0) == (S == 0), "segments iff pages");
  std::vector<int> seen(B, 0);
  int64_t min_len = INT64_MAX, max_len = 0;
  int max_parts = 1;
  for (int i = 0; i < S; ++i) {
    const int32_t* r = seg + 4 * i;
    CHECK(r[0] <= r[1] && r[1] <= s.num_pieces, "segment piece range");
    CHECK(i == 0 || r[0] == seg[4 * (i - 1) + 1], "segments contiguous in pieces");
    CHECK(r[2] == (i == 0 ? 0 : seg[4 * (i - 1) + 2] + seg[4 * (i - 1) + 3]), "segments contiguous in slots");
    CHECK(r[3] >= 1 && (i + 1 < S || r[2] + r[3] == total), "segment pages");
    min_len = std::min<int64_t>(min_len, r[3]);
    max_len = std::max<int64_t>(max_len, r[3]);
    int64_t slot = r[2];
    for (int k = r[0]; k < r[1]; ++k) {
      const int32_t* p = pc + 8 * k;
      CHECK(p[0] >= 0 && p[0] < B, "piece request");
      CHECK(p[1] == slot && p[2] > p[1], "pieces contiguous and non-empty");
      CHECK(p[1] >= indptr[p[0]] && p[2] <= indptr[p[0] + 1], "piece inside its request");
      CHECK(p[4] == indptr[p[0] + 1] - 1 && p[5] == lpl[p[0]], "piece tail");
      slot = p[2];
      ++seen[p[0]];
    }
    CHECK(slot == r[2] + r[3], "segment fully covered");
  }
  if (S) CHECK(min_len >= 1 && max_len <= 128, "segments within 1..128 pages");
  for (int b = 0; b < B; ++b) {
    CHECK(seen[b] == np[b], "nparts");
    CHECK((indptr[b + 1] == indptr[b]) == (np[b] == 0), "empty requests have no piece");
    max_parts = std::max(max_parts, np[b]);
  }
  CHECK(s.max_partitions == max_parts, "max_partitions");
  CHECK(s.workspace_bytes ==
            kvc_decode_workspace_bytes(B, s.num_qo_heads, s.head_dim, s.max_partitions),
        "workspace bytes");
  return 0;
}

int check_prefill(const std::vector<int32_t>& qo, const std::vector<int32_t>& kv, int hkv,
                  const kvc_prefill_schedule& s, const std::vector<int32_t>& img, int it) {
  const int B = s.batch;
  const int64_t units = int64_t(s.num_items) * hkv;
  const int64_t W = std::min<int64_t>(256, units);
  const int64_t table = (2 * W + 3) / 4 * 4;
  CHECK(s.plan_ints == table + 8 * units, "prefill plan_ints");
  // the workgroup table covers the unit records once, in order, none empty
  int64_t next = 0;
  std::vector<int64_t> load(W, 0);
  int64_t max_cost = 0;
  for (int64_t w = 0; w < W; ++w) {
    CHECK(img[2 * w] == next && img[2 * w + 1] >= 1, "workgroup table");
    for (int64_t u = next; u < next + img[2 * w + 1]; ++u) {
      const int64_t c = img[table + 8 * u + 6] + 2;
      load[w] += c;
      max_cost = std::max(max_cost, c);
    }
    next += img[2 * w + 1];
  }
  CHECK(next == units, "every unit in one workgroup");
  // list scheduling: within each XCD's workgroups, loads within one unit's cost
  const int groups = W % 8 == 0 ? 8 : 1;
  for (int x = 0; x < groups; ++x) {
    int64_t lo = INT64_MAX, hi = 0;
    for (int64_t w = x; w < W; w += groups) lo = std::min(lo, load[w]), hi = std::max(hi, load[w]);
    CHECK(hi - lo <= max_cost, "workgroup balance");
  }
  // every query of every request in exactly one unit per KV head
  std::vector<int> req_of_q(qo.empty() ? 0 : size_t(qo[B]) + 1, -1);
  for (int b = 0; b < B; ++b)
    if (qo[b + 1] > qo[b]) req_of_q[size_t(qo[b])] = b;
  std::vector<int64_t> covered(size_t(B) * hkv, 0);
  for (int64_t u = 0; u < units; ++u) {
    const int32_t* r = img.data() + table + 8 * u;
    CHECK(r[0] >= 0 && r[0] < hkv, "unit head");
    CHECK(r[4] >= 0 && r[4] < int64_t(req_of_q.size()) && req_of_q[size_t(r[4])] >= 0,
          "unit request");
    const int b = req_of_q[size_t(r[4])];
    CHECK(r[2] == qo[b + 1] - qo[b] && r[5] == kv[b], "unit offsets");
    CHECK(r[1] >= 0 && r[1] < r[2] && r[1] % s.tile_tokens == 0, "unit first query");
    covered[size_t(b) * hkv + r[0]] += std::min(r[1] + s.tile_tokens, r[2]) - r[1];
  }
  for (int b = 0; b < B; ++b)
    for (int h = 0; h < hkv; ++h)
      CHECK(covered[size_t(b) * hkv + h] == qo[b + 1] - qo[b], "queries covered once per head");
  return 0;
}

// int32 entries the wrapper reserves (BatchPrefillWithPagedKVCacheWrapper._plan_capacity).
int64_t prefill_capacity(const std::vector<int32_t>& qo, int group, int hkv) {
  const int64_t tile = 256 / group;
  int64_t units = 0;
  for (size_t b = 0; b + 1 < qo.size(); ++b) units += (qo[b + 1] - qo[b] + tile - 1) / tile;
  units *= hkv;
  const int64_t table = (2 * std::min<int64_t>(256, units) + 3) / 4 * 4;
  return units <= 512 ? 2 * 256 + 9 * (512 + 256) + 8 * units + table + 8 * units + 8
                      : table + 8 * units + 8;
}

int check_split(const kvc_prefill_schedule& whole, const std::vector<int32_t>& base,
                const kvc_prefill_schedule& s, const kvc_prefill_split& p,
                const std::vector<int32_t>& img, int hkv, int group, int it) {
  const int64_t units = int64_t(whole.num_items) * hkv;
  const int64_t base_table = (2 * std::min<int64_t>(256, units) + 3) / 4 * 4;
  CHECK(s.plan_ints == p.base_offset + whole.plan_ints, "split plan_ints");
  CHECK(std::equal(base.begin(), base.begin() + whole.plan_ints, img.begin() + p.base_offset),
        "the whole units' image behind the split one");
  if (p.num_parts == 0) {
    CHECK(p.base_offset == 0 && p.num_merges == 0 && p.workspace_bytes == 0 &&
              p.num_units == units, "nothing cut");
    return 0;
  }
  CHECK(p.num_workgroups >= 1 && p.num_workgroups <= 256, "split workgroups");
  CHECK(p.workspace_bytes == int64_t(p.num_parts) * 256 * 129 * 4, "split workspace");
  const int64_t table = (2 * int64_t(p.num_workgroups) + 3) / 4 * 4;
  CHECK(p.parts_offset == table + 8 * int64_t(p.num_units) &&
            p.merges_offset == p.parts_offset + (p.num_units + 3) / 4 * 4 &&
            p.base_offset == p.merges_offset + 8 * p.num_merges, "split offsets");
  int64_t next = 0;
  for (int w = 0; w < p.num_workgroups; ++w) {
    CHECK(img[2 * w] == next && img[2 * w + 1] >= 1, "split workgroup table");
    next += img[2 * w + 1];
  }
  CHECK(next == p.num_units, "every piece in one workgroup");
  // The pieces of each (head, q offset, first query), by their first key.
  typedef std::array<int32_t, 3> Key;
  std::map<Key, std::vector<int64_t>> pieces;
  const int32_t* rec = img.data() + table;
  const int32_t* part = img.data() + p.parts_offset;
  for (int64_t u = 0; u < p.num_units; ++u)
    pieces[Key{rec[8 * u], rec[8 * u + 4], rec[8 * u + 1]}].push_back(u);
  std::vector<int> seen(size_t(p.num_parts), 0);
  int64_t cut = 0;
  const int32_t* merges = img.data() + p.merges_offset;
  for (int64_t u = 0; u < units; ++u) {
    const int32_t* r = base.data() + base_table + 8 * u;
    auto at = pieces.find(Key{r[0], r[4], r[1]});
    CHECK(at != pieces.end(), "a unit is in the split plan");
    std::vector<int64_t> list = at->second;
    pieces.erase(at);
    std::sort(list.begin(), list.end(),
              [&](int64_t x, int64_t y) { return rec[8 * x + 3] > rec[8 * y + 3]; });
    int64_t first = 0;
    for (size_t i = 0; i < list.size(); ++i) {
      const int32_t* q = rec + 8 * list[i];
      const int pages = std::min<int64_t>(r[7], 4 * first);
      CHECK(q[2] == r[2] && q[3] == r[3] - 64 * first && q[5] == r[5] + pages &&
                q[7] == r[7] - pages, "a piece's record starts at its first key");
      CHECK(q[6] >= (list.size() > 1 ? 1 : 0), "a piece has tiles");
      if (list.size() == 1) {
        CHECK(part[list[i]] == -1, "a whole unit writes the output");
      } else {
        CHECK(part[list[i]] >= 0 && part[list[i]] < p.num_parts &&
                  part[list[i]] == part[list[0]] + int(i), "partials in order");
        ++seen[size_t(part[list[i]])];
      }
      first += q[6];
    }
    CHECK(first == r[6], "every key tile in one piece");
    if (list.size() > 1) {
      ++cut;
      int found = 0;
      for (int m = 0; m < p.num_merges; ++m) {
        const int32_t* g = merges + 8 * m;
        if (g[3] != part[list[0]]) continue;
        ++found;
        CHECK(g[0] == r[0] && g[1] == r[4] + r[1] && g[4] == int(list.size()) &&
                  g[2] == std::min(256 / group, r[2] - r[1]) * group, "merge record");
      }
      CHECK(found == 1, "one merge record per cut unit");
    }
  }
  CHECK(pieces.empty() && cut == p.num_merges, "no other pieces or merges");
  CHECK(std::count(seen.begin(), seen.end(), 1) == p.num_parts, "every partial once");
  return 0;
}

int fuzz_split(std::mt19937& rng, int it, int* cut) {
  const int B = int(rng() % 12) + 1;
  const int hkv = int(rng() % 8) + 1, g = 1 << (rng() % 4), causal = int(rng() % 4) != 0;
  std::vector<int32_t> qo(B + 1, 0), kv(B + 1, 0), lpl(B, 0);
  for (int b = 0; b < B; ++b) {
    const int len = rng() % 6 == 0 ? 0 : int(rng() % (rng() % 2 ? 40000 : 3000));
    const int top = std::min(len, rng() % 4 == 0 ? 3000 : 200);
    kv[b + 1] = kv[b] + (len + 15) / 16;
    lpl[b] = len == 0 ? 0 : (len % 16 ? len % 16 : 16);
    qo[b + 1] = qo[b] + (top ? int(rng() % (top + 1)) : int(rng() % 3));  // also more queries than keys
  }
  const int64_t cap = prefill_capacity(qo, g, hkv);
  std::vector<int32_t> base(size_t(cap), -7), img(size_t(cap), -7);
  kvc_prefill_schedule ws{}, ps{};
  kvc_prefill_split split{};
  CHECK(kvc_prefill_plan(qo.data(), kv.data(), lpl.data(), B, hkv * g, hkv, 128, 16, causal, &ws,
                         base.data(), cap) == KVC_OK, "prefill plan within the capacity");
  CHECK(kvc_prefill_plan_split(qo.data(), kv.data(), lpl.data(), B, hkv * g, hkv, 128, 16, causal,
                               &ps, &split, img.data(), cap) == KVC_OK,
        "split plan within the capacity");
  for (int64_t i = ps.plan_ints; i < cap; ++i) CHECK(img[size_t(i)] == -7, "nothing past plan_ints");
  *cut += split.num_parts > 0;
  return check_split(ws, base, ps, split, img, hkv, g, it);
}

}  // namespace

int main(int argc, char** argv) {
  const int iters = argc > 1 ? std::atoi(argv[1]) : 2000;
  std::mt19937 rng(20261202);
  const int dims[3] = {64, 128, 256};
  for (int it = 0; it < iters; ++it) {
    const int B = int(rng() % 300);
    const bool short_ctx = rng() % 3 == 0;
    std::vector<int32_t> indptr(B + 1, 0), lpl(B, 0);
    for (int b = 0; b < B; ++b) {
      const int len = rng() % 5 == 0 ? 0
                      : short_ctx    ? int(rng() % 300)
                                     : int(rng() % (rng() % 4 == 0 ? 40000 : 3000));
      indptr[b + 1] = indptr[b] + (len + 15) / 16;
      lpl[b] = len == 0 ? 0 : (len % 16 ? len % 16 : 16);
    }
    const int hkv = 1 << (rng() % 5), g = 1 << (rng() % 4);
    const int d = dims[rng() % 3];
    const int hint = rng() % 4 == 0 ? int(rng() % 2000) : 0;
    const int cus = int(rng() % 300) + 1;
    kvc_decode_schedule s{};
    std::vector<int32_t> img(size_t(rng() % 64 + 1));
    int st = kvc_decode_plan(indptr.data(), lpl.data(), B, hkv * g, hkv, d, 16, hint, cus, &s,
                             img.data(), int64_t(img.size()));
    if (st == KVC_ERR_WORKSPACE) {
      CHECK(s.plan_ints > int64_t(img.size()), "capacity report");
      img.assign(size_t(s.plan_ints), -7);
      st = kvc_decode_plan(indptr.data(), lpl.data(), B, hkv * g, hkv, d, 16, hint, cus, &s,
                           img.data(), int64_t(img.size()));
    }
    CHECK(st == KVC_OK, "decode plan of a valid batch");
    if (check_decode(indptr, lpl, s, img, it)) return 1;

    // Prefill: chunks of at most each request's cached tokens.
    std::vector<int32_t> qo(B + 1, 0);
    for (int b = 0; b < B; ++b) {
      const int len = (indptr[b + 1] - indptr[b]) * 16 - (lpl[b] ? 16 - lpl[b] : 0);
      qo[b + 1] = qo[b] + (len ? int(rng() % (len + 1)) : 0);
    }
    kvc_prefill_schedule ps{};
    std::vector<int32_t> pimg(size_t(rng() % 256 + 1));
    const int causal = int(rng() % 2);
    st = kvc_prefill_plan(qo.data(), indptr.data(), lpl.data(), B, hkv * g, hkv, 128, 16,
                          causal, &ps, pimg.data(), int64_t(pimg.size()));
    if (st == KVC_ERR_WORKSPACE) {
      CHECK(ps.plan_ints > int64_t(pimg.size()), "prefill capacity report");
      pimg.assign(size_t(ps.plan_ints), -7);
      st = kvc_prefill_plan(qo.data(), indptr.data(), lpl.data(), B, hkv * g, hkv, 128, 16,
                            causal, &ps, pimg.data(), int64_t(pimg.size()));
    }
    CHECK(st == KVC_OK, "prefill plan of a valid batch");
    if (check_prefill(qo, indptr, hkv, ps, pimg, it)) return 1;
  }
  std::mt19937 split_rng(20261204);
  int cut = 0;
  for (int it = 0; it < iters; ++it)
    if (fuzz_split(split_rng, it, &cut)) return 1;
  if (cut < iters / 4) {
    std::printf("only %d of %d batches were cut\n", cut, iters);
    return 1;
  }
  std::printf("ok %d\n", iters);
  return 0;
}
