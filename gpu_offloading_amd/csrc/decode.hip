// (a6/a7/a8) Paged GQA decode attention for gfx950.
//
// Semantics: FlashInfer BatchDecodeWithPagedKVCacheWrapper.run as the reference
// engine calls it (src/MoE/moe_engine.py:3907-3909, planned at :1949-1955 with
// pos_encoding_mode="NONE", default sm_scale = 1/sqrt(head_dim)): for request b
// and query head hq, attention over the tokens held in pages
// indices[indptr[b] .. indptr[b+1]) (final page: last_page_len[b] tokens) of KV
// head hq / group.  Split-K partials are merged with the log-sum-exp rule of
// src/dense/offload_kv_attn.py:24-39 (done in base 2 here).
//
// Decode is a GEMV: every K/V byte feeds only `group` query heads, so the
// kernels are HBM-bound.
//
// Schedule (balanced split-KV, computed on the host by kvc_decode_plan like
// FlashInfer's plan()): the flattened page list indices[0 .. P) of the whole
// batch is cut into S segments of equal cost, S ~ the number of workgroups
// the GPU holds at once, so every workgroup streams about the same number of
// pages and all finish together whatever the spread of request lengths (a
// switch to another request inside a segment costs about one page more; see
// cut_segments).  A segment crosses request boundaries; the part of a request
// inside one segment is a "piece".  A request covered by one piece is written
// straight to the output; otherwise each piece leaves an fp32 partial +
// log2-sum-exp in the workspace and decode_merge_kernel folds them.
//
// Three streaming kernels, chosen by the plan; all read K/V from HBM exactly
// once and serve the `group` query heads of a KV head together:
//
//   decode_lds_kernel<G>   head_dim 128, group <= 4, a multiple of 8 KV heads:
//         one workgroup of 8 waves per (segment, 8 heads), pages staged in LDS
//         as whole 2 KB token rows;
//   decode_wave_kernel<G, D>   everything else (head_dim 64 / 256, group 8,
//         other head counts) and small batches: each wave streams pages of one
//         head straight into registers, no barrier in its loop;
//   decode_small_kernel<G>  head_dim 128, requests of at most 16 pages: one
//         workgroup per (request, KV head), no partials.
//
// decode_lds_kernel: the waves stage each page together: wave w loads 256
// consecutive 16-byte chunks of the page's (token row x head slice) image (two
// whole 2 KB token rows for Mixtral), so the workgroup reads the page's K and V
// blocks as contiguous runs, into a double-buffered LDS tile; one barrier per
// page; the next two pages are in flight in two register stages meanwhile.
// K/V are loaded with the non-temporal hint (read once; 5.7 -> 6.3 TB/s at 32K
// contexts).  Tile rows are padded by 16 B, which keeps both read patterns
// below free of LDS bank conflicts and makes every LDS address a lane base
// plus an immediate:
//   q.k : lane (token t, query head g) computes the whole 128-dim dot product
//         with v_dot2_f32_bf16 from 16 ds_read_b128 of row t (the four lanes
//         of a token read the same address); no cross-lane reduction;
//   p.v : lane l owns dims 2l, 2l+1 for every query head; per token one
//         ds_read_b32 of V and one broadcast read of p[t][0..G).
// Softmax statistics live per 16-lane DPP row (one query head per row).
// A wave's page ids are loaded once, one per lane (2 registers: up to 128
// pages per segment), and broadcast with v_readlane, so no dependent global
// load sits in the streaming loop.
#include "kvc_common.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

namespace kvc {
namespace {

constexpr int kPage = 16;      // tokens per page (the engine's page_size)
constexpr int kLdsHeads = 8;   // KV heads per workgroup of the LDS kernel
constexpr int kMaxWaveHeads = 4;   // KV heads per workgroup of the wave kernel, at most
constexpr int64_t kChipCus = 256;  // an MI355X's CUs
constexpr int kIdRegs = 2;     // page-id registers per lane
constexpr int kMaxSegPages = 64 * kIdRegs;
constexpr int kReadGroup = 4;  // LDS reads scheduled together
constexpr float kRescaleLog2 = 8.f;  // lazy-rescale threshold (base 2)
constexpr float kLn2 = 0.69314718055994530942f;
constexpr float kLog2e = 1.44269504088896340736f;

struct DecodeArgs {
  const uint16_t* q;
  int64_t q_stride;        // elements between requests
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  int64_t block_stride;    // elements between cache blocks
  int64_t token_stride;    // elements between tokens of a block
  int64_t num_blocks;
  const int32_t* indices;
  int64_t num_indices;
  const int4* segments;    // [S]: (first piece, end piece, first slot, pages)
  int32_t total_pages;     // pages of the whole batch
  int32_t num_segments;
  const int4* pieces;      // [N][2]: (request, first slot, end slot, partial or -1),
                           //         (request's last slot, its tokens, 0, 0)
  float scale_log2;        // sm_scale * log2(e)
  int32_t num_kv_heads;
  int32_t max_parts;
  float* part_o;           // [batch][Hkv][max_parts][G][D]
  float* part_lse;         // [batch][Hkv][max_parts][G]   (log2 domain)
  uint16_t* out;
  int64_t out_stride;      // elements between requests
  float* lse;              // [batch][Hq] natural log, may be null
  // Fused append: row b of new_k / new_v is written as request b's last token
  // before it is attended; null: none.
  const uint16_t* new_k;
  const uint16_t* new_v;
  int64_t new_k_stride;    // elements between requests
  int64_t new_v_stride;
  int32_t heads_per_group; // KV heads per workgroup of the wave kernel
  int32_t q_splits;        // workgroups that share a KV head's query heads
};

// Pieces, counted from a segment's first, within which a request's end may lie
// for the LDS kernel's fused append (the plan reports the most any segment
// needs).
constexpr int kNewMax = 4;

// Compiler-level ordering point for LDS traffic between lanes of one wave
// (the LDS unit itself executes one wave's instructions in order).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}


// First slot and page count of a segment, from its record (the plan's cuts
// balance pages and piece switches, so they do not follow from the index).
__device__ __forceinline__ void segment_span(const int4& segment, int& g0, int& n) {
  g0 = segment.z;
  n = min(segment.w, kMaxSegPages);
}

// Page ids of a segment: lane l of register r holds indices[g0 + l + 64 r].
// The registers are only ever indexed by constants (v_readlane picks the
// lane): a runtime index would turn them into a per-thread LDS array.
struct SegmentIds {
  int32_t r[kIdRegs];

  __device__ __forceinline__ void load(const DecodeArgs& a, int g0, int n, int lane) {
    // Clamped addresses, uniform branches: the loads issue back to back.
    const int64_t last = a.num_indices - 1;
#pragma unroll
    for (int i = 0; i < kIdRegs; ++i) {
      r[i] = -1;
      if (64 * i < n) {
        const int j = lane + 64 * i;
        const int64_t slot = int64_t(g0) + j;
        const int32_t v = a.indices[min(slot, last)];
        r[i] = (j < n && slot <= last) ? v : -1;
      }
    }
  }
  // Block id of the segment's j-th page (j uniform).
  __device__ __forceinline__ int32_t at(int j) const {
    const int l = j & 63;
    const int w = j >> 6;
    int32_t v = __builtin_amdgcn_readlane(r[0], l);
#pragma unroll
    for (int i = 1; i < kIdRegs; ++i) {
      const int32_t x = __builtin_amdgcn_readlane(r[i], l);
      v = w == i ? x : v;
    }
    return v;
  }
};

// The piece being streamed by a wave and what the page loop needs of it.
struct Piece {
  int4 desc;     // (request, first slot, end slot, partial index or -1)
  int req_last;  // slot of the request's final page
  int last_len;  // tokens in that page

  __device__ __forceinline__ void load(const DecodeArgs& a, int k) {
    desc = a.pieces[2 * k];
    const int4 tail = a.pieces[2 * k + 1];
    req_last = tail.x;
    last_len = min(max(tail.y, 0), kPage);
  }
  __device__ __forceinline__ int valid(int slot, int32_t blk, int64_t num_blocks) const {
    if (blk < 0 || blk >= num_blocks) return 0;
    return slot == req_last ? last_len : kPage;
  }
};

// Output of a finished piece for query head hq = h * group + g: the final
// bf16 row (a request covered by one piece) or an fp32 partial; `o` holds
// this lane's NDIM normalised values starting at dim d0.
template <int D, int NDIM>
__device__ __forceinline__ void write_piece(const DecodeArgs& a, const int4& pc, int h,
                                            int group, int g, int d0, const float (&o)[NDIM],
                                            float lse2, bool lse_lane) {
  const int b = pc.x;
  const int hq = h * group + g;
  if (pc.w < 0) {
    uint16_t* dst = a.out + int64_t(b) * a.out_stride + int64_t(hq) * D + d0;
    static_assert(NDIM % 2 == 0, "dims are stored in pairs");
#pragma unroll
    for (int e = 0; e < NDIM; e += 2)
      *reinterpret_cast<uint32_t*>(dst + e) =
          uint32_t(f32_to_bf16(o[e])) | (uint32_t(f32_to_bf16(o[e + 1])) << 16);
    if (a.lse && lse_lane)
      a.lse[int64_t(b) * a.num_kv_heads * group + hq] = lse2 * kLn2;
  } else {
    const int64_t pr = ((int64_t(b) * a.num_kv_heads + h) * a.max_parts + pc.w) * group + g;
    float* dst = a.part_o + pr * D + d0;
#pragma unroll
    for (int e = 0; e < NDIM; ++e) dst[e] = o[e];
    if (lse_lane) a.part_lse[pr] = lse2;
  }
}

// ---------------------------------------------------------------------------
// head_dim 128: LDS-staged kernel.
// ---------------------------------------------------------------------------
template <int G>
struct LdsCfg {
  static constexpr int QL = G > 4 ? G / 4 : 1;  // query heads per lane in q.k
  static constexpr int GP = G < 4 ? G : 4;      // distinct query heads over the 4 rows
  static constexpr int NS = G < 4 ? 4 / G : 1;  // lanes sharing one dot product
  static constexpr int CH = 16 / NS;            // 16-byte chunks of a K row per lane
};

// The LDS tile of one page for the HPW KV heads of a workgroup: K and V, 16
// token rows of HPW x 256 B, each row padded by 16 B.  With the pad, the 16
// rows read by one q.k instruction start on 16 different 4-bank groups, and
// every lane address is a lane base plus an immediate offset.
template <int HPW>
struct BlockTile {
  static constexpr int kRowBytes = HPW * 256 + 16;
  static constexpr int kRowChunks = kRowBytes / 16;
  uint4 k[kPage * kRowChunks];
  uint4 v[kPage * kRowChunks];
};

// Workgroup = 8 waves = 8 neighbouring KV heads of one segment.  The waves
// stage each page together: wave w loads 256 consecutive 16-byte chunks
// of the page's (token row x head slice) image, so the workgroup reads the
// block's rows as long contiguous runs (2 KB per token row for 8 heads), into
// a double-buffered tile; one barrier per page; then each wave computes its
// own head from the tile.
template <int G>
__global__ __launch_bounds__(64 * kLdsHeads) void decode_lds_kernel(DecodeArgs a) {
  constexpr int HPW = kLdsHeads;
  using C = LdsCfg<G>;
  using Tile = BlockTile<HPW>;
  constexpr int D = 128;
  constexpr int kSliceChunks = HPW * 16;  // 16-byte chunks per token row of the slice
  __shared__ Tile s_tile[2];
  __shared__ float s_p[HPW][kPage * 8];   // softmax weights p[token][query head]
  // Fused append: the new rows (K, V) of the requests that end inside the
  // segment, by piece index.
  __shared__ uint4 s_new[kNewMax][2][kSliceChunks];

  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int h0 = blockIdx.y * HPW;  // first KV head of the workgroup
  const int h = h0 + wave;
  const int4 segment = a.segments[blockIdx.x];
  int g0, n;
  segment_span(segment, g0, n);
  int k = segment.x;
  const int k_end = segment.y;
  if (k >= k_end || n <= 0) return;  // uniform over the workgroup
  float* p_buf = s_p[wave];

  // q.k role: token t, query head gq (and gq + 4 when G == 8), dim split.
  const int t = lane & 15;
  const int row = lane >> 4;
  const int gq = row % C::GP;
  const int split = row / C::GP;
  // Staging role: chunk u of this lane is chunk q = 256 wave + 64 u + lane of
  // the page image (token q / kSliceChunks, 16-byte chunk q % kSliceChunks).
  uint32_t st_goff[4];
  int st_loff[4], st_tok[4];
  const uint32_t ts_bytes = uint32_t(a.token_stride * 2);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int q = 256 * wave + 64 * u + lane;
    st_tok[u] = q / kSliceChunks;
    const int cc = q % kSliceChunks;
    st_goff[u] = uint32_t(st_tok[u]) * ts_bytes + uint32_t(h0 * D * 2 + cc * 16);
    st_loff[u] = st_tok[u] * Tile::kRowChunks + cc;
  }
  const char* kbytes = reinterpret_cast<const char*>(a.k_cache);
  const char* vbytes = reinterpret_cast<const char*>(a.v_cache);
  const int64_t block_bytes = a.block_stride * 2;

  SegmentIds ids;
  ids.load(a, g0, n, lane);
  Piece pc;
  pc.load(a, k);
  const int k0 = k;
  const bool appending = a.new_k != nullptr;
  // Thread i < 2 x kSliceChunks loads chunk i % kSliceChunks of the K (or V)
  // slice of each new row; the rows land in s_new after the first pages'
  // loads are issued.
  // The loads are issued on every path (a piece past the segment's last
  // re-reads that one's row), so the compiler's count of loads in flight stays
  // exact and staging s_new does not wait for the first pages' loads.
  uint4 nrow[kNewMax];
#pragma unroll
  for (int i = 0; i < kNewMax; ++i) nrow[i] = make_uint4(0, 0, 0, 0);
  {
    if (appending) {
      const int is_v = (threadIdx.x & (2 * kSliceChunks - 1)) >= kSliceChunks;
      const int cc = threadIdx.x & (kSliceChunks - 1);
#pragma unroll
      for (int i = 0; i < kNewMax; ++i) {
        const int b = a.pieces[2 * min(k + i, k_end - 1)].x;
        const uint16_t* src = is_v ? a.new_v + int64_t(b) * a.new_v_stride
                                   : a.new_k + int64_t(b) * a.new_k_stride;
        nrow[i] = reinterpret_cast<const uint4*>(src + h0 * D)[cc];
      }
    }
  }

  uint32_t qw[C::QL][C::CH * 4];
  auto load_q = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) {
      const uint4* qp = reinterpret_cast<const uint4*>(
          a.q + int64_t(b) * a.q_stride + int64_t(h * G + gq + 4 * ql) * D + split * C::CH * 8);
#pragma unroll
      for (int i = 0; i < C::CH; ++i) {
        const uint4 x = qp[i];
        qw[ql][4 * i + 0] = x.x;
        qw[ql][4 * i + 1] = x.y;
        qw[ql][4 * i + 2] = x.z;
        qw[ql][4 * i + 3] = x.w;
      }
    }
  };
  float m_run[C::QL], l_run[C::QL], acc[G][2];
  auto reset = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) {
      m_run[ql] = kNegBig;
      l_run[ql] = 0.f;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g][0] = acc[g][1] = 0.f;
  };
  auto finalize = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float l = readlane_f(l_run[g / 4], 16 * (g % 4));
      const float m = readlane_f(m_run[g / 4], 16 * (g % 4));
      const float inv = l > 0.f ? 1.f / l : 0.f;
      const float o[2] = {acc[g][0] * inv, acc[g][1] * inv};
      write_piece<D, 2>(a, pc.desc, h, G, g, 2 * lane, o,
                        l > 0.f ? m + fast_log2(l) : -INFINITY, lane == 0);
    }
  };

  // Two register stages: while page j is consumed, pages j+1 and j+2 are in
  // flight (2 x 8 KB per wave, 2 x 8 KB x HPW per workgroup).
  struct Stage {
    uint4 k[4], v[4];
  };
  auto issue = [&](Stage& r, int32_t blk) __attribute__((always_inline)) {
    // Uniform block base (SGPRs) + 32-bit lane offset.
    const char* kb = kbytes + int64_t(blk) * block_bytes;
    const char* vb = vbytes + int64_t(blk) * block_bytes;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r.k[u] = load_stream(kb + st_goff[u]);
      r.v[u] = load_stream(vb + st_goff[u]);
    }
  };
  auto safe_id = [&](int32_t id) __attribute__((always_inline)) { return (id >= 0 && id < a.num_blocks) ? id : 0; };
  auto stage_tile = [&](Stage& r, Tile& tile, int valid) __attribute__((always_inline)) {
    if (valid < kPage) {
      // Rows past the end may hold anything (even NaN bits): stage zeros so
      // that 0 * v stays 0.
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (st_tok[u] >= valid) r.k[u] = r.v[u] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      tile.k[st_loff[u]] = r.k[u];
      tile.v[st_loff[u]] = r.v[u];
    }
  };
  auto consume = [&](const Tile& tile, int valid) __attribute__((always_inline)) {
    // q.k: lane (t, gq) over its chunks of K row t, head `wave` of the tile.
    float dots[C::QL];
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) dots[ql] = 0.f;
    const uint4* krow = tile.k + t * Tile::kRowChunks + wave * 16 + split * C::CH;
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      const uint4 kv = krow[i];
#pragma unroll
      for (int ql = 0; ql < C::QL; ++ql) {
        dots[ql] = dot2_bf16(qw[ql][4 * i + 0], kv.x, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * i + 1], kv.y, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * i + 2], kv.z, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * i + 3], kv.w, dots[ql]);
      }
      // Keep a bounded number of LDS reads in flight: hoisting all of them
      // would cost registers, and with them a wave per SIMD.
      if ((i + 1) % kReadGroup == 0) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int off = 16 * C::GP; off < 64; off <<= 1)
#pragma unroll
      for (int ql = 0; ql < C::QL; ++ql) dots[ql] += __shfl_xor(dots[ql], off);

    // Online softmax per row (one query head per 16-lane row).
    const bool live = t < valid;
    float alpha[C::QL];
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) {
      const float s = live ? dots[ql] * a.scale_log2 : kNegBig;
      const float m_new = fmaxf(m_run[ql], row16_max(s));
      const float p = live ? fast_exp2(s - m_new) : 0.f;
      alpha[ql] = fast_exp2(m_run[ql] - m_new);
      l_run[ql] = fmaf(l_run[ql], alpha[ql], row16_sum(p));
      m_run[ql] = m_new;
      if (row < C::GP) p_buf[t * G + gq + 4 * ql] = p;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float al = readlane_f(alpha[g / 4], 16 * (g % 4));
      acc[g][0] *= al;
      acc[g][1] *= al;
    }
    wave_lds_fence();

    // p.v over the 16 tokens of the page (rows past `valid` are zero).
    const uint32_t* vcol = reinterpret_cast<const uint32_t*>(tile.v + wave * 16) + lane;
#pragma unroll
    for (int tt = 0; tt < kPage; ++tt) {
      const uint32_t vw = vcol[tt * Tile::kRowChunks * 4];
      const float v0 = bf16lo(vw);
      const float v1 = bf16hi(vw);
      float pg[G];
      if constexpr (G >= 4) {
#pragma unroll
        for (int q4 = 0; q4 < G / 4; ++q4) {
          const float4 x = reinterpret_cast<const float4*>(p_buf + tt * G)[q4];
          pg[4 * q4 + 0] = x.x;
          pg[4 * q4 + 1] = x.y;
          pg[4 * q4 + 2] = x.z;
          pg[4 * q4 + 3] = x.w;
        }
      } else {
#pragma unroll
        for (int g = 0; g < G; ++g) pg[g] = p_buf[tt * G + g];
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        acc[g][0] = fmaf(pg[g], v0, acc[g][0]);
        acc[g][1] = fmaf(pg[g], v1, acc[g][1]);
      }
      if ((tt + 1) % kReadGroup == 0) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Page j: stage it into tile j%2, refill its register stage with page j+2,
  // wait for the whole workgroup's part of the tile (one barrier per page:
  // every wave has also finished reading the tile's previous page j-2),
  // consume, and close the piece if page j is its last.
  auto step = [&](int j, Stage& r, int32_t& id, Tile& tile) __attribute__((always_inline)) {
    const int slot = g0 + j;
    const int valid = pc.valid(slot, id, a.num_blocks);
    {
      // The request's last page: its new token row comes from s_new (the
      // loaded row is stale) and is written to the cache.
      if (appending && slot == pc.req_last && valid > 0 && k - k0 < kNewMax) {
        const int tnew = valid - 1;
        const int i = k - k0;
        char* kdst = const_cast<char*>(kbytes) + int64_t(id) * block_bytes;
        char* vdst = const_cast<char*>(vbytes) + int64_t(id) * block_bytes;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (st_tok[u] == tnew) {
            const int cc = st_loff[u] - st_tok[u] * Tile::kRowChunks;
            r.k[u] = s_new[i][0][cc];
            r.v[u] = s_new[i][1][cc];
            store_stream(kdst + st_goff[u], r.k[u]);
            store_stream(vdst + st_goff[u], r.v[u]);
          }
        }
      }
    }
    stage_tile(r, tile, valid);
    if (j + 2 < n) {
      id = ids.at(j + 2);
      issue(r, safe_id(id));
    }
    __syncthreads();
    consume(tile, valid);
    wave_lds_fence();
    if (slot + 1 == pc.desc.z) {
      finalize();
      if (++k < k_end) {
        pc.load(a, k);
        load_q(pc.desc.x);
        reset();
      }
    }
  };

  load_q(pc.desc.x);
  reset();
  Stage ra, rb;
  int32_t ida = ids.at(0), idb = 0;
  issue(ra, safe_id(ida));
  if (n > 1) {
    idb = ids.at(1);
    issue(rb, safe_id(idb));
  }
  {
    if (appending) {
      if (threadIdx.x < 2 * kSliceChunks) {
        const int is_v = threadIdx.x >= kSliceChunks;
        const int cc = threadIdx.x & (kSliceChunks - 1);
#pragma unroll
        for (int i = 0; i < kNewMax; ++i) s_new[i][is_v][cc] = nrow[i];
      }
      __syncthreads();
    }
  }
  for (int j = 0; j < n; j += 2) {
    step(j, ra, ida, s_tile[0]);
    if (j + 1 < n) step(j + 1, rb, idb, s_tile[1]);
  }
}

// ---------------------------------------------------------------------------
// head_dim 128, small batches: one workgroup per (request, KV head), its
// kSmallWaves waves splitting the request's pages (wave w takes pages w,
// w + kSmallWaves, ...), the waves' softmax states merged in LDS.  One launch,
// no partials in memory and no merge kernel: for batches whose requests fit
// in kSmallMaxPages pages but would otherwise be cut into one-page segments
// and merged (batch 1 at a 128-token context: 9 pages).  The plan image holds
// one segment and one piece per request (empty requests included), so the
// request's record sits at piece index b.
// ---------------------------------------------------------------------------
constexpr int kSmallWaves = 8;
constexpr int kSmallMaxPages = 2 * kSmallWaves;

template <int G>
__global__ __launch_bounds__(64 * kSmallWaves) void decode_small_kernel(DecodeArgs a) {
  using C = LdsCfg<G>;
  using Tile = BlockTile<1>;
  constexpr int D = 128;
  constexpr int kPagesPerWave = kSmallMaxPages / kSmallWaves;
  __shared__ Tile s_tile[kSmallWaves];
  __shared__ float s_p[kSmallWaves][kPage * 8];
  __shared__ float s_m[kSmallWaves][G];
  __shared__ float s_l[kSmallWaves][G];
  __shared__ float s_o[kSmallWaves][G][D];

  const int b = blockIdx.x;
  const int h = blockIdx.y;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int4 desc = a.pieces[2 * b];        // (request, first slot, end slot, -1)
  const int4 tail = a.pieces[2 * b + 1];    // (request's last slot, its tokens, 0, 0)
  const int first = desc.y;
  const int npages = min(desc.z - desc.y, kSmallMaxPages);
  const int last_len = min(max(tail.y, 0), kPage);
  Tile& tile = s_tile[wave];
  float* p_buf = s_p[wave];

  const int t = lane & 15;
  const int row = lane >> 4;
  const int gq = row % C::GP;
  const int split = row / C::GP;
  // Staging: chunk u of this lane is chunk 64 u + lane of the (16 tokens x
  // 256 B) image of head h in a page: token (64 u + lane) / 16, chunk lane % 16.
  const int cc = lane & 15;
  const uint32_t ts_bytes = uint32_t(a.token_stride * 2);
  uint32_t st_goff[4];
  int st_tok[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    st_tok[u] = (64 * u + lane) >> 4;
    st_goff[u] = uint32_t(st_tok[u]) * ts_bytes + uint32_t(h * D * 2 + cc * 16);
  }
  const char* kbytes = reinterpret_cast<const char*>(a.k_cache);
  const char* vbytes = reinterpret_cast<const char*>(a.v_cache);
  const int64_t block_bytes = a.block_stride * 2;

  // This wave's pages, their ids and their loads, all issued up front.
  struct Stage {
    uint4 k[4], v[4];
  };
  Stage st[kPagesPerWave];
  int32_t ids[kPagesPerWave];
#pragma unroll
  for (int i = 0; i < kPagesPerWave; ++i) {
    const int j = wave + kSmallWaves * i;
    ids[i] = -1;
    if (j < npages) {
      const int64_t slot = int64_t(first) + j;
      ids[i] = slot < a.num_indices ? a.indices[slot] : -1;
    }
  }
#pragma unroll
  for (int i = 0; i < kPagesPerWave; ++i) {
    const int32_t id = (ids[i] >= 0 && ids[i] < a.num_blocks) ? ids[i] : 0;
    const char* kb = kbytes + int64_t(id) * block_bytes;
    const char* vb = vbytes + int64_t(id) * block_bytes;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      st[i].k[u] = make_uint4(0, 0, 0, 0);
      st[i].v[u] = make_uint4(0, 0, 0, 0);
    }
    if (wave + kSmallWaves * i < npages) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        st[i].k[u] = load_stream(kb + st_goff[u]);
        st[i].v[u] = load_stream(vb + st_goff[u]);
      }
    }
  }
  // Fused append: lane chunk cc of head h of the request's new K / V row.
  const bool appending = a.new_k != nullptr && npages > 0 && last_len > 0;
  uint4 nk = make_uint4(0, 0, 0, 0), nv = make_uint4(0, 0, 0, 0);
  if (appending) {
    nk = reinterpret_cast<const uint4*>(a.new_k + int64_t(b) * a.new_k_stride + h * D)[cc];
    nv = reinterpret_cast<const uint4*>(a.new_v + int64_t(b) * a.new_v_stride + h * D)[cc];
  }

  uint32_t qw[C::QL][C::CH * 4];
#pragma unroll
  for (int ql = 0; ql < C::QL; ++ql) {
    const uint4* qp = reinterpret_cast<const uint4*>(
        a.q + int64_t(b) * a.q_stride + int64_t(h * G + gq + 4 * ql) * D + split * C::CH * 8);
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      const uint4 x = qp[i];
      qw[ql][4 * i + 0] = x.x;
      qw[ql][4 * i + 1] = x.y;
      qw[ql][4 * i + 2] = x.z;
      qw[ql][4 * i + 3] = x.w;
    }
  }
  float m_run[C::QL], l_run[C::QL], acc[G][2];
#pragma unroll
  for (int ql = 0; ql < C::QL; ++ql) {
    m_run[ql] = kNegBig;
    l_run[ql] = 0.f;
  }
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g][0] = acc[g][1] = 0.f;

#pragma unroll
  for (int i = 0; i < kPagesPerWave; ++i) {
    const int j = wave + kSmallWaves * i;
    if (j >= npages) break;  // uniform over the wave
    const int slot = first + j;
    const int32_t id = ids[i];
    const bool ok = id >= 0 && id < a.num_blocks;
    const int valid = !ok ? 0 : (slot == tail.x ? last_len : kPage);
    Stage& r = st[i];
    if (appending && slot == tail.x && ok) {
      // The request's last page: its new token row (row valid - 1) comes
      // from the step's rows and is written to the cache.
      char* kdst = const_cast<char*>(kbytes) + int64_t(id) * block_bytes;
      char* vdst = const_cast<char*>(vbytes) + int64_t(id) * block_bytes;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (st_tok[u] == valid - 1) {
          r.k[u] = nk;
          r.v[u] = nv;
          store_stream(kdst + st_goff[u], nk);
          store_stream(vdst + st_goff[u], nv);
        }
      }
    }
    // Stage the page into this wave's tile (rows past `valid` as zeros).
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool live = st_tok[u] < valid;
      tile.k[st_tok[u] * Tile::kRowChunks + cc] = live ? r.k[u] : make_uint4(0, 0, 0, 0);
      tile.v[st_tok[u] * Tile::kRowChunks + cc] = live ? r.v[u] : make_uint4(0, 0, 0, 0);
    }
    wave_lds_fence();
    // q.k: lane (t, gq) over its chunks of K row t.
    float dots[C::QL];
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) dots[ql] = 0.f;
    const uint4* krow = tile.k + t * Tile::kRowChunks + split * C::CH;
#pragma unroll
    for (int c = 0; c < C::CH; ++c) {
      const uint4 kv = krow[c];
#pragma unroll
      for (int ql = 0; ql < C::QL; ++ql) {
        dots[ql] = dot2_bf16(qw[ql][4 * c + 0], kv.x, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * c + 1], kv.y, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * c + 2], kv.z, dots[ql]);
        dots[ql] = dot2_bf16(qw[ql][4 * c + 3], kv.w, dots[ql]);
      }
    }
#pragma unroll
    for (int off = 16 * C::GP; off < 64; off <<= 1)
#pragma unroll
      for (int ql = 0; ql < C::QL; ++ql) dots[ql] += __shfl_xor(dots[ql], off);
    const bool live = t < valid;
    float alpha[C::QL];
#pragma unroll
    for (int ql = 0; ql < C::QL; ++ql) {
      const float s = live ? dots[ql] * a.scale_log2 : kNegBig;
      const float m_new = fmaxf(m_run[ql], row16_max(s));
      const float p = live ? fast_exp2(s - m_new) : 0.f;
      alpha[ql] = fast_exp2(m_run[ql] - m_new);
      l_run[ql] = fmaf(l_run[ql], alpha[ql], row16_sum(p));
      m_run[ql] = m_new;
      if (row < C::GP) p_buf[t * G + gq + 4 * ql] = p;
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float al = readlane_f(alpha[g / 4], 16 * (g % 4));
      acc[g][0] *= al;
      acc[g][1] *= al;
    }
    wave_lds_fence();
    // p.v over the page's rows: all 16 for a full page, else four at a time
    // up to `valid` (rows past it have p = 0 and zero V rows, so leaving
    // them out changes nothing).
    const uint32_t* vcol = reinterpret_cast<const uint32_t*>(tile.v) + lane;
    auto pv_row = [&](int tt) {
      const uint32_t vw = vcol[tt * Tile::kRowChunks * 4];
      const float v0 = bf16lo(vw);
      const float v1 = bf16hi(vw);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float pg = p_buf[tt * G + g];
        acc[g][0] = fmaf(pg, v0, acc[g][0]);
        acc[g][1] = fmaf(pg, v1, acc[g][1]);
      }
    };
    if (valid == kPage) {
#pragma unroll
      for (int tt = 0; tt < kPage; ++tt) pv_row(tt);
    } else {
      for (int t4 = 0; t4 < valid; t4 += 4) {
#pragma unroll
        for (int tt = t4; tt < t4 + 4; ++tt) pv_row(tt);
      }
    }
    wave_lds_fence();  // the tile and p_buf are rewritten by the next page
  }

  // The waves' states (log2 domain) into LDS, then one merged output row per
  // query head; lanes cover (query head, dim).
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float l = readlane_f(l_run[g / 4], 16 * (g % 4));
    const float m = readlane_f(m_run[g / 4], 16 * (g % 4));
    if (lane == 0) {
      s_m[wave][g] = m;
      s_l[wave][g] = l;
    }
    s_o[wave][g][2 * lane] = acc[g][0];
    s_o[wave][g][2 * lane + 1] = acc[g][1];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < G * D; e += 64 * kSmallWaves) {
    const int g = e / D;
    const int d = e - g * D;
    float mx = kNegBig;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w)
      if (s_l[w][g] > 0.f) mx = fmaxf(mx, s_m[w][g]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      if (s_l[w][g] > 0.f) {
        const float wt = fast_exp2(s_m[w][g] - mx);
        L = fmaf(s_l[w][g], wt, L);
        O = fmaf(s_o[w][g][d], wt, O);
      }
    }
    const int hq = h * G + g;
    a.out[int64_t(b) * a.out_stride + int64_t(hq) * D + d] = f32_to_bf16(L > 0.f ? O / L : 0.f);
    if (a.lse && d == 0)
      a.lse[int64_t(b) * a.num_kv_heads * G + hq] =
          L > 0.f ? (mx + fast_log2(L)) * kLn2 : -INFINITY;
  }
}

// ---------------------------------------------------------------------------
// Wave streaming kernel (any head_dim, group and head count).
//
// Bound by HBM, so built to keep loads in flight and the arithmetic per byte
// small: K and V go from memory into registers, nothing is staged in LDS, and
// no barrier sits in the page loop.  A workgroup's waves are its KV heads times
// TS page shares: wave (head, ts) streams units ts, ts + TS, ... of the
// segment (a unit is one page, at head_dim 64 below group 8 two); in the narrow
// form, for many requests per segment, a workgroup is its heads' waves alone, each
// on all units, and several workgroups share a CU.  One unit is in flight per wave
// while another is consumed -- K's registers are refilled as soon as q.k has read
// them, V's after p.v -- 64 KB and more a CU with the waves of WaveCfg.
// Every K and V load of the wave reads whole token rows (four rows of 256 B at
// head_dim 128), which the layouts of the 4x4 matrix instructions allow:
//   q.k : v_mfma_f32_4x4x4_16b_bf16, block b = 16-byte chunk b of a row, rows =
//         four tokens, columns = four query heads; the blocks (chunks) are
//         summed with lane swaps and row rotations that leave row c of 16
//         lanes with four tokens, head l % 4 in lane l.  (The 16x16x32 layout
//         needs no such sum, but its loads touch 16 rows of 16 B per quarter
//         wave: 5.95 against 6.84 TB/s of plain reads.)
//   softmax : each row of 16 lanes keeps its own maximum and sum over its
//         tokens, so pages need no exchange; the rows meet once per piece.
//         The rescale is skipped unless a maximum grows by more than 2^8.
//   p.v : v_mfma_f32_4x4x1_16b_f32 with p in fp32 as it lies in the lanes and
//         V widened to fp32 (exact): lane l holds eight dims of its row's token
//         for the four heads.  A group of one multiplies on the VALU instead.
// At a piece's end the rows' states are merged in the wave, then (a piece of more
// than one unit) the TS waves' through LDS with one barrier, and the piece is
// written.  Uniform plan records come by scalar loads, which the loads in flight
// do not delay.
//
// One layer with its append (start: the kernel it replaces with the merge of
// its time), us:
//   32 requests of 500-3001 tokens, 8 KV heads, group 8, head_dim 64: 63.8 -> 30.6
//   64 of 512-4096, 8 KV heads, group 8, head_dim 128: 149 -> 110 (5.6 TB/s)
//   64 of 512-4096, one KV head, group 4, head_dim 128: 35.6 -> 20.1
//   32 of 500-3000, 8 KV heads, head_dim 256, group 4: 100 -> 87 (5.5 TB/s)
//   64 of 512-4096, 16 KV heads, head_dim 64, group 1: 109 -> 100
// ---------------------------------------------------------------------------
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
// Vectors at the element alignment the callers guarantee (head_dim 64 takes
// 8-byte aligned rows, the output 4-byte aligned ones); gfx950 moves them with
// one dwordx4 all the same.
typedef u32x4_t u32x4_a8_t __attribute__((aligned(8)));
typedef u32x4_t u32x4_a4_t __attribute__((aligned(4)));

// Word 3 of a raw buffer resource (32-bit data, no swizzle; loads past
// num_records return zeros) and the non-temporal bit of a buffer load.
constexpr int kBufferRsrcWord3 = 0x00020000;
constexpr int kNonTemporal = 2;

constexpr int wave_kernel_waves(int group, int head_dim) {
  return head_dim == 256 ? (group == 1 ? 12 : 8) : head_dim == 128 ? 8 : (group == 1 ? 16 : 12);
}

// G: query heads of a KV head that one workgroup serves.  At head_dim 256 a
// group of 8 is served as two workgroups of four (q_splits 2): its accumulators
// alone would fill a wave's registers.
template <int G, int D>
struct WaveCfg {
  static_assert(G <= 4 || D < 256, "four query heads per wave at head_dim 256");
  // Waves per workgroup.  At head_dim 64 and 256 as many as registers allow
  // without spills, at most 16 (12 for groups 2 and 4 at 64: 16 took 16.8 ->
  // 19.0 us on 64 requests of one KV head, 8 took 17.2).  At head_dim 128 a
  // page is 8 KB per wave, so eight waves have 64 KB in flight, enough for the
  // CU's share of HBM; more only start later and meet in more states at a
  // piece's end.  16 waves at group 1 or 12 else -> 8, one layer, us:
  //   64 requests of 512-4096, one KV head: group 1 21.0 -> 18.7, 4 21.2 -> 20.4,
  //   8 24.9 -> 24.1; 8 of 300-2000, 8 heads: group 4 16.0 -> 15.1, 8 22.2 -> 21.2;
  //   one of 32000: 29.6 -> 28.8.  (16 at groups 2 and 4: 1 to 15% slower than 12.)
  static constexpr int kWaves = wave_kernel_waves(G, D);
  static constexpr int kPages = D == 64 && G < 8 ? 2 : 1;  // pages a wave takes at a time
  static constexpr int kGroups = G == 8 ? 2 : 1;   // query heads in fours
  static constexpr int kGroupHeads = G < 4 ? G : 4;
  static constexpr int kLoads = D / 32;            // 16-byte K (and V) loads per lane and page
  static constexpr int kQ = D == 256 ? 2 : 1;      // 16-byte q chunks per lane and group
  static constexpr int kDims = D == 256 ? 16 : 8;  // output dims per lane
};

// x and y summed over the wave's halves: lanes < 32 get x's sum, the others y's.
__device__ __forceinline__ float swap32_add(float x, float y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// x and y summed over pairs of 16-lane rows (0 + 1, 2 + 3): even rows get x's
// sum, odd rows y's.
__device__ __forceinline__ float swap16_add(float x, float y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// D += A B over 16 blocks of four lanes: A row l % 4 and B column l % 4 of
// block l / 4, four bf16 each (a0, a1 / b0, b1); D register r: row r, column l % 4.
__device__ __forceinline__ f32x4_t mfma_4x4x4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                              f32x4_t d) {
  return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(
      __builtin_bit_cast(i16x4_t, (uint64_t(a1) << 32) | a0),
      __builtin_bit_cast(i16x4_t, (uint64_t(b1) << 32) | b0), d, 0, 0, 0);
}

// Eight output dims (from d0) of a finished piece for query head h * group + g.
template <int D>
__device__ __forceinline__ void write_dims8(const DecodeArgs& a, const int4& pc, int h, int group,
                                            int g, int d0, const float* o) {
  const int hq = h * group + g;
  if (pc.w < 0) {
    u32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = uint32_t(f32_to_bf16(o[2 * e])) | (uint32_t(f32_to_bf16(o[2 * e + 1])) << 16);
    *reinterpret_cast<u32x4_a4_t*>(a.out + int64_t(pc.x) * a.out_stride + int64_t(hq) * D + d0) = w;
  } else {
    const int64_t pr = ((int64_t(pc.x) * a.num_kv_heads + h) * a.max_parts + pc.w) * group + g;
    float4* dst = reinterpret_cast<float4*>(a.part_o + pr * D + d0);
    dst[0] = make_float4(o[0], o[1], o[2], o[3]);
    dst[1] = make_float4(o[4], o[5], o[6], o[7]);
  }
}
__device__ __forceinline__ void write_lse(const DecodeArgs& a, const int4& pc, int h, int group,
                                          int g, float lse2) {
  const int hq = h * group + g;
  if (pc.w < 0) {
    if (a.lse) a.lse[int64_t(pc.x) * a.num_kv_heads * group + hq] = lse2 * kLn2;
  } else {
    a.part_lse[((int64_t(pc.x) * a.num_kv_heads + h) * a.max_parts + pc.w) * group + g] = lse2;
  }
}

// A uniform int4 of the plan image as a scalar load: waiting for it does not
// wait for the page loads in flight (those are counted apart).
__device__ __forceinline__ int4 scalar_int4(const int4* p, int i) {
  typedef int i32x4_t __attribute__((ext_vector_type(4)));
  typedef const __attribute__((address_space(4))) i32x4_t* cptr;
  const i32x4_t v = ((cptr)(uintptr_t)(p))[i];
  return make_int4(v[0], v[1], v[2], v[3]);
}

// Workgroup barrier that orders LDS traffic only: global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The lane index as a value that what is computed from it cannot be hoisted
// past: the rare paths of a loop then hold no registers through it.
__device__ __forceinline__ int local_lane() {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));
  return l;
}

// Value of lane 4 (l / 4) + V for every lane l.
template <int V>
__device__ __forceinline__ float quad_lane(float x) {
  return dpp<V * 0x55>(x);
}

// kNarrow: a workgroup is one wave per head, each streaming the whole segment.
template <int G, int D, bool kNarrow>
__global__ __launch_bounds__((64 * (kNarrow ? kMaxWaveHeads : WaveCfg<G, D>::kWaves)),
                             (WaveCfg<G, D>::kWaves / 4)) void decode_wave_kernel(DecodeArgs a) {
  using C = WaveCfg<G, D>;
  constexpr int W = C::kWaves, NG = C::kGroups, NL = C::kLoads, NE = C::kDims, PU = C::kPages;
  __shared__ float s_o[2][W][G][D];
  __shared__ float s_m[2][W][G], s_l[2][W][G];

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int hpw = a.heads_per_group;
  const int hw = kNarrow ? wave : wave % hpw, ts = kNarrow ? 0 : wave / hpw;
  const int TS = kNarrow ? 1 : W / hpw;
  const int split = blockIdx.y % a.q_splits, h0 = blockIdx.y / a.q_splits * hpw;
  const int h = h0 + hw;
  const int group = G * a.q_splits;  // query heads of a KV head
  const int4 segment = scalar_int4(a.segments, blockIdx.x);
  int k = segment.x;
  const int k_end = segment.y;
  int g0, n;
  segment_span(segment, g0, n);
  if (k >= k_end) return;  // uniform over the workgroup

  // Lane roles.  K (and q.k): row of four consecutive tokens l % 4, 16-byte
  // chunk l / 4.  V (and p.v): tokens t_row .. t_row + 3 of the page, chunk
  // l % 16.
  const int c = lane >> 4, nn = lane & 15;
  const int t_row = D == 64 ? 8 * (c & 1) + 4 * (c >> 1) : 4 * c;
  const uint32_t tsb = uint32_t(a.token_stride * 2);
  const int k_chunk = D == 64 ? (lane >> 2) & 7 : lane >> 2;
  const int k_tok = (D == 64 ? 4 * (lane >> 5) : 0) + (lane & 3);
  const int v_chunk = D == 64 ? nn & 7 : nn;
  const int v_tok = t_row + (D == 64 ? nn >> 3 : 0);
  // Byte offset of load u inside a page block (head_dim 256's second half is
  // 256 bytes further), and its token.
  constexpr int NT = NL < 4 ? NL : 4;
  uint32_t k_off[NT], v_off[NT];
  auto k_step = [](int u) { return D == 64 ? 8 * u : 4 * (u & 3); };
  auto v_step = [](int u) { return D == 64 ? 2 * u : u & 3; };
  auto d_step = [](int u) { return D == 256 ? (u >> 2) * 256 : 0; };
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    k_off[u] = uint32_t(k_tok + k_step(u)) * tsb + uint32_t(h * D * 2 + k_chunk * 16);
    v_off[u] = uint32_t(v_tok + v_step(u)) * tsb + uint32_t(h * D * 2 + v_chunk * 16);
  }
  const char* kbytes = reinterpret_cast<const char*>(a.k_cache);
  const char* vbytes = reinterpret_cast<const char*>(a.v_cache);
  const int64_t block_bytes = a.block_stride * 2;

  // This wave's units of PU consecutive pages: unit ts, ts + TS, ... of the
  // segment; the pages' ids one per lane (a wave that shares the segment has at most
  // half of its pages; at head_dim 64 the second register stays all the same, for the
  // code that the compiler makes of it: 8 KV heads, group 8, 16 requests of 8000
  // 56.8 us without, 55.4 with; of one request of 96 tokens, 2 heads 9.0 and 8.6).
  const int nw = n > PU * ts ? (n - PU * ts + PU * TS - 1) / (PU * TS) : 0;
  auto page_slot = [&](int j, int x) { return g0 + PU * (ts + TS * j) + x; };
  constexpr int IR = kNarrow || D == 64 ? kIdRegs : kIdRegs / 2;
  static_assert(kNarrow || W >= 2 * kMaxWaveHeads, "two waves at least share a segment");
  int32_t idr[IR];
  {
    const int64_t last = a.num_indices - 1;
#pragma unroll
    for (int i = 0; i < IR; ++i) {
      idr[i] = -1;
      if (64 * i < PU * nw) {
        const int j = lane + 64 * i;
        const int64_t slot = page_slot(j / PU, j % PU);
        const int32_t v = a.indices[min(slot, last)];
        idr[i] = (slot < g0 + n && slot <= last) ? v : -1;
      }
    }
  }
  auto id_at = [&](int j) __attribute__((always_inline)) {
    int32_t v = __builtin_amdgcn_readlane(idr[0], j & 63);
#pragma unroll
    for (int i = 1; i < IR; ++i) {
      const int32_t x = __builtin_amdgcn_readlane(idr[i], j & 63);
      v = (j >> 6) == i ? x : v;
    }
    return v;
  };

  int4 cp = scalar_int4(a.pieces, 2 * k), ct = scalar_int4(a.pieces, 2 * k + 1);
  // The piece of the next page to be requested.
  int ki = k;
  int4 ip = cp, it = ct;
  // q: head l % 4 of each four, the 16-byte chunk(s) of this lane's K loads.
  const int q_head = (lane & 3) % C::kGroupHeads;
  const uint32_t q_off = uint32_t((h * group + G * split + q_head) * D + k_chunk * 8) * 2;
  const int page_bytes = kPage * int(tsb);  // under 2 GiB (host check)
  u32x4_t q[NG][C::kQ], qn[NG][C::kQ];  // of the current piece and the next
  auto load_q = [&](u32x4_t (&dst)[NG][C::kQ], int b) __attribute__((always_inline)) {
    const char* qb = reinterpret_cast<const char*>(a.q + int64_t(b) * a.q_stride);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int x = 0; x < C::kQ; ++x)
        dst[g][x] = *reinterpret_cast<const u32x4_a8_t*>(qb + (4 * g * D + 128 * x) * 2 + q_off);
  };

  // The unit in the K and V registers: K's next unit is requested once q.k has
  // read them, V's after p.v, so one set of registers keeps a unit in flight.
  // A missing page, or one past the segment's last, loads nothing.
  struct Ids {
    int32_t v[PU];
  };
  u32x4_t kr[PU][NL], vr[PU][NL];
  auto unit_ids = [&](int j) __attribute__((always_inline)) {
    Ids r;
#pragma unroll
    for (int x = 0; x < PU; ++x) {
      const int32_t id = j < nw ? id_at(PU * j + x) : -1;
      r.v[x] = id < a.num_blocks ? id : -1;
    }
    return r;
  };
  auto load_unit = [&](u32x4_t (&dst)[PU][NL], const char* base, const uint32_t (&off)[NT],
                       const Ids& ids) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < PU; ++x) {
      const int32_t id = ids.v[x];
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(base + int64_t(max(id, 0)) * block_bytes), 0, id < 0 ? 0 : page_bytes,
          kBufferRsrcWord3);
#pragma unroll
      for (int u = 0; u < NL; ++u)
        dst[x][u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, int(off[u & 3]) + d_step(u), 0,
                                                          kNonTemporal);
    }
  };

  float m[NG], l[NG];
  // acc[g][e]: this lane's dim e for the four query heads of g (G 1: one head).
  constexpr int NH = G == 1 ? 1 : 4;
  typedef float acc_t __attribute__((ext_vector_type(NH)));
  acc_t acc[NG][NE];
  auto reset = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      m[g] = kNegBig;
      l[g] = 0.f;
#pragma unroll
      for (int e = 0; e < NE; ++e) acc[g][e] = 0.f;
    }
  };

  int parity = 0;
  bool holds = false;  // this wave has consumed pages of the piece (uniform)
  // Close piece k: the four rows' states of every wave are merged, then those of
  // the waves that shared the piece, and the piece is written.  A piece of one
  // unit is written by the wave that holds it, and the others go on: no barrier.
  // (Every wave closing every piece together cost about 2 us a piece: 40 requests
  // of 3 tokens before 30 of 1590, 8 KV heads, group 4, head_dim 64 took 49.5 us,
  // now 33.7; group 8 at 128 79 -> 51.)
  auto finish = [&]() __attribute__((always_inline)) {
    const bool alone = kNarrow || (cp.y - g0) / PU == (cp.z - 1 - g0) / PU;  // the same in every wave
    if (!kNarrow && alone && !holds) return;
    const int fl = local_lane();
    const int c = fl >> 4, nn = fl & 15, v_chunk = D == 64 ? nn & 7 : nn;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      float M = fmaxf(m[g], __shfl_xor(m[g], 16));
      M = fmaxf(M, __shfl_xor(M, 32));
      const float w = fast_exp2(m[g] - M);
      float L = l[g] * w;
      L += __shfl_xor(L, 16);
      L += __shfl_xor(L, 32);
      const float w0 = quad_lane<0>(w), w1 = quad_lane<1>(w), w2 = quad_lane<2>(w),
                  w3 = quad_lane<3>(w);
      // Row c ends up with head c: swap halves, then odd and even rows.
      float o[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        float x0 = acc[g][e][0] * w0, x1 = acc[g][e][1 % NH] * w1;
        float x2 = acc[g][e][2 % NH] * w2, x3 = acc[g][e][3 % NH] * w3;
        if constexpr (D == 64) {
          x0 += dpp<kDppRowRor8>(x0);
          x1 += dpp<kDppRowRor8>(x1);
          x2 += dpp<kDppRowRor8>(x2);
          x3 += dpp<kDppRowRor8>(x3);
        }
        o[e] = swap16_add(swap32_add(x0, x2), swap32_add(x1, x3));
      }
      const float Lc = __shfl(L, c), Mc = __shfl(M, c);
      const int gl = 4 * g + c, gq = G * split + gl;  // query head of the workgroup, of the KV head
      if (alone) {
        if (c < C::kGroupHeads) {
          const float inv = Lc > 0.f ? 1.f / Lc : 0.f;
#pragma unroll
          for (int e = 0; e < NE; ++e) o[e] *= inv;
          if (D != 64 || nn < 8) {
#pragma unroll
            for (int x = 0; x < NE / 8; ++x)
              write_dims8<D>(a, cp, h, group, gq, 128 * x + 8 * v_chunk, o + 8 * x);
          }
          if (nn == 0) write_lse(a, cp, h, group, gq, Lc > 0.f ? Mc + fast_log2(Lc) : -INFINITY);
        }
      } else if (c < C::kGroupHeads) {
        if (D != 64 || nn < 8) {
#pragma unroll
          for (int x = 0; x < NE / 8; ++x) {
            float4* dst = reinterpret_cast<float4*>(&s_o[parity][wave][gl][128 * x + 8 * v_chunk]);
            dst[0] = make_float4(o[8 * x], o[8 * x + 1], o[8 * x + 2], o[8 * x + 3]);
            dst[1] = make_float4(o[8 * x + 4], o[8 * x + 5], o[8 * x + 6], o[8 * x + 7]);
          }
        }
        if (nn == 0) {
          s_m[parity][wave][gl] = Mc;
          s_l[parity][wave][gl] = Lc;
        }
      }
    }
    if (!alone) {
      // One barrier per piece: the other parity's buffers are only written
      // again after the next such piece's barrier.
      lds_barrier();
      for (int i = 64 * wave + fl; i < hpw * G * (D / 2); i += 64 * W) {
        const int d = 2 * (i % (D / 2)), r = i / (D / 2);
        const int gq = r % G, hh = r / G;
        float M = kNegBig;
        for (int t = 0; t < TS; ++t) M = fmaxf(M, s_m[parity][hh + hpw * t][gq]);
        float L = 0.f, o0 = 0.f, o1 = 0.f;
        for (int t = 0; t < TS; ++t) {
          const int ww = hh + hpw * t;
          const float w = fast_exp2(s_m[parity][ww][gq] - M);
          L = fmaf(s_l[parity][ww][gq], w, L);
          const float2 x = *reinterpret_cast<const float2*>(&s_o[parity][ww][gq][d]);
          o0 = fmaf(x.x, w, o0);
          o1 = fmaf(x.y, w, o1);
        }
        const float inv = L > 0.f ? 1.f / L : 0.f;
        const float o[2] = {o0 * inv, o1 * inv};
        write_piece<D, 2>(a, cp, h0 + hh, group, G * split + gq, d, o,
                          L > 0.f ? M + fast_log2(L) : -INFINITY, d == 0);
      }
      parity ^= 1;
    }
  };

  // Fused append.  The wave that owns a request's last page writes the new
  // token's row of its head just before it requests the page: one wave's memory
  // operations are performed in order, so the page comes back with the row.
  // Lane l holds 16-byte chunk l % (D / 8) of the K (or V) row; the row of the
  // first such page among the segment's leading pieces is loaded ahead.
  const bool appending = a.new_k != nullptr;
  auto load_new = [&](int b) __attribute__((always_inline)) {
    const int nl = local_lane();
    const uint16_t* src = nl >= D / 8 ? a.new_v + int64_t(b) * a.new_v_stride
                                      : a.new_k + int64_t(b) * a.new_k_stride;
    u32x4_t r = {0, 0, 0, 0};
    if (nl < D / 4) r = *reinterpret_cast<const u32x4_a4_t*>(src + h * D + (nl % (D / 8)) * 8);
    return r;
  };
  u32x4_t nrow = {0, 0, 0, 0};
  int nslot = -1;
  if (appending) {
    for (int i = 0; i < kNewMax && k + i < k_end && nslot < 0; ++i) {
      const int4 pd = scalar_int4(a.pieces, 2 * (k + i)), pt = scalar_int4(a.pieces, 2 * (k + i) + 1);
      if (pd.z == pt.x + 1 && (pt.x - g0) / PU % TS == ts) {
        nslot = pt.x;
        nrow = load_new(pd.x);
      }
    }
  }
  auto append_page = [&](int slot, int32_t id) __attribute__((always_inline)) {
    if (id < 0) return;
    while (slot >= ip.z && ki + 1 < k_end) {
      ++ki;
      ip = scalar_int4(a.pieces, 2 * ki);
      it = scalar_int4(a.pieces, 2 * ki + 1);
    }
    const int tnew = min(max(it.y, 0), kPage) - 1;
    if (slot != it.x || tnew < 0) return;
    if (slot != nslot) nrow = load_new(ip.x);
    const int nl = local_lane();
    const char* dst = (nl >= D / 8 ? vbytes : kbytes) + int64_t(id) * block_bytes +
                      int64_t(tnew) * tsb + h * D * 2 + (nl % (D / 8)) * 16;
    if (nl < D / 4)
      __builtin_nontemporal_store(nrow, reinterpret_cast<u32x4_a8_t*>(const_cast<char*>(dst)));
    wave_lds_fence();
  };

  auto append_unit = [&](int j, const Ids& ids) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < PU; ++x) append_page(page_slot(j, x), ids.v[x]);
  };

  Ids id = unit_ids(0);
  if (appending) append_unit(0, id);
  load_unit(kr, kbytes, k_off, id);
  load_unit(vr, vbytes, v_off, id);
  load_q(q, cp.x);
  load_q(qn, scalar_int4(a.pieces, 2 * min(k + 1, k_end - 1)).x);
  reset();
  int pos = nw > 0 ? page_slot(0, 0) : INT32_MAX;  // first page not yet consumed
  for (int j = 0;;) {
    while (pos >= cp.z) {
      finish();
      if (++k >= k_end) return;
      cp = scalar_int4(a.pieces, 2 * k);
      ct = scalar_int4(a.pieces, 2 * k + 1);
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int x = 0; x < C::kQ; ++x) q[g][x] = qn[g][x];
      load_q(qn, scalar_int4(a.pieces, 2 * min(k + 1, k_end - 1)).x);
      reset();
      holds = false;
    }
    holds = true;
    // The tokens of each page that the piece holds: none of a missing page, or
    // of one that lies in another piece (a unit may cross into the next piece:
    // it is then consumed once for each, and refilled after the last).
    int valid[PU];
#pragma unroll
    for (int x = 0; x < PU; ++x) {
      const int slot = page_slot(j, x);
      const bool in = PU == 1 || (slot >= pos && slot < cp.z);
      valid[x] = id.v[x] < 0 || !in ? 0 : (slot == ct.x ? min(max(ct.y, 0), kPage) : kPage);
    }
    const bool crosses = PU > 1 && page_slot(j, PU - 1) >= cp.z && cp.z < g0 + n;  // uniform
    const Ids next = unit_ids(j + 1);
    float p[NG][PU][4];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
      for (int y = 0; y < PU; ++y) {
        f32x4_t d[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          d[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < C::kQ; ++x) {
            const u32x4_t kk = kr[y][i + 4 * x], qq = q[g][x];
            d[i] = mfma_4x4x4(kk[0], kk[1], qq[0], qq[1], d[i]);
            d[i] = mfma_4x4x4(kk[2], kk[3], qq[2], qq[3], d[i]);
          }
        }
        // Sum over the chunks of a row; lane row c keeps tokens t_row .. +3.
        // The quads of a row must end up with the same bits, as they decide alone
        // on the rescale and share the row's l: turned by two quads first, quads j
        // and j + 2 hold the same sum, and turned by one then, every quad adds the
        // same two.  (By one first, the quads' sums differ by fp32 rounding.)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x;
          if constexpr (D == 64)
            x = swap16_add(d[0][r], d[1][r]);
          else
            x = swap16_add(swap32_add(d[0][r], d[2][r]), swap32_add(d[1][r], d[3][r]));
          x += dpp<kDppRowRor8>(x);
          x += dpp<kDppRowRor4>(x);
          p[g][y][r] = x;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!crosses) {
      if (appending) append_unit(j + 1, next);
      load_unit(kr, kbytes, k_off, next);
    }
#pragma unroll
    for (int y = 0; y < PU; ++y) {
      if (valid[y] < kPage) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p[g][y][r] = t_row + r < valid[y] ? p[g][y][r] : -INFINITY;
        // Rows past the end may hold anything (even NaN bits): 0 * v stays 0.
        // (A page without tokens is left out of p.v.)
        if (PU == 1 || valid[y] > 0) {
#pragma unroll
          for (int u = 0; u < NL; ++u)
            if (v_tok + v_step(u) >= valid[y]) vr[y][u] = u32x4_t{0, 0, 0, 0};
        }
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      float mx = -INFINITY;
#pragma unroll
      for (int y = 0; y < PU; ++y)
        mx = fmaxf(mx, fmaxf(fmaxf(p[g][y][0], p[g][y][1]), fmaxf(p[g][y][2], p[g][y][3])));
      const float cand = fmaxf(m[g], mx * a.scale_log2);
      const bool grow = cand > m[g] + kRescaleLog2;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float al = grow ? fast_exp2(m[g] - cand) : 1.f;
        m[g] = grow ? cand : m[g];
        l[g] *= al;
        const float a0 = quad_lane<0>(al), a1 = quad_lane<1>(al), a2 = quad_lane<2>(al),
                    a3 = quad_lane<3>(al);
#pragma unroll
        for (int e = 0; e < NE; ++e) {
          acc[g][e][0] *= a0;
          if constexpr (G > 1) {
            acc[g][e][1] *= a1;
            acc[g][e][2] *= a2;
            acc[g][e][3] *= a3;
          }
        }
      }
#pragma unroll
      for (int y = 0; y < PU; ++y) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          p[g][y][r] = fast_exp2(fmaf(p[g][y][r], a.scale_log2, -m[g]));
        l[g] += (p[g][y][0] + p[g][y][1]) + (p[g][y][2] + p[g][y][3]);
      }
    }
#pragma unroll
    for (int i = 0; i < PU * NL; ++i) {
      const int y = i / NL, u = i % NL;
      if (PU > 1 && valid[y] == 0) continue;  // uniform
      float pu[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if constexpr (D == 64)
          pu[g] = nn < 8 ? p[g][y][2 * u] : p[g][y][2 * u + 1];
        else
          pu[g] = p[g][y][u & 3];
      }
      const int e0 = D == 256 ? 8 * (u >> 2) : 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float v0 = bf16lo(vr[y][u][w]), v1 = bf16hi(vr[y][u][w]);
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          if constexpr (G == 1) {
            acc[g][e0 + 2 * w][0] = fmaf(pu[g], v0, acc[g][e0 + 2 * w][0]);
            acc[g][e0 + 2 * w + 1][0] = fmaf(pu[g], v1, acc[g][e0 + 2 * w + 1][0]);
          } else {
            acc[g][e0 + 2 * w] =
                __builtin_amdgcn_mfma_f32_4x4x1f32(pu[g], v0, acc[g][e0 + 2 * w], 0, 0, 0);
            acc[g][e0 + 2 * w + 1] =
                __builtin_amdgcn_mfma_f32_4x4x1f32(pu[g], v1, acc[g][e0 + 2 * w + 1], 0, 0, 0);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // (bounds the widened V held at once)
    }
    if (!crosses) {
      load_unit(vr, vbytes, v_off, next);
      id = next;
      ++j;
      pos = j < nw ? page_slot(j, 0) : INT32_MAX;
    } else {
      pos = cp.z;
    }
  }
}

// ---------------------------------------------------------------------------
// Split-K merge.
// ---------------------------------------------------------------------------
struct MergeArgs {
  const float* part_o;
  const float* part_lse;
  const int32_t* req_nparts;
  int32_t max_parts;
  int32_t num_kv_heads;
  int32_t group;
  uint16_t* out;
  int64_t out_stride;
  float* lse;
};

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// One wave per (request, query head), for plans with at most kSpecParts pieces
// per request.  The partials and the log2-sum-exps are loaded together with the request's piece
// count (all inside the max_parts rows the workspace holds for the request),
// so the common case costs one memory round trip; lane p weighs piece p and
// every lane folds its D/64 dims.  Requests with a single piece were finished
// by the streaming kernel; requests with no pages get a zero output and
// lse = -inf.
//
// With no split request in the batch (max_parts == 1) the launch only zeroes
// the empty requests and the workspace is absent (part_o == part_lse ==
// null): then no partial is read, and every request counts at most one
// piece.
constexpr int kSpecParts = 16;
constexpr int64_t kNarrowPerCu = 8;  // narrow segments per CU, at most

template <int D>
__global__ __launch_bounds__(64) void decode_merge_kernel(MergeArgs a) {
  constexpr int EPL = D / 64;  // dims per lane
  const int hq = blockIdx.x;
  const int b = blockIdx.y;
  const int lane = threadIdx.x;
  const int G = a.group;
  const int Hq = a.num_kv_heads * G;
  const int h = hq / G;
  const int g = hq - h * G;
  const bool have_parts = a.part_o != nullptr && a.part_lse != nullptr;  // uniform
  const int max_parts = have_parts ? a.max_parts : 1;
  const int64_t base = (int64_t(b) * a.num_kv_heads + h) * max_parts;
  const int64_t lse0 = base * G + g;  // piece p at part_lse[lse0 + p * G]
  const int nparts_raw = a.req_nparts[b];
  const int nspec = have_parts ? min(max_parts, kSpecParts) : 0;
  const float lse_spec = (have_parts && lane < max_parts)
                             ? a.part_lse[lse0 + int64_t(lane) * G] : -INFINITY;
  float po[kSpecParts][EPL];
#pragma unroll
  for (int p = 0; p < kSpecParts; ++p) {
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      po[p][e] = p < nspec ? a.part_o[((base + p) * G + g) * D + lane * EPL + e] : 0.f;
  }
  const int nparts = min(nparts_raw, max_parts);
  if (nparts == 1) return;
  uint16_t* out = a.out + int64_t(b) * a.out_stride + int64_t(hq) * D;

  float mx = lane < nparts ? lse_spec : -INFINITY;
  mx = wave_max(mx);
  if (nparts <= 0 || mx == -INFINITY) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) out[lane * EPL + e] = 0;
    if (a.lse && lane == 0) a.lse[int64_t(b) * Hq + hq] = -INFINITY;
    return;
  }
  float acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
  const float w0 = lane < nparts ? fast_exp2(lse_spec - mx) : 0.f;
  float S = w0;
#pragma unroll
  for (int p = 0; p < kSpecParts; ++p) {
    if (p < nparts) {
      const float wp = readlane_f(w0, p);
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[e] = fmaf(wp, po[p][e], acc[e]);
    }
  }
  S = wave_sum(S);
  const float inv = 1.f / S;
#pragma unroll
  for (int e = 0; e < EPL; ++e) out[lane * EPL + e] = f32_to_bf16(acc[e] * inv);
  if (a.lse && lane == 0) a.lse[int64_t(b) * Hq + hq] = (mx + fast_log2(S)) * kLn2;
}

// Plans whose requests may have more than kSpecParts pieces (few requests over
// many segments): the same merge by four waves per (request, query head), wave
// w folding pieces w, w + 4, ... with four partials in flight, the waves' sums
// added through LDS.  One wave alone folds them as a chain of single loads:
// 15.7 us at 65 pieces (8 requests of 300-2000 tokens, 8 KV heads) and 57 us
// at 256 (one request of 4096), against 5.1 and 9.1 us this way.  At 16 pieces
// and fewer the chain is already one batch of loads and the smaller workgroup
// starts sooner.
constexpr int kManyWaves = 4;

template <int D>
__global__ __launch_bounds__(64 * kManyWaves) void decode_merge_many_kernel(MergeArgs a) {
  constexpr int EPL = D / 64;     // dims per lane
  constexpr int kAhead = 4;       // partials in flight per wave
  __shared__ float s_acc[kManyWaves][D];
  const int hq = blockIdx.x;
  const int b = blockIdx.y;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int G = a.group;
  const int h = hq / G;
  const int g = hq - h * G;
  const int64_t base = (int64_t(b) * a.num_kv_heads + h) * a.max_parts;
  const float* lp = a.part_lse + base * G + g;                    // piece p at lp[p * G]
  const float* op = a.part_o + (base * G + g) * D + lane * EPL;   // piece p at op[p * G * D]
  const int nparts = min(a.req_nparts[b], a.max_parts);
  if (nparts == 1) return;  // (uniform) written by the streaming kernel
  // Every wave finds the maximum and the sum of the weights over all pieces.
  float mx = -INFINITY;
  for (int p = lane; p < nparts; p += 64) mx = fmaxf(mx, lp[int64_t(p) * G]);
  mx = wave_max(mx);
  float acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
  float S = 0.f;
  if (mx != -INFINITY) {
    for (int q0 = 0; q0 < nparts; q0 += 64) {
      const float w = q0 + lane < nparts ? fast_exp2(lp[int64_t(q0 + lane) * G] - mx) : 0.f;
      S += w;
      const int cnt = min(64, nparts - q0);
      for (int j0 = wave; j0 < cnt; j0 += kManyWaves * kAhead) {
        float x[kAhead][EPL];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          const int j = min(j0 + kManyWaves * i, cnt - 1);  // (past the end: weight 0 below)
#pragma unroll
          for (int e = 0; e < EPL; ++e) x[i][e] = op[int64_t(q0 + j) * G * D + e];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
          const int j = j0 + kManyWaves * i;
          if (j < cnt) {  // uniform
            const float wj = readlane_f(w, j);
#pragma unroll
            for (int e = 0; e < EPL; ++e) acc[e] = fmaf(wj, x[i][e], acc[e]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EPL; ++e) s_acc[wave][lane * EPL + e] = acc[e];
  __syncthreads();
  S = wave_sum(S);
  const bool none = mx == -INFINITY;  // no pages, or none present: 0 and -inf
  const float inv = none ? 0.f : 1.f / S;
  uint16_t* out = a.out + int64_t(b) * a.out_stride + int64_t(hq) * D;
  for (int d = threadIdx.x; d < D; d += 64 * kManyWaves) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < kManyWaves; ++w) o += s_acc[w][d];
    out[d] = f32_to_bf16(o * inv);
  }
  if (a.lse && threadIdx.x == 0)
    a.lse[int64_t(b) * a.num_kv_heads * G + hq] = none ? -INFINITY : (mx + fast_log2(S)) * kLn2;
}

template <int D>
void launch_merge(const MergeArgs& m, int num_qo_heads, int batch, hipStream_t s) {
  const dim3 grid{unsigned(num_qo_heads), unsigned(batch)};
  if (m.max_parts > kSpecParts)
    decode_merge_many_kernel<D><<<grid, 64 * kManyWaves, 0, s>>>(m);
  else
    decode_merge_kernel<D><<<grid, 64, 0, s>>>(m);
}

// Segment cuts of the flattened page list [0, total): cut[s] is segment s's
// first page, cut[segs] = total.  The segments cost the same, a page counting
// kPageCost and every request that starts strictly inside a segment
// kSwitchCost more: at such a piece switch the workgroup loads the next
// request's record and q while its page pipeline drains by about one page
// (a 35-page segment with one switch was measured 2.5 us = 1.15 pages slower
// than one without).  Every segment keeps at least one page; if the balanced
// cuts would give a segment more than kMaxSegPages pages, equal page counts
// are used instead.
constexpr int64_t kPageCost = 8;
constexpr int64_t kSwitchCost = 9;

std::vector<int64_t> cut_segments(const int32_t* indptr, int batch, int64_t total,
                                  int64_t segs) {
  std::vector<int64_t> cut(size_t(segs) + 1);
  cut[0] = 0;
  cut[size_t(segs)] = total;
  if (segs <= 1) return cut;
  // first pages of the requests after the first non-empty one
  std::vector<int64_t> starts;
  for (int b = 1; b < batch; ++b)
    if (indptr[b + 1] > indptr[b] && indptr[b] > 0) starts.push_back(indptr[b]);
  // F(x) = cost of pages [0, x): cut s goes where F is nearest to s/segs of
  // the total, so a cut can land exactly on a request's first page (which
  // then costs no switch: F counts it in the segment it starts).  F is linear
  // between starts, so the walk goes from start to start and not page by page
  // (a plan of 70 requests with 3040 pages, cut twice: 19.1 -> 11.1 us).
  const int64_t num_starts = int64_t(starts.size());
  const int64_t T = kPageCost * total + kSwitchCost * num_starts;  // below 2^35
  auto F = [&](int64_t x, int64_t below) { return kPageCost * x + kSwitchCost * below; };
  int64_t x = 0, below = 0;  // below = starts < x
  int64_t target = 0, rest = 0;  // s T / segs and its remainder
  bool ok = true;
  for (int64_t s = 1; s < segs; ++s) {
    target += T / segs;
    rest += T % segs;
    if (rest >= segs) rest -= segs, ++target;
    while (x < total && F(x, below) < target) {
      const int64_t end = below < num_starts ? starts[size_t(below)] : total;
      if (x < end) {
        x = std::min(end, x + (target - F(x, below) + kPageCost - 1) / kPageCost);
      } else {  // on a start: the page after it costs the switch, too
        ++x;
        ++below;
      }
    }
    // x is the first page with F(x) >= target; x - 1 may be nearer
    int64_t pick = x;
    if (x > 0) {
      const int64_t below_prev = below - ((below > 0 && starts[size_t(below) - 1] == x - 1) ? 1 : 0);
      if (target - F(x - 1, below_prev) < F(x, below) - target) pick = x - 1;
    }
    cut[size_t(s)] = std::min(std::max(pick, cut[size_t(s) - 1] + 1), total - (segs - s));
    ok = ok && cut[size_t(s)] - cut[size_t(s) - 1] <= kMaxSegPages;
  }
  ok = ok && total - cut[size_t(segs) - 1] <= kMaxSegPages;
  if (!ok)
    for (int64_t s = 1; s < segs; ++s) cut[size_t(s)] = s * total / segs;
  return cut;
}

// Whether a request lies in more than one segment.
bool cuts_a_request(const int32_t* indptr, int batch, const std::vector<int64_t>& cut) {
  int b = 0;
  for (size_t s = 1; s + 1 < cut.size(); ++s) {
    while (b < batch && indptr[b + 1] <= cut[s]) ++b;
    if (b < batch && indptr[b] < cut[s]) return true;
  }
  return false;
}

// The most leading pieces of a segment that reach the end of a request.
int32_t leading_ends(const int32_t* indptr, int batch, const std::vector<int64_t>& cut) {
  int32_t most = 0;
  int b = 0;
  for (size_t s = 0; s + 1 < cut.size(); ++s) {
    while (b < batch && indptr[b + 1] <= cut[s]) ++b;
    int32_t ends = 0;
    for (int i = b; i < batch && indptr[i + 1] <= cut[s + 1]; ++i) ends += indptr[i + 1] > indptr[i];
    most = std::max(most, ends);
  }
  return most;
}

// The most segments that one request lies in.
int32_t most_pieces(const int32_t* indptr, int batch, const std::vector<int64_t>& cut) {
  int64_t most = 1;
  size_t s = 1;
  for (int b = 0; b < batch; ++b) {
    while (s + 1 < cut.size() && cut[s] <= indptr[b]) ++s;  // the first cut past its start
    size_t e = s;
    while (e + 1 < cut.size() && cut[e] < indptr[b + 1]) ++e;
    most = std::max<int64_t>(most, int64_t(e - s) + 1);
    s = e;
  }
  return int32_t(most);
}

// Whether a head layout has the LDS kernel.
bool lds_layout(int group, int head_dim, int num_kv_heads) {
  return head_dim == 128 && group <= 4 && num_kv_heads % kLdsHeads == 0;
}

// KV heads per workgroup of the wave kernel: its waves are split between heads
// and pages.  More heads read longer runs of each token row, fewer leave longer
// segments and so fewer pieces to merge.  Heads in twos (6, 10, 14) are taken two
// at a time where rows are short or long: 6 heads, 1 -> 2 per workgroup, us: 8
// requests of 300-2000 tokens, head_dim 64, groups 1 and 4 14.6 -> 13.9, 14.3 -> 13.0
// (narrow form, 32 of 500-3000: 24.6 -> 24.9, 25.0 -> 26.0); 32 of 500-3000, head_dim
// 256 63.2 -> 59.9, 61.7 -> 59.6; at 128 33.5 and 33.6, 36.5 and 36.4.
int wave_heads(int head_dim, int num_kv_heads) {
  if (num_kv_heads % 4 == 0) return 4;
  return num_kv_heads == 2 || (head_dim != 128 && num_kv_heads % 2 == 0) ? 2 : 1;
}

// Whether a kernel takes a schedule's KV heads per workgroup.
bool valid_heads_per_group(int group, int head_dim, int num_kv_heads, int hpw) {
  if (hpw == kLdsHeads) return lds_layout(group, head_dim, num_kv_heads);
  return (hpw == 1 || hpw == 2 || hpw == 4) && num_kv_heads % hpw == 0;
}

// The wave kernel's form follows from the grid: all its waves on a segment, or,
// with more segments than one workgroup per CU can take, one wave per head of
// each, several workgroups per CU.  (Either form runs any plan.)  Plans have that
// many segments where they were made for the narrow form, or where the page cap
// asks for them; those of the latter, long segments, run narrow only if that
// leaves no more than a quarter of the chip's waves out.
template <int G, int D>
void launch_wave(const DecodeArgs& a, dim3 grid, int hpw, hipStream_t s) {
  constexpr int kWaves = WaveCfg<G, D>::kWaves;
  const int64_t workgroups = int64_t(grid.x) * grid.y;
  const bool capped = a.total_pages > kMaxSegPages / 2 * int64_t(grid.x);
  if (workgroups > kChipCus && (!capped || workgroups * hpw >= kChipCus * kWaves * 3 / 4))
    decode_wave_kernel<G, D, true><<<grid, 64 * hpw, 0, s>>>(a);
  else
    decode_wave_kernel<G, D, false><<<grid, 64 * kWaves, 0, s>>>(a);
}

template <int G, int D>
void launch_segments(const DecodeArgs& a, int segments, int head_groups, int hpw,
                     hipStream_t s) {
  const dim3 grid{unsigned(segments), unsigned(head_groups)};
  if constexpr (D == 128 && G <= 4) {
    if (hpw == kLdsHeads) {
      decode_lds_kernel<G><<<grid, 64 * kLdsHeads, 0, s>>>(a);
      return;
    }
  }
  if constexpr (D == 256 && G == 8) {
    DecodeArgs b = a;
    b.q_splits = 2;
    launch_wave<4, D>(b, dim3{grid.x, 2 * grid.y}, hpw, s);
  } else {
    launch_wave<G, D>(a, grid, hpw, s);
  }
}

template <int D>
bool dispatch_group(int group, const DecodeArgs& a, int segments, int head_groups, int hpw,
                    hipStream_t s) {
  switch (group) {
    case 1: launch_segments<1, D>(a, segments, head_groups, hpw, s); return true;
    case 2: launch_segments<2, D>(a, segments, head_groups, hpw, s); return true;
    case 4: launch_segments<4, D>(a, segments, head_groups, hpw, s); return true;
    case 8: launch_segments<8, D>(a, segments, head_groups, hpw, s); return true;
    default: return false;
  }
}

// Merge of two bf16 attention states (a8 as a standalone op).
__global__ __launch_bounds__(256) void merge_states_kernel(
    const uint16_t* o1, const float* lse1, const uint16_t* o2,
    const float* lse2, int64_t n, int head_dim, uint16_t* out, float* lse) {
  const int64_t total = n * head_dim;
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * 256) {
    const int64_t r = i / head_dim;
    const float l1 = lse1[r], l2 = lse2[r];
    const float mx = fmaxf(l1, l2);
    float w1, w2, nl;
    if (mx == -INFINITY) {
      w1 = w2 = 0.f;
      nl = -INFINITY;
    } else {
      const float e1 = expf(l1 - mx), e2 = expf(l2 - mx);
      nl = mx + logf(e1 + e2);
      w1 = e1 / (e1 + e2);
      w2 = e2 / (e1 + e2);
    }
    const float a1 = __uint_as_float(uint32_t(o1[i]) << 16);
    const float a2 = __uint_as_float(uint32_t(o2[i]) << 16);
    // Element i is read and written by the same thread, so out may alias o1
    // or o2; lse may not alias lse1/lse2 (checked on the host).
    out[i] = f32_to_bf16(a1 * w1 + a2 * w2);
    if (lse && i - r * head_dim == 0) lse[r] = nl;
  }
}

}  // namespace
}  // namespace kvc

using namespace kvc;

extern "C" int64_t kvc_decode_workspace_bytes(int32_t batch, int32_t num_qo_heads,
                                              int32_t head_dim,
                                              int32_t max_partitions) {
  if (batch <= 0 || num_qo_heads <= 0 || head_dim <= 0 || max_partitions <= 1)
    return 0;
  const int64_t rows = int64_t(batch) * num_qo_heads * max_partitions;
  const int64_t o_bytes = (rows * head_dim * 4 + 255) / 256 * 256;
  const int64_t l_bytes = (rows * 4 + 255) / 256 * 256;
  return o_bytes + l_bytes;
}

extern "C" int64_t kvc_decode_plan_ints(int32_t batch, int32_t num_segments) {
  if (batch < 0 || num_segments < 0) return -1;
  return 4 * int64_t(num_segments) + 8 * (int64_t(num_segments) + batch) + batch;
}

extern "C" int kvc_decode_plan(const int32_t* indptr_host, const int32_t* last_page_len_host,
                               int32_t batch, int32_t num_qo_heads, int32_t num_kv_heads,
                               int32_t head_dim, int32_t page_size,
                               int32_t num_segments_hint, int32_t num_cus,
                               kvc_decode_schedule* sched, int32_t* plan_host,
                               int64_t plan_capacity) {
  KVC_REQUIRE(sched, KVC_ERR_INVALID_ARG, "null schedule");
  KVC_REQUIRE(batch >= 0 && batch <= 65535, KVC_ERR_INVALID_ARG,
              "batch must be in [0, 65535]");
  KVC_REQUIRE(batch == 0 || (indptr_host && last_page_len_host), KVC_ERR_INVALID_ARG,
              "null indptr or last_page_len");
  KVC_REQUIRE(num_qo_heads > 0 && num_kv_heads > 0 &&
                  num_qo_heads % num_kv_heads == 0,
              KVC_ERR_INVALID_ARG, "num_qo_heads must be a multiple of num_kv_heads");
  const int group = num_qo_heads / num_kv_heads;
  KVC_REQUIRE(group == 1 || group == 2 || group == 4 || group == 8,
              KVC_ERR_UNSUPPORTED, "group size must be 1, 2, 4 or 8");
  KVC_REQUIRE(head_dim == 64 || head_dim == 128 || head_dim == 256,
              KVC_ERR_UNSUPPORTED, "head_dim must be 64, 128 or 256");
  KVC_REQUIRE(page_size == kPage, KVC_ERR_UNSUPPORTED, "page_size must be 16");
  KVC_REQUIRE(num_kv_heads <= 65535, KVC_ERR_INVALID_ARG, "too many KV heads");
  KVC_REQUIRE(batch == 0 || indptr_host[0] == 0, KVC_ERR_INVALID_ARG,
              "indptr[0] must be 0");
  int32_t num_empty = 0;
  for (int b = 0; b < batch; ++b) {
    KVC_REQUIRE(indptr_host[b + 1] >= indptr_host[b], KVC_ERR_INVALID_ARG,
                "indptr must be non-decreasing");
    num_empty += indptr_host[b + 1] == indptr_host[b];
  }
  const int64_t total = batch > 0 ? indptr_host[batch] : 0;
  const bool lds = lds_layout(group, head_dim, num_kv_heads);
  int hpw = lds ? kLdsHeads : wave_heads(head_dim, num_kv_heads);
  // Workgroups a KV head group's segments share the CUs with (head_dim 256
  // serves a group of 8 as two).
  const int q_splits = head_dim == 256 && group == 8 ? 2 : 1;

  // Segments per KV-head group: one workgroup per CU, at most
  // kMaxSegPages pages each, at least one page each.  When the page cap
  // forces more segments than there are slots, the count is rounded
  // up to whole rounds of slots, so no round runs a few stragglers alone.
  // A round of the wave kernel has no more workgroups than slots: one fills a CU
  // (at head_dim 64 and 256 and for groups of 8), so of the 258 that 3, 6 or 12
  // KV heads gave rounded up, two ran a second full length alone (32 requests of
  // 500-3000 tokens, rounded up -> down, us: 6 heads, head_dim 64, group 4 31.9 ->
  // 24.1; 6 at 256 103 -> 71; 6 at 128, group 8 66 -> 44; 3 at 64 26.4 -> 19.7).
  // The LDS kernel's count stays rounded up (24 KV heads: 258).
  const int64_t slots = num_cus > 0 ? num_cus : 256;
  auto segment_count = [&](int heads) -> int64_t {
    if (total == 0) return 0;
    const int64_t at_least = (total + kMaxSegPages - 1) / kMaxSegPages;
    int64_t n;
    if (num_segments_hint > 0) {
      n = std::max<int64_t>(num_segments_hint, at_least);
    } else {
      const int64_t groups = int64_t(num_kv_heads / heads) * q_splits;
      const int64_t per_round = heads == kLdsHeads ? (slots + groups - 1) / groups
                                                   : std::max<int64_t>(1, slots / groups);
      n = (std::max(per_round, at_least) + per_round - 1) / per_round * per_round;
    }
    return std::min<int64_t>(n, total);
  };
  auto fine_segments = [&]() -> int64_t {
    const int64_t round = (slots * (group == 8 ? 4 : 8) + num_kv_heads - 1) / num_kv_heads;
    const int64_t at_least = (total + kMaxSegPages - 1) / kMaxSegPages;
    return std::min((std::max(round, at_least) + round - 1) / round * round, total);
  };
  int64_t segs = segment_count(hpw);
  KVC_REQUIRE(segs <= (int64_t(1) << 30), KVC_ERR_INVALID_ARG, "too many segments");

  std::vector<int64_t> cut = cut_segments(indptr_host, batch, total, segs);

  // Small batches (head_dim 128, no forced segment count): when every request
  // fits in kSmallMaxPages pages and the segments would cut a request,
  // one workgroup per (request, KV head) streams it and merges its waves'
  // states in LDS instead (no partials, no merge launch).
  int64_t max_pages = 0;
  for (int b = 0; b < batch; ++b)
    max_pages = std::max<int64_t>(max_pages, indptr_host[b + 1] - indptr_host[b]);
  // Layouts without the LDS kernel are cut here as finely as eight workgroups per
  // CU (four for groups of 8) would be: that takes nearly every batch of requests
  // of two pages and more but those that line up with the segments, many of a
  // length (1024 of 26 tokens, 4 KV heads, group 4: 59 us this way, 18.6 in the
  // wave kernel's narrow form).
  if (num_segments_hint <= 0 && head_dim == 128 && total > 0 && max_pages <= kSmallMaxPages &&
      cuts_a_request(indptr_host, batch,
                     lds ? cut : cut_segments(indptr_host, batch, total, fine_segments()))) {
    const int64_t need = kvc_decode_plan_ints(batch, batch);
    sched->batch = batch;
    sched->num_qo_heads = num_qo_heads;
    sched->num_kv_heads = num_kv_heads;
    sched->head_dim = head_dim;
    sched->page_size = page_size;
    sched->num_segments = batch;
    sched->num_head_groups = num_kv_heads;
    sched->heads_per_group = 1;
    sched->total_pages = int32_t(total);
    sched->num_empty = num_empty;
    sched->plan_ints = need;
    sched->small_batch = 1;
    KVC_REQUIRE(plan_host && plan_capacity >= need, KVC_ERR_WORKSPACE,
                "plan buffer too small: need " + std::to_string(need) + " int32");
    // One segment and one piece per request, empty requests included.
    int32_t* segments = plan_host;
    int32_t* pieces = plan_host + 4 * int64_t(batch);
    int32_t* nparts = pieces + 8 * (2 * int64_t(batch));
    for (int b = 0; b < batch; ++b) {
      const int32_t p0 = indptr_host[b], p1 = indptr_host[b + 1];
      int32_t* rec = segments + 4 * b;
      rec[0] = b;
      rec[1] = b + 1;
      rec[2] = p0;
      rec[3] = p1 - p0;
      int32_t* pc = pieces + 8 * b;
      pc[0] = b;
      pc[1] = p0;
      pc[2] = p1;
      pc[3] = -1;
      pc[4] = p1 - 1;
      pc[5] = last_page_len_host[b];
      pc[6] = 0;
      pc[7] = 0;
      nparts[b] = p1 > p0 ? 1 : 0;
    }
    sched->num_pieces = batch;
    sched->pieces_offset = 4 * batch;
    sched->nparts_offset = 4 * batch + 16 * batch;
    sched->max_partitions = 1;
    sched->workspace_bytes = 0;
    sched->append_pieces = 1;
    return ok();
  }

  // Few pages for the LDS kernel's 8-head workgroups: at two or three pages
  // each they are all start-up and cut a long request into up to 256 pieces.
  // The wave kernel streams longer segments on 1, 2 or 4 heads per workgroup, of
  // which the shorter the requests, the more (in its narrow form, below, they are
  // alike).  Measured with 8 KV heads, one layer with its append, LDS kernel ->
  // 1 / 2 / 4 heads, in us:
  //   group 4, requests x pages:  1 x 256  26.0 -> 12.8 / 13.9 / 18.1
  //     2 x 500 28.3 -> 19.3 / 19.8 / 21.3     4 x 40    13.1 -> 11.1 / 11.2 / 13.0
  //     8 x 68  20.1 -> 14.4 / 14.0 / 14.7     16 x 110  29.1 -> 26.0 / 25.9 / 25.9
  //     20 x 37 19.7 -> 17.4 / 17.3 / 17.4     60 x 27   29.4 -> 26.4 / 26.6 / 26.4
  //     150 x 20 44.2 -> 42.6 / 43.3 / 42.6    12 x 250  41.6 -> 37.9 / 38.0 / 38.2
  //   groups 1, 2 (the LDS kernel's arithmetic is a quarter or half of that; group
  //   1's figures):
  //     2 x 138 16.7 -> 11.7 / 11.8 / 13.0     4 x 131   16.2 -> 13.7 / 13.2 / 13.8
  //     8 x 72  15.0 -> 14.1 / 13.4 / 13.6     1 x 2900  48.0 -> 39.1 / 38.0 / 40.2
  //     30 x 50 23.2 -> 22.7 / 22.6 / 22.7     30 x 100  37.1 -> 36.3 / 36.5 / 36.3
  //     20 x 37 15.4 -> 15.8 / 15.7 / 15.6
  //   above 12 pages per CU and KV head group the LDS kernel has long segments, too
  //   (64 requests of 512-4096 tokens: at 6.2 of 7.0 TB/s)
  const int64_t work = total * (num_kv_heads / kLdsHeads);  // pages of 8 heads
  const int64_t mean = total / std::max(1, batch - num_empty);  // pages per request
  // Batches for which the LDS kernel cannot append keep its plan, and with it which
  // calls take the append and which rows (40 requests of 3 tokens + 30 of 1590: 46
  // us with the append's launch, 42 here).
  if (lds && num_segments_hint <= 0 && work <= 12 * slots && mean >= (group == 4 ? 16 : 48) &&
      leading_ends(indptr_host, batch, cut) <= kNewMax) {
    hpw = group < 4 ? 2 : mean < 48 ? 4 : work <= 3 * slots ? 1 : 2;
    segs = segment_count(hpw);
    cut = cut_segments(indptr_host, batch, total, segs);
  }

  // Many requests per segment of the wave kernel: its waves would share every
  // request and meet at its end.  The narrow form, a wave per head and segment,
  // closes pieces without meeting; its segments are as many as the chip has waves
  // for (at most 8 per CU, at least two pages each), or three quarters of that (seven
  // eighths for groups 2 and 4 at head_dim 64: five sixths of them take 54.7 us
  // against the other form's 52.7 for 20 of 1100-11000 tokens, 8 KV heads, 35.9
  // against 33.2 for 40 of 2000-5000, 4 heads; group 8 53.3 against 54.0).  It
  // is taken where a request has at most about kSpecParts of them, so that the
  // merge stays one batch of loads, where they are more than the other form runs at
  // once, and where its partials fit the allocation-free run or are no more than
  // the other's.
  // Measured, waves on a segment together -> narrow, us a layer:
  //   1000 requests of 1-300 tokens, group 4, head_dim 128: 1 KV head 38.1 -> 25.9,
  //     2 50.9 -> 42.3, 3 85.9 -> 60.5, 4 82.0 -> 75.4; 8, group 8 182 -> 161
  //   the same, 8 KV heads, head_dim 64: group 1 81.2 -> 69.5, 4 93.0 -> 79.0,
  //     8 133 -> 98; 64 of 200-600, group 1 20.8 -> 18.9, 4 21.7 -> 20.0
  //   128 of 100-2000, head_dim 128, group 4: 1 KV head 22.9 -> 21.6, 4 55.0 -> 54.5
  // Not at head_dim 256: 128 of 100-2000, 2 KV heads, group 8 80 -> 91.
  if (hpw < kLdsHeads && num_segments_hint <= 0) {
    const int64_t requests = batch - num_empty;
    const int64_t waves = slots * wave_kernel_waves(group, head_dim);
    const int64_t heads = int64_t(num_kv_heads) * q_splits;  // waves of a narrow segment
    int64_t narrow =
        std::min({std::max<int64_t>(1, waves / heads), total / 2, kNarrowPerCu * slots});
    const int64_t most = kSpecParts * requests;
    const int eighths = head_dim == 64 && (group == 2 || group == 4) ? 7 : 6;
    if (8 * most * heads >= eighths * waves) narrow = std::min(narrow, most);
    const bool fits = num_segments_hint == 0 && head_dim < 256 && narrow <= most &&
                      2 * narrow * heads > 3 * slots * hpw;
    auto partials = [&](const std::vector<int64_t>& c) {
      return kvc_decode_workspace_bytes(batch, num_qo_heads, head_dim,
                                        most_pieces(indptr_host, batch, c));
    };
    // Short requests: one segment each, so that none is cut and no merge follows.
    // At head_dim 128 these are the many, alike in length, that the kernel above
    // leaves; the narrow form's balanced segments would cut them all but for a few
    // head counts (group 4, 6 KV heads: 342 of 26 tokens 20.7 -> 10.9 us, 1368 of 180
    // 170 -> 146; group 8, 1 head, 1024 of 66 23.3 -> 13.9; 4 heads, where 1024 of
    // 66 are not cut, 37.8 and 40.8).
    // At head_dim 64 and 256, in the narrow form where they fill three quarters of
    // its waves, else where they are one round of the other form's workgroups (two
    // for groups, whose merge costs more).
    //   8 KV heads, 1024 of 17-32 tokens: head_dim 64, group 1 40.4 -> 22.3 us, 4
    //   51.2 -> 24.5; head_dim 256, group 4 95 -> 69.  256 of 17-100, narrow
    //   segments against one each: head_dim 64, group 1 17.7 and 20.2, 4 21.7 and 19.4
    // While CUs are left over, with fewer heads per workgroup (few), so that more
    // waves share a request's pages.  8 requests, 4 KV heads, us by pages of a
    // request, 4 heads per workgroup -> 1 (and cut, 4 heads per workgroup):
    //   head_dim 64, group 1    3  6.6 -> 7.2 (7.9)    7  8.7 -> 7.3 (8.0)
    //                          16 12.6 -> 8.7 (8.8)
    //     group 4               3  7.4 -> 6.5 (8.2)   16 12.1 -> 8.9 (9.1)
    //   head_dim 256, group 1   4 12.0 -> 8.2 (10.2)  16 28.0 -> 12.7 (11.1)
    //     group 4               4 14.0 -> 8.2 (10.7)  16 28.1 -> 13.4 (11.8)
    //   2 heads at least for group 1 up to 6 pages, head_dim 64 (3 pages, 2 KV heads,
    //   2 -> 1: 5.9 -> 7.0)
    // At head_dim 256 not where the workgroup is on its pages longer than the
    // segments on theirs and a merge, which costs more for groups; with no partials to
    // be had (a negative hint), or more than the allocation-free run has, the
    // requests stay whole.
    const int fewest = head_dim == 64 && group == 1 && max_pages <= 6 ? 2 : 1;
    int few = hpw;
    while (few > fewest && 2 * requests * heads <= slots * few) few /= 2;
    const int64_t longest = segs > 0 ? (total + segs - 1) / segs : 0;
    const int64_t alone = group == 1 ? 6 : group == 2 ? 10 : 14;  // pages of a head
    const bool whole =
        max_pages > 1 && max_pages <= kSmallMaxPages &&
        (head_dim == 128 ? !lds
                         : (4 * requests * heads >= 3 * waves ||
                            requests * heads <= (group == 1 ? 1 : 2) * slots * hpw || !fits) &&
                               (head_dim == 64 || num_segments_hint < 0 ||
                                (max_pages - 2 * longest) * few <= alone ||
                                partials(cut) > KVC_NOALLOC_SCRATCH_BYTES));
    if (whole) {
      hpw = few;
      cut.clear();
      for (int i = 0; i < batch; ++i)
        if (indptr_host[i + 1] > indptr_host[i]) cut.push_back(indptr_host[i]);
      segs = int64_t(cut.size());
      cut.push_back(total);
    } else if (fits) {
      const int64_t rounds = (total + kMaxSegPages * narrow - 1) / (kMaxSegPages * narrow);
      std::vector<int64_t> cut_n = cut_segments(indptr_host, batch, total, rounds * narrow);
      if (partials(cut_n) <= std::max<int64_t>(KVC_NOALLOC_SCRATCH_BYTES, partials(cut))) {
        segs = rounds * narrow;
        cut = std::move(cut_n);
      }
    }
  }
  const int head_groups = num_kv_heads / hpw;

  const int64_t need = kvc_decode_plan_ints(batch, int32_t(segs));
  sched->batch = batch;
  sched->num_qo_heads = num_qo_heads;
  sched->num_kv_heads = num_kv_heads;
  sched->head_dim = head_dim;
  sched->page_size = page_size;
  sched->num_segments = int32_t(segs);
  sched->num_head_groups = head_groups;
  sched->heads_per_group = hpw;
  sched->total_pages = int32_t(total);
  sched->num_empty = num_empty;
  sched->plan_ints = need;
  sched->small_batch = 0;
  KVC_REQUIRE(plan_host && plan_capacity >= need, KVC_ERR_WORKSPACE,
              "plan buffer too small: need " + std::to_string(need) + " int32");

  // Plan image: segments [segs][4], pieces [num_pieces][8], req_nparts [batch].
  int32_t* segments = plan_host;
  const int64_t pieces_off = 4 * segs;
  int32_t* pieces = plan_host + pieces_off;
  int32_t* nparts = pieces + 8 * (segs + batch);
  std::fill(nparts, nparts + batch, 0);
  int64_t np = 0;
  int b = 0;
  int32_t append_pieces = 0;
  for (int64_t s = 0; s < segs; ++s) {
    const int64_t g0 = cut[size_t(s)];
    const int64_t g1 = cut[size_t(s) + 1];
    int32_t* rec = segments + 4 * s;
    rec[0] = int32_t(np);
    rec[2] = int32_t(g0);
    rec[3] = int32_t(g1 - g0);
    while (b < batch && indptr_host[b + 1] <= g0) ++b;
    for (int bb = b; bb < batch && indptr_host[bb] < g1; ++bb) {
      const int64_t sb = std::max<int64_t>(g0, indptr_host[bb]);
      const int64_t se = std::min<int64_t>(g1, indptr_host[bb + 1]);
      if (se > sb) {
        int32_t* pc = pieces + 8 * np++;
        pc[0] = bb;
        pc[1] = int32_t(sb);
        pc[2] = int32_t(se);
        pc[3] = nparts[bb]++;
        pc[4] = indptr_host[bb + 1] - 1;
        pc[5] = last_page_len_host ? last_page_len_host[bb] : kPage;
        pc[6] = 0;
        pc[7] = 0;
        // a request ending here: the fused append stages its new row by the
        // piece's index within the segment
        if (se == indptr_host[bb + 1])
          append_pieces = std::max<int32_t>(append_pieces, int32_t(np - rec[0]));
      }
    }
    rec[1] = int32_t(np);
  }
  int32_t max_parts = 1;
  for (int i = 0; i < batch; ++i) max_parts = std::max(max_parts, nparts[i]);
  // A request covered by a single piece is written directly (index -1).
  for (int64_t i = 0; i < np; ++i)
    if (nparts[pieces[8 * i]] == 1) pieces[8 * i + 3] = -1;
  sched->num_pieces = int32_t(np);
  sched->pieces_offset = int32_t(pieces_off);
  sched->nparts_offset = int32_t(pieces_off + 8 * (segs + batch));
  sched->max_partitions = max_parts;
  sched->workspace_bytes =
      kvc_decode_workspace_bytes(batch, num_qo_heads, head_dim, max_parts);
  sched->append_pieces = append_pieces;
  return ok();
}

namespace {
int decode_run(const kvc_decode_schedule* sched, const int32_t* plan, const void* q,
               int64_t q_batch_stride, const void* key_cache, const void* value_cache,
               int64_t cache_block_stride, int64_t cache_token_stride, int64_t num_blocks,
               const int32_t* indptr, const int32_t* indices, int64_t num_indices,
               const int32_t* last_page_len, const void* new_key, int64_t new_key_stride,
               const void* new_value, int64_t new_value_stride, float sm_scale,
               void* workspace, int64_t workspace_bytes, void* out, int64_t out_batch_stride,
               float* lse, void* stream) {
  KVC_REQUIRE(sched, KVC_ERR_INVALID_ARG, "null schedule");
  const int batch = sched->batch;
  if (batch == 0) return ok();
  // indices may be null (an empty tensor) when no request has a page; the
  // device indptr / last_page_len are not read (the plan image carries both).
  KVC_REQUIRE(plan && q && key_cache && value_cache && (indices || sched->total_pages == 0) &&
                  out,
              KVC_ERR_INVALID_ARG, "null pointer");
  const int Hq = sched->num_qo_heads, Hkv = sched->num_kv_heads, D = sched->head_dim;
  KVC_REQUIRE(Hkv > 0 && Hq % Hkv == 0, KVC_ERR_INVALID_ARG, "bad head counts");
  const int group = Hq / Hkv;
  KVC_REQUIRE(sched->page_size == kPage, KVC_ERR_UNSUPPORTED, "page_size must be 16");
  const bool small = sched->small_batch != 0;
  KVC_REQUIRE(sched->num_segments >= 0 && sched->max_partitions >= 1 &&
                  (small ? (D == 128 && sched->heads_per_group == 1 &&
                            sched->num_head_groups == Hkv && sched->num_segments == batch &&
                            sched->num_pieces == batch && sched->max_partitions == 1)
                         : (valid_heads_per_group(group, D, Hkv, sched->heads_per_group) &&
                            sched->num_head_groups == Hkv / sched->heads_per_group)) &&
                  sched->plan_ints == kvc_decode_plan_ints(batch, sched->num_segments),
              KVC_ERR_INVALID_ARG, "schedule not produced by kvc_decode_plan");
  KVC_REQUIRE(num_blocks > 0 && num_indices >= sched->total_pages, KVC_ERR_INVALID_ARG,
              "bad num_blocks or fewer indices than planned pages");
  KVC_REQUIRE(cache_token_stride >= int64_t(Hkv) * D &&
                  cache_block_stride >= cache_token_stride * kPage,
              KVC_ERR_INVALID_ARG, "cache strides smaller than the block");
  KVC_REQUIRE(cache_token_stride * kPage * 2 < (int64_t(1) << 31), KVC_ERR_INVALID_ARG,
              "a cache block spans more than 2 GiB");
  KVC_REQUIRE(q_batch_stride >= int64_t(Hq) * D && out_batch_stride >= int64_t(Hq) * D,
              KVC_ERR_INVALID_ARG, "q/out batch stride smaller than Hq*head_dim");
  KVC_REQUIRE(sm_scale > 0.f, KVC_ERR_INVALID_ARG, "sm_scale must be positive");
  const int vec_bytes = D == 64 ? 8 : 16;
  KVC_REQUIRE(aligned(q, vec_bytes) && aligned(key_cache, vec_bytes) &&
                  aligned(value_cache, vec_bytes) &&
                  (q_batch_stride * 2) % vec_bytes == 0 &&
                  (cache_block_stride * 2) % vec_bytes == 0 &&
                  (cache_token_stride * 2) % vec_bytes == 0,
              KVC_ERR_ALIGNMENT, "q/cache pointers or strides not vector aligned");
  KVC_REQUIRE(aligned(out, 4) && out_batch_stride % 2 == 0 && aligned(plan, 16),
              KVC_ERR_ALIGNMENT, "out must be 4-byte aligned with an even batch stride, "
                                 "plan 16-byte aligned");
  const int64_t need = kvc_decode_workspace_bytes(batch, Hq, D, sched->max_partitions);
  KVC_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), KVC_ERR_WORKSPACE,
              "decode workspace too small: need " + std::to_string(need) + " bytes");

  DecodeArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.q_stride = q_batch_stride;
  a.k_cache = static_cast<const uint16_t*>(key_cache);
  a.v_cache = static_cast<const uint16_t*>(value_cache);
  a.block_stride = cache_block_stride;
  a.token_stride = cache_token_stride;
  a.num_blocks = num_blocks;
  a.indices = indices;
  a.num_indices = num_indices;
  a.segments = reinterpret_cast<const int4*>(plan);
  a.pieces = reinterpret_cast<const int4*>(plan + sched->pieces_offset);
  a.total_pages = sched->total_pages;
  a.num_segments = sched->num_segments;
  a.scale_log2 = sm_scale * kLog2e;
  a.num_kv_heads = Hkv;
  a.max_parts = sched->max_partitions;
  const int64_t rows = int64_t(batch) * Hq * sched->max_partitions;
  a.part_o = need ? static_cast<float*>(workspace) : nullptr;
  a.part_lse = need ? reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                              (rows * D * 4 + 255) / 256 * 256)
                    : nullptr;
  // Partials are written (streaming kernel) and read (merge) only for split
  // requests, which exist only when max_partitions > 1; with one piece per
  // request both kernels get null partials and never touch them.
  KVC_REQUIRE(sched->max_partitions == 1 || (a.part_o && a.part_lse), KVC_ERR_WORKSPACE,
              "a plan with split requests needs the partials workspace");
  a.out = static_cast<uint16_t*>(out);
  a.out_stride = out_batch_stride;
  a.lse = lse;
  a.new_k = static_cast<const uint16_t*>(new_key);
  a.new_v = static_cast<const uint16_t*>(new_value);
  a.new_k_stride = new_key_stride;
  a.new_v_stride = new_value_stride;
  a.heads_per_group = sched->heads_per_group;
  a.q_splits = 1;
  if (new_key || new_value) {
    KVC_REQUIRE(new_key && new_value, KVC_ERR_INVALID_ARG, "new_key and new_value go together");
    const bool lds = !small && sched->heads_per_group == kLdsHeads;
    KVC_REQUIRE(!lds || sched->append_pieces <= kNewMax, KVC_ERR_UNSUPPORTED,
                "with 8 KV heads per workgroup the append takes at most " +
                    std::to_string(kNewMax) + " leading pieces per segment holding request "
                    "ends (schedule->append_pieces)");
    KVC_REQUIRE(new_key_stride >= int64_t(Hkv) * D && new_value_stride >= int64_t(Hkv) * D,
                KVC_ERR_INVALID_ARG, "new row stride smaller than a row");
    // The wave kernel takes any 4-byte aligned rows, the others 16-byte ones.
    const int row_bytes = small || lds ? 16 : 4;
    KVC_REQUIRE(aligned(new_key, row_bytes) && aligned(new_value, row_bytes) &&
                    (new_key_stride * 2) % row_bytes == 0 && (new_value_stride * 2) % row_bytes == 0,
                KVC_ERR_ALIGNMENT, "new rows must be " + std::to_string(row_bytes) + "-byte aligned");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);

  if (small) {
    // One workgroup per (request, KV head); outputs (empty requests too)
    // are written in the launch, no merge follows.
    const dim3 grid{unsigned(batch), unsigned(Hkv)};
    switch (group) {
      case 1: decode_small_kernel<1><<<grid, 64 * kSmallWaves, 0, s>>>(a); break;
      case 2: decode_small_kernel<2><<<grid, 64 * kSmallWaves, 0, s>>>(a); break;
      case 4: decode_small_kernel<4><<<grid, 64 * kSmallWaves, 0, s>>>(a); break;
      case 8: decode_small_kernel<8><<<grid, 64 * kSmallWaves, 0, s>>>(a); break;
      default:
        return set_error(KVC_ERR_UNSUPPORTED, "decode_run: unsupported group size " +
                                                  std::to_string(group));
    }
    KVC_LAUNCH_CHECK();
    return ok();
  }

  if (sched->num_segments > 0) {
    bool launched = false;
    const int segs = sched->num_segments, hg = sched->num_head_groups;
    const int hpw = sched->heads_per_group;
    if (D == 128) launched = dispatch_group<128>(group, a, segs, hg, hpw, s);
    else if (D == 64) launched = dispatch_group<64>(group, a, segs, hg, hpw, s);
    else if (D == 256) launched = dispatch_group<256>(group, a, segs, hg, hpw, s);
    KVC_REQUIRE(launched, KVC_ERR_UNSUPPORTED,
                "unsupported (group, head_dim) = (" + std::to_string(group) + ", " +
                    std::to_string(D) + ")");
    KVC_LAUNCH_CHECK();
  }
  // Single-piece requests were written by the streaming kernel; the merge
  // pass is needed for split requests and to zero empty ones.
  if (sched->max_partitions == 1 && sched->num_empty == 0) return ok();

  MergeArgs m;
  m.part_o = a.part_o;
  m.part_lse = a.part_lse;
  m.req_nparts = plan + sched->nparts_offset;
  m.max_parts = a.max_parts;
  m.num_kv_heads = Hkv;
  m.group = group;
  m.out = a.out;
  m.out_stride = out_batch_stride;
  m.lse = lse;
  if (D == 128) launch_merge<128>(m, Hq, batch, s);
  else if (D == 64) launch_merge<64>(m, Hq, batch, s);
  else launch_merge<256>(m, Hq, batch, s);
  KVC_LAUNCH_CHECK();
  return ok();
}

}  // namespace

extern "C" int kvc_batch_decode_run(
    const kvc_decode_schedule* sched, const int32_t* plan, const void* q,
    int64_t q_batch_stride, const void* key_cache, const void* value_cache,
    int64_t cache_block_stride, int64_t cache_token_stride, int64_t num_blocks,
    const int32_t* indptr, const int32_t* indices, int64_t num_indices,
    const int32_t* last_page_len, float sm_scale, void* workspace,
    int64_t workspace_bytes, void* out, int64_t out_batch_stride, float* lse,
    void* stream) {
  return decode_run(sched, plan, q, q_batch_stride, key_cache, value_cache, cache_block_stride,
                    cache_token_stride, num_blocks, indptr, indices, num_indices, last_page_len,
                    nullptr, 0, nullptr, 0, sm_scale, workspace, workspace_bytes, out,
                    out_batch_stride, lse, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free decode run: the split-K partials live in this library's own
// device array instead of a caller workspace.  Each GPU the library runs on
// holds one copy of the array until the process ends; all calls on one GPU
// share it (calls that overlap on one GPU race on it).  The partials are
// written before they are read within a call, so nothing needs clearing.
// ---------------------------------------------------------------------------
static __device__ __align__(256) char scratch[KVC_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on `device`, which must be the current device:
// looked up once per device (hipGetSymbolAddress; the array's host-side name
// is not a device address and is never passed to a kernel or a copy).
int scratch_address(int device, void** out) {
  KVC_REQUIRE(device >= 0 && device < kMaxDevices, KVC_ERR_INVALID_ARG,
              "device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    KVC_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    KVC_REQUIRE(p != nullptr, KVC_ERR_HIP, "hipGetSymbolAddress gave a null address");
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return ok();
}

}  // namespace

extern "C" int kvc_batch_decode_run_noalloc(
    const kvc_decode_schedule* sched, const int32_t* plan, const void* q,
    int64_t q_batch_stride, const void* key_cache, const void* value_cache,
    int64_t cache_block_stride, int64_t cache_token_stride, int64_t num_blocks,
    const int32_t* indptr, const int32_t* indices, int64_t num_indices,
    const int32_t* last_page_len, float sm_scale, void* out, int64_t out_batch_stride,
    float* lse, void* stream) {
  KVC_REQUIRE(sched, KVC_ERR_INVALID_ARG, "null schedule");
  if (sched->batch == 0) return ok();
  const int64_t need =
      kvc_decode_workspace_bytes(sched->batch, sched->num_qo_heads, sched->head_dim,
                                 sched->max_partitions);
  KVC_REQUIRE(need <= KVC_NOALLOC_SCRATCH_BYTES, KVC_ERR_WORKSPACE,
              "the batch needs " + std::to_string(need) +
                  " bytes of split-K partials; the allocation-free run holds at most " +
                  std::to_string(int64_t(KVC_NOALLOC_SCRATCH_BYTES)) +
                  " (use kvc_batch_decode_run with a workspace)");
  int device = -1;
  KVC_HIP_CHECK(hipGetDevice(&device));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (s) {
    hipDevice_t sdev = -1;
    KVC_HIP_CHECK(hipStreamGetDevice(s, &sdev));
    KVC_REQUIRE(int(sdev) == device, KVC_ERR_INVALID_ARG,
                "the stream belongs to device " + std::to_string(int(sdev)) +
                    ", the current device is " + std::to_string(device));
  }
  void* ws = nullptr;
  const int st = scratch_address(device, &ws);
  if (st != KVC_OK) return st;
  return decode_run(sched, plan, q, q_batch_stride, key_cache, value_cache, cache_block_stride,
                    cache_token_stride, num_blocks, indptr, indices, num_indices, last_page_len,
                    nullptr, 0, nullptr, 0, sm_scale, ws, KVC_NOALLOC_SCRATCH_BYTES, out,
                    out_batch_stride, lse, stream);
}

extern "C" int kvc_batch_decode_append_run(
    const kvc_decode_schedule* sched, const int32_t* plan, const void* q,
    int64_t q_batch_stride, void* key_cache, void* value_cache,
    int64_t cache_block_stride, int64_t cache_token_stride, int64_t num_blocks,
    const int32_t* indptr, const int32_t* indices, int64_t num_indices,
    const int32_t* last_page_len, const void* new_key, int64_t new_key_stride,
    const void* new_value, int64_t new_value_stride, float sm_scale, void* workspace,
    int64_t workspace_bytes, void* out, int64_t out_batch_stride, float* lse,
    void* stream) {
  KVC_REQUIRE(new_key && new_value, KVC_ERR_INVALID_ARG, "null new_key or new_value");
  KVC_REQUIRE(sched, KVC_ERR_INVALID_ARG, "null schedule");
  if (sched->batch > 0) {
    const bool small = sched->small_batch != 0;
    KVC_REQUIRE(sched->num_kv_heads > 0 && sched->head_dim == 128 &&
                    (small || (lds_layout(sched->num_qo_heads / sched->num_kv_heads, 128,
                                          sched->num_kv_heads) &&
                               (sched->heads_per_group != kLdsHeads ||
                                sched->append_pieces <= kNewMax))),
                KVC_ERR_UNSUPPORTED,
                "fused append needs head_dim 128 and either a small-batch schedule or a "
                "multiple of 8 KV heads with group <= 4 and at most " +
                    std::to_string(kNewMax) + " leading pieces per segment holding request "
                    "ends (schedule->append_pieces)");
    KVC_REQUIRE(aligned(new_key, 16) && aligned(new_value, 16) && new_key_stride % 8 == 0 &&
                    new_value_stride % 8 == 0,
                KVC_ERR_ALIGNMENT, "new rows must be 16-byte aligned");
  }
  return decode_run(sched, plan, q, q_batch_stride, key_cache, value_cache, cache_block_stride,
                    cache_token_stride, num_blocks, indptr, indices, num_indices, last_page_len,
                    new_key, new_key_stride, new_value, new_value_stride, sm_scale, workspace,
                    workspace_bytes, out, out_batch_stride, lse, stream);
}

extern "C" int kvc_batch_decode_step_run(
    const kvc_decode_schedule* sched, const int32_t* plan, const void* q,
    int64_t q_batch_stride, void* key_cache, void* value_cache,
    int64_t cache_block_stride, int64_t cache_token_stride, int64_t num_blocks,
    const int32_t* indptr, const int32_t* indices, int64_t num_indices,
    const int32_t* last_page_len, const void* new_key, int64_t new_key_stride,
    const void* new_value, int64_t new_value_stride, float sm_scale, void* workspace,
    int64_t workspace_bytes, void* out, int64_t out_batch_stride, float* lse,
    void* stream) {
  KVC_REQUIRE(new_key && new_value, KVC_ERR_INVALID_ARG, "null new_key or new_value");
  return decode_run(sched, plan, q, q_batch_stride, key_cache, value_cache, cache_block_stride,
                    cache_token_stride, num_blocks, indptr, indices, num_indices, last_page_len,
                    new_key, new_key_stride, new_value, new_value_stride, sm_scale, workspace,
                    workspace_bytes, out, out_batch_stride, lse, stream);
}

extern "C" int kvc_merge_attention_states(const void* out1, const float* lse1,
                                          const void* out2, const float* lse2,
                                          int64_t n, int32_t head_dim, void* out,
                                          float* lse, void* stream) {
  KVC_REQUIRE(n >= 0 && head_dim > 0, KVC_ERR_INVALID_ARG, "bad shape");
  if (n == 0) return ok();
  KVC_REQUIRE(out1 && lse1 && out2 && lse2 && out, KVC_ERR_INVALID_ARG, "null pointer");
  KVC_REQUIRE(lse != lse1 && lse != lse2, KVC_ERR_INVALID_ARG,
              "lse must not alias lse1 or lse2");
  const int64_t total = n * head_dim;
  const int64_t grid = std::min<int64_t>((total + 255) / 256, 1 << 16);
  merge_states_kernel<<<dim3(unsigned(grid)), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(out1), lse1, static_cast<const uint16_t*>(out2), lse2,
      n, head_dim, static_cast<uint16_t*>(out), lse);
  KVC_LAUNCH_CHECK();
  return ok();
}
