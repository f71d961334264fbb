// Kernel argument blocks and launcher declarations shared by the kernel
// translation units and the C-ABI front end (cra_api.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace cra {

// Documents of one launch: sequences packed along S (varlen), or the single
// sequence of a plain call. Each document has its own window, relay switch
// and packed global rows; nothing is attended across documents. A kernel's
// work items are numbered document by document: item0[d] is the first item
// of document d and item0[n] the total.
constexpr int kMaxDocs = 64;

// Division of a 32-bit unsigned by a launch constant (Granlund and Montgomery,
// "Division by Invariant Integers using Multiplication", 1994): a multiply, a
// subtraction and two shifts where the compiler's 32-bit division is about
// forty instructions.
struct FastDiv {
  uint32_t m, sh;  // multiplier; the two shifts, the second in bits 8..
};
inline FastDiv fast_div(uint32_t d) {
  int l = 0;
  while (l < 32 && (uint64_t(1) << l) < d) ++l;
  const uint64_t m = ((((uint64_t(1) << l) - d) << 32) / d) + 1;
  return FastDiv{(uint32_t)m, (uint32_t)((l > 0 ? 1 : 0) | (l > 1 ? l - 1 : 0) << 8)};
}
__host__ __device__ inline uint32_t div_by(uint32_t n, FastDiv f) {
  const uint32_t t = (uint32_t)(((uint64_t)f.m * n) >> 32);
  return (t + ((n - t) >> (f.sh & 0xff))) >> (f.sh >> 8);
}

template <int N>
struct DocsT {
  int n;
  int off[N];   // first row along S
  int len[N];   // rows
  int W[N];     // window = block size
  FastDiv dW[N];
  int rpb[N];   // packed global rows per block: 1 + top_k with relay, else 1
  FastDiv drpb[N];
  int gofs[N];  // first packed global row
  int bofs[N];  // first block (relay_src rows)
  int pofs[N];  // backward: first row of the global-row partials, per (b, kv head)
  int item0[N + 1];
};
using Docs = DocsT<kMaxDocs>;

// One document, resolved for a work item.
struct Doc {
  int off, len, W, rpb, gofs, bofs, pofs;
  FastDiv dW, drpb;
  int item;  // work item index within the document
};

// A launch of one document (every plain call) takes a table of one: a tenth
// of the kernel arguments, and no lookup on the way to the first load. With
// the divisions above, each kernel of a short call is 0.5-1 us shorter (H=12
// S=1000 D=64: forward 8.9 -> 8.4 us, dQ 10.4 -> 9.7; H=8 S=8192 forward 17.5
// -> 17.0, global-row build 7.5 -> 6.5; B=2 H=32 S=4096 D=128 forward 77.5 ->
// 72 us).
template <int N>
__device__ __forceinline__ Doc find_doc(const DocsT<N>& t, int item) {
  int d = 0;
  if constexpr (N > 1) {
    // the last d with item0[d] <= item (item0 is non-decreasing): a search
    // of log2(n) dependent loads, not a scan of n
    int hi = t.n - 1;
    while (d < hi) {
      const int mid = (d + hi + 1) >> 1;
      if (item >= t.item0[mid]) d = mid; else hi = mid - 1;
    }
  }
  return Doc{t.off[d],  t.len[d],  t.W[d],  t.rpb[d],  t.gofs[d],
             t.bofs[d], t.pofs[d], t.dW[d], t.drpb[d], item - (N > 1 ? t.item0[d] : 0)};
}

// XCD-aware work order for launches of nbh heads x nt tiles (one document)
// when nbh is not a multiple of 8. The dispatcher sends block i to XCD i % 8;
// the plain order (item = rank * nbh + head, rank 0 the heaviest tile) then
// spreads a head's neighbouring tiles over several XCDs, whose L2s do not
// share the K/V (or Q/dO) rows those tiles overlap on. Here a head's tiles
// pair up as units {rank p, rank nt - 1 - p} (a heavy and a light tile: every
// unit costs about the same), units are numbered head by head (u = head * P +
// p), and XCD x takes a contiguous eighth of them, so it holds about nbh / 8
// heads with an equal share of the work. Its blocks take its tiles in the
// plain order's sequence (by rank, then head): heaviest first, as there.
// xcd_item returns the plain order's item index, or -1 for a padding block.
struct XcdChunk {
  int P, Pl;    // units per head; units with a light tile (the middle tile of
                // an odd nt is its unit's only tile)
  int q0, r0;   // first unit of this XCD: head q0, p = r0
  int q1, r1;   // one past its last unit
};

__host__ __device__ inline XcdChunk xcd_chunk(int x, int nbh, int nt) {
  const int P = (nt + 1) >> 1, U = nbh * P;
  const int base = U >> 3, extra = U & 7;
  const int u0 = x * base + (x < extra ? x : extra);
  const int u1 = u0 + base + (x < extra ? 1 : 0);
  return XcdChunk{P, nt >> 1, u0 / P, u0 % P, u1 / P, u1 % P};
}

// units of the chunk with p in [a, b)
__host__ __device__ inline int xcd_units(const XcdChunk& c, int a, int b) {
  if (a >= b) return 0;
  const int e1 = c.r1 < a ? a : c.r1 > b ? b : c.r1;
  const int e0 = c.r0 < a ? a : c.r0 > b ? b : c.r0;
  return (c.q1 - c.q0) * (b - a) + e1 - e0;
}

// tiles of the chunk with rank < r
__host__ __device__ inline int xcd_before(const XcdChunk& c, int nt, int r) {
  const int heavy = xcd_units(c, 0, r < c.P ? r : c.P);
  const int a = nt - r > 0 ? nt - r : 0;
  return heavy + xcd_units(c, a < c.Pl ? a : c.Pl, c.Pl);
}

__host__ __device__ inline int xcd_grid(int nbh, int nt) {
  int most = 0;
  for (int x = 0; x < 8; ++x) {
    const XcdChunk c = xcd_chunk(x, nbh, nt);
    const int n = xcd_before(c, nt, nt);
    most = n > most ? n : most;
  }
  return 8 * most;
}

__host__ __device__ inline int xcd_item(int block, int nbh, int nt) {
  const XcdChunk c = xcd_chunk(block & 7, nbh, nt);
  const int k = block >> 3;
  if (k >= xcd_before(c, nt, nt)) return -1;  // padding block
  // the rank r with xcd_before(r) <= k < xcd_before(r + 1)
  int lo = 0, hi = nt - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (xcd_before(c, nt, mid) <= k) lo = mid; else hi = mid - 1;
  }
  const int r = lo;
  const int p = r < c.P ? r : nt - 1 - r;
  // heads whose unit p lies in the chunk form a run from head q0 (q0 + 1
  // when unit (q0, p) precedes the chunk); take the j-th
  return r * nbh + c.q0 + (p < c.r0 ? 1 : 0) + (k - xcd_before(c, nt, r));
}

struct GlobalCommon {
  const void* k;
  const void* v;
  int64_t ksb, ksh, kss, vsb, vsh, vss;
  void* gk;
  void* gv;
  int32_t* src;        // [B, H_kv, NB, top_k], doc-relative rows
  const float* scale;
  int Hkv, top_k;
  int NB;              // blocks of all documents (rows of relay_src per head)
  int64_t G;           // packed global rows of all documents, per head
};
template <int N>
struct GlobalArgsT : GlobalCommon {
  using Common = GlobalCommon;
  static constexpr int kDocs = N;
  DocsT<N> docs;  // items: W-blocks
};
using GlobalArgs = GlobalArgsT<kMaxDocs>;

struct FwdCommon {
  const void* q;
  const void* k;
  const void* v;
  const void* gk;
  const void* gv;
  void* o;
  float* lse;
  int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss, osb, osh, oss;
  int B, Hq, Hkv;
  int direct;  // one document without relay: the global rows are read from k and v
  FastDiv d_bhq, d_hq, d_bhkv, d_hkv, d_grp;  // by B * Hq, Hq, B * Hkv, Hkv, Hq / Hkv
  int S;       // rows along S of all documents (row stride of lse)
  int64_t G;   // packed global rows of all documents, per head
  float scale;
  int phases;  // bit 0: local window, bit 1: global rows
  int* work_counter;  // persistent launch: zeroed item counter, else null
  int xcd_nt;  // > 0: XCD-aware order (xcd_item) over this many tiles per head
};
template <int N>
struct FwdArgsT : FwdCommon {
  using Common = FwdCommon;
  static constexpr int kDocs = N;
  DocsT<N> docs;  // items: query tiles (set by the launcher for its tile size)
};
using FwdArgs = FwdArgsT<kMaxDocs>;

struct BwdCommon {
  const void* q;
  const void* k;
  const void* v;
  const void* o;
  const void* dout;
  const float* lse;
  const void* gk;
  const void* gv;
  const int32_t* src;
  const float* rscale;
  void* dq;
  void* dk;
  void* dv;
  float* delta;    // [B, Hq, S] -rowsum(o * do)
  float* nlse2;    // [B, Hq, S] -lse * log2(e)
  float* gpart;    // fp32 partial dK/dV of the global rows (part_row)
  float* dalpha;   // [Hkv] or null
  int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss, osb, osh, oss;
  int64_t dosb, dosh, doss, dqsb, dqsh, dqss, dksb, dksh, dkss, dvsb, dvsh, dvss;
  int B, Hq, Hkv, top_k;
  int direct;  // one document without relay: the global rows are read from k and v
  FastDiv d_bhq, d_hq, d_bhkv, d_hkv, d_grp;  // by B * Hq, Hq, B * Hkv, Hkv, Hq / Hkv
  int S;           // rows along S of all documents (row stride of lse, delta)
  int NB;          // blocks of all documents (rows of relay_src per head)
  int64_t G;       // packed global rows of all documents, per head
  float scale;
  int cus;         // compute units of the device (launch rules)
  int chunk_len;   // most queries per chunk of the global-row kernel
  int nchunk;      // most query chunks of a document
  int even;        // packed documents that fill the chip evenly uncut (ChunkPlan)
  int group;       // 0: first launch of a call (writes dalpha);
                   // later document groups of the call add to dalpha
  int xcd_nt;      // > 0: XCD-aware order (xcd_item) over this many tiles per head
};
template <int N>
struct BwdArgsT : BwdCommon {
  using Common = BwdCommon;
  static constexpr int kDocs = N;
  DocsT<N> docs;  // items: set by the launcher per kernel
};
using BwdArgs = BwdArgsT<kMaxDocs>;

// Calls launch(args) with the arguments over a table of one document if there
// is one, else with the table as it is.
template <template <int> class A, typename F>
inline void by_docs(const A<kMaxDocs>& a, F launch) {
  if (a.docs.n != 1) {
    launch(a);
    return;
  }
  A<1> o;
  using Common = typename A<1>::Common;
  static_cast<Common&>(o) = a;
  const Docs& t = a.docs;
  o.docs = DocsT<1>{1,           {t.off[0]},    {t.len[0]},  {t.W[0]},    {t.dW[0]}, {t.rpb[0]},
                    {t.drpb[0]}, {t.gofs[0]},   {t.bofs[0]}, {t.pofs[0]}, {t.item0[0], t.item0[1]}};
  launch(o);
}

// Calls f(std::bool_constant): the direct form exists for one document only.
template <int ND, typename F>
inline void dispatch_direct(bool direct, F f) {
  if constexpr (ND == 1) {
    if (direct) {
      f(std::true_type{});
      return;
    }
  }
  f(std::false_type{});
}

template <typename A>
inline void set_divs(A& a) {
  a.d_bhq = fast_div(a.B * a.Hq);
  a.d_hq = fast_div(a.Hq);
  a.d_bhkv = fast_div(a.B * a.Hkv);
  a.d_hkv = fast_div(a.Hkv);
  a.d_grp = fast_div(a.Hq / a.Hkv);
}

// (batch, head) of a work item, items numbered heads first.
struct QHead {
  int rest, bh, b, h, hk;
};
template <typename A>
__device__ __forceinline__ QHead q_head(const A& a, int item) {
  const int rest = div_by(item, a.d_bhq), bh = item - rest * (a.B * a.Hq);
  const int b = div_by(bh, a.d_hq), h = bh - b * a.Hq;
  return QHead{rest, bh, b, h, (int)div_by(h, a.d_grp)};
}
struct KvHead {
  int rest, bhk, b, hk;
};
template <typename A>
__device__ __forceinline__ KvHead kv_head(const A& a, int item) {
  const int rest = div_by(item, a.d_bhkv), bhk = item - rest * (a.B * a.Hkv);
  const int b = div_by(bhk, a.d_hkv);
  return KvHead{rest, bhk, b, bhk - b * a.Hkv};
}

// Global rows of a document for a kernel: the packed rows, or with DIRECT (a
// document without relay, k and v of one row stride) row r is row r * W of k
// and v, read in place. The tiled forward and dQ kernels take it at compile
// time: with one row stride for k and v the direct form needs no more
// registers than the packed one, with two it needs four more (dQ at D = 64
// then drops from 3 to 2 waves per SIMD). GPU time of a call, packed / direct:
// H=8 S=512 D=64 forward 11.0 / 8.2 us; H=12 S=1000 D=64 step 41 / 38 us; B=8
// H=32 S=1000 D=64 forward 35 / 27.6 us, S=2048 step 301 / 290 us.
struct GlobRows {
  const char *k, *v;     // row 0
  int64_t kstep, vstep;  // bytes from row to row
};
template <typename T, int D, typename A>
__device__ __forceinline__ GlobRows glob_rows(const A& a, const Doc& dc, int b, int hk,
                                              const void* kp, const void* vp, bool direct) {
  if (direct)
    return GlobRows{(const char*)kp, (const char*)vp, dc.W * a.kss * (int64_t)sizeof(T),
                    dc.W * a.kss * (int64_t)sizeof(T)};
  const int64_t off = (((int64_t)(b * a.Hkv + hk) * a.G + dc.gofs) * D) * (int64_t)sizeof(T);
  return GlobRows{(const char*)a.gk + off, (const char*)a.gv + off, D * (int64_t)sizeof(T),
                  D * (int64_t)sizeof(T)};
}

// Number the work items document by document: count(d) items for document d.
template <typename F>
inline void set_items(Docs& t, F count) {
  int s = 0;
  for (int d = 0; d < t.n; ++d) {
    t.item0[d] = s;
    s += count(d);
  }
  t.item0[t.n] = s;
}

// Queries per chunk of document length len split nchunk ways (multiple of 64).
__host__ __device__ inline int chunk_len_for(int len, int nchunk) {
  const int c = (len + nchunk - 1) / nchunk;
  return (c + 63) / 64 * 64;
}

// Query chunks of a document of length len.
__host__ __device__ inline int num_chunks(int len, int chunk_len) {
  return (len + chunk_len - 1) / chunk_len;
}

// Queries per chunk of a document cut into `nck`: packed documents (ND > 1)
// are cut evenly, so that a document a little longer than chunk_len does not
// end in a short piece; one document's chunk_len is even already.
template <int ND>
__device__ __forceinline__ int doc_chunk_len(int len, int nck, int chunk_len) {
  return ND > 1 ? chunk_len_for(len, nck) : chunk_len;
}

// Packed global rows of a document.
__host__ __device__ inline int doc_rows(int len, int W, int rpb) { return (len + W - 1) / W * rpb; }

// sqrt(N) geometry (reference core.py:957, 1038-1061, 1112-1117): length of the
// global-row prefix query i attends to. With relay each W-block contributes
// rpb = 1 + top_k rows (strided row first); without, rpb = 1.
__device__ __forceinline__ int glob_prefix(int i, const Doc& dc) {
  const int a = i - dc.W + 1 > 0 ? i - dc.W + 1 : 0;
  const int f = div_by(a, dc.dW);
  return dc.rpb * f + ((a - f * dc.W) != 0 ? 1 : 0);
}

// First query that sees packed global row gr (inverse of glob_prefix).
__device__ __forceinline__ int glob_row_first_query(int gr, const Doc& dc) {
  const int r = div_by(gr, dc.drpb);
  return (gr - r * dc.rpb) == 0 ? r * dc.W + dc.W : (r + 1) * dc.W + dc.W - 1;
}

// Partial dK/dV of global row `row` of a document from query chunk `chunk`:
// row index into gpart ([2, D] each). A document's partials are
// [chunks, B * Hkv, rows], behind those of the documents before it.
__device__ __forceinline__ int64_t part_row(const Doc& dc, int chunk, int nbh, int bhk, int row) {
  const int rows = doc_rows(dc.len, dc.W, dc.rpb);
  return (int64_t)dc.pofs * nbh + ((int64_t)chunk * nbh + bhk) * rows + row;
}

// Compiled tile geometry (dtype 0 f16, 1 bf16, 2 f32; D 32/64/128): the forward's
// {waves, queries, key rows per tile} and the backward's {waves, rows, tile} of
// dQ, global-row dK/dV and local dK/dV. Returns false for an unbuilt (dtype, D).
bool fwd_tile_config(int dtype, int D, int out[3]);
bool bwd_tile_config(int dtype, int D, int out[9]);

// dtype: 0 f16, 1 bf16, 2 f32. Each returns hipError_t of the launch.
hipError_t launch_build_global(int dtype, int D, const GlobalArgs& a, int B, hipStream_t st);
hipError_t launch_fwd(int dtype, int D, const FwdArgs& a, hipStream_t st);
hipError_t launch_bwd(int dtype, int D, const BwdArgs& a, hipStream_t st);
// Query chunks of the global-row kernel and its fp32 partials for n documents
// of lengths len[], windows W[] and packed rows per block rpb[] on a device
// with `cus` compute units.
struct ChunkPlan {
  int chunk_len;      // most queries per chunk (multiple of 64)
  int nchunk;         // most chunks of a document
  bool even;          // packed documents that fill the chip evenly uncut
  int64_t part_rows;  // partial rows per (b, kv head), all documents
};
ChunkPlan plan_chunks(int D, int B, int Hq, int Hkv, int n, const int* len, const int* W,
                      const int* rpb, int cus);
// Workspace of the backward: Delta and -lse*log2(e), [B*Hq*S] fp32 each
// (rounded up to 256 bytes), then the partials, part_rows * B * Hkv rows of
// [2, D] fp32.
size_t bwd_workspace_layout(int D, int B, int Hq, int Hkv, int S, int64_t part_rows);

}  // namespace cra
