// Backward of the three-phase sqrt(N) attention.
//
// Reference: `CronRootAttentionV14Function.backward` (core.py:3626-3759) runs
// dQ (core.py:1165-1316), local dK/dV (core.py:1650-1745), strided dK/dV with
// fp16 atomics (core.py:1755-1889), relay dK/dV (core.py:2381-2492) and a
// read-add-store scatter of the relay gradients onto their source rows
// (core.py:2767-2815). Math per pair (i, j): P = exp(s - LSE_i),
// dP = dO_i . v_j, dS = P (dP - Delta_i), Delta_i = O_i . dO_i;
// dQ_i += scale dS k_j, dK_j += scale dS q_i, dV_j += P dO_i.
//
// This build keeps every accumulation in fp32 and rounds once:
//   1. dq2_kernel        query-centric: local band + global prefix -> dQ; it
//      (dq_wide, dq_f32) also forms Delta = rowsum(O * dO) of its queries and
//                        stores -Delta and -lse * log2(e) for the dK/dV kernels
//   2. dkdv2_kernel<GLOB> packed global rows (strided + relay), query range
//      (dkdv_f32)        split in chunks -> fp32 partials in the workspace
//   3. gsum_kernel       sums the chunk partials of each global row
//   4. dalpha_kernel     (optional) gradient of the relay log-scale
//   5. dkdv2_kernel<LOC> key-centric local band; its epilogue adds the
//                        summed partials of the global rows whose source is
//                        the key row (strided row r*W, relay source rows) and
//                        writes dK/dV once.
// No atomics: every output row has exactly one writer and the partial sums
// are reduced in a fixed order, so two runs give identical bits.
#include <algorithm>
#include <type_traits>

#include "cra_common.hpp"
#include "cra_internal.hpp"

namespace cra {

namespace {

template <typename T>
__device__ __forceinline__ void zero_frag(Frag<T>& f) {
#pragma unroll
  for (int w = 0; w < Frag<T>::kWords; ++w) f.w[w] = make_uint4(0, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ void store4(T* p, const f32x4& v, float mul) {
  T e[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) e[r] = from_f32<T>(v[r] * mul);
  if constexpr (sizeof(T) == 2)
    *reinterpret_cast<uint2*>(p) = *reinterpret_cast<const uint2*>(e);
  else
    *reinterpret_cast<uint4*>(p) = *reinterpret_cast<const uint4*>(e);
}

// ---------------------------------------------------------------------------
// 3. Chunk partials of the global rows summed into chunk 0, in chunk order
// (one float4 per thread; work items: the documents' rows x 2D / 4 / 256).
// Only chunks with a query that sees the row are read.
// ---------------------------------------------------------------------------
// kGsumU partials' loads are in flight together (past the last chunk that
// chunk is read again and left out): one at a time, the sum is a chain of
// memory latencies
constexpr int kGsumU = 8;
template <int D, int ND>
__global__ __launch_bounds__(256) void gsum_kernel(BwdArgsT<ND> a) {
  constexpr int kVec = 2 * D / 4;  // float4 per row (dK and dV)
  const int nbh = a.B * a.Hkv;
  const KvHead hd = kv_head(a, blockIdx.x);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bhk = hd.bhk;
  const int rows = doc_rows(dc.len, dc.W, dc.rpb);
  const int e = dc.item * 256 + (int)threadIdx.x;
  if (e >= rows * kVec) return;
  // Chunks [c_lo, c_hi) hold queries that see the row; the global-row
  // kernel wrote no partial for the others (their workgroups had no query
  // that sees the tile), so they are skipped rather than read.
  const int first = glob_row_first_query(e / kVec, dc);
  const int nck = num_chunks(dc.len, a.chunk_len);
  const int c_lo = first / doc_chunk_len<ND>(dc.len, nck, a.chunk_len);
  const int c_hi = first < dc.len ? nck : c_lo;
  float* p0 = a.gpart + part_row(dc, 0, nbh, bhk, 0) * 2 * D + 4 * (int64_t)e;
  const int64_t cstride = (int64_t)nbh * rows * 2 * D;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c = c_lo; c < c_hi; c += kGsumU) {
    f32x4 x[kGsumU];
#pragma unroll
    for (int u = 0; u < kGsumU; ++u)
      x[u] = *reinterpret_cast<const f32x4*>(p0 + min(c + u, c_hi - 1) * cstride);
#pragma unroll
    for (int u = 0; u < kGsumU; ++u)
      if (c + u < c_hi) acc += x[u];
  }
  *reinterpret_cast<f32x4*>(p0) = acc;
}

// ---------------------------------------------------------------------------
// 4. d(relay_log_scale)[hk] = sum over b and relay rows of dRK.RK + dRV.RV
// (reference core.py:3363-3366), one workgroup per kv head, fixed order.
// ---------------------------------------------------------------------------
// 1024 threads with four elements each per step, four rows' loads in flight:
// the sum is latency-bound (one element per thread and step of a 256-thread
// workgroup took 66 us at B=1 H_kv=4 S=8191 D=256, this one 9.8 us).
template <typename T, int D>
__global__ __launch_bounds__(1024) void dalpha_kernel(BwdArgs a) {
  constexpr int kVec = D / 4;  // four-element groups per row
  const int hk = blockIdx.x;
  const int tid = threadIdx.x;
  const int nbh = a.B * a.Hkv;
  float acc = 0.f;
  for (int b = 0; b < a.B; ++b) {
    const int bhk = b * a.Hkv + hk;
    const T* gk = static_cast<const T*>(a.gk) + (int64_t)bhk * a.G * D;
    const T* gv = static_cast<const T*>(a.gv) + (int64_t)bhk * a.G * D;
    for (int doc = 0; doc < a.docs.n; ++doc) {
      const int rpb = a.docs.rpb[doc];
      if (rpb == 1) continue;  // no relay rows in this document
      const int rows = doc_rows(a.docs.len[doc], a.docs.W[doc], rpb);
      const int nrel = rows / rpb * a.top_k;
      const int64_t part = (int64_t)a.docs.pofs[doc] * nbh + (int64_t)bhk * rows;  // summed chunks
      const int64_t gofs = a.docs.gofs[doc];
#pragma unroll 4
      for (int e = tid; e < nrel * kVec; e += 1024) {
        const int t = e / kVec, d = e % kVec * 4;
        const int row = (t / a.top_k) * rpb + 1 + t % a.top_k;
        const float* pk = a.gpart + (part + row) * 2 * D + d;
        const f32x4 dk = *reinterpret_cast<const f32x4*>(pk);
        const f32x4 dv = *reinterpret_cast<const f32x4*>(pk + D);
        T ek[4], ev[4];
        __builtin_memcpy(ek, gk + (gofs + row) * D + d, sizeof(ek));
        __builtin_memcpy(ev, gv + (gofs + row) * D + d, sizeof(ev));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc += dk[i] * to_f32(ek[i]) + dv[i] * to_f32(ev[i]);
      }
    }
  }
  __shared__ float red[1024];
  red[tid] = acc;
  __syncthreads();
  for (int off = 512; off >= 1; off >>= 1) {
    if (tid < off) red[tid] += red[tid + off];
    __syncthreads();
  }
  if (tid == 0) a.dalpha[hk] = (a.group ? a.dalpha[hk] : 0.f) + red[0];
}

// ---------------------------------------------------------------------------
// fp16/bf16 backward kernels on the gfx950 tile machinery (see SwzTile):
// K/V (dq2) or Q/dO (dkdv2) tiles of 64 rows double-buffered in swizzled LDS,
// filled by buffer loads straight into LDS while the previous tile is
// computed; transposed operands (K^T for dQ, Q^T and dO^T for dK/dV) are
// read with ds_read_b64_tr_b16 from the same row-major tiles.
// ---------------------------------------------------------------------------
// At D = 256 Delta is subtracted from the finished dP, one rounding of the
// difference: accumulating onto -Delta (below D = 256, one operation less per
// element) rounds every partial sum at Delta's magnitude, over twice the
// products.
template <int D>
constexpr bool kSubDelta = D > 128;

// Query-centric dQ for QB blocks of 16 queries per wave against one BN-key
// tile, in 32-key halves: S = K . Q^T and dP - Delta = V . dO^T - Delta (key
// on rows; the products accumulate onto -Delta, so no subtraction per
// element), dS = P * (dP - Delta), dQ^T += K^T . dS^T.
//
// dq2_ds: dS of 32-key half kc.
template <typename T, int D, int QB, int BN, bool MASK>
__device__ __forceinline__ void dq2_ds(const char* tK, const char* tV, int kc,
                                       const LaneOffs<D>& lo, const Frag<T> (&qf)[QB][D / 32],
                                       const Frag<T> (&df)[QB][D / 32], const float (&lse2)[QB],
                                       const float (&ndl)[QB], float c2, int g,
                                       const TileMask<QB>& mk, Frag<T> (&dsf)[QB]) {
  using Tile = SwzTile<D, BN>;
  constexpr int NC = D / 32;
  float ds[2][QB][4];  // [h][qb][r]
  // K and V row fragments are read two steps ahead of their MFMAs; fences
  // keep the compiler from moving the reads next to their uses
  constexpr int NT = 2 * NC;
  auto row_kv = [&](int t, Frag<T>& k_, Frag<T>& v_) {
    const int kn = 2 * kc + t / NC, cn = t % NC;
    k_ = Tile::template row_frag_at<T>(tK + kn * Tile::kBlk16 + lo.row_at(cn));
    v_ = Tile::template row_frag_at<T>(tV + kn * Tile::kBlk16 + lo.row_at(cn));
  };
  Frag<T> kf[3], vf[3];
  row_kv(0, kf[0], vf[0]);
  row_kv(1, kf[1], vf[1]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f32x4 sc[QB], dp[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      sc[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      const float d0 = kSubDelta<D> ? 0.f : ndl[qb];
      dp[qb] = f32x4{d0, d0, d0, d0};
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int t = h * NC + c;
      if (t + 2 < NT) row_kv(t + 2, kf[(t + 2) % 3], vf[(t + 2) % 3]);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        sc[qb] = mma(sc[qb], kf[t % 3], qf[qb][c]);
        dp[qb] = mma(dp[qb], vf[t % 3], df[qb][c]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int kb = 2 * kc + h;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ko = 16 * kb + 4 * g + r;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        float x = fmaf(sc[qb][r], c2, -lse2[qb]);
        if (MASK && !mk.ok(ko, qb)) x = -__builtin_huge_valf();
        ds[h][qb][r] =
            __builtin_amdgcn_exp2f(x) * (kSubDelta<D> ? dp[qb][r] + ndl[qb] : dp[qb][r]);
      }
    }
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float v8[8] = {ds[0][qb][0], ds[0][qb][1], ds[0][qb][2], ds[0][qb][3],
                         ds[1][qb][0], ds[1][qb][1], ds[1][qb][2], ds[1][qb][3]};
    dsf[qb] = pack8<T>(v8);
  }
}

// dQ^T += K^T . dS^T of 32-key half kc; transposed K fragments two steps ahead.
template <typename T, int D, int QB, int BN>
__device__ __forceinline__ void dq2_acc(const char* tK, int kc, const LaneOffs<D>& lo,
                                        const Frag<T> (&dsf)[QB], f32x4 (&dqa)[D / 16][QB]) {
  using Tile = SwzTile<D, BN>;
  Frag<T> kt[3];
  auto tr_k = [&](int db) {
    const char* pa = tK + (2 * kc) * Tile::kBlk16 + lo.tr_at(db);
    return Tile::template tr_frag_at<T>(pa, pa + Tile::kBlk16);
  };
  kt[0] = tr_k(0);
  kt[1] = tr_k(1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int db = 0; db < D / 16; ++db) {
    if (db + 2 < D / 16) kt[(db + 2) % 3] = tr_k(db + 2);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) dqa[db][qb] = mma(dqa[db][qb], kt[db % 3], dsf[qb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, int D, int QB, int BN, bool MASK>
__device__ __forceinline__ void dq2_tile(const char* tK, const char* tV, const LaneOffs<D>& lo,
                                         const Frag<T> (&qf)[QB][D / 32],
                                         const Frag<T> (&df)[QB][D / 32],
                                         f32x4 (&dqa)[D / 16][QB], const float (&lse2)[QB],
                                         const float (&ndl)[QB], float c2, int g,
                                         const TileMask<QB>& mk, bool half0, bool half1) {
#pragma unroll
  for (int kc = 0; kc < BN / 32; ++kc) {
    // masked tiles: a 32-key half with no key visible to the wave is skipped
    if (MASK && !(kc ? half1 : half0)) continue;
    Frag<T> dsf[QB];
    dq2_ds<T, D, QB, BN, MASK>(tK, tV, kc, lo, qf, df, lse2, ndl, c2, g, mk, dsf);
    dq2_acc<T, D, QB, BN>(tK, kc, lo, dsf, dqa);
  }
}

// NW waves of QB blocks of 16 queries each cover the workgroup's
// 16 * NW * QB queries; key tiles of BN rows; at least WPE waves per SIMD.
template <typename T, int D, int NW, int QB, int BN, int WPE, int ND, bool DIR = false>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE)))
void dq2_kernel(BwdArgsT<ND> a) {
  using Tile = SwzTile<D, BN>;
  constexpr int kQW = 16 * QB, kBM = NW * kQW, kBN = BN;
  // Two pipeline stages as separate LDS objects (see fwd2_kernel).
  __shared__ __attribute__((aligned(1024))) char stage0[2][Tile::kBytes];  // K, V
  __shared__ __attribute__((aligned(1024))) char stage1[2][Tile::kBytes];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int nbh = a.B * a.Hq;
  int item = (int)blockIdx.x;
  if (a.xcd_nt > 0) {
    item = xcd_item(item, nbh, a.xcd_nt);
    if (item < 0) return;  // padding block
  }
  const QHead hd = q_head(a, item);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bh = hd.bh, b = hd.b, h = hd.h, hk = hd.hk;
  const int tile = (dc.len + kBM - 1) / kBM - 1 - dc.item;  // heaviest first
  const int m0 = tile * kBM;
  const int q0 = m0 + wave * kQW;
  const int S = dc.len, W = dc.W;

  const T* qp = static_cast<const T*>(a.q) + b * a.qsb + h * a.qsh + (int64_t)dc.off * a.qss;
  const T* dop =
      static_cast<const T*>(a.dout) + b * a.dosb + h * a.dosh + (int64_t)dc.off * a.doss;
  const T* kp = static_cast<const T*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const T* vp = static_cast<const T*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  const float* lse = a.lse + (int64_t)bh * a.S + dc.off;
  float* delta = a.delta + (int64_t)bh * a.S + dc.off;
  float* nlse2 = a.nlse2 + (int64_t)bh * a.S + dc.off;
  const GlobRows gr = glob_rows<T, D>(a, dc, b, hk, kp, vp, DIR);

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (hi - lo_k + kBN - 1) / kBN;
  // global tiles first: their first fill is an L2 hit; then the local
  // window from its highest key tile down, in step with the neighbouring
  // query tile's workgroup (see fwd2_kernel; 7% fewer HBM reads)
  const int nglob = (gmax + kBN - 1) / kBN;
  const int ntot = nloc + nglob;
  // Buffer resources over the rows this workgroup may read (local rows below
  // hi, global rows below gmax): loads past them return zeros.
  using Fill = typename Tile::template Fill<NW>;
  const int kbytes = (int)(a.kss * 2), vbytes = DIR ? kbytes : (int)(a.vss * 2);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(kp, (uint32_t)((hi - 1) * kbytes + D * 2));
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(vp, (uint32_t)((hi - 1) * vbytes + D * 2));
  const int gkb = (int)gr.kstep, gvb = (int)gr.vstep;
  const __amdgpu_buffer_rsrc_t rgk = make_rsrc(gr.k, gmax > 0 ? (uint32_t)((gmax - 1) * gkb + D * 2) : 0);
  const __amdgpu_buffer_rsrc_t rgv = make_rsrc(gr.v, gmax > 0 ? (uint32_t)((gmax - 1) * gvb + D * 2) : 0);
  const int fk = Fill::lane_off(wave, lane, kbytes);
  const int fv = Fill::lane_off(wave, lane, vbytes);
  const int fgk = Fill::lane_off(wave, lane, gkb), fgv = Fill::lane_off(wave, lane, gvb);
  auto issue = [&](int it, char* dst) {
    if (it >= nglob) {
      const int ts = lo_k + (nloc - 1 - (it - nglob)) * kBN;
      Fill::load(dst, rk, fk, kbytes, ts, wave);
      Fill::load(dst + Tile::kBytes, rv, fv, vbytes, ts, wave);
    } else {
      const int ts = it * kBN;
      Fill::load(dst, rgk, fgk, gkb, ts, wave);
      Fill::load(dst + Tile::kBytes, rgv, fgv, gvb, ts, wave);
    }
  };
  issue(0, stage0[0]);

  LaneOffs<D> lo;
  lo.init(lane);
  Frag<T> qf[QB][D / 32], df[QB][D / 32];
  int qi[QB];
  float lse2[QB], ndl[QB];
  // Delta = rowsum(O * dO) of this wave's queries, computed here and stored
  // negated (-Delta, the initial value of the dP accumulators) for the dK/dV
  // kernels, with -lse * log2(e) (their exponent's offset): lane (l16, g)
  // sums its 32 columns, then the four lanes of a query add theirs in a
  // fixed order.
  const T* opp = static_cast<const T*>(a.o) + b * a.osb + h * a.osh + (int64_t)dc.off * a.oss;
  // All of the wave's Q, dO and O fragments are loaded before any is used
  // (rows past the document read its last row: those queries' results are
  // never stored), so the loads are in flight together.
  Frag<T> of[QB][D / 32];
  float lv[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    qi[qb] = q0 + 16 * qb + l16;
    const int qr = min(qi[qb], S - 1);
    lv[qb] = lse[qr];
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
      qf[qb][c] = lds_frag_row<T>(qp + (int64_t)qr * a.qss + 32 * c + 8 * g);
      df[qb][c] = lds_frag_row<T>(dop + (int64_t)qr * a.doss + 32 * c + 8 * g);
      of[qb][c] = lds_frag_row<T>(opp + (int64_t)qr * a.oss + 32 * c + 8 * g);
    }
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const bool ok = qi[qb] < S;
    lse2[qb] = ok ? lv[qb] * kLog2e : 0.f;
    float od = 0.f;
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
      const T* eo = reinterpret_cast<const T*>(of[qb][c].w);
      const T* ed = reinterpret_cast<const T*>(df[qb][c].w);
#pragma unroll
      for (int i = 0; i < 8; ++i) od = fmaf(to_f32(eo[i]), to_f32(ed[i]), od);
    }
    od += __shfl_xor(od, 16);
    od += __shfl_xor(od, 32);
    ndl[qb] = -od;
    if (ok && g == 0) {
      delta[qi[qb]] = -od;
      nlse2[qi[qb]] = -lse2[qb];
    }
  }
  const float c2 = a.scale * kLog2e;
  f32x4 dqa[D / 16][QB];
#pragma unroll
  for (int db = 0; db < D / 16; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) dqa[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = q0 < S;
  const int q_last = min(q0 + kQW, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  int glen[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) glen[qb] = glob_prefix(qi[qb], dc);

  // Local and global tiles share one body (parameters chosen per tile); the
  // loop is unrolled over the two stages.
  auto step = [&](auto stage_c, int it) {
    constexpr int kStage = decltype(stage_c)::value;
    char(&cur)[2][Tile::kBytes] = kStage ? stage1 : stage0;
    char(&nxt)[2][Tile::kBytes] = kStage ? stage0 : stage1;
    wait_vmem();
    __syncthreads();
    if (it + 1 < ntot) issue(it + 1, nxt[0]);
    const char* tK = cur[0];
    const char* tV = cur[1];
    const bool loc = it >= nglob;
    const int ts = loc ? lo_k + (nloc - 1 - (it - nglob)) * kBN : it * kBN;
    const bool work = active && (loc ? (ts <= q_last && ts + kBN - 1 >= w_lo) : ts < wg_hi);
    const bool full = loc ? (ts >= q_last - W + 1 && ts + kBN - 1 <= q0) : ts + kBN <= wg_lo;
    TileMask<QB> mk;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      mk.hi[qb] = loc ? qi[qb] - ts : glen[qb] - 1 - ts;
      mk.span[qb] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
    }
    if (work) {
      // keys of the tile visible to some query of the wave: [vis_lo, vis_hi]
      const int vis_lo = loc ? w_lo - ts : 0;
      const int vis_hi = loc ? q_last - ts : wg_hi - 1 - ts;
      const bool half0 = vis_lo <= 31, half1 = vis_hi >= 32;
      if (full)
        dq2_tile<T, D, QB, BN, false>(tK, tV, lo, qf, df, dqa, lse2, ndl, c2, g, mk, true, true);
      else
        dq2_tile<T, D, QB, BN, true>(tK, tV, lo, qf, df, dqa, lse2, ndl, c2, g, mk, half0, half1);
    }
  };
  for (int it = 0; it < ntot; it += 2) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 < ntot) step(std::integral_constant<int, 1>{}, it + 1);
  }

  T* dqp = static_cast<T*>(a.dq) + b * a.dqsb + h * a.dqsh + (int64_t)dc.off * a.dqss;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    if (!active || qi[qb] >= S) continue;
    T* row = dqp + (int64_t)qi[qb] * a.dqss;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) store4<T>(row + 16 * db + 4 * g, dqa[db][qb], a.scale);
  }
}

// Delta of the lane's query from sums of eight products, chunk c of the lane's
// group in x[c]: by pairs, so that the error grows with the logarithm of D.
template <int D>
__device__ __forceinline__ float delta_sum(float (&x)[D / 32]) {
#pragma unroll
  for (int n = D / 64; n >= 1; n /= 2)
#pragma unroll
    for (int c = 0; c < n; ++c) x[c] += x[c + n];
  x[0] += __shfl_xor(x[0], 32);
  return x[0] + __shfl_xor(x[0], 16);
}

// dQ of the 2-byte types at head dim 256: 4 waves of 16 queries (Q, dO and dQ
// take 128 registers of a wave per 16 queries), 32-key tiles. V is staged one
// tile at a time and K two, 48 KB of LDS per workgroup: the next K arrives
// during this tile's S and dP, the next V during its K^T . dS^T. Bound by
// LDS reads (one K, V or K^T fragment per MFMA: at most about 60% MFMA-busy)
// and 2 waves per SIMD (211 VGPRs). B=1 H=8 S=32768 bf16: 340 us; with tiles
// through registers and V and K^T stored transposed by 2-byte LDS writes, one
// stage, it took 479 us and a Delta pass before it 46 us.
constexpr int kWideWaves = 4, kWideBN = 32;
template <typename T, int D, int ND, bool DIR = false>
__global__ __launch_bounds__(64 * kWideWaves) __attribute__((amdgpu_waves_per_eu(2)))
void dq_wide_kernel(BwdArgsT<ND> a) {
  constexpr int NW = kWideWaves, BN = kWideBN, kBM = 16 * NW;
  using Tile = SwzTile<D, BN>;
  __shared__ __attribute__((aligned(1024))) char sK0[Tile::kBytes];
  __shared__ __attribute__((aligned(1024))) char sK1[Tile::kBytes];
  __shared__ __attribute__((aligned(1024))) char sV[Tile::kBytes];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const QHead hd = q_head(a, blockIdx.x);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bh = hd.bh, b = hd.b, h = hd.h, hk = hd.hk;
  const int tile = (dc.len + kBM - 1) / kBM - 1 - dc.item;  // heaviest first
  const int m0 = tile * kBM;
  const int q0 = m0 + wave * 16;
  const int S = dc.len, W = dc.W;

  const T* qp = static_cast<const T*>(a.q) + b * a.qsb + h * a.qsh + (int64_t)dc.off * a.qss;
  const T* dop =
      static_cast<const T*>(a.dout) + b * a.dosb + h * a.dosh + (int64_t)dc.off * a.doss;
  const T* opp = static_cast<const T*>(a.o) + b * a.osb + h * a.osh + (int64_t)dc.off * a.oss;
  const T* kp = static_cast<const T*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const T* vp = static_cast<const T*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  const int64_t row_bh = (int64_t)bh * a.S + dc.off;
  const GlobRows gr = glob_rows<T, D>(a, dc, b, hk, kp, vp, DIR);

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (hi - lo_k + BN - 1) / BN;
  const int nglob = (gmax + BN - 1) / BN;
  const int ntot = nloc + nglob;
  using Fill = typename Tile::template Fill<NW>;
  const int kbytes = (int)(a.kss * 2), vbytes = DIR ? kbytes : (int)(a.vss * 2);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(kp, (uint32_t)((hi - 1) * kbytes + D * 2));
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(vp, (uint32_t)((hi - 1) * vbytes + D * 2));
  const int gkb = (int)gr.kstep, gvb = (int)gr.vstep;
  const __amdgpu_buffer_rsrc_t rgk = make_rsrc(gr.k, gmax > 0 ? (uint32_t)((gmax - 1) * gkb + D * 2) : 0);
  const __amdgpu_buffer_rsrc_t rgv = make_rsrc(gr.v, gmax > 0 ? (uint32_t)((gmax - 1) * gvb + D * 2) : 0);
  const int fk = Fill::lane_off(wave, lane, kbytes);
  const int fv = Fill::lane_off(wave, lane, vbytes);
  const int fgk = Fill::lane_off(wave, lane, gkb), fgv = Fill::lane_off(wave, lane, gvb);
  // the local window, then the global rows, as the forward
  auto row0 = [&](int it) { return it < nloc ? lo_k + it * BN : (it - nloc) * BN; };
  auto issue_k = [&](int it, char* dst) {
    if (it < nloc)
      Fill::load(dst, rk, fk, kbytes, row0(it), wave);
    else
      Fill::load(dst, rgk, fgk, gkb, row0(it), wave);
  };
  auto issue_v = [&](int it) {
    if (it < nloc)
      Fill::load(sV, rv, fv, vbytes, row0(it), wave);
    else
      Fill::load(sV, rgv, fgv, gvb, row0(it), wave);
  };
  issue_k(0, sK0);
  issue_v(0);

  LaneOffs<D> lo;
  lo.init(lane);
  // Delta = rowsum(O * dO) of the wave's queries, stored negated with
  // -lse * log2(e) for the dK/dV kernels (see dq2_kernel). Rows past the
  // document read its last row; their results are never stored.
  Frag<T> qf[1][D / 32], df[1][D / 32];
  const int qi = q0 + l16;
  const int qr = min(qi, S - 1);
  const bool ok = qi < S;
  const float lse2[1] = {ok ? a.lse[row_bh + qr] * kLog2e : 0.f};
  float od8[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    qf[0][c] = lds_frag_row<T>(qp + (int64_t)qr * a.qss + 32 * c + 8 * g);
    df[0][c] = lds_frag_row<T>(dop + (int64_t)qr * a.doss + 32 * c + 8 * g);
    const Frag<T> of = lds_frag_row<T>(opp + (int64_t)qr * a.oss + 32 * c + 8 * g);
    const T* eo = reinterpret_cast<const T*>(of.w);
    const T* ed = reinterpret_cast<const T*>(df[0][c].w);
    od8[c] = 0.f;
    if constexpr (std::is_same<T, f16>::value) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        od8[c] = __builtin_amdgcn_fdot2(reinterpret_cast<const f16x2*>(eo)[i],
                                        reinterpret_cast<const f16x2*>(ed)[i], od8[c], false);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) od8[c] = fmaf(to_f32(eo[i]), to_f32(ed[i]), od8[c]);
    }
  }
  const float od = delta_sum<D>(od8);
  const float ndl[1] = {-od};
  if (ok && g == 0) {
    a.delta[row_bh + qi] = -od;
    a.nlse2[row_bh + qi] = -lse2[0];
  }
  const float c2 = a.scale * kLog2e;
  f32x4 dqa[D / 16][1];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) dqa[db][0] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = q0 < S;
  const int q_last = min(q0 + 16, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  const int glen = glob_prefix(qi, dc);

  auto step = [&](auto buf_c, int it) {
    char(&cur)[Tile::kBytes] = decltype(buf_c)::value ? sK1 : sK0;
    char(&nxt)[Tile::kBytes] = decltype(buf_c)::value ? sK0 : sK1;
    wait_vmem();
    __syncthreads();  // this tile's K and V landed; every wave is done with the other K
    if (it + 1 < ntot) issue_k(it + 1, nxt);
    const bool loc = it < nloc;
    const int ts = row0(it);
    const bool work = active && (loc ? (ts <= q_last && ts + BN - 1 >= w_lo) : ts < wg_hi);
    Frag<T> dsf[1];
    if (work) {
      const bool full = loc ? (ts >= q_last - W + 1 && ts + BN - 1 <= q0) : ts + BN <= wg_lo;
      TileMask<1> mk;
      mk.hi[0] = loc ? qi - ts : glen - 1 - ts;
      mk.span[0] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
      if (full)
        dq2_ds<T, D, 1, BN, false>(cur, sV, 0, lo, qf, df, lse2, ndl, c2, g, mk, dsf);
      else
        dq2_ds<T, D, 1, BN, true>(cur, sV, 0, lo, qf, df, lse2, ndl, c2, g, mk, dsf);
    }
    __syncthreads();  // every wave is done with this tile's V
    if (it + 1 < ntot) issue_v(it + 1);
    if (work) dq2_acc<T, D, 1, BN>(cur, 0, lo, dsf, dqa);
  };
  for (int it = 0; it < ntot; it += 2) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 < ntot) step(std::integral_constant<int, 1>{}, it + 1);
  }

  if (!active || qi >= S) return;
  T* row = static_cast<T*>(a.dq) + b * a.dqsb + h * a.dqsh + (int64_t)(dc.off + qi) * a.dqss;
#pragma unroll
  for (int db = 0; db < D / 16; ++db) store4<T>(row + 16 * db + 4 * g, dqa[db][0], a.scale);
}

// Epilogues of the dK/dV kernels: lane (l16, g) owns key row kw + 16kb + l16,
// dims 16db + 4g .. +4 of each block. Global rows: the chunk's fp32 partial.
template <int D, int KB>
__device__ __forceinline__ void write_part(const BwdCommon& a, const Doc& dc, int chunk, int nbh,
                                           int bhk, int kw, int nrows, int l16, int g,
                                           const f32x4 (&dka)[D / 16][KB],
                                           const f32x4 (&dva)[D / 16][KB]) {
  float* part = a.gpart + part_row(dc, chunk, nbh, bhk, 0) * 2 * D;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int row = kw + 16 * kb + l16;
    if (row >= nrows) continue;
    float* pk = part + (int64_t)row * 2 * D;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      *reinterpret_cast<f32x4*>(pk + 16 * db + 4 * g) = dka[db][kb] * a.scale;
      *reinterpret_cast<f32x4*>(pk + D + 16 * db + 4 * g) = dva[db][kb];
    }
  }
}

// Local rows: dK/dV of row j, with the global rows whose source is row j (the
// strided row of its block and any relay row selected from it; reference
// scatter, core.py:2767-2815).
template <typename T, int D, int KB>
__device__ __forceinline__ void write_local(const BwdCommon& a, const Doc& dc, int nbh, int b, int hk,
                                            int kw, int l16, int g, f32x4 (&dka)[D / 16][KB],
                                            f32x4 (&dva)[D / 16][KB]) {
  const int S = dc.len, W = dc.W, rpb = dc.rpb;
  const bool relay = rpb > 1;
  const int bhk = b * a.Hkv + hk;
  T* dkp = static_cast<T*>(a.dk) + b * a.dksb + hk * a.dksh + (int64_t)dc.off * a.dkss;
  T* dvp = static_cast<T*>(a.dv) + b * a.dvsb + hk * a.dvsh + (int64_t)dc.off * a.dvss;
  const float rsc = (relay && a.rscale) ? a.rscale[hk] : 1.f;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int j = kw + 16 * kb + l16;
    if (j >= S) continue;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) dka[db][kb] *= a.scale;
    // (a plain division: with div_by the D = 64 local kernel, at its register
    // cap, spills 21 and is 45% slower)
    const int rblk = j / W;
    int grow[5];
    float gsc[5];
    int nm = 0;
    if (j == rblk * W) {
      grow[nm] = rblk * rpb;
      gsc[nm++] = 1.f;
    }
    if (relay) {
      const int32_t* src = a.src + ((int64_t)bhk * a.NB + dc.bofs + rblk) * a.top_k;
      for (int t = 0; t < a.top_k; ++t) {
        if (src[t] == j) {
          grow[nm] = rblk * rpb + 1 + t;
          gsc[nm++] = rsc;
        }
      }
    }
    // the chunk partials of the global rows are summed into chunk 0
    for (int m = 0; m < nm; ++m) {
      const float* pk = a.gpart + part_row(dc, 0, nbh, bhk, grow[m]) * 2 * D;
#pragma unroll
      for (int db = 0; db < D / 16; ++db) {
        dka[db][kb] += *reinterpret_cast<const f32x4*>(pk + 16 * db + 4 * g) * gsc[m];
        dva[db][kb] += *reinterpret_cast<const f32x4*>(pk + D + 16 * db + 4 * g) * gsc[m];
      }
    }
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      store4<T>(dkp + (int64_t)j * a.dkss + 16 * db + 4 * g, dka[db][kb], 1.f);
      store4<T>(dvp + (int64_t)j * a.dvss + 16 * db + 4 * g, dva[db][kb], 1.f);
    }
  }
}

// Key-centric dK/dV: each wave owns KB blocks of 16 key rows (rows of k/v,
// or packed global rows with GLOB), B operands in registers; query tiles of
// BQ rows of Q and dO stream through LDS with their -lse * log2(e) (sL) and
// -Delta (sDl), both written by dq2_kernel. A key row
// j sees the queries [j, j+W-1] (local) or [first_query(j), S) (global rows),
// so every mask is a per-key interval.
template <typename T, int D, int KB, int BQ, bool MASK, bool LOC>
__device__ __forceinline__ void dkdv2_tile(const char* tQ, const char* tO, const float* sL,
                                           const float* sDl, const LaneOffs<D>& lo,
                                           const Frag<T> (&kf)[KB][D / 32],
                                           const Frag<T> (&vf)[KB][D / 32],
                                           f32x4 (&dka)[D / 16][KB], f32x4 (&dva)[D / 16][KB],
                                           float c2, int g, int ts, const int (&qmin)[KB],
                                           const int (&qmax)[KB], const unsigned (&qspan)[KB]) {
  using Tile = SwzTile<D, BQ>;
  constexpr int NS = BQ / 32;  // 32-query subtiles
  // LDS fragments are read PF MFMA steps ahead of their use; scheduling
  // fences keep the compiler from moving the reads next to their uses
  constexpr int PF = 2;
  // S = Q . K^T and dP - Delta = dO . V^T - Delta of subtile qs (two
  // 16-query blocks; sDl holds -Delta, the dP accumulators' initial value)
  auto scores = [&](int qs, f32x4 (&sc)[2][KB], f32x4 (&dp)[2][KB]) {
    constexpr int NC = D / 32, NT = 2 * NC;
    auto row_qo = [&](int t, Frag<T>& q_, Frag<T>& o_) {
      const int qn = 2 * qs + t / NC, cn = t % NC;
      q_ = Tile::template row_frag_at<T>(tQ + qn * Tile::kBlk16 + lo.row_at(cn));
      o_ = Tile::template row_frag_at<T>(tO + qn * Tile::kBlk16 + lo.row_at(cn));
    };
    Frag<T> qa[PF + 1], oa[PF + 1];
#pragma unroll
    for (int t = 0; t < PF; ++t) row_qo(t, qa[t], oa[t]);
#pragma unroll
    for (int qb2 = 0; qb2 < 2; ++qb2) {
      const f32x4 ndq = *reinterpret_cast<const f32x4*>(sDl + 16 * (2 * qs + qb2) + 4 * g);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        sc[qb2][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
        dp[qb2][kb] = kSubDelta<D> ? f32x4{0.f, 0.f, 0.f, 0.f} : ndq;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int qb2 = t / NC, c = t % NC;
      if (t + PF < NT) row_qo(t + PF, qa[(t + PF) % (PF + 1)], oa[(t + PF) % (PF + 1)]);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        sc[qb2][kb] = mma(sc[qb2][kb], qa[t % (PF + 1)], kf[kb][c]);
        dp[qb2][kb] = mma(dp[qb2][kb], oa[t % (PF + 1)], vf[kb][c]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Each subtile's scores, then its exponentials, in sequence: 165 VGPRs,
  // 3 waves per SIMD. (A software pipeline over the subtiles, the next
  // subtile's score MFMAs beside this one's exponentials, needs 225
  // registers and 2 waves per SIMD: 4.2% slower backward with the local
  // kernel.) LOC (local rows) tests each mask with one unsigned compare;
  // the global-row kernel keeps two compares. Unrolled by two only: the four
  // subtiles of a 128-row tile fully unrolled spill (the compiler hoists the
  // next subtiles' fragment reads).
  f32x4 sc[2][KB], dp[2][KB];  // [qb2][kb]
#pragma unroll 2
  for (int qs = 0; qs < NS; ++qs) {
    scores(qs, sc, dp);
    float p[2][KB][4], ds[2][KB][4];  // [qb2][kb][r]
    // query 16 qblk + 4g + r of the tile is visible to key kb iff
    // (unsigned)(16 qblk + r - q0[kb]) <= qspan[kb]
    int q0[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) q0[kb] = qmin[kb] - ts - 4 * g;
#pragma unroll
    for (int qb2 = 0; qb2 < 2; ++qb2) {
      const int qblk = 2 * qs + qb2;
      const f32x4 nlq = *reinterpret_cast<const f32x4*>(sL + 16 * qblk + 4 * g);
      f32x4 ndq{};
      if (kSubDelta<D>) ndq = *reinterpret_cast<const f32x4*>(sDl + 16 * qblk + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          float x = fmaf(sc[qb2][kb][r], c2, nlq[r]);
          if (MASK) {
            const bool out = LOC ? (unsigned)(16 * qblk + r - q0[kb]) > qspan[kb]
                                 : (ts + 16 * qblk + 4 * g + r < qmin[kb] ||
                                    ts + 16 * qblk + 4 * g + r > qmax[kb]);
            if (out) x = -__builtin_huge_valf();
          }
          p[qb2][kb][r] = __builtin_amdgcn_exp2f(x);
          ds[qb2][kb][r] =
              p[qb2][kb][r] * (kSubDelta<D> ? dp[qb2][kb][r] + ndq[r] : dp[qb2][kb][r]);
        }
      }
    }
    Frag<T> pf[KB], sf[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const float pv[8] = {p[0][kb][0], p[0][kb][1], p[0][kb][2], p[0][kb][3],
                           p[1][kb][0], p[1][kb][1], p[1][kb][2], p[1][kb][3]};
      const float sv[8] = {ds[0][kb][0], ds[0][kb][1], ds[0][kb][2], ds[0][kb][3],
                           ds[1][kb][0], ds[1][kb][1], ds[1][kb][2], ds[1][kb][3]};
      pf[kb] = pack8<T>(pv);
      sf[kb] = pack8<T>(sv);
    }
    // each transposed Q/dO fragment pair serves every key block of the wave
    Frag<T> ot[PF + 1], qt[PF + 1];
    auto tr_pair = [&](int db, Frag<T>& o_, Frag<T>& q_) {
      const char* po = tO + (2 * qs) * Tile::kBlk16 + lo.tr_at(db);
      const char* pq = tQ + (2 * qs) * Tile::kBlk16 + lo.tr_at(db);
      o_ = Tile::template tr_frag_at<T>(po, po + Tile::kBlk16);
      q_ = Tile::template tr_frag_at<T>(pq, pq + Tile::kBlk16);
    };
#pragma unroll
    for (int db = 0; db < PF; ++db) tr_pair(db, ot[db], qt[db]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      if (db + PF < D / 16) tr_pair(db + PF, ot[(db + PF) % (PF + 1)], qt[(db + PF) % (PF + 1)]);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        dva[db][kb] = mma(dva[db][kb], ot[db % (PF + 1)], pf[kb]);
        dka[db][kb] = mma(dka[db][kb], qt[db % (PF + 1)], sf[kb]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// NW waves of KB key blocks each cover the workgroup's 16 * NW * KB key
// rows; query tiles of BQ rows. At most 168 VGPRs: 3 waves per SIMD (the
// global-row kernel below D = 128: at most 128, 4 waves per SIMD). At D = 256
// the accumulators and the resident K/V fragments take 192 registers of a
// 16-row wave: 256 VGPRs (9-10 spilled), 2 waves per SIMD, 4-wave workgroups
// with 32-query tiles (66 KB of LDS, two per CU). B=1 H=8 S=32768 bf16:
// global rows 224 us, local 323 us; with one LDS stage and transposed tiles
// written by 2-byte LDS stores 721 and 638 us.
template <typename T, int D, bool GLOB, int NW, int KB, int BQ, int ND>
__global__ __launch_bounds__(64 * NW)
__attribute__((amdgpu_waves_per_eu(D > 128 ? 2 : GLOB && D < 128 ? 4 : 3)))
void dkdv2_kernel(BwdArgsT<ND> a) {
  using Tile = SwzTile<D, BQ>;
  constexpr int kKW = 16 * KB, kBK = NW * kKW, kBQ = BQ;
  static_assert(BQ == 32 || BQ == 64 || BQ == 128, "query tile rows");
  // Two pipeline stages as separate LDS objects (see fwd2_kernel): Q and dO
  // rows, and their -lse * log2(e) and -Delta.
  __shared__ __attribute__((aligned(1024))) char stage0[2][Tile::kBytes];
  __shared__ __attribute__((aligned(1024))) char stage1[2][Tile::kBytes];
  __shared__ __attribute__((aligned(16))) float sld0[2][kBQ];  // [-lse log2 e, -delta][q]
  __shared__ __attribute__((aligned(16))) float sld1[2][kBQ];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int nbh = a.B * a.Hkv;
  int item = (int)blockIdx.x;
  if (!GLOB && a.xcd_nt > 0) {
    item = xcd_item(item, nbh, a.xcd_nt);
    if (item < 0) return;  // padding block
  }
  const KvHead hd = kv_head(a, item);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bhk = hd.bhk, b = hd.b, hk = hd.hk;
  const int nck = GLOB ? num_chunks(dc.len, a.chunk_len) : 1;
  const int tile = GLOB ? dc.item / nck : dc.item;
  const int chunk = GLOB ? dc.item - tile * nck : 0;
  const int grp = a.Hq / a.Hkv;
  const int S = dc.len, W = dc.W, rpb = dc.rpb;
  const int nrows = GLOB ? doc_rows(S, W, rpb) : S;  // keys: global rows or rows
  const int k0 = tile * kBK;
  const int kw = k0 + wave * kKW;

  const T* kbase;
  const T* vbase;
  int64_t kstride, vstride;
  kbase = static_cast<const T*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  vbase = static_cast<const T*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  kstride = a.kss;
  vstride = a.vss;
  if (GLOB) {
    const GlobRows gr = glob_rows<T, D>(a, dc, b, hk, kbase, vbase, a.direct);
    kbase = (const T*)gr.k;
    vbase = (const T*)gr.v;
    kstride = gr.kstep / (int)sizeof(T);
    vstride = gr.vstep / (int)sizeof(T);
  }

  // query interval of the workgroup; per-key intervals for the masks
  int q_lo, q_hi;
  if (GLOB) {
    const int chunk_len = doc_chunk_len<ND>(S, nck, a.chunk_len);
    const int c_lo = chunk * chunk_len;
    q_hi = min(S, c_lo + chunk_len);
    q_lo = max(c_lo, glob_row_first_query(k0, dc));
    // no query of this chunk sees the tile's rows: gsum_kernel skips the
    // chunk for them (with a single chunk the zeros are written instead)
    if (q_hi <= q_lo && a.nchunk > 1) return;
  } else {
    q_lo = k0;
    q_hi = min(S, k0 + kBK - 1 + W);
  }
  const int ntile_q = q_hi > q_lo ? (q_hi - q_lo + kBQ - 1) / kBQ : 0;
  const int ntot = ntile_q * grp;

  const int qbytes = (int)(a.qss * 2), obytes = (int)(a.doss * 2);
  // the first FW (a power of two) waves fill the tiles
  constexpr int FW = NW >= 8 ? 8 : NW;
  using Fill = typename Tile::template Fill<FW>;
  const int fq = Fill::lane_off(wave & (FW - 1), lane, qbytes);
  const int fo = Fill::lane_off(wave & (FW - 1), lane, obytes);

  LaneOffs<D> lo;
  lo.init(lane);
  Frag<T> kf[KB][D / 32], vf[KB][D / 32];
  int qmin[KB], qmax[KB];
  unsigned qspan[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int row = kw + 16 * kb + l16;
    // query rows at or past q_hi load as zeros: excluded
    if (GLOB) {
      qmin[kb] = row < nrows ? glob_row_first_query(row, dc) : S;
      qmax[kb] = q_hi - 1;
    } else {
      qmin[kb] = row;
      qmax[kb] = min(row + W, q_hi) - 1;
    }
    // masks test (unsigned)(q - qmin) <= qspan; an empty interval gets a qmin
    // no query reaches
    qspan[kb] = qmax[kb] >= qmin[kb] ? (unsigned)(qmax[kb] - qmin[kb]) : 0u;
    if (!GLOB && qmax[kb] < qmin[kb]) qmin[kb] = 1 << 30;
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
      if (row < nrows) {
        kf[kb][c] = lds_frag_row<T>(kbase + (int64_t)row * kstride + 32 * c + 8 * g);
        vf[kb][c] = lds_frag_row<T>(vbase + (int64_t)row * vstride + 32 * c + 8 * g);
      } else {
        zero_frag(kf[kb][c]);
        zero_frag(vf[kb][c]);
      }
    }
  }
  f32x4 dka[D / 16][KB], dva[D / 16][KB];
#pragma unroll
  for (int db = 0; db < D / 16; ++db)
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) dka[db][kb] = dva[db][kb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = kw < nrows;
  const int k_last = min(kw + kKW, nrows) - 1;
  // queries this wave can see at all
  const int wq_lo = GLOB ? (active ? max(q_lo, glob_row_first_query(kw, dc)) : S) : kw;
  const int wq_hi = GLOB ? q_hi : min(q_hi, kw + kKW - 1 + W);
  const int full_lo = GLOB ? (active ? glob_row_first_query(k_last, dc) : S) : k_last;
  const int full_hi = GLOB ? q_hi : kw + W;  // exclusive
  const float c2 = a.scale * kLog2e;

  // Tiles run head by head of the kv group (tile `it` is query tile
  // it % ntile_q of group head it / ntile_q). The (head, tile) counters of
  // the next tile to load and of the tile being computed advance by one per
  // step, and the buffer resources are rebuilt only when the head changes:
  // no per-tile division or 64-bit address arithmetic.
  struct HeadRes {
    __amdgpu_buffer_rsrc_t q, o, l, d;
  };
  auto head_res = [&](int j) {
    const int hq = hk * grp + j;
    const int64_t bh = (int64_t)b * a.Hq + hq;
    // query rows at or past q_hi load as zeros
    HeadRes r;
    r.q = make_rsrc(static_cast<const T*>(a.q) + b * a.qsb + hq * a.qsh + (int64_t)dc.off * a.qss,
                    (uint32_t)((q_hi - 1) * qbytes + D * 2));
    r.o = make_rsrc(
        static_cast<const T*>(a.dout) + b * a.dosb + hq * a.dosh + (int64_t)dc.off * a.doss,
        (uint32_t)((q_hi - 1) * obytes + D * 2));
    r.l = make_rsrc(a.nlse2 + bh * a.S + dc.off, (uint32_t)(S * 4));
    r.d = make_rsrc(a.delta + bh * a.S + dc.off, (uint32_t)(S * 4));
    return r;
  };
  HeadRes ld_res = head_res(0);
  int ld_j = 0, ld_t = 0;  // next tile to load
  auto load_tile = [&](char (&dst)[2][Tile::kBytes], float (&dsl)[2][kBQ]) {
    const int ts = q_lo + ld_t * kBQ;
    if (NW == FW || wave < FW) {
      Fill::load(dst[0], ld_res.q, fq, qbytes, ts, wave);
      Fill::load(dst[1], ld_res.o, fo, obytes, ts, wave);
    }
    // one lane per query row of the tile (lane i of pass c lands at
    // dsl[.][64 c + i])
    if (wave == 0) {
#pragma unroll
      for (int c = 0; c < (kBQ + 63) / 64; ++c) {
        if (kBQ >= 64 || lane < kBQ) {
          const int qrow = min(ts + 64 * c + lane, q_hi - 1);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(ld_res.l, CRA_LDS(&dsl[0][64 * c]), 4,
                                                   qrow * 4, 0, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(ld_res.d, CRA_LDS(&dsl[1][64 * c]), 4,
                                                   qrow * 4, 0, 0, 0);
        }
      }
    }
    if (++ld_t == ntile_q) {
      ld_t = 0;
      if (++ld_j < grp) ld_res = head_res(ld_j);
    }
  };
  if (ntot > 0) load_tile(stage0, sld0);
  int cu_t = 0;  // query tile being computed

  auto step = [&](auto BUFC, int it) {
    constexpr int BUF = decltype(BUFC)::value;
    char(&cur)[2][Tile::kBytes] = BUF ? stage1 : stage0;
    float(&csl)[2][kBQ] = BUF ? sld1 : sld0;
    wait_vmem();
    __syncthreads();
    if (it + 1 < ntot) {
      if (BUF)
        load_tile(stage0, sld0);
      else
        load_tile(stage1, sld1);
    }
    const int ts = q_lo + cu_t * kBQ;
    if (++cu_t == ntile_q) cu_t = 0;
    const int t_last = min(ts + kBQ, q_hi) - 1;
    if (active && t_last >= wq_lo && ts < wq_hi) {
      const bool full = ts >= full_lo && ts + kBQ <= full_hi && ts + kBQ <= q_hi;
      if (full)
        dkdv2_tile<T, D, KB, BQ, false, !GLOB>(cur[0], cur[1], csl[0], csl[1], lo, kf, vf, dka,
                                               dva, c2, g, ts, qmin, qmax, qspan);
      else
        dkdv2_tile<T, D, KB, BQ, true, !GLOB>(cur[0], cur[1], csl[0], csl[1], lo, kf, vf, dka, dva, c2, g,
                                   ts, qmin, qmax, qspan);
    }
  };
  for (int it = 0; it < ntot; it += 2) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 < ntot) step(std::integral_constant<int, 1>{}, it + 1);
  }

  if (GLOB)
    write_part<D, KB>(a, dc, chunk, nbh, bhk, kw, nrows, l16, g, dka, dva);
  else
    write_local<T, D, KB>(a, dc, nbh, b, hk, kw, l16, g, dka, dva);
}

// ---------------------------------------------------------------------------
// fp32 backward: dq2 and dkdv2 with every operand split in three bf16 pieces
// (Split). 4 waves of 16 queries (dQ) or 16 key rows (dK/dV), whose own
// operands stay split in registers; 32-row tiles of K and V (Q and dO) are
// staged through registers and split once per workgroup, up to D = 64 in two
// LDS stages with one barrier per tile; dS and P are split in registers. Delta
// is subtracted from the finished dP, as at D = 256 in 2 bytes (kSubDelta).
// Against the fp32-MFMA kernels before them (dQ with the separate Delta pass /
// global rows / local rows), H=8: S=32768 D=64 547 / 566 / 469 -> 336 / 324 /
// 247 us, D=128 1248 / 1603 / 1040 -> 629 / 674 / 487 us, S=4096 D=64 58 / 49 /
// 42 -> 26 / 29 / 21 us; H=4 S=8192 D=256 199 / 211 / 146 -> 147 / 148 / 120 us.
// ---------------------------------------------------------------------------
constexpr int kF32Waves = 4, kF32BN = 32;

template <int D, bool MASK>
__device__ __forceinline__ void dq_f32_tile(const char* tK, const char* tV, const LaneOffs<D>& lo,
                                            const Split (&qf)[D / 32], const Split (&df)[D / 32],
                                            f32x4 (&dqa)[D / 16], float lse2, float ndl, float c2,
                                            int g, const TileMask<1>& mk) {
  using Stage = SplitStage<D, kF32BN, 64 * kF32Waves>;
  using Tile = typename Stage::Tile;
  f32x4 sc[2], dp[2], sl[2], dl[2];  // sl, dl: the small products (kSmallApart)
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    sc[h] = dp[h] = sl[h] = dl[h] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    Split kf[2], vf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      kf[h] = Stage::row_frag(tK + h * Tile::kBlk16 + lo.row_at(c));
      vf[h] = Stage::row_frag(tV + h * Tile::kBlk16 + lo.row_at(c));
    }
    // consecutive MFMAs go to different accumulators
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4& s_ = t < kSmallApart<D> ? sl[h] : sc[h];
        f32x4& d_ = t < kSmallApart<D> ? dl[h] : dp[h];
        s_ = mma(s_, kf[h].p[split_a(t)], qf[c].p[split_b(t)]);
        d_ = mma(d_, vf[h].p[split_a(t)], df[c].p[split_b(t)]);
      }
  }
  if (kSmallApart<D> > 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] += sl[h];
      dp[h] += dl[h];
    }
  }
  float ds[8];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = fmaf(sc[h][r], c2, -lse2);
      if (MASK && !mk.ok(16 * h + 4 * g + r, 0)) x = -__builtin_huge_valf();
      ds[4 * h + r] = __builtin_amdgcn_exp2f(x) * (dp[h][r] + ndl);
    }
  const Split dsf = split8<true>(ds);
#pragma unroll
  for (int db = 0; db < D / 16; db += 2) {
    Split kt[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) kt[e] = Stage::tr_frag(tK + lo.tr_at(db + e));
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e)
        dqa[db + e] = mma(dqa[db + e], kt[e].p[split_a(t)], dsf.p[split_b(t)]);
  }
}

// (D = 64: at most 168 registers, three workgroups per CU; at 170 and two it
// took 1249 us against 1039 at B=1 H=4 S=131072)
template <int D, int ND>
__global__ __launch_bounds__(64 * kF32Waves)
__attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : D > 64 ? 2 : 3)))
void dq_f32_kernel(BwdArgsT<ND> a) {
  constexpr int NW = kF32Waves, BN = kF32BN, kBM = 16 * NW;
  constexpr int kStages = D <= 64 ? 2 : 1;
  using Stage = SplitStage<D, BN, 64 * NW>;
  __shared__ __attribute__((aligned(1024))) char lds[kStages][2][Stage::kBytes];  // K, V

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const QHead hd = q_head(a, blockIdx.x);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bh = hd.bh, b = hd.b, h = hd.h, hk = hd.hk;
  const int tile = (dc.len + kBM - 1) / kBM - 1 - dc.item;  // heaviest first
  const int m0 = tile * kBM;
  const int q0 = m0 + wave * 16;
  const int S = dc.len, W = dc.W;

  const float* qp = static_cast<const float*>(a.q) + b * a.qsb + h * a.qsh + (int64_t)dc.off * a.qss;
  const float* dop =
      static_cast<const float*>(a.dout) + b * a.dosb + h * a.dosh + (int64_t)dc.off * a.doss;
  const float* opp = static_cast<const float*>(a.o) + b * a.osb + h * a.osh + (int64_t)dc.off * a.oss;
  const float* kp = static_cast<const float*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const float* vp = static_cast<const float*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  const int64_t row_bh = (int64_t)bh * a.S + dc.off;
  const GlobRows gr = glob_rows<float, D>(a, dc, b, hk, kp, vp, a.direct);
  const float *gkp = (const float*)gr.k, *gvp = (const float*)gr.v;

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (hi - lo_k + BN - 1) / BN;
  const int nglob = (gmax + BN - 1) / BN;
  const int ntot = nloc + nglob;
  // global tiles first, then the local window from its highest tile down
  auto row0 = [&](int it) { return it >= nglob ? lo_k + (nloc - 1 - (it - nglob)) * BN : it * BN; };
  Stage stk, stv;
  auto load = [&](int it) {
    if (it >= nglob) {
      stk.load(kp, a.kss, row0(it), hi, tid);
      stv.load(vp, a.vss, row0(it), hi, tid);
    } else {
      stk.load(gkp, gr.kstep / 4, row0(it), gmax, tid);
      stv.load(gvp, gr.vstep / 4, row0(it), gmax, tid);
    }
  };
  auto store = [&](int it) {
    char(&dst)[2][Stage::kBytes] = lds[kStages == 2 ? it & 1 : 0];
    stk.store(dst[0], tid);
    stv.store(dst[1], tid);
  };
  load(0);

  LaneOffs<D> lo;
  lo.init(lane);
  // Delta = rowsum(O * dO) of the wave's queries, stored negated with
  // -lse * log2(e) for the dK/dV kernels (see dq2_kernel). Rows past the
  // document read its last row; their results are never stored.
  Split qf[D / 32], df[D / 32];
  const int qi = q0 + l16;
  const int qr = min(qi, S - 1);
  const bool ok = qi < S;
  const float lse2 = ok ? a.lse[row_bh + qr] * kLog2e : 0.f;
  float od8[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    qf[c] = load_split(qp + (int64_t)qr * a.qss + 32 * c + 8 * g);
    const float* pd = dop + (int64_t)qr * a.doss + 32 * c + 8 * g;
    const float* po = opp + (int64_t)qr * a.oss + 32 * c + 8 * g;
    float xd[8];
    od8[c] = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4 d4 = reinterpret_cast<const f32x4*>(pd)[i], o4 = reinterpret_cast<const f32x4*>(po)[i];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        xd[4 * i + r] = d4[r];
        od8[c] = fmaf(o4[r], d4[r], od8[c]);
      }
    }
    df[c] = split8<true>(xd);
  }
  const float od = delta_sum<D>(od8);
  if (ok && g == 0) {
    a.delta[row_bh + qi] = -od;
    a.nlse2[row_bh + qi] = -lse2;
  }
  const float c2 = a.scale * kLog2e;
  f32x4 dqa[D / 16];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) dqa[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool active = q0 < S;
  const int q_last = min(q0 + 16, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  const int glen = glob_prefix(qi, dc);

  store(0);
  __syncthreads();
  for (int it = 0; it < ntot; ++it) {
    if (it + 1 < ntot) load(it + 1);
    const char(&cur)[2][Stage::kBytes] = lds[kStages == 2 ? it & 1 : 0];
    const bool loc = it >= nglob;
    const int ts = row0(it);
    if (active && (loc ? (ts <= q_last && ts + BN - 1 >= w_lo) : ts < wg_hi)) {
      const bool full = loc ? (ts >= q_last - W + 1 && ts + BN - 1 <= q0) : ts + BN <= wg_lo;
      TileMask<1> mk;
      mk.hi[0] = loc ? qi - ts : glen - 1 - ts;
      mk.span[0] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
      if (full)
        dq_f32_tile<D, false>(cur[0], cur[1], lo, qf, df, dqa, lse2, -od, c2, g, mk);
      else
        dq_f32_tile<D, true>(cur[0], cur[1], lo, qf, df, dqa, lse2, -od, c2, g, mk);
    }
    if (kStages == 1) __syncthreads();  // every wave is done with this tile
    if (it + 1 < ntot) store(it + 1);
    __syncthreads();
  }

  if (!active || qi >= S) return;
  float* row = static_cast<float*>(a.dq) + b * a.dqsb + h * a.dqsh + (int64_t)(dc.off + qi) * a.dqss;
#pragma unroll
  for (int db = 0; db < D / 16; ++db) store4<float>(row + 16 * db + 4 * g, dqa[db], a.scale);
}

// A key row sees the queries [qmin, qmin + qspan] (see dkdv2_kernel).
template <int D, bool MASK, bool SUM>
__device__ __forceinline__ void dkdv_f32_tile(const char* tQ, const char* tO, const float* sL,
                                              const float* sDl, const LaneOffs<D>& lo,
                                              const Split (&kf)[D / 32], const Split (&vf)[D / 32],
                                              f32x4 (&dka)[D / 16][1], f32x4 (&dva)[D / 16][1],
                                              float c2, int g, int q_off, unsigned qspan) {
  using Stage = SplitStage<D, kF32BN, 64 * kF32Waves>;
  using Tile = typename Stage::Tile;
  f32x4 sc[2], dp[2], sl[2], dl[2];  // sl, dl: the small products (kSmallApart)
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    sc[h] = dp[h] = sl[h] = dl[h] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    Split qa[2], oa[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      qa[h] = Stage::row_frag(tQ + h * Tile::kBlk16 + lo.row_at(c));
      oa[h] = Stage::row_frag(tO + h * Tile::kBlk16 + lo.row_at(c));
    }
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4& s_ = t < kSmallApart<D> ? sl[h] : sc[h];
        f32x4& d_ = t < kSmallApart<D> ? dl[h] : dp[h];
        s_ = mma(s_, qa[h].p[split_a(t)], kf[c].p[split_b(t)]);
        d_ = mma(d_, oa[h].p[split_a(t)], vf[c].p[split_b(t)]);
      }
  }
  if (kSmallApart<D> > 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] += sl[h];
      dp[h] += dl[h];
    }
  }
  float p[8], ds[8];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const f32x4 nlq = *reinterpret_cast<const f32x4*>(sL + 16 * h + 4 * g);
    const f32x4 ndq = *reinterpret_cast<const f32x4*>(sDl + 16 * h + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = fmaf(sc[h][r], c2, nlq[r]);
      if (MASK && (unsigned)(16 * h + r + q_off) > qspan) x = -__builtin_huge_valf();
      p[4 * h + r] = __builtin_amdgcn_exp2f(x);
      ds[4 * h + r] = p[4 * h + r] * (dp[h][r] + ndq[r]);
    }
  }
  const Split pf = split8<false>(p), sf = split8<true>(ds);
  // SUM (global rows): a tile's six products are summed from zero and added
  // once. A row of the first blocks sums over thousands of queries, where six
  // roundings of the long sum per tile would show (dK at S = 131072: relative
  // error 1.4e-6, and 5.6e-7 so; the fp32 MFMA's 9.5e-7). A local row sums over
  // W queries of each head of its kv group: added up straight its error stays
  // below the fp32 MFMA's with the longest sums too (H=32/1 S=131072 D=64, 11.6K
  // queries: dK 2.1e-6 against 3.4e-6; H=16/1 S=65536 D=128 1.2e-6 against
  // 1.7e-6), and per-tile sums would take the D = 128 kernel, at its register
  // cap, 7% longer for a sixth less of it.
#pragma unroll
  for (int db = 0; db < D / 16; ++db) {
    const Split ot = Stage::tr_frag(tO + lo.tr_at(db));
    const Split qt = Stage::tr_frag(tQ + lo.tr_at(db));
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 tv = SUM ? zero : dva[db][0], tk = SUM ? zero : dka[db][0];
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      tv = mma(tv, ot.p[split_a(t)], pf.p[split_b(t)]);
      tk = mma(tk, qt.p[split_a(t)], sf.p[split_b(t)]);
    }
    dva[db][0] = SUM ? dva[db][0] + tv : tv;
    dka[db][0] = SUM ? dka[db][0] + tk : tk;
  }
}

// At D = 128 the global-row kernel needs 343 registers: one wave per SIMD and
// two LDS stages (at 256 registers it spilled 82: 835 us against 761, B=1 H=8
// S=32768); the local one keeps 256 (22 spilled) and two workgroups per CU. At
// D = 256 both take the 512 of one wave per SIMD (9 and 24 spilled).
template <int D, bool GLOB>
constexpr bool kF32OneWave = D > 128 || (GLOB && D == 128);

template <int D, bool GLOB, int ND>
__global__ __launch_bounds__(64 * kF32Waves)
__attribute__((amdgpu_waves_per_eu(kF32OneWave<D, GLOB> ? 1 : 2)))
void dkdv_f32_kernel(BwdArgsT<ND> a) {
  constexpr int NW = kF32Waves, kBK = 16 * NW, kBQ = kF32BN;
  constexpr int kStages = D <= 64 || (GLOB && D == 128) ? 2 : 1;
  using Stage = SplitStage<D, kBQ, 64 * NW>;
  __shared__ __attribute__((aligned(1024))) char lds[kStages][2][Stage::kBytes];  // Q, dO
  __shared__ __attribute__((aligned(16))) float sld[kStages][2][kBQ];  // -lse log2(e), -Delta

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int nbh = a.B * a.Hkv;
  const KvHead hd = kv_head(a, blockIdx.x);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bhk = hd.bhk, b = hd.b, hk = hd.hk;
  const int nck = GLOB ? num_chunks(dc.len, a.chunk_len) : 1;
  const int tile = GLOB ? dc.item / nck : dc.item;
  const int chunk = GLOB ? dc.item - tile * nck : 0;
  const int grp = a.Hq / a.Hkv;
  const int S = dc.len, W = dc.W, rpb = dc.rpb;
  const int nrows = GLOB ? doc_rows(S, W, rpb) : S;  // keys: global rows or rows
  const int k0 = tile * kBK;
  const int kw = k0 + wave * 16;

  const float *kbase, *vbase;
  int64_t kstride, vstride;
  kbase = static_cast<const float*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  vbase = static_cast<const float*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  kstride = a.kss;
  vstride = a.vss;
  if (GLOB) {
    const GlobRows gr = glob_rows<float, D>(a, dc, b, hk, kbase, vbase, a.direct);
    kbase = (const float*)gr.k;
    vbase = (const float*)gr.v;
    kstride = gr.kstep / (int)sizeof(float);
    vstride = gr.vstep / (int)sizeof(float);
  }

  // queries of the workgroup
  int q_lo, q_hi;
  if (GLOB) {
    const int chunk_len = doc_chunk_len<ND>(S, nck, a.chunk_len);
    const int c_lo = chunk * chunk_len;
    q_hi = min(S, c_lo + chunk_len);
    q_lo = max(c_lo, glob_row_first_query(k0, dc));
    // see dkdv2_kernel
    if (q_hi <= q_lo && a.nchunk > 1) return;
  } else {
    q_lo = k0;
    q_hi = min(S, k0 + kBK - 1 + W);
  }
  const int ntile_q = q_hi > q_lo ? (q_hi - q_lo + kBQ - 1) / kBQ : 0;
  const int ntot = ntile_q * grp;

  LaneOffs<D> lo;
  lo.init(lane);
  const int row = kw + l16;
  const int rr = min(row, nrows - 1);  // rows past the last one see no query
  Split kf[D / 32], vf[D / 32];
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    kf[c] = load_split(kbase + (int64_t)rr * kstride + 32 * c + 8 * g);
    vf[c] = load_split(vbase + (int64_t)rr * vstride + 32 * c + 8 * g);
  }
  int qmin = GLOB ? (row < nrows ? glob_row_first_query(row, dc) : S) : row;
  const int qmax = GLOB ? q_hi - 1 : min(row + W, q_hi) - 1;
  // an empty interval gets a qmin no query reaches
  const unsigned qspan = qmax >= qmin ? (unsigned)(qmax - qmin) : 0u;
  if (qmax < qmin) qmin = 1 << 30;
  f32x4 dka[D / 16][1], dva[D / 16][1];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) dka[db][0] = dva[db][0] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = kw < nrows;
  const int k_last = min(kw + 16, nrows) - 1;
  // queries this wave can see at all, and those every row of it sees
  const int wq_lo = GLOB ? (active ? max(q_lo, glob_row_first_query(kw, dc)) : S) : kw;
  const int wq_hi = GLOB ? q_hi : min(q_hi, kw + 15 + W);
  const int full_lo = GLOB ? (active ? glob_row_first_query(k_last, dc) : S) : k_last;
  const int full_hi = GLOB ? q_hi : kw + W;  // exclusive
  const float c2 = a.scale * kLog2e;

  // tiles run head by head of the kv group
  Stage stq, sto;
  float st_l = 0.f, st_d = 0.f;
  int ld_j = 0, ld_t = 0;  // next tile to load
  auto load = [&]() {
    const int hq = hk * grp + ld_j;
    const int ts = q_lo + ld_t * kBQ;
    stq.load(static_cast<const float*>(a.q) + b * a.qsb + hq * a.qsh + (int64_t)dc.off * a.qss,
             a.qss, ts, q_hi, tid);
    sto.load(static_cast<const float*>(a.dout) + b * a.dosb + hq * a.dosh + (int64_t)dc.off * a.doss,
             a.doss, ts, q_hi, tid);
    if (tid < kBQ) {
      const int64_t q = ((int64_t)b * a.Hq + hq) * a.S + dc.off + min(ts + tid, q_hi - 1);
      st_l = a.nlse2[q];
      st_d = a.delta[q];
    }
    if (++ld_t == ntile_q) {
      ld_t = 0;
      ++ld_j;
    }
  };
  auto store = [&](int it) {
    const int st = kStages == 2 ? it & 1 : 0;
    stq.store(lds[st][0], tid);
    sto.store(lds[st][1], tid);
    if (tid < kBQ) {
      sld[st][0][tid] = st_l;
      sld[st][1][tid] = st_d;
    }
  };
  if (ntot > 0) {
    load();
    store(0);
  }
  __syncthreads();
  int cu_t = 0;  // query tile being computed
  for (int it = 0; it < ntot; ++it) {
    if (it + 1 < ntot) load();
    const int st = kStages == 2 ? it & 1 : 0;
    const int ts = q_lo + cu_t * kBQ;
    if (++cu_t == ntile_q) cu_t = 0;
    const int t_last = min(ts + kBQ, q_hi) - 1;
    if (active && t_last >= wq_lo && ts < wq_hi) {
      const bool full = ts >= full_lo && ts + kBQ <= full_hi && ts + kBQ <= q_hi;
      const int q_off = ts + 4 * g - qmin;
      if (full)
        dkdv_f32_tile<D, false, GLOB>(lds[st][0], lds[st][1], sld[st][0], sld[st][1], lo, kf, vf, dka,
                                dva, c2, g, q_off, qspan);
      else
        dkdv_f32_tile<D, true, GLOB>(lds[st][0], lds[st][1], sld[st][0], sld[st][1], lo, kf, vf, dka,
                               dva, c2, g, q_off, qspan);
    }
    if (kStages == 1) __syncthreads();  // every wave is done with this tile
    if (it + 1 < ntot) store(it + 1);
    __syncthreads();
  }
  if (GLOB)
    write_part<D, 1>(a, dc, chunk, nbh, bhk, kw, nrows, l16, g, dka, dva);
  else
    write_local<float, D, 1>(a, dc, nbh, b, hk, kw, l16, g, dka, dva);
}

// dK/dV workgroups: waves of 16 key rows (no register file spill into AGPR
// copies at D = 128; 32 rows per wave measured 14% slower). The global-row
// kernel uses 12 waves (192 rows): at 166 VGPRs a SIMD holds 3 of its
// waves, and one 12-wave workgroup fills them, where a second 8-wave
// workgroup did not fit beside the first (8 waves measured 1.7% slower
// backward, 4 waves 3% slower than 8); the local
// kernel 4 waves (64 rows: its band of queries, 64 + W - 1, wastes fewer
// pairs than with 128 rows; measured 7% faster). dQ workgroups: 4 waves of
// 32 queries, 64-key tiles, 2 waves per SIMD at 254 VGPRs (each K/V
// fragment read from LDS serves two query blocks). 16 queries per wave
// lose that reuse: 8 waves measured 27% slower, and with 32-key tiles at
// 3 or 4 waves per SIMD still 5-10% slower backward at D = 128.
// Below D = 128 the global-row kernel needs at most 128 VGPRs (114 at
// D = 64), so two 8-wave workgroups share a CU at 4 waves per SIMD, where
// one 12-wave workgroup left it at 3: backward 1.4% faster at B=1 H=12
// S=131072 D=64 and 3.3% at H=8 S=65536 (16-wave workgroups: 0.8%).
// Below D = 128 the local kernel's waves take 32 key rows each (two 16-key
// blocks sharing every Q/dO fragment read from LDS; 168 VGPRs, 3 waves per
// SIMD): twice the MFMAs per LDS read and per barrier of its 32-query
// tiles. Config 4 training (B=1 H=12 D=64) 1.2-1.7% faster at S = 8192,
// 32768 and 131072 (three alternating runs).
template <int D>
constexpr int kDkdvGlobWaves = D > 128 ? 4 : D == 128 ? 12 : 8;
constexpr int kDkdvLocalWaves = 4;
constexpr int kDkdvKB = 1;  // 16-key blocks per wave (global-row kernel)
template <int D>
constexpr int kDkdvLocalKB = D >= 128 ? 1 : 2;  // local kernel
constexpr int kDqWaves = 4;
constexpr int kDqQB = 2;    // 16-query blocks per dQ wave
constexpr int kDqBN = 64;   // key rows per dQ tile
constexpr int kDqWPE = 2;   // dQ waves per SIMD (register budget)
// Query rows per dK/dV tile. The local kernel's 32-row tiles keep its LDS
// at 33 KB, so three 4-wave workgroups (3 waves per SIMD, 165 VGPRs) fit on
// a CU; with 64-row tiles only two fit. The global-row kernel (one 12-wave
// workgroup per CU, 130 KB of LDS) takes 128-row tiles: one barrier per 128
// queries instead of 64 (backward 1.7% faster).
template <int D>
constexpr int kDkdvGlobBQ = D > 128 ? 32 : 128;
constexpr int kDkdvLocalBQ = 32;

// The global-row kernel's second geometry: 4-wave workgroups of 64 rows with
// 32-query tiles (the local kernel's: 33 KB of LDS, 3 workgroups per CU at
// D = 128). It is finer: where the wide workgroups (192 rows at D = 128, 128
// below) are fewer than two rounds of the CUs their last round leaves the chip
// half idle, and rows padded to a wide tile, or not yet visible to a chunk,
// idle their waves. Against that, 64-row tiles sweep the queries once per 64
// rows. Kernel time, wide / 64-row workgroups (wide workgroups in the launch;
// H: query / kv heads; G: packed rows):
//   D=128  H=8/8 S=4096        (256; G = 192)   21 /   17 us
//          B=2 H=32/32 S=4096  (384; G = 192)   65 /   48 us
//          H=16/16 S=16384     (384; G = 384)  100 /   79 us
//          H=8/8 S=65536       (384; G = 768)  331 /  278 us
//          H=16/4 S=65536      (384; G = 768)  700 /  543 us
//          B=8 H=32/32 S=2048  (512; G =  45)   69 /   59 us
//          H=32/4 S=4096       (G = 192)        55 /   34 us
//          B=4 H=32/32 S=8192  (512; G = 273)  200 /  219 us
//          H=16/16 S=32768     (G = 546)       198 /  209 us
//          H=16/16 S=65536     (704; G = 768)  537 /  513 us
//          B=4 H=32/8  S=32768 (576; G = 546) 1712 / 1720 us
//          B=2 H=32/32 S=65536 (2816; G = 768) 2051 / 2520 us
//   D=64   H=8/8 S=2100        (G = 138)       9.4 /  8.2 us
//          H=8/8 S=4096        (G = 192)      10.2 / 10.8 us
//          H=4/4 S=8192        (G = 273)      11.7 / 12.6 us
//          H=16/16 S=3000      (G = 165)      12.0 / 12.0 us
//          B=8 H=32/32 S=2048  (512; G =  45)   33 /   29 us
//          H=8/8 S=16384       (768; G = 384)   32 /   27 us
//          H=16/16 S=16384     (768; G = 384)   51 /   45 us
//          B=4 H=32/32 S=8192  (768; G = 273)  129 /  128 us
//          H=8/8 S=32768       (G = 546)        67 /   71 us
//          H=12/12 S=65536     (792; G = 768)  227 /  242 us
// So: the 64-row workgroups for launches of fewer than two wide workgroups
// per CU (up to 768 rows, the most that was measured), and where the documents'
// rows padded to wide tiles are at least 1.75 times those padded to 64 (one
// document of up to 64 rows, packed ones with many short among them). At D = 64
// the line is a rough one: it misses 15% at S = 16384 and gives away 6% at S =
// 4096 and 8192 with few heads. Packed documents of up to 768 rows take them
// too where their sweeps are cut (plan_chunks): the pieces are made for them
// (over 190 such batches 0.86 times the wide kernel's time on average, with
// gsum_kernel; at most 1.07 times). Uncut ones keep the wide workgroups (eight
// documents of 4096, H=32/32 D=128: 164 / 222 us).
constexpr int kNarrowWaves = 4, kNarrowBQ = 32, kNarrowMaxRows = 768;

template <int D>
bool narrow_glob(const BwdArgs& a) {
  constexpr int kWide = 16 * kDkdvGlobWaves<D> * kDkdvKB, kNarrow = 16 * kNarrowWaves;
  int64_t items = 0, wide = 0, narrow = 0;
  int most = 0;
  for (int d = 0; d < a.docs.n; ++d) {
    const int rows = doc_rows(a.docs.len[d], a.docs.W[d], a.docs.rpb[d]);
    const int chunks = num_chunks(a.docs.len[d], a.chunk_len);
    const int tiles = (rows + kWide - 1) / kWide;
    most = std::max(most, rows);
    items += (int64_t)tiles * chunks * a.B * a.Hkv;
    wide += (int64_t)tiles * kWide;
    narrow += (int64_t)(rows + kNarrow - 1) / kNarrow * kNarrow;
  }
  const bool few = a.docs.n > 1 ? !a.even : items < 2 * a.cus;
  return D <= 128 && ((few && most <= kNarrowMaxRows) || 4 * wide >= 7 * narrow);
}

// Below D = 128 a local workgroup takes 128 keys, 32 a wave; where that gives
// no more than one workgroup per CU it takes 64, 16 a wave: the chip has room
// for twice the workgroups, and each is shorter. Local kernel, 128 / 64 keys
// (128-key workgroups in the launch): B=2 H=16/2 S=2048 D=64 (64) 39 / 21.5
// us, H=16/2 S=1000 (16) 34 / 16.6, H=12 S=1000 (96) 9.7 / 7.0, H=8 S=4096
// (256) 12.3 / 10.4, H=16/4 S=8192 (256) 29 / 24, H=12 S=8192 (768) 22.7 / 26.5.
template <int D>
bool half_local_tiles(const BwdArgs& a) {
  if (kDkdvLocalKB<D> == 1) return false;
  constexpr int kKeys = 16 * kDkdvLocalWaves * kDkdvLocalKB<D>;
  int64_t items = 0;
  for (int d = 0; d < a.docs.n; ++d) items += (a.docs.len[d] + kKeys - 1) / kKeys;
  return items * a.B * a.Hkv <= a.cus;
}

template <typename T, int D>
hipError_t launch_TD(const BwdArgs& a, hipStream_t st) {
  constexpr bool kF32 = sizeof(T) == 4;
  // work items per document: query tiles (dQ), global-row tiles x query
  // chunks (global dK/dV), key tiles (local dK/dV), each of its kernel's
  // workgroup size
  BwdArgs aq = a, ag = a, al = a;
  constexpr int kQM = kF32 ? 16 * kF32Waves : D > 128 ? 16 * kWideWaves : 16 * kDqWaves * kDqQB;  // dQ queries per workgroup
  set_items(aq.docs, [&](int d) { return (a.docs.len[d] + kQM - 1) / kQM; });
  const bool narrow = !kF32 && narrow_glob<D>(a);
  const int kGK = kF32     ? 16 * kF32Waves
                  : narrow ? 16 * kNarrowWaves
                           : 16 * kDkdvGlobWaves<D> * kDkdvKB;  // rows per workgroup
  const bool half_local = !kF32 && half_local_tiles<D>(a);
  const int kLK = kF32 ? 16 * kF32Waves : 16 * kDkdvLocalWaves * (half_local ? 1 : kDkdvLocalKB<D>);
  set_items(ag.docs, [&](int d) {
    return (doc_rows(a.docs.len[d], a.docs.W[d], a.docs.rpb[d]) + kGK - 1) / kGK *
           num_chunks(a.docs.len[d], a.chunk_len);
  });
  set_items(al.docs, [&](int d) { return (a.docs.len[d] + kLK - 1) / kLK; });
  const int nq = aq.docs.item0[a.docs.n], ng = ag.docs.item0[a.docs.n];
  const int nl = al.docs.item0[a.docs.n];
  // one document, D = 128 and a head count that is not a multiple of 8: the
  // dQ and local dK/dV kernels run in the XCD-aware order (as the forward)
  const bool xq = !kF32 && D == 128 && a.docs.n == 1 && (a.B * a.Hq) % 8 != 0;
  const bool xl = !kF32 && D == 128 && a.docs.n == 1 && (a.B * a.Hkv) % 8 != 0;
  aq.xcd_nt = xq ? nq : 0;
  al.xcd_nt = xl ? nl : 0;
  const int gq = xq ? xcd_grid(a.B * a.Hq, nq) : nq * a.B * a.Hq;
  const int gl = xl ? xcd_grid(a.B * a.Hkv, nl) : nl * a.B * a.Hkv;
  const dim3 qgrid(gq), ggrid(ng * a.B * a.Hkv), lgrid(gl);
  by_docs(aq, [&](const auto& x) {
    constexpr int ND = std::decay_t<decltype(x)>::kDocs;
    if constexpr (kF32)
      hipLaunchKernelGGL((dq_f32_kernel<D, ND>), qgrid, dim3(64 * kF32Waves), 0, st, x);
    else
      dispatch_direct<ND>(a.direct, [&](auto dir) {
        constexpr bool DIR = decltype(dir)::value;
        if constexpr (D > 128)
          hipLaunchKernelGGL((dq_wide_kernel<T, D, ND, DIR>), qgrid, dim3(64 * kWideWaves), 0, st, x);
        else
          hipLaunchKernelGGL((dq2_kernel<T, D, kDqWaves, kDqQB, kDqBN, kDqWPE, ND, DIR>), qgrid,
                             dim3(64 * kDqWaves), 0, st, x);
      });
  });
  by_docs(ag, [&](const auto& x) {
    constexpr int ND = std::decay_t<decltype(x)>::kDocs;
    if constexpr (kF32) {
      hipLaunchKernelGGL((dkdv_f32_kernel<D, true, ND>), ggrid, dim3(64 * kF32Waves), 0, st, x);
    } else {
      if constexpr (D <= 128) {  // (at D = 256 the one geometry has 64 rows)
        if (narrow) {
          hipLaunchKernelGGL((dkdv2_kernel<T, D, true, kNarrowWaves, kDkdvKB, kNarrowBQ, ND>),
                             ggrid, dim3(64 * kNarrowWaves), 0, st, x);
          return;
        }
      }
      hipLaunchKernelGGL((dkdv2_kernel<T, D, true, kDkdvGlobWaves<D>, kDkdvKB, kDkdvGlobBQ<D>, ND>),
                         ggrid, dim3(64 * kDkdvGlobWaves<D>), 0, st, x);
    }
  });
  if (a.nchunk > 1) {
    BwdArgs as = a;
    set_items(as.docs, [&](int d) {
      return (doc_rows(a.docs.len[d], a.docs.W[d], a.docs.rpb[d]) * (2 * D / 4) + 255) / 256;
    });
    by_docs(as, [&](const auto& x) {
      constexpr int ND = std::decay_t<decltype(x)>::kDocs;
      hipLaunchKernelGGL((gsum_kernel<D, ND>), dim3(x.docs.item0[x.docs.n] * a.B * a.Hkv),
                         dim3(256), 0, st, x);
    });
  }
  if (a.dalpha) hipLaunchKernelGGL((dalpha_kernel<T, D>), dim3(a.Hkv), dim3(1024), 0, st, a);
  by_docs(al, [&](const auto& x) {
    constexpr int ND = std::decay_t<decltype(x)>::kDocs;
    if constexpr (kF32)
      hipLaunchKernelGGL((dkdv_f32_kernel<D, false, ND>), lgrid, dim3(64 * kF32Waves), 0, st, x);
    else if (half_local)
      hipLaunchKernelGGL((dkdv2_kernel<T, D, false, kDkdvLocalWaves, 1, kDkdvLocalBQ, ND>), lgrid,
                         dim3(64 * kDkdvLocalWaves), 0, st, x);
    else
      hipLaunchKernelGGL(
          (dkdv2_kernel<T, D, false, kDkdvLocalWaves, kDkdvLocalKB<D>, kDkdvLocalBQ, ND>), lgrid,
          dim3(64 * kDkdvLocalWaves), 0, st, x);
  });
  return hipGetLastError();
}

template <typename T>
hipError_t launch_T(int D, const BwdArgs& a, hipStream_t st) {
  switch (D) {
    case 32: return launch_TD<T, 32>(a, st);
    case 64: return launch_TD<T, 64>(a, st);
    case 128: return launch_TD<T, 128>(a, st);
    case 256: return launch_TD<T, 256>(a, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace

ChunkPlan plan_chunks(int D, int B, int Hq, int Hkv, int n, const int* len,
                      const int* W, const int* rpb, int cus) {
  // Query chunks of the global-row kernel: each document's query range is
  // cut into chunks of chunk_len queries (a multiple of 64), one
  // workgroup per (row tile, chunk). More chunks balance the uneven
  // workgroups better (a late row tile sees only the last queries) and
  // shorten the last round; each chunk costs a partial dK/dV of its rows,
  // written once and summed once by gsum_kernel. Measured on gfx950 over
  // 1-48 chunks (training step, 2 sweeps): the best counts fill the kernel's
  // resident slots about 1.5 times over (the device's CUs, one 12-wave
  // workgroup per CU at D = 128, two 8-wave ones below) until chunks would
  // exceed about 6144 queries, from which on 6144-query chunks keep the
  // balance. On the 256-CU MI355X:
  //   B=1 H=16 D=128 S=131072: 22 chunks (16 and 32 within 0.6%)
  //   B=1 H=12 D=64 S=8192 / 32768 / 131072: 22 / 13 / 22 chunks
  //   B=2 H=32 D=128 S=4096: 6 (the previous rule's 16 was 12% slower)
  //   B=1 H=8 D=64 S=16384: 32 (64 was 10% slower)
  // (D = 256: 64 rows per 4-wave workgroup, two workgroups per CU by their
  // 66 KB of LDS)
  const int rows = D > 128    ? 16 * kDkdvGlobWaves<256> * kDkdvKB
                   : D == 128 ? 16 * kDkdvGlobWaves<128> * kDkdvKB
                              : 16 * kDkdvGlobWaves<64> * kDkdvKB;
  const int slots = (cus > 0 ? cus : 256) * (D == 128 ? 1 : 2);
  int64_t row_tiles = 0;
  int max_len = 1;
  for (int d = 0; d < n; ++d) {
    row_tiles += (doc_rows(len[d], W[d], rpb[d]) + rows - 1) / rows;
    if (len[d] > max_len) max_len = len[d];
  }
  const int64_t base = row_tiles * B * Hkv;
  ChunkPlan c{};
  if (n > 1) {
    // Several documents: pieces of about one length, so that a long document
    // gets more of them than a short one. The sweeps (queries that see a 64-row
    // tile, over the tiles, batches and kv heads) are cut into about three
    // pieces per CU, the 64-row kernel's resident workgroups, unless the longest
    // is at most 0.6 of a CU's load: those fill the chip evenly as they are, and
    // pieces would only add partials. Global-row kernel and gsum_kernel over 226
    // batches (1 to 131072 tokens, 2 to 200 documents, 1 to 32 kv heads) against
    // the same number of chunks for every document, where the longest
    // document's workgroups run alone at the end: 0.81 times the time on
    // average (1.5, 2 and 4 pieces per CU 0.87, 0.83 and 0.83; always cut
    // 0.82), at most 1.17 times, 3.4% of the step (16 documents of 1 to 9001
    // tokens, H=16/4 D=128: 244 -> 91 us; six of 5000, H=32/32 D=128: uncut 204
    // us, cut 232).
    double sweeps = 0;
    int longest = 0;
    for (int d = 0; d < n; ++d) {
      const int g = doc_rows(len[d], W[d], rpb[d]);
      longest = std::max(longest, len[d] - W[d]);
      for (int t = 0; t < g; t += 64)
        sweeps += std::max(0, len[d] - (t / rpb[d] + 1) * W[d]);
    }
    sweeps *= (double)B * Hkv / (cus > 0 ? cus : 256);  // per CU
    c.even = longest <= 0.6 * sweeps;
    const double L = c.even ? 6144.0 : std::min(std::max(sweeps / 3, 64.0), 6144.0);
    c.chunk_len = chunk_len_for((int)L, 1);
    for (;;) {
      c.part_rows = 0;
      for (int d = 0; d < n; ++d)
        c.part_rows += (int64_t)num_chunks(len[d], c.chunk_len) * doc_rows(len[d], W[d], rpb[d]);
      if (c.part_rows < ((int64_t)1 << 31)) break;  // pofs is 32-bit
      c.chunk_len *= 2;
    }
    c.nchunk = num_chunks(max_len, c.chunk_len);
    return c;
  }
  int64_t nc = (3 * slots + 2 * base - 1) / (2 * base);  // 1.5 rounds of workgroups
  const int64_t by_len = (max_len + 6143) / 6144;
  if (nc < by_len) nc = by_len;
  // At least 256 queries a chunk, counted over the heads of the kv group: a
  // workgroup sweeps its chunk once per head of the group, and with few kv
  // heads the chunks are all the workgroups there are. Global-row kernel with
  // 256 queries of each head / of all: B=2 H=16/2 S=2048 D=64 37 / 12 us, B=1
  // H=8/1 S=4096 D=128 51 / 18, H=32/4 S=8192 D=128 95 / 66, H=32/8 S=2000
  // D=128 26 / 11, fp32 H=8/2 S=3000 D=64 67 / 27 us.
  const int grp = Hq / Hkv;
  const int64_t max_nc = ((int64_t)max_len * grp + 255) / 256;
  if (nc > max_nc) nc = max_nc;
  if (nc < 1) nc = 1;
  if (grp > 1) {  // (with one head per kv head 64-query rounding can leave the last chunks empty)
    c.chunk_len = chunk_len_for(max_len, (int)nc);
    nc = num_chunks(max_len, c.chunk_len);
  }
  c.nchunk = (int)nc;
  c.chunk_len = chunk_len_for(max_len, c.nchunk);
  c.part_rows = nc * doc_rows(len[0], W[0], rpb[0]);
  return c;
}

size_t bwd_workspace_layout(int D, int B, int Hq, int Hkv, int S, int64_t part_rows) {
  // -Delta and -lse * log2(e) per query, then the chunk
  // partials
  const size_t delta = (((size_t)B * Hq * S * 4) + 255) / 256 * 256;
  const size_t part = (size_t)part_rows * B * Hkv * 2 * D * 4;
  return 2 * delta + part;
}

bool bwd_tile_config(int dtype, int D, int out[9]) {
  if (dtype < 0 || dtype > 2 || (D != 32 && D != 64 && D != 128 && D != 256)) return false;
  if (dtype == 2) {
    constexpr int w = kF32Waves, r = 16 * kF32Waves, n = kF32BN;
    const int v[9] = {w, r, n, w, r, n, w, r, n};
    for (int i = 0; i < 9; ++i) out[i] = v[i];
  } else if (D == 256) {
    const int v[9] = {kWideWaves,      16 * kWideWaves,                     kWideBN,
                      kDkdvGlobWaves<256>, 16 * kDkdvGlobWaves<256> * kDkdvKB, kDkdvGlobBQ<256>,
                      kDkdvLocalWaves, 16 * kDkdvLocalWaves * kDkdvLocalKB<256>, kDkdvLocalBQ};
    for (int i = 0; i < 9; ++i) out[i] = v[i];
  } else {
    const int gw = D == 128 ? kDkdvGlobWaves<128> : kDkdvGlobWaves<64>;
    const int lkb = D == 128 ? kDkdvLocalKB<128> : kDkdvLocalKB<64>;
    const int v[9] = {kDqWaves,        16 * kDqWaves * kDqQB,        kDqBN,
                      gw,              16 * gw * kDkdvKB,            kDkdvGlobBQ<128>,
                      kDkdvLocalWaves, 16 * kDkdvLocalWaves * lkb,   kDkdvLocalBQ};
    for (int i = 0; i < 9; ++i) out[i] = v[i];
  }
  return true;
}

hipError_t launch_bwd(int dtype, int D, const BwdArgs& args, hipStream_t st) {
  BwdArgs a = args;
  set_divs(a);
  switch (dtype) {
    case 0: return launch_T<f16>(D, a, st);
    case 1: return launch_T<bf16>(D, a, st);
    case 2: return launch_T<float>(D, a, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace cra
