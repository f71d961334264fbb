// Forward: three-phase sqrt(N) attention with one online softmax.
//
// Reference semantics: `_cron_root_attn_fwd_v14_tiled` (core.py:907-1158).
// Per query i (ls = max(0, i-W+1)) the keys are the local window [ls, i]
// (core.py:976-1028) and the global rows -- strided rows s*W < ls
// (core.py:1042-1087) and the relay rows of blocks ending before ls
// (core.py:1097-1142). The global rows arrive packed per block
// (cra_global.hip), so the global set of query i is a prefix of one array and
// both phases are dense MFMA contractions with a mask only on edge tiles
// (the reference streams every relay row for every tile).
// Scores are fp32 dot(q, k) * scale; P is rounded to the input dtype before
// P.V (core.py:1027, 1086, 1141); O = acc / l and LSE = m + ln(l)
// (core.py:1147-1158). Unlike the reference, whose l sums the unrounded P
// (core.py:1028), l sums the rounded P of the 2-byte types.
//
// Mapping: one workgroup = 4 waves = 128 consecutive queries of one (b, h);
// each wave owns 32 queries. K/V tiles of 64 rows (32 for fp32) are staged
// row-major in LDS. S^T = K . Q^T puts a query on lane%16 so
// the per-query softmax state is lane-local; O^T = V^T . P^T consumes P^T
// straight from the S^T registers. Tiles are launched heaviest first (work
// per query grows with i) and consecutive workgroups are different heads of
// the same tile, so each XCD keeps a fixed pair of heads.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "cra_common.hpp"
#include "cra_internal.hpp"

namespace cra {

namespace {

// ---------------------------------------------------------------------------
// fp32 forward: the mapping of fwd2 (below) with every operand split in three
// bf16 pieces (Split): Q in registers, K and V tiles of 32 rows as three
// planes in LDS, staged through registers (the split happens there, once per
// workgroup), P split in registers. 4 waves of 16 QB queries; up to D = 64
// two LDS stages, one barrier per tile. The running maximum is raised lazily
// as in fwd2 (an fp32 P keeps its precision at any magnitude). Bound by
// the matrix core and the splits' VALU work about equally (per wave and 32-key
// tile at D = 64: 96 MFMAs, 1536 cycles, beside about 300 VALU). Against the
// fp32-MFMA kernel before it (V transposed by LDS writes, one stage): H=8
// S=32768 D=64 377 -> 246 us, D=128 963 -> 598 us, S=4096 D=64 45 -> 28 us,
// H=4 S=8192 D=256 153 -> 122 us.
// ---------------------------------------------------------------------------
constexpr float kSumMaxF32 = 32768.f;
constexpr int kF32Waves = 4, kF32BN = 32;
template <int D>
constexpr int kF32QB = D > 128 ? 1 : 2;  // 16-query blocks per wave

template <int D, int QB, bool MASK>
__device__ __forceinline__ void attend_f32(const char* tK, const char* tV, const LaneOffs<D>& lo,
                                           const Split (&qf)[QB][D / 32], f32x4 (&acc)[D / 16][QB],
                                           float (&m_run)[QB], float (&l_run)[QB], float c2, int g,
                                           const TileMask<QB>& mk) {
  using Stage = SplitStage<D, kF32BN, 64 * kF32Waves>;
  using Tile = typename Stage::Tile;
  f32x4 s[2][QB], sl[2][QB];  // sl: the small products (kSmallApart)
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) s[h][qb] = sl[h][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    Split kf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) kf[h] = Stage::row_frag(tK + h * Tile::kBlk16 + lo.row_at(c));
    // consecutive MFMAs go to different accumulators
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          f32x4& s_ = t < kSmallApart<D> ? sl[h][qb] : s[h][qb];
          s_ = mma(s_, kf[h].p[split_a(t)], qf[qb][c].p[split_b(t)]);
        }
  }
  if (kSmallApart<D> > 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) s[h][qb] += sl[h][qb];
  }
  Split pf[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    float pv[8], ps = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (MASK && !mk.ok(16 * h + 4 * g + r, qb)) s[h][qb][r] = -__builtin_huge_valf();
        pv[4 * h + r] = __builtin_amdgcn_exp2f(fmaf(s[h][qb][r], c2, -m_run[qb]));
        ps += pv[4 * h + r];
      }
    if (__any(!(ps <= kSumMaxF32))) {
      float mx = -__builtin_huge_valf();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[h][qb][r]);
      const float m_new = fmaxf(m_run[qb], group_max(mx * c2));
      const float mu = m_new == -__builtin_huge_valf() ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run[qb] - mu);
      l_run[qb] *= alpha;
#pragma unroll
      for (int db = 0; db < D / 16; ++db) acc[db][qb] *= alpha;
      m_run[qb] = m_new;
      ps = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pv[4 * h + r] = __builtin_amdgcn_exp2f(fmaf(s[h][qb][r], c2, -mu));
          ps += pv[4 * h + r];
        }
    }
    l_run[qb] += ps;
    pf[qb] = split8<false>(pv);
  }
#pragma unroll
  for (int db = 0; db < D / 16; db += 2) {
    Split vt[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) vt[e] = Stage::tr_frag(tV + lo.tr_at(db + e));
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          acc[db + e][qb] = mma(acc[db + e][qb], vt[e].p[split_a(t)], pf[qb].p[split_b(t)]);
  }
}

template <int D, int QB, int ND>
__global__ __launch_bounds__(64 * kF32Waves) __attribute__((amdgpu_waves_per_eu(D > 64 ? 1 : 2)))
void fwd_f32_kernel(FwdArgsT<ND> a) {
  constexpr int NW = kF32Waves, BN = kF32BN, kQW = 16 * QB, kBM = NW * kQW;
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
  const int q0 = m0 + wave * kQW;
  const int S = dc.len, W = dc.W;

  const float* qp = static_cast<const float*>(a.q) + b * a.qsb + h * a.qsh + (int64_t)dc.off * a.qss;
  const float* kp = static_cast<const float*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const float* vp = static_cast<const float*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  const GlobRows gr = glob_rows<float, D>(a, dc, b, hk, kp, vp, a.direct);
  const float *gkp = (const float*)gr.k, *gvp = (const float*)gr.v;

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (a.phases & 1) ? (hi - lo_k + BN - 1) / BN : 0;
  const int nglob = (a.phases & 2) ? (gmax + BN - 1) / BN : 0;
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
  if (ntot > 0) load(0);

  LaneOffs<D> lo;
  lo.init(lane);
  Split qf[QB][D / 32];
  int qi[QB];
  float m_run[QB], l_run[QB];
  f32x4 acc[D / 16][QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    qi[qb] = q0 + 16 * qb + l16;
    const int qr = min(qi[qb], S - 1);  // queries past the document are never stored
#pragma unroll
    for (int c = 0; c < D / 32; ++c)
      qf[qb][c] = load_split(qp + (int64_t)qr * a.qss + 32 * c + 8 * g);
    m_run[qb] = -__builtin_huge_valf();
    l_run[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float c2 = a.scale * kLog2e;
  const bool active = q0 < S;
  const int q_last = min(q0 + kQW, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  int glen[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) glen[qb] = glob_prefix(qi[qb], dc);

  auto store = [&](int it) {
    char(&dst)[2][Stage::kBytes] = lds[kStages == 2 ? it & 1 : 0];
    stk.store(dst[0], tid);
    stv.store(dst[1], tid);
  };
  if (ntot > 0) store(0);
  __syncthreads();
  for (int it = 0; it < ntot; ++it) {
    if (it + 1 < ntot) load(it + 1);
    const char(&cur)[2][Stage::kBytes] = lds[kStages == 2 ? it & 1 : 0];
    const bool loc = it >= nglob;
    const int ts = row0(it);
    if (active && (loc ? (ts <= q_last && ts + BN - 1 >= w_lo) : ts < wg_hi)) {
      const bool full = loc ? (ts >= q_last - W + 1 && ts + BN - 1 <= q0) : ts + BN <= wg_lo;
      TileMask<QB> mk;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        mk.hi[qb] = loc ? qi[qb] - ts : glen[qb] - 1 - ts;
        mk.span[qb] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
      }
      if (full)
        attend_f32<D, QB, false>(cur[0], cur[1], lo, qf, acc, m_run, l_run, c2, g, mk);
      else
        attend_f32<D, QB, true>(cur[0], cur[1], lo, qf, acc, m_run, l_run, c2, g, mk);
    }
    if (kStages == 1) __syncthreads();  // every wave is done with this tile
    if (it + 1 < ntot) store(it + 1);
    __syncthreads();
  }

  float* op = static_cast<float*>(a.o) + b * a.osb + h * a.osh + (int64_t)dc.off * a.oss;
  float* lse = a.lse + (int64_t)bh * a.S + dc.off;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l = fmaxf(group_sum(l_run[qb]), 1e-6f);
    if (!active || qi[qb] >= S) continue;
    const float inv = 1.f / l;
    float* orow = op + (int64_t)qi[qb] * a.oss;
#pragma unroll
    for (int db = 0; db < D / 16; ++db)
      *reinterpret_cast<f32x4*>(orow + 16 * db + 4 * g) = acc[db][qb] * inv;
    if (g == 0) lse[qi[qb]] = (m_run[qb] + __builtin_amdgcn_logf(l)) * kLn2;
  }
}

// ---------------------------------------------------------------------------
// fp16/bf16 forward: 4 waves x 32 queries. K/V tiles (64 rows) are
// double-buffered in swizzled LDS, filled with
// global_load_lds while the previous tile is computed, V^T operands come from
// ds_read_b64_tr_b16 on the row-major V tile, each tile is processed in two
// 32-key halves, and the running max is raised only when the rounded
// exponentials of a half against it sum past 2^15 (each P stays <= 2^15;
// O and LSE are exact for any reference max). The normaliser l sums the
// rounded P that the P.V MFMAs use.
// ---------------------------------------------------------------------------
// MFMA steps by which the forward's LDS operand reads run ahead of their use
// (K row fragments and transposed V fragments). Three measured 0.6% faster
// than two and four no better than two (D = 128: 242, 238 and 246 VGPRs, 2
// waves per SIMD either way; D = 64 stays at 168, 3 waves per SIMD).
#ifndef CRA_FWD_PF
#define CRA_FWD_PF 3
#endif

template <typename T, int D, int BN, int QB>
__device__ __forceinline__ void tile_scores(const char* tK, const LaneOffs<D>& lo,
                                            const Frag<T> (&qf)[QB][D / 32], int kc,
                                            f32x4 (&s)[2][QB]) {
  using Tile = SwzTile<D, BN>;
  constexpr int NC = D / 32, NK = 2 * NC;
  // K fragments are read CRA_FWD_PF steps ahead of the MFMAs that use them; fences
  // keep the compiler from moving the reads next to their uses. Step t takes
  // key block t % 2 and D-chunk t / 2, so the four accumulators alternate and
  // each MFMA's accumulator was last written four MFMAs earlier (key block
  // major, two apart, measured 0.5% slower).
  auto k_frag = [&](int t) {
    return Tile::template row_frag_at<T>(tK + (2 * kc + t % 2) * Tile::kBlk16 + lo.row_at(t / 2));
  };
  constexpr int PF = CRA_FWD_PF < NK ? CRA_FWD_PF : NK;
  Frag<T> kf[PF + 1];
#pragma unroll
  for (int t = 0; t < PF; ++t) kf[t] = k_frag(t);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < NK; ++t) {
    if (t + PF < NK) kf[(t + PF) % (PF + 1)] = k_frag(t + PF);
    const int h = t % 2, c = t / 2;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      if (c == 0) s[h][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      s[h][qb] = mma(s[h][qb], kf[t % (PF + 1)], qf[qb][c]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// O^T += V^T . P^T for 32-key half kh: transposed V fragments read
// CRA_FWD_PF steps ahead of the MFMAs that use them.
template <typename T, int D, int BN, int QB>
__device__ __forceinline__ void pv_half(const char* tV, int kh, const LaneOffs<D>& lo,
                                        const Frag<T> (&pf)[QB], f32x4 (&acc)[D / 16][QB]) {
  using Tile = SwzTile<D, BN>;
  constexpr int NDB = D / 16;
  auto tr_v = [&](int db) {
    const char* pa = tV + (2 * kh) * Tile::kBlk16 + lo.tr_at(db);
    return Tile::template tr_frag_at<T>(pa, pa + Tile::kBlk16);
  };
  constexpr int PF = CRA_FWD_PF < NDB ? CRA_FWD_PF : NDB;
  Frag<T> vt[PF + 1];
#pragma unroll
  for (int db = 0; db < PF; ++db) vt[db] = tr_v(db);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    if (db + PF < NDB) vt[(db + PF) % (PF + 1)] = tr_v(db + PF);
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) acc[db][qb] = mma(acc[db][qb], vt[db % (PF + 1)], pf[qb]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Largest sum of a half's 32 rounded exponentials accepted against the
// running maximum: each term is then at most 2^15 and finite in fp16.
constexpr float kSumMax = 32768.f;

// All-ones A operand: ones . P^T puts the sum over the 32 keys of each query
// (column of P^T) in all four of that query's lanes' result rows.
template <typename T>
__device__ __forceinline__ Frag<T> ones_frag() {
  Frag<T> f;
  const uint32_t w = sizeof(T) == 2 ? (std::is_same<T, bf16>::value ? 0x3f803f80u : 0x3c003c00u)
                                    : 0u;
  f.w[0] = make_uint4(w, w, w, w);
  return f;
}

// Sum of the rounded P of a 32-key half for each query, on the matrix core
// (one MFMA in place of four v_dot2 per lane plus a cross-lane sum).
template <typename T>
__device__ __forceinline__ float half_sum(const Frag<T>& pk, const Frag<T>& one) {
  return mma(f32x4{0.f, 0.f, 0.f, 0.f}, one, pk)[0];
}

// Exponentials of one 32-key half (8 per lane and query block) against the
// running maximum, rounded to the input type, and the sum of the rounded
// values over the half's 32 keys (the P.V operand and its normaliser).
template <typename T, bool MASK, int QB>
__device__ __forceinline__ void half_exp(f32x4 (&s)[2][QB], int kc, int qb, float c2, float m,
                                         int g, const TileMask<QB>& mk, const Frag<T>& one,
                                         Frag<T>& pk, float& ps) {
  float pv[8];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (MASK && !mk.ok(32 * kc + 16 * h + 4 * g + r, qb)) s[h][qb][r] = -__builtin_huge_valf();
      pv[4 * h + r] = __builtin_amdgcn_exp2f(fmaf(s[h][qb][r], c2, -m));
    }
  pk = pack8<T>(pv);
  ps = half_sum(pk, one);
}

// Raise the running maximum of query block qb to this half's maximum,
// rescale its accumulators and redo the half's exponentials. Taken for the
// first visible keys and whenever a score exceeds the running maximum by
// enough to push a sum of 8 rounded terms past kSumMax (inf and NaN sums
// included).
template <typename T, int D, int QB>
__device__ __forceinline__ void half_rescale(f32x4 (&s)[2][QB], int qb, float c2,
                                             f32x4 (&acc)[D / 16][QB], float (&m_run)[QB],
                                             float (&l_run)[QB], const Frag<T>& one, Frag<T>& pk,
                                             float& ps) {
  float mx = -__builtin_huge_valf();
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[h][qb][r]);
  const float m_new = fmaxf(m_run[qb], group_max(mx * c2));
  // Until a query's first visible key its accumulators and l are zero; the
  // whole wave's first rescale (its first tile) has nothing to scale.
  if (!__all(m_run[qb] == -__builtin_huge_valf())) {
    const float alpha =
        m_run[qb] == -__builtin_huge_valf() ? 0.f : __builtin_amdgcn_exp2f(m_run[qb] - m_new);
    l_run[qb] *= alpha;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db][qb] *= alpha;
  }
  m_run[qb] = m_new;
  const float mu = m_new == -__builtin_huge_valf() ? 0.f : m_new;
  float pv[8];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) pv[4 * h + r] = __builtin_amdgcn_exp2f(fmaf(s[h][qb][r], c2, -mu));
  pk = pack8<T>(pv);
  ps = half_sum(pk, one);
}

// One BN-key tile for the wave's 32 queries, in 32-key halves. The online
// softmax keeps a lazily raised running maximum: exponentials are taken
// against it first and the maximum is recomputed only when their sum says a
// term got too large. Program order puts the next half's score MFMAs and the
// previous half's PV MFMAs beside each half's exponentials, in one basic
// block, so matrix and vector work can overlap.
template <typename T, int D, int BN, bool MASK>
__device__ __forceinline__ void attend_tile2(const char* tK, const char* tV, const LaneOffs<D>& lo,
                                             const Frag<T> (&qf)[2][D / 32],
                                             f32x4 (&acc)[D / 16][2], float (&m_run)[2],
                                             float (&l_run)[2], float c2, int g,
                                             const TileMask<2>& mk, const Frag<T>& one) {
  using Tile = SwzTile<D, BN>;
  constexpr int kHalves = BN / 32;
  f32x4 s[kHalves][2][2];
  tile_scores<T, D, BN, 2>(tK, lo, qf, 0, s[0]);
  Frag<T> pf[2];
#pragma unroll
  for (int kc = 0; kc < kHalves; ++kc) {
    Frag<T> pn[2];
    float ps[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
      half_exp<T, MASK, 2>(s[kc], kc, qb, c2, m_run[qb], g, mk, one, pn[qb], ps[qb]);
    if (kc > 0) pv_half<T, D, BN, 2>(tV, kc - 1, lo, pf, acc);  // beside this half's exponentials
    if (kc + 1 < kHalves) tile_scores<T, D, BN, 2>(tK, lo, qf, kc + 1, s[kc + 1]);
    // one branch for both query blocks (a branch each measured 0.5% slower:
    // forward kernel at H=16 S=131072 D=128 1207 against 1201 us, at H=12
    // S=32768 D=64 87.2 against 86.5 us)
    if (__any(!(ps[0] <= kSumMax) || !(ps[1] <= kSumMax))) {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        if (__any(!(ps[qb] <= kSumMax)))
          half_rescale<T, D, 2>(s[kc], qb, c2, acc, m_run, l_run, one, pn[qb], ps[qb]);
    }
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      l_run[qb] += ps[qb];
      pf[qb] = pn[qb];
    }
  }
  pv_half<T, D, BN, 2>(tV, kHalves - 1, lo, pf, acc);
}

// One 32-key half kc of a masked tile, for tiles whose other half has no
// key visible to any of the wave's queries (window and prefix edges).
template <typename T, int D, int BN>
__device__ __forceinline__ void attend_half(const char* tK, const char* tV, int kc,
                                            const LaneOffs<D>& lo, const Frag<T> (&qf)[2][D / 32],
                                            f32x4 (&acc)[D / 16][2], float (&m_run)[2],
                                            float (&l_run)[2], float c2, int g,
                                            const TileMask<2>& mk, const Frag<T>& one) {
  using Tile = SwzTile<D, BN>;
  f32x4 s[2][2];
  tile_scores<T, D, BN, 2>(tK, lo, qf, kc, s);
  float ps[2];
  Frag<T> pf[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
    half_exp<T, true, 2>(s, kc, qb, c2, m_run[qb], g, mk, one, pf[qb], ps[qb]);
  if (__any(!(ps[0] <= kSumMax) || !(ps[1] <= kSumMax))) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
      if (__any(!(ps[qb] <= kSumMax)))
        half_rescale<T, D, 2>(s, qb, c2, acc, m_run, l_run, one, pf[qb], ps[qb]);
  }
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) l_run[qb] += ps[qb];
  pv_half<T, D, BN, 2>(tV, kc, lo, pf, acc);
}

// NW waves of 32 queries share each K/V tile of BN = 64 rows (2 x 32 KB
// double buffer at D = 128); at least 2 waves per SIMD at D = 128 (240
// VGPRs), 3 below it (168 VGPRs at D = 64, where the compiler's own choice
// of 174 allowed only 2: the D = 64 forward is 8% faster at 3). PH selects the key
// phases (bit 0 local window, bit 1 global rows) at compile time, so the
// phase-restricted launches are kernels of their own in a trace.
template <int D>
using FwdStage = char[2][SwzTile<D, 64>::kBytes];  // K and V tiles of one pipeline stage

// One work item (a 128-query tile of one (b, h); items numbered heaviest
// first, consecutive items on different heads) with its LDS stages.
template <typename T, int D, int NW, int PH, int ND, bool DIR>
__device__ __forceinline__ void fwd2_item(const FwdArgsT<ND>& a, const int item, FwdStage<D>& stage0,
                                          FwdStage<D>& stage1) {
  constexpr int BN = 64;
  using Tile = SwzTile<D, BN>;
  constexpr int kQW = 32, kBM = NW * kQW, kBN = BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const QHead hd = q_head(a, item);
  const Doc dc = find_doc(a.docs, hd.rest);
  const int bh = hd.bh, b = hd.b, h = hd.h, hk = hd.hk;
  const int tile = (dc.len + kBM - 1) / kBM - 1 - dc.item;  // heaviest first
  const int m0 = tile * kBM;
  const int q0 = m0 + wave * kQW;
  const int S = dc.len, W = dc.W;

  const T* qp = static_cast<const T*>(a.q) + b * a.qsb + h * a.qsh + (int64_t)dc.off * a.qss;
  const T* kp = static_cast<const T*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const T* vp = static_cast<const T*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  float* lse = a.lse + (int64_t)bh * a.S + dc.off;
  const GlobRows gr = glob_rows<T, D>(a, dc, b, hk, kp, vp, DIR);

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (PH & 1) ? (hi - lo_k + kBN - 1) / kBN : 0;
  // Global tiles come first: every workgroup of the head reads them, so the
  // first fill (issued before anything can hide it) is an L2 hit, and the
  // cold local rows are fetched while global tiles are computed. The local
  // window is then walked from its highest key tile down: the workgroup of
  // the next lower query tile (launched next for this head) walks down the
  // same keys one or two tiles behind and finds them in L2 (the forward's HBM
  // reads drop from 1.32 to 1.14 times the compulsory bytes).
  const int nglob = (PH & 2) ? (gmax + kBN - 1) / kBN : 0;
  const int ntot = nloc + nglob;

  // Buffer resources over the rows this workgroup may read (local rows below
  // hi, global rows below gmax): loads past them return zeros. 32-bit
  // offsets, uniform bases.
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
  Frag<T> qf[2][D / 32];
  int qi[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    qi[qb] = q0 + 16 * qb + l16;
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
      if (qi[qb] < S)
        qf[qb][c] = lds_frag_row<T>(qp + (int64_t)qi[qb] * a.qss + 32 * c + 8 * g);
      else
        qf[qb][c].w[0] = make_uint4(0, 0, 0, 0);
    }
  }
  const float c2 = a.scale * kLog2e;
  float m_run[2] = {-__builtin_huge_valf(), -__builtin_huge_valf()};
  float l_run[2] = {0.f, 0.f};
  f32x4 acc[D / 16][2];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) acc[db][0] = acc[db][1] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = q0 < S;
  const int q_last = min(q0 + kQW, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  const int glen[2] = {glob_prefix(qi[0], dc), glob_prefix(qi[1], dc)};

  const Frag<T> one = ones_frag<T>();
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
    TileMask<2> mk;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      mk.hi[qb] = loc ? qi[qb] - ts : glen[qb] - 1 - ts;
      mk.span[qb] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
    }
    if (work) {
      // keys of the tile visible to some query of the wave: [vis_lo, vis_hi]
      const int vis_lo = loc ? w_lo - ts : 0;
      const int vis_hi = loc ? q_last - ts : wg_hi - 1 - ts;
      const bool half0 = vis_lo <= 31, half1 = vis_hi >= 32;
      if (full)
        attend_tile2<T, D, BN, false>(tK, tV, lo, qf, acc, m_run, l_run, c2, g, mk, one);
      else if (half0 && half1)
        attend_tile2<T, D, BN, true>(tK, tV, lo, qf, acc, m_run, l_run, c2, g, mk, one);
      else
        attend_half<T, D, BN>(tK, tV, half0 ? 0 : 1, lo, qf, acc, m_run, l_run, c2, g, mk, one);
    }
  };
  for (int it = 0; it < ntot; it += 2) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 < ntot) step(std::integral_constant<int, 1>{}, it + 1);
  }

  T* op = static_cast<T*>(a.o) + b * a.osb + h * a.osh + (int64_t)dc.off * a.oss;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const float l = l_run[qb];  // each lane holds its query's whole sum
    if (!active || qi[qb] >= S) continue;
    // O is rounded to the 2-byte type: the reciprocal's 1-ulp error is invisible
    const float inv = __builtin_amdgcn_rcpf(fmaxf(l, 1e-6f));
    T* orow = op + (int64_t)qi[qb] * a.oss;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      T e[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) e[r] = from_f32<T>(acc[db][qb][r] * inv);
      *reinterpret_cast<uint2*>(orow + 16 * db + 4 * g) = *reinterpret_cast<const uint2*>(e);
    }
    if (g == 0)
      lse[qi[qb]] = (m_run[qb] + __builtin_amdgcn_logf(fmaxf(l, 1e-6f))) * kLn2;
  }
}

// Two pipeline stages as separate LDS objects, each selected at compile
// time: the compiler can then tell the fill of one stage from reads of the
// other and does not wait for the fill before those reads.
template <typename T, int D, int NW, int PH, int ND, bool DIR = false>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 3)))
void fwd2_kernel(FwdArgsT<ND> a) {
  __shared__ __attribute__((aligned(1024))) FwdStage<D> stage0;
  __shared__ __attribute__((aligned(1024))) FwdStage<D> stage1;
  int item = (int)blockIdx.x;
  if (a.xcd_nt > 0) {
    item = xcd_item(item, a.B * a.Hq, a.xcd_nt);
    if (item < 0) return;  // padding block
  }
  fwd2_item<T, D, NW, PH, ND, DIR>(a, item, stage0, stage1);
}

// Persistent form (use_persistent; the reference's work-queue kernel,
// core.py:711-900): a grid of at most one round of resident workgroups, each
// taking items in order (heaviest first) from a counter in device memory
// that the caller zeroes, until none is left. Every workgroup ends once the
// counter passes the item count.
template <typename T, int D, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 3)))
void fwd2_persistent_kernel(FwdArgsT<1> a) {
  __shared__ __attribute__((aligned(1024))) FwdStage<D> stage0;
  __shared__ __attribute__((aligned(1024))) FwdStage<D> stage1;
  __shared__ int next_item;
  const int n_items = a.docs.item0[a.docs.n] * a.B * a.Hq;
  for (;;) {
    if (threadIdx.x == 0) next_item = atomicAdd(a.work_counter, 1);
    __syncthreads();  // also: every wave is done with the previous item's LDS tiles
    const int item = next_item;
    __syncthreads();  // read before the next overwrite
    if (item >= n_items) break;
    fwd2_item<T, D, NW, 3, 1, false>(a, item, stage0, stage1);
  }
}

// fp16/bf16 forward at head dim 256: 4 waves of 16 queries (two blocks per
// wave would hold 192 registers of accumulators and Q operands), 32-key tiles.
// K and V are staged in turn, one tile of each in LDS: while a tile's scores
// and softmax are computed its V is on the way, and the next tile's K during
// P.V, so 32 KB of LDS per workgroup hide the fills and three workgroups (3
// waves per SIMD at 168 VGPRs) share a CU. Bound by LDS reads: a K or V
// fragment serves one MFMA, which caps MFMA-busy at about 60%.
//
// The softmax is the plain online one: the maximum is raised with every tile
// (a query's largest P is exactly 1), l sums the unrounded P and O is divided
// by it. fwd2's lazy maximum, sum of the rounded P and reciprocal would be 10%
// faster here and put O and the gradients 2% farther from fp64 (B=1 H=8/4
// S=8191 bf16 training step: relative error 3.53e-3 against 3.45e-3).
//
// B=1 H=8 S=32768 bf16: 234 us (514 effective TFLOP/s; 211 with the lazy
// maximum); with tiles through registers and V stored transposed by 2-byte
// LDS writes it took 470 us.
constexpr int kWideWaves = 4, kWideBN = 32;

// Softmax of a 32-key tile: raises the maximum, rescales l and O^T where it
// rose and rounds P to the input type. l is the lane's own share of the sum.
template <typename T, int D, bool MASK>
__device__ __forceinline__ void wide_softmax(const f32x4 (&s)[2][1], float c2, int g,
                                             const TileMask<1>& mk, f32x4 (&acc)[D / 16][1],
                                             float& m_run, float& l_run, Frag<T>& pf) {
  float t[8];  // scores (scaled in masked tiles), then P
  float mx = -__builtin_huge_valf();
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = s[h][0][r];
      if (MASK) x = mk.ok(16 * h + 4 * g + r, 0) ? x * c2 : -__builtin_huge_valf();
      t[4 * h + r] = x;
      mx = fmaxf(mx, x);
    }
  mx = group_max(MASK ? mx : mx * c2);
  const float m_new = fmaxf(m_run, mx);
  const float m_use = m_new == -__builtin_huge_valf() ? 0.f : m_new;  // no visible key yet
  const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    t[i] = __builtin_amdgcn_exp2f(MASK ? t[i] - m_use : fmaf(t[i], c2, -m_use));
    psum += t[i];
  }
  l_run = l_run * alpha + psum;
  m_run = m_new;
  if (__any(alpha != 1.f)) {
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db][0] *= alpha;
  }
  pf = pack8<T>(t);
}

template <typename T, int D, int ND, bool DIR = false>
__global__ __launch_bounds__(64 * kWideWaves) __attribute__((amdgpu_waves_per_eu(3)))
void fwd_wide_kernel(FwdArgsT<ND> a) {
  constexpr int NW = kWideWaves, BN = kWideBN, kBM = 16 * NW;
  using Tile = SwzTile<D, BN>;
  __shared__ __attribute__((aligned(1024))) char sK[Tile::kBytes];
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
  const T* kp = static_cast<const T*>(a.k) + b * a.ksb + hk * a.ksh + (int64_t)dc.off * a.kss;
  const T* vp = static_cast<const T*>(a.v) + b * a.vsb + hk * a.vsh + (int64_t)dc.off * a.vss;
  const GlobRows gr = glob_rows<T, D>(a, dc, b, hk, kp, vp, DIR);

  const int lo_k = max(0, m0 - W + 1);
  const int hi = min(S, m0 + kBM);
  const int gmax = glob_prefix(hi - 1, dc);
  const int nloc = (a.phases & 1) ? (hi - lo_k + BN - 1) / BN : 0;
  const int nglob = (a.phases & 2) ? (gmax + BN - 1) / BN : 0;
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
  // the local window, then the global rows
  auto row0 = [&](int it) { return it < nloc ? lo_k + it * BN : (it - nloc) * BN; };
  auto issue_k = [&](int it) {
    if (it < nloc)
      Fill::load(sK, rk, fk, kbytes, row0(it), wave);
    else
      Fill::load(sK, rgk, fgk, gkb, row0(it), wave);
  };
  auto issue_v = [&](int it) {
    if (it < nloc)
      Fill::load(sV, rv, fv, vbytes, row0(it), wave);
    else
      Fill::load(sV, rgv, fgv, gvb, row0(it), wave);
  };
  if (ntot > 0) issue_k(0);

  LaneOffs<D> lo;
  lo.init(lane);
  Frag<T> qf[1][D / 32];
  const int qi = q0 + l16;
  const int qr = min(qi, S - 1);  // queries past the document are never stored
#pragma unroll
  for (int c = 0; c < D / 32; ++c)
    qf[0][c] = lds_frag_row<T>(qp + (int64_t)qr * a.qss + 32 * c + 8 * g);
  const float c2 = a.scale * kLog2e;
  float m_run[1] = {-__builtin_huge_valf()}, l_run[1] = {0.f};
  f32x4 acc[D / 16][1];
#pragma unroll
  for (int db = 0; db < D / 16; ++db) acc[db][0] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool active = q0 < S;
  const int q_last = min(q0 + 16, S) - 1;
  const int w_lo = max(0, q0 - W + 1);
  const int wg_lo = active ? glob_prefix(q0, dc) : 0;
  const int wg_hi = active ? glob_prefix(q_last, dc) : 0;
  const int glen = glob_prefix(qi, dc);

  for (int it = 0; it < ntot; ++it) {
    wait_vmem();
    __syncthreads();  // K of this tile landed; every wave is done with the previous V
    issue_v(it);
    const bool loc = it < nloc;
    const int ts = row0(it);
    const bool work = active && (loc ? (ts <= q_last && ts + BN - 1 >= w_lo) : ts < wg_hi);
    Frag<T> pf[1];
    if (work) {
      const bool full = loc ? (ts >= q_last - W + 1 && ts + BN - 1 <= q0) : ts + BN <= wg_lo;
      TileMask<1> mk;
      mk.hi[0] = loc ? qi - ts : glen - 1 - ts;
      mk.span[0] = loc ? (unsigned)(W - 1) : 0x7fffffffu;
      f32x4 s[2][1];
      tile_scores<T, D, BN, 1>(sK, lo, qf, 0, s);
      if (full)
        wide_softmax<T, D, false>(s, c2, g, mk, acc, m_run[0], l_run[0], pf[0]);
      else
        wide_softmax<T, D, true>(s, c2, g, mk, acc, m_run[0], l_run[0], pf[0]);
    }
    wait_vmem();
    __syncthreads();  // V landed; every wave is done with this tile's K
    if (it + 1 < ntot) issue_k(it + 1);
    if (work) pv_half<T, D, BN, 1>(sV, 0, lo, pf, acc);
  }

  const float l = fmaxf(group_sum(l_run[0]), 1e-6f);
  if (!active || qi >= S) return;
  T* orow = static_cast<T*>(a.o) + b * a.osb + h * a.osh + (int64_t)(dc.off + qi) * a.oss;
  const float inv = 1.f / l;
#pragma unroll
  for (int db = 0; db < D / 16; ++db) {
    T e[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = from_f32<T>(acc[db][0][r] * inv);
    *reinterpret_cast<uint2*>(orow + 16 * db + 4 * g) = *reinterpret_cast<const uint2*>(e);
  }
  if (g == 0)
    a.lse[(int64_t)bh * a.S + dc.off + qi] = (m_run[0] + __builtin_amdgcn_logf(l)) * kLn2;
}

// Resident workgroups of `kern` on the current device (CUs x workgroups per
// CU), looked up once per device and instantiation: the persistent launch
// serves small problems, where per-call host queries would cost more than
// the kernel.
template <typename T, int D, typename K>
hipError_t resident_slots(K kern, int threads, int* out) {
  constexpr int kMaxDev = 64;
  static std::mutex mu;
  static int cache[kMaxDev] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDev) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!cache[dev]) {
    int per_cu = 0, cus = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    cache[dev] = std::max(1, per_cu) * std::max(1, cus);
  }
  *out = cache[dev];
  return hipSuccess;
}

// Waves per forward workgroup (32 queries each) for 2-byte types. 8 waves
// (256 queries sharing each K/V tile) halve the tile loads per query but
// measured 4% slower at D = 128: the wider local window adds key tiles.
constexpr int kFwdWaves = 4;

// Kernels that take one grid for every order of work: fp32 (every head dim)
// and the 2-byte types at head dim 256. A persistent request runs the same
// tiled kernel there (the work-queue form is built for fwd2 only; the results
// are the same function of the inputs).
hipError_t launch_f32(int D, const FwdArgs& a, hipStream_t st) {
  FwdArgs b = a;
  auto go = [&](auto dc) {
    constexpr int Dc = decltype(dc)::value;
    constexpr int kBM = 16 * kF32Waves * kF32QB<Dc>;
    set_items(b.docs, [&](int d) { return (b.docs.len[d] + kBM - 1) / kBM; });
    const dim3 grid(b.docs.item0[b.docs.n] * b.B * b.Hq);
    by_docs(b, [&](const auto& x) {
      constexpr int ND = std::decay_t<decltype(x)>::kDocs;
      hipLaunchKernelGGL((fwd_f32_kernel<Dc, kF32QB<Dc>, ND>), grid, dim3(64 * kF32Waves), 0, st, x);
    });
  };
  switch (D) {
    case 32: go(std::integral_constant<int, 32>{}); break;
    case 64: go(std::integral_constant<int, 64>{}); break;
    case 128: go(std::integral_constant<int, 128>{}); break;
    case 256: go(std::integral_constant<int, 256>{}); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_wide(const FwdArgs& a, hipStream_t st) {
  constexpr int kBM = 16 * kWideWaves;
  FwdArgs b = a;
  set_items(b.docs, [&](int d) { return (b.docs.len[d] + kBM - 1) / kBM; });
  const dim3 grid(b.docs.item0[b.docs.n] * b.B * b.Hq);
  by_docs(b, [&](const auto& x) {
    constexpr int ND = std::decay_t<decltype(x)>::kDocs;
    dispatch_direct<ND>(a.direct, [&](auto dir) {
      hipLaunchKernelGGL((fwd_wide_kernel<T, 256, ND, decltype(dir)::value>), grid,
                         dim3(64 * kWideWaves), 0, st, x);
    });
  });
  return hipGetLastError();
}

template <typename T>
hipError_t launch_T(int D, const FwdArgs& a, hipStream_t st) {
  if (D == 256) return launch_wide<T>(a, st);
  FwdArgs b = a;
  constexpr int kBM = 32 * kFwdWaves;
  set_items(b.docs, [&](int d) { return (b.docs.len[d] + kBM - 1) / kBM; });
  const dim3 grid(b.docs.item0[b.docs.n] * b.B * b.Hq), block(64 * kFwdWaves);
  // one document, D = 128 and a head count that is not a multiple of 8:
  // XCD-aware order (measured 2.5-5% faster at D = 128; at D = 64, with
  // 45% less HBM traffic, 0.5% faster to 3.6% slower)
  const bool xcd = b.docs.n == 1 && (b.B * b.Hq) % 8 != 0 && D == 128;
  FwdArgs bx = b;
  bx.xcd_nt = xcd ? b.docs.item0[1] : 0;
  const dim3 xgrid(xcd ? xcd_grid(b.B * b.Hq, b.docs.item0[1]) : grid.x);
  hipError_t qerr = hipSuccess;
  auto go = [&](auto dc) {
    constexpr int Dc = decltype(dc)::value;
    by_docs(bx, [&](const auto& x) {
      constexpr int ND = std::decay_t<decltype(x)>::kDocs;
      if constexpr (ND == 1) {
        // one document: also the persistent and the phase-restricted forms
        if (a.work_counter && a.phases == 3) {
          // one round of resident workgroups: CUs x workgroups per CU
          auto kern = fwd2_persistent_kernel<T, Dc, kFwdWaves>;
          int slots = 0;
          qerr = resident_slots<T, Dc>(kern, 64 * kFwdWaves, &slots);
          if (qerr != hipSuccess) return;
          const dim3 pgrid(std::max(1, std::min((int)grid.x, slots)));
          hipLaunchKernelGGL(kern, pgrid, block, 0, st, x);
          return;
        }
        if (a.direct) {
          hipLaunchKernelGGL((fwd2_kernel<T, Dc, kFwdWaves, 3, 1, true>), xgrid, block, 0, st, x);
          return;
        }
        if (a.phases == 1) {
          hipLaunchKernelGGL((fwd2_kernel<T, Dc, kFwdWaves, 1, 1>), xgrid, block, 0, st, x);
          return;
        }
        if (a.phases == 2) {
          hipLaunchKernelGGL((fwd2_kernel<T, Dc, kFwdWaves, 2, 1>), xgrid, block, 0, st, x);
          return;
        }
      }
      hipLaunchKernelGGL((fwd2_kernel<T, Dc, kFwdWaves, 3, ND>), xgrid, block, 0, st, x);
    });
  };
  switch (D) {
    case 32: go(std::integral_constant<int, 32>{}); break;
    case 64: go(std::integral_constant<int, 64>{}); break;
    case 128: go(std::integral_constant<int, 128>{}); break;
    default: return hipErrorInvalidValue;
  }
  if (qerr != hipSuccess) return qerr;
  return hipGetLastError();
}

}  // namespace


bool fwd_tile_config(int dtype, int D, int out[3]) {
  if (dtype < 0 || dtype > 2 || (D != 32 && D != 64 && D != 128 && D != 256)) return false;
  if (D == 256 && dtype != 2) {
    out[0] = kWideWaves; out[1] = 16 * kWideWaves; out[2] = kWideBN;
  } else if (dtype == 2) {
    out[0] = kF32Waves; out[1] = 16 * kF32Waves * (D == 256 ? kF32QB<256> : kF32QB<128>);
    out[2] = kF32BN;
  } else {
    out[0] = kFwdWaves; out[1] = 32 * kFwdWaves; out[2] = 64;
  }
  return true;
}

hipError_t launch_fwd(int dtype, int D, const FwdArgs& args, hipStream_t st) {
  FwdArgs a = args;
  set_divs(a);
  switch (dtype) {
    case 0: return launch_T<f16>(D, a, st);
    case 1: return launch_T<bf16>(D, a, st);
    case 2: return launch_f32(D, a, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace cra
