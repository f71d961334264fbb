// Shared building blocks for the gfx950 kernels: element types, MFMA
// fragments, LDS tile staging and the sqrt(N) index geometry.
//
// MFMA shape used everywhere: v_mfma_f32_16x16x32_{f16,bf16} (fp32 inputs:
// six of them, see Split). Register layout of one wave (64 lanes),
// l16 = lane % 16, g = lane / 16:
//   A operand (16 x 32):  lane holds A[row = l16][k = kappa(g, s)], s = 0..7
//   B operand (32 x 16):  lane holds B[k = kappa(g, s)][col = l16]
//   C result  (16 x 16):  lane holds C[row = 4g + r][col = l16], r = 0..3
// Any bijection kappa works as long as A and B use the same one; a fragment
// loaded from a row-major tile uses kappa(g, s) = 8g + s, a fragment built
// from two C results (rows 16kb0.. and 16kb1..) uses
// kappa(g, s) = 16kb0 + 4g + s (s < 4), 16kb1 + 4g + s - 4 (s >= 4).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cra {

typedef _Float16 f16;
typedef __bf16 bf16;
typedef f16 f16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

static constexpr float kLog2e = 1.4426950408889634f;
static constexpr float kLn2 = 0.6931471805599453f;

// ---------------------------------------------------------------------------
// Eight-element operand fragment, stored as raw 16-byte words.
// ---------------------------------------------------------------------------
template <typename T>
struct Frag {
  static constexpr int kWords = sizeof(T) / 2;  // 16-byte words: 1 (f16/bf16) or 2 (f32)
  uint4 w[kWords];
};

__device__ __forceinline__ f32x4 mma(f32x4 c, const Frag<f16>& a, const Frag<f16>& b) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a.w[0]),
                                                __builtin_bit_cast(f16x8, b.w[0]), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma(f32x4 c, const Frag<bf16>& a, const Frag<bf16>& b) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.w[0]),
                                                 __builtin_bit_cast(bf16x8, b.w[0]), c, 0, 0, 0);
}
// Element conversions (round to nearest even, as torch's .to(dtype)).
template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ f16 from_f32<f16>(float x) { return (f16)x; }
template <>
__device__ __forceinline__ bf16 from_f32<bf16>(float x) { return (bf16)x; }
template <>
__device__ __forceinline__ float from_f32<float>(float x) { return x; }

template <typename T>
__device__ __forceinline__ float to_f32(T x) { return (float)x; }

// Packs eight fp32 values into a fragment of a 2-byte T (pairwise conversions,
// round to nearest even).
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef f16 f16x2 __attribute__((ext_vector_type(2)));
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ Frag<T> pack8(const float (&v)[8]) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  Frag<T> f;
  uint32_t* w = reinterpret_cast<uint32_t*>(f.w);
#pragma unroll
  for (int s = 0; s < 4; ++s)
    w[s] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2 * s], v[2 * s + 1]}, t2));
  return f;
}

// ---------------------------------------------------------------------------
// LDS operand reads.
// ---------------------------------------------------------------------------
// Eight consecutive elements of a row-major tile (16-byte aligned).
template <typename T>
__device__ __forceinline__ Frag<T> lds_frag_row(const T* p) {
  Frag<T> f;
#pragma unroll
  for (int i = 0; i < Frag<T>::kWords; ++i) f.w[i] = reinterpret_cast<const uint4*>(p)[i];
  return f;
}

// Cross-lane helpers on the 4 lane groups of a wave (lanes l, l^16, l^32, l^48).
// The swaps exchange 16- or 32-lane halves of two registers in the VALU: both
// holding x, they come back as x of the lane and of its partner in some order
// (__shfl_xor goes through the LDS pipe, the bound of the kernels that ask for a
// maximum with every tile).
template <int OFF, typename F>
__device__ __forceinline__ float with_partner(float x, F f) {
  static_assert(OFF == 16 || OFF == 32, "lane group distance");
  const uint32_t u = __float_as_uint(x);
  const auto r = OFF == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false)
                           : __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return f(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float group_max(float x) {
  auto mx = [](float a, float b) { return fmaxf(a, b); };
  return with_partner<32>(with_partner<16>(x, mx), mx);
}
__device__ __forceinline__ float group_sum(float x) {
  auto add = [](float a, float b) { return a + b; };
  return with_partner<32>(with_partner<16>(x, add), add);
}

// ---------------------------------------------------------------------------
// gfx950 LDS tiles for 2-byte elements: ROWS x D, row-major, no padding,
// 16-byte chunks XOR-swizzled per row so that 16 lanes reading the same
// chunk of 16 consecutive rows hit 16 different bank groups.
//
// Filled straight from HBM with global_load_lds (16 B per lane; lane i of an
// instruction lands at LDS base + 16 i, so each lane fetches the global chunk
// that belongs at its LDS position). Read either as 16-byte row fragments or
// transposed with ds_read_b64_tr_b16: in each 16-lane group, result lane L,
// slot j receives element L%4 of what source lane 4j + L/4 addressed, so if
// source lane 4j+m addresses row r_j, columns c0+4m .. c0+4m+3, result lane L
// holds column c0+L of rows r_0..r_3 -- a transposed MFMA operand.
// ---------------------------------------------------------------------------
typedef short i16x4 __attribute__((ext_vector_type(4)));
#define CRA_LDS(p) ((__attribute__((address_space(3))) void*)(p))

template <int D, int ROWS>
struct SwzTile {
  static_assert(D == 32 || D == 64 || D == 128 || D == 256, "head dim");
  static constexpr int kCPR = D / 8;      // 16-byte chunks per row
  static constexpr int kRPL = D < 128 ? 128 / D : 1;  // rows sharing one 256-byte line
  static constexpr int kSwz = kCPR < 16 ? kCPR : 16;  // chunks the swizzle permutes
  static constexpr int kBytes = ROWS * D * 2;
  static constexpr int kInstr = ROWS * kCPR / 64;  // 1 KB global_load_lds per instruction

  __device__ __forceinline__ static int swz(int row) { return (row / kRPL) % kSwz; }
  // byte offset of logical 16-byte chunk `chunk` of `row`
  __device__ __forceinline__ static int off(int row, int chunk) {
    return row * (D * 2) + ((chunk ^ swz(row)) << 4);
  }

  // Cooperative fill by NWAVES waves: instruction t = t0 * NWAVES + wave
  // moves tile rows [4t, 4t + 4) (D = 128; 64 / kCPR rows in general), so a
  // wave's successive instructions are kRowStep rows apart. kRowStep is a
  // multiple of the swizzle period, so a lane's in-row chunk is the same for
  // all of its instructions and its offset is one precomputed VGPR plus a
  // wave-uniform row offset. At D = 256 with 4 waves it is half the period:
  // every other instruction takes the chunk with bit 3 flipped (kAlt).
  template <int NWAVES>
  struct Fill {
    static constexpr int kPer = (kInstr + NWAVES - 1) / NWAVES;
    static constexpr int kRowsPerInstr = 64 / kCPR;
    static constexpr int kRowStep = NWAVES * kRowsPerInstr;
    static constexpr bool kAlt = kPer > 1 && D == 256 && kRowStep == 8;
    static_assert(kPer == 1 || kAlt || (kRowStep % kRPL == 0 && (kRowStep / kRPL) % kSwz == 0),
                  "swizzle must repeat every instruction step");

    // Lane's byte offset for its first instruction, relative to tile row 0 of
    // a source whose rows are row_bytes apart.
    __device__ __forceinline__ static int lane_off(int wave, int lane, int row_bytes) {
      const int row = wave * kRowsPerInstr + lane / kCPR;
      return row * row_bytes + (((lane % kCPR) ^ swz(row)) << 4);
    }

    // Tile row i <- source row row0 + i. The buffer resource's record count
    // bounds the rows that may be read: lanes past it load zeros.
    __device__ __forceinline__ static void load(char* lds, __amdgpu_buffer_rsrc_t rsrc,
                                                int lane_off, int row_bytes, int row0,
                                                int wave) {
      // The LDS destination goes to M0: make the wave index visibly uniform,
      // and keep its range visible, or the compiler cannot tell this fill
      // from reads of the other buffer and waits for it before them.
      static_assert((NWAVES & (NWAVES - 1)) == 0, "power-of-two wave count");
      const int w = __builtin_amdgcn_readfirstlane(wave) & (NWAVES - 1);
      int alt = 0;  // byte distance of the flipped chunk
      if (kAlt) {
        const int lane = threadIdx.x & 63;
        alt = (((lane % kCPR) ^ swz(wave * kRowsPerInstr + lane / kCPR)) & 8) ? -128 : 128;
      }
#pragma unroll
      for (int t0 = 0; t0 < kPer; ++t0) {
        const int t = t0 * NWAVES + w;
        if (kInstr % NWAVES != 0 && t >= kInstr) break;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, CRA_LDS(lds + t * 1024), 16,
                                                 lane_off + (row0 + t0 * kRowStep) * row_bytes +
                                                     (kAlt && t0 % 2 ? alt : 0),
                                                 0, 0, 0);
      }
    }
  };

  // 8 consecutive elements (16 B) of `row` starting at column 8*chunk.
  template <typename T>
  __device__ __forceinline__ static Frag<T> row_frag(const char* lds, int row, int chunk) {
    Frag<T> f;
    f.w[0] = *reinterpret_cast<const uint4*>(lds + off(row, chunk));
    return f;
  }

  // The swizzle repeats every 16 rows (16 / kRPL is a multiple of kSwz), so
  // for rows 16*blk + r the offset is blk * 16 * row_bytes + lane_off(r, ..):
  // lane-constant parts are computed once and the block term folds into the
  // instruction's immediate offset.
  static constexpr int kBlk16 = 16 * D * 2;
  // row fragment of row 16*blk + (lane%16), chunk `chunk`
  __device__ __forceinline__ static int row_lane_off(int lane, int chunk) {
    return off(lane & 15, chunk);
  }
  // transposed fragment at column c0: rows 16*blk + 4g + j, this lane's part
  __device__ __forceinline__ static int tr_lane_off(int lane, int c0) {
    const int L = lane & 15, g = lane >> 4;
    const int col = c0 + 4 * (L & 3);
    return off(4 * g + (L >> 2), col >> 3) + ((col & 7) << 1);
  }
  template <typename T>
  __device__ __forceinline__ static Frag<T> row_frag_at(const char* p) {
    Frag<T> f;
    f.w[0] = *reinterpret_cast<const uint4*>(p);
    return f;
  }
  // pa: rows 16*blk_a + ..; pb: rows 16*blk_b + .. (both already offset)
  template <typename T>
  __device__ __forceinline__ static Frag<T> tr_frag_at(const char* pa, const char* pb) {
    i16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)pa);
    i16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)pb);
    Frag<T> f;
    const uint2 ux = __builtin_bit_cast(uint2, x);
    const uint2 uy = __builtin_bit_cast(uint2, y);
    f.w[0] = make_uint4(ux.x, ux.y, uy.x, uy.y);
    return f;
  }

  // Transposed operand: lane (L = lane%16, g = lane/16) gets column c0 + L of
  // rows ra + 4g + j (slots 0..3) and rb + 4g + j (slots 4..7).
  template <typename T>
  __device__ __forceinline__ static Frag<T> tr_frag(const char* lds, int ra, int rb, int c0,
                                                    int lane) {
    const int L = lane & 15, g = lane >> 4;
    const int j = L >> 2, m = L & 3;
    const int col = c0 + 4 * m;
    const int ca = ra + 4 * g + j, cb = rb + 4 * g + j;
    const int oa = off(ca, col >> 3) + ((col & 7) << 1);
    const int ob = off(cb, col >> 3) + ((col & 7) << 1);
    i16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(lds + oa));
    i16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(lds + ob));
    Frag<T> f;
    const uint2 ux = __builtin_bit_cast(uint2, x);
    const uint2 uy = __builtin_bit_cast(uint2, y);
    f.w[0] = make_uint4(ux.x, ux.y, uy.x, uy.y);
    return f;
  }
};

// ---------------------------------------------------------------------------
// fp32 operands on the bf16 matrix core. A float's 24-bit significand is cut
// into three bf16 pieces of 8 bits, x = hi + mid + lo exactly: hi and mid are
// rounded to nearest, so mid is at most 2^-8 and lo 2^-17 of x's power of two
// (below 2^-110 the last bits fall under the smallest bf16). A product takes
// the six piece products down to 2^-16 of it; the three left out are at most
// 2^-24 of |x y| together (2^-28 on average, of either sign), what one fp32
// multiply-add rounds by. (Pieces cut off instead leave up to 2^-21, always
// toward zero: sums of one sign lose it. dq of positive inputs at H=2 S=131072
// D=64: relative error 1.8e-4 against 3.1e-5.) Six 16x16x32 MFMAs (16 cycles
// each) stand for eight 16x16x4 fp32 ones (32 cycles each) and round the sum
// six times where those did eight times. Relative error of o, dq, dk, dv
// against fp64, x 1e-7, fp32 MFMA / this:
//   H=8 S=4096 D=64         3.4, 4.5, 4.7, 4.5 / 2.6, 4.1, 3.7, 3.6
//   H=4 S=4096 D=32         2.9, 4.1, 4.2, 4.3 / 2.2, 3.8, 3.3, 3.3
//   H=4 S=4096 D=128        4.3, 5.4, 5.5, 5.2 / 3.3, 4.7, 4.4, 4.2
//   H=4 S=8192 D=256        5.8, 6.9, 6.9, 6.5 / 2.9, 4.2, 3.9, 3.8
//   H=2 S=131072 D=64       5.8, 6.8, 9.5, 9.3 / 5.2, 6.4, 5.7, 5.4
//   H=32/1 S=131072 D=64    5.8, 6.8, 34, 34   / 5.1, 6.4, 21, 20
// Inputs of one sign keep the fp32 MFMA's error up to D = 128 (H=4 S=4096
// D=128 1.9, 127, 2.0, 1.9 / 1.7, 127, 1.9, 1.7; dq is a difference of
// near-equal sums there) within a fifth, dk at D = 256 within a third.
// An infinite x is kept in the piece that meets only the other operand's hi,
// so that infinity times a number stays infinite.
// ---------------------------------------------------------------------------
struct Split {
  Frag<bf16> p[3];  // hi, mid, lo
};

constexpr float kMaxBf16 = 0x1.fep127f;

// INF: x may be infinite, or finite above the largest bf16 (which is its hi then).
template <bool INF>
__device__ __forceinline__ Split split8(const float (&x)[8]) {
  auto pack = [](const float (&v)[2]) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[0], v[1]}, bf16x2));
  };
  auto value = [](uint32_t u, int i) { return __uint_as_float(i ? u & 0xffff0000u : u << 16); };
  Split f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float v[2], c[2];
    bool inf[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      inf[i] = INF && __builtin_isinf(x[2 * w + i]);
      v[i] = inf[i] ? 0.f : x[2 * w + i];
      c[i] = INF ? __builtin_amdgcn_fmed3f(v[i], -kMaxBf16, kMaxBf16) : v[i];
    }
    const uint32_t h = pack(c);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] -= value(h, i);
    const uint32_t m = pack(v);
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = inf[i] ? x[2 * w + i] : v[i] - value(m, i);
    reinterpret_cast<uint32_t*>(f.p[0].w)[w] = h;
    reinterpret_cast<uint32_t*>(f.p[1].w)[w] = m;
    reinterpret_cast<uint32_t*>(f.p[2].w)[w] = pack(v);
  }
  return f;
}

// Piece pairs of a product, the small ones first.
__device__ __forceinline__ constexpr int split_a(int t) { return t == 0 ? 2 : t == 2 || t == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int split_b(int t) { return t == 1 ? 2 : t == 2 || t == 4 ? 1 : 0; }
// t:      0 1 2 3 4 5
// a, b:   lo.hi hi.lo mid.mid mid.hi hi.mid hi.hi

// Products of the scores and dP that are summed apart from hi.hi and added at
// the end: all but hi.hi at D = 256, whose sums over eight chunks would round 48
// times at full magnitude (now 8). Relative error of o, dq, dk, dv at B=1 H=4
// S=8192: 4.7, 5.9, 5.7, 5.3e-7 in one sum, 2.9, 4.2, 3.9, 3.8e-7 so, for 1-4%
// of the kernels' time; at D = 128 a fourth less error would cost dQ 9%.
template <int D>
constexpr int kSmallApart = D > 128 ? 5 : 0;

// ROWS x D tile of fp32 rows as three planes of SwzTile, filled through
// registers by NT threads: load() issues the reads, store() splits and writes.
template <int D, int ROWS, int NT>
struct SplitStage {
  using Tile = SwzTile<D, ROWS>;
  static constexpr int kBytes = 3 * Tile::kBytes;
  static constexpr int kRowGroups = NT / Tile::kCPR < ROWS ? NT / Tile::kCPR : ROWS;
  static constexpr int kRPT = ROWS / kRowGroups;  // rows per thread
  static_assert(kRowGroups * kRPT == ROWS, "tile/thread mismatch");
  uint4 r[kRPT][2];

  __device__ __forceinline__ void load(const float* base, int64_t row_stride, int row0, int row_hi,
                                       int tid) {
    const int cg = tid % Tile::kCPR, rg = tid / Tile::kCPR;
#pragma unroll
    for (int i = 0; i < kRPT; ++i) {
      const int row = row0 + i * kRowGroups + rg;
      if (rg < kRowGroups && row < row_hi) {
        const uint4* src = reinterpret_cast<const uint4*>(base + (int64_t)row * row_stride + cg * 8);
        r[i][0] = src[0];
        r[i][1] = src[1];
      } else {
        r[i][0] = r[i][1] = make_uint4(0, 0, 0, 0);
      }
    }
  }
  __device__ __forceinline__ void store(char* lds, int tid) const {
    const int cg = tid % Tile::kCPR, rg = tid / Tile::kCPR;
    if (rg >= kRowGroups) return;
    // values above the largest bf16 are rare: tested together
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < kRPT; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(reinterpret_cast<const float*>(r[i])[j]));
    if (__any(mx > kMaxBf16))
      store_split<true>(lds, cg, rg);
    else
      store_split<false>(lds, cg, rg);
  }
  template <bool INF>
  __device__ __forceinline__ void store_split(char* lds, int cg, int rg) const {
#pragma unroll
    for (int i = 0; i < kRPT; ++i) {
      const Split f = split8<INF>(*reinterpret_cast<const float(*)[8]>(&r[i][0]));
      char* dst = lds + Tile::off(i * kRowGroups + rg, cg);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<uint4*>(dst + k * Tile::kBytes) = f.p[k].w[0];
    }
  }

  __device__ __forceinline__ static Split row_frag(const char* p) {
    Split f;
#pragma unroll
    for (int k = 0; k < 3; ++k) f.p[k] = Tile::template row_frag_at<bf16>(p + k * Tile::kBytes);
    return f;
  }
  __device__ __forceinline__ static Split tr_frag(const char* p) {
    Split f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const char* q = p + k * Tile::kBytes;
      f.p[k] = Tile::template tr_frag_at<bf16>(q, q + Tile::kBlk16);
    }
    return f;
  }
};

// Eight floats of a row, split.
__device__ __forceinline__ Split load_split(const float* p) {
  float x[8];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    *reinterpret_cast<uint4*>(&x[4 * i]) = reinterpret_cast<const uint4*>(p)[i];
  return split8<true>(x);
}

// Lane offsets into the swizzled tiles. The swizzle permutes 16 chunks (256
// bytes) of a row, so at D = 256 the upper half of a row is 256 bytes behind
// the lower half: an immediate of the read, no further register.
template <int D>
struct LaneOffs {
  static constexpr int kD = D < 128 ? D : 128;
  int row[kD / 32];  // row fragment, chunk 4c + g, row lane%16
  int tr[kD / 16];   // transposed fragment, columns 16 db ..
  __device__ __forceinline__ void init(int lane) {
    using Tile = SwzTile<D, 64>;
#pragma unroll
    for (int c = 0; c < kD / 32; ++c) row[c] = Tile::row_lane_off(lane, 4 * c + (lane >> 4));
#pragma unroll
    for (int db = 0; db < kD / 16; ++db) tr[db] = Tile::tr_lane_off(lane, 16 * db);
  }
  __device__ __forceinline__ int row_at(int c) const {
    return row[c % (kD / 32)] + c / (kD / 32) * 256;
  }
  __device__ __forceinline__ int tr_at(int db) const {
    return tr[db % (kD / 16)] + db / (kD / 16) * 256;
  }
};

// Wait until this wave's outstanding global loads (incl. loads to LDS) landed.
// Mask of one tile for one query block: key row `ts + ko` is visible to the
// lane's query iff (unsigned)(hi - ko) <= span. Local window: hi = qi - ts,
// span = W - 1 (qi - W + 1 <= ts + ko <= qi); global prefix: hi = glen - 1 - ts,
// span = 2^31 - 1 (ts + ko < glen).
template <int NQB = 2>  // query blocks of the wave
struct TileMask {
  int hi[NQB];
  unsigned span[NQB];
  __device__ __forceinline__ bool ok(int ko, int qb) const {
    return (unsigned)(hi[qb] - ko) <= span[qb];
  }
};

__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0); }

// Raw buffer resource over `bytes` bytes at `base` (gfx9 descriptor word 3).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

}  // namespace cra
