// tpr_gen.hip -- general prefix-reuse attention kernels on the matrix cores.
//
// The path for fp32 inputs, for bf16 head sizes the tuned bf16 families do
// not cover (any multiple of 8 up to 256) and for physical key masks. One
// template for both types; a unit of this file is compiled per (type, padded
// head size): TPR_GEN_FP32 (0 / 1) and TPR_GEN_DP.
//
// Precision. Nothing is held in less than 32 bits:
//   fp32   v_mfma_f32_32x32x2_f32: fp32 operands, products and sums. Its rate
//          is 1/16 of the bf16 MFMA's, so these kernels are bound by it
//          (154 TFLOP/s in a large fp32 matrix product on this card).
//   bf16   the dot products q . k and dout . v take the inputs' own bf16
//          values. Probabilities and dS stay fp32: an fp32 value is the exact
//          sum of three bf16 values (8 mantissa bits each, split3), so
//          P V, P^T dO, dS K and dS^T Q are three bf16 MFMAs into one fp32
//          accumulator -- 3/16 of the time the fp32 MFMA takes.
//
// Measured against the vector-ALU kernels they replace (forward / dK/dV / dQ,
// us): fp32, prefix 1024 + 2 x 1024, GQA 32/8, d128: 1222 / 4094 / 1260 ->
// 403 / 930 / 590 (128 TFLOP/s in the forward, of 154); fp32, prefix 512 + 2 x
// 512, 4 heads, d64: 375 / 485 / 317 -> 26 / 47 / 33; bf16, prefix 1024 + 3 x
// 1024, GQA 32/8, d96: 1276 / 6116 / 1703 -> 165 / 441 / 187 (before split3
// kept its terms nonzero); bf16 under a causal mask with padding, 1024 + 2048,
// GQA 32/8, d128: 2409 / 4707 / 2590 -> 241 / 740 / 298. What is left in bf16
// is the serial chain product - exp - split - product of the one wave a SIMD
// holds in dK/dV.
//
// A wave owns 32 stationary rows -- queries of one head in the forward and dQ,
// keys of one KV head in dK/dV -- and streams 32-row tiles of the other side
// through LDS. With the tile rows as A operand (in the order sigma32) and the
// stationary rows as B, a lane of the score tile holds one stationary row and
// two runs of 8 tile rows, which are the k-slots of the second product
// (row_product, then col_product). MFMA layout: see tpr_mfma.hip; for
// 32x32x2 f32, A and B lane l hold (row / column l % 32, k-slot l / 32).
//
// Math (per leaf, per query head; reference: _fa_fp32_reference.py:12-28):
//   s_j = scale * q . k_j over keys j = cat(ancestor nodes, suffix keys <= i)
//   out = sum_j softmax(s)_j v_j,  lse = log sum_j exp(s_j)
// Backward (standard softmax-attention gradients, recomputing P from lse):
//   p_j = exp(s_j - lse), dv_j += p_j dout, dp_j = dout . v_j,
//   ds_j = p_j (dp_j - delta), delta = dout . out,
//   dq = scale sum_j ds_j k_j, dk_j += scale ds_j q.
// Key streams: the leaf's own suffix, then its ancestors' key runs (the
// plan's run table: ancestors root first, rows adjacent in prefix_k/v merged).
//
// Masked plans (kMask): a physical key mask replaces the causal rule, as in
// the reference's custom-mask mode (rectangular_attention.py:112-122): key
// c of a leaf's sequence cat(ancestors, suffix) is visible to query row r iff
// mask[r][c] == 0, so every suffix key is streamed, and the dK/dV items of a
// suffix tile cover every query block of the leaf. A wave skips the products
// of a tile that none of its rows sees. A row with no visible key ends with
// l = 0: its output is 0, its lse -inf, and every p of it is 0 in the backward
// (p is selected by visibility, never computed from that lse).

#include "tpr_kernel_util.h"

#ifndef TPR_GEN_FP32
#error "compile with -DTPR_GEN_FP32=0|1 -DTPR_GEN_DP=64|96|128|256"
#endif

namespace tpr {
namespace {

#if TPR_GEN_FP32
typedef float elem;
constexpr bool kF32 = true;
#else
typedef bf16 elem;
constexpr bool kF32 = false;
#endif

constexpr int kDP = TPR_GEN_DP;                   // head size, padded with zeros
constexpr int kRows = kGenRows;                   // rows per tile and per wave
constexpr int kElems = 16 / sizeof(elem);         // elements of a 16-byte chunk
constexpr int kFrags = kF32 ? kDP / 8 : kDP / 16;  // 16-byte operand chunks a lane holds of a row
constexpr int kDB = kDP / 32;                     // 32-column blocks of an output row
// LDS row pitch: fp32 rows are padded by one chunk (16 rows at one chunk then
// cover all banks); bf16 rows fill whole 256-byte groups, chunk-swizzled as
// in swz_chunk (row reads and transposed reads are conflict-free).
constexpr int kPitch = kF32 ? kDP * 4 + 16 : (kDP <= 128 ? 256 : 512);
constexpr int kTile = kRows * kPitch;
constexpr int kChunks = kF32 ? kDP / 4 : (kDP <= 64 ? 8 : kDP <= 128 ? 16 : 32);  // staged chunks per row (2^n)

// memory accesses with the element's own alignment: neither the C ABI nor a
// head offset promises 16 bytes here
typedef f32x4 chunk_u __attribute__((aligned(sizeof(elem))));
struct Frag { f32x4 c[kFrags]; };

__device__ __forceinline__ f32x4 load_chunk(const elem* p) { return *reinterpret_cast<const chunk_u*>(p); }

__device__ __forceinline__ int lds_off(int row, int chunk) {
  if constexpr (kF32) return row * kPitch + 16 * chunk;
  else return row * kPitch + (chunk >> 4) * 256 + ((swz_chunk(row, chunk & 15)) << 4);
}

// A lane's stationary operand: chunks of its row at k-slots of its half
// (columns at or beyond d are 0), times `mul` (fp32 only).
__device__ __forceinline__ void load_frag(Frag& f, const elem* row, int d, int h, float mul) {
#pragma unroll
  for (int g = 0; g < kFrags; g++) {
    const int e = kElems * (2 * g + h);
    f.c[g] = e < d ? load_chunk(row + e) : f32x4{};
    if constexpr (kF32) f.c[g] *= mul;
  }
}

// fp32 at head size 256: Q, dO, dQ and the score tiles together are over the
// 512 registers of a wave, so dO's chunks are read again for each tile (from
// L2: 32 KB beside 400 MFMAs of 64 cycles).
constexpr bool kReload = kF32 && kDP == 256;

// S tile: 32 tile rows (A, order sigma32) x the wave's 32 stationary rows.
// Register r of a lane: tile row 16 (r / 8) + 8 h + r % 8, stationary row n.
__device__ __forceinline__ f32x16 row_product(const char* tile, const Frag& f, int n, int h) {
  f32x16 s = {};
  const int row = sigma32(n);
#pragma unroll
  for (int g = 0; g < kFrags; g++) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(tile + lds_off(row, 2 * g + h));
    if constexpr (kF32) {
#pragma unroll
      for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], f.c[g][i], s, 0, 0, 0);
    } else {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, f.c[g]), s,
                                                  0, 0, 0);
    }
  }
  return s;
}

// The same with the stationary row read from memory.
__device__ __forceinline__ f32x16 row_product_reload(const char* tile, const elem* row, int d, int n, int h) {
  f32x16 s = {};
  if constexpr (kReload) {
    const int r = sigma32(n);
#pragma unroll
    for (int g = 0; g < kFrags; g++) {
      const int e = kElems * (2 * g + h);
      const f32x4 b = e < d ? load_chunk(row + e) : f32x4{};
      const f32x4 a = *reinterpret_cast<const f32x4*>(tile + lds_off(r, 2 * g + h));
#pragma unroll
      for (int i = 0; i < 4; i++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], s, 0, 0, 0);
    }
  }
  return s;
}

// Bits whose high half is the bf16 next to x towards 0 (0 for x = +0): the
// integer below x's bits, cut to bf16, is always smaller than x.
__device__ __forceinline__ uint32_t below(float x) { return __builtin_elementwise_sub_sat(__float_as_uint(x), 1u); }
__device__ __forceinline__ float high_half(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }

// x = hi + mid + lo exactly (up to underflow), each a bf16 and, for x != 0,
// each nonzero and of x's sign: hi is the bf16 below x, mid the bf16 below the
// rest (at most 2^16 units of x's last place), lo what is left (at most 2^8 of
// them, or a power of two). A zero term would make NaN of a product with an
// infinite V, dO, K or Q where the fp32 product is infinite; an infinite x
// ends in lo, behind two finite terms of its sign. (With the terms cut at x's
// own bits, 1 = 1 + 0 + 0, two VALU instructions less a value: bf16 under a
// causal mask, 1024 + 2048, GQA 32/8, d128, forward / dK/dV / dQ 223 / 684 /
// 281 us against 241 / 740 / 298.) kSigned: x may be -0, which below() does
// not take.
template <bool kSigned>
__device__ __forceinline__ void split3(const float (&x)[8], bf16x8& hi, bf16x8& mid, bf16x8& lo) {
  uint32_t a[4], b[4], c[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float y0 = kSigned ? x[2 * i] + 0.f : x[2 * i], y1 = kSigned ? x[2 * i + 1] + 0.f : x[2 * i + 1];
    const uint32_t x0 = below(y0), x1 = below(y1);
    const float r0 = y0 - high_half(x0), r1 = y1 - high_half(x1);
    const uint32_t u0 = below(r0), u1 = below(r1);
    const float t0 = r0 - high_half(u0), t1 = r1 - high_half(u1);
    a[i] = __builtin_amdgcn_perm(x1, x0, 0x07060302u);  // the high halves of the two words
    b[i] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    c[i] = __builtin_amdgcn_perm(__float_as_uint(t1), __float_as_uint(t0), 0x07060302u);
  }
  hi = __builtin_bit_cast(bf16x8, a);
  mid = __builtin_bit_cast(bf16x8, b);
  lo = __builtin_bit_cast(bf16x8, c);
}

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// acc[db] += (tile columns)^T x: acc rows are output columns (out_col), acc
// columns the wave's stationary rows; x[r] belongs to tile row
// 16 (r / 8) + 8 h + r % 8. kNB column blocks from block db0 on. kSigned: x is
// not a probability (split3).
template <bool kSigned, int kNB>
__device__ __forceinline__ void col_product(const char* tile, const f32x16& x, f32x16 (&acc)[kNB], int db0, int lane) {
  const int n = lane & 31, h = lane >> 5;
  if constexpr (kF32) {
    // blocks of kVec columns per lane: one LDS read feeds kVec MFMAs
    constexpr int kVec = kNB < 4 ? kNB : 4;
    static_assert(kNB % kVec == 0, "whole column groups");
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const char* row = tile + (16 * (r >> 3) + (r & 7)) * kPitch + 8 * kPitch * h;
#pragma unroll
      for (int vb = 0; vb < kNB / kVec; vb++) {
        const float* p = reinterpret_cast<const float*>(row) + 32 * (db0 + kVec * vb) + kVec * n;
        float a[kVec];
        if constexpr (kVec == 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(p);
          a[0] = v[0]; a[1] = v[1]; a[2] = v[2]; a[3] = v[3];
        } else {
#pragma unroll
          for (int i = 0; i < kVec; i++) a[i] = p[i];
        }
#pragma unroll
        for (int i = 0; i < kVec; i++)
          acc[kVec * vb + i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], x[r], acc[kVec * vb + i], 0, 0, 0);
      }
    }
  } else {
    const int i = lane & 15, g = (lane >> 4) & 1;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; e++) p[e] = x[8 * c + e];
      bf16x8 hi, mid, lo;
      split3<kSigned>(p, hi, mid, lo);
      const int row = 16 * c + 8 * h + (i >> 2);
#pragma unroll
      for (int db = 0; db < kNB; db++) {
        const int col = 32 * (db0 + db) + 16 * g + 4 * (i & 3);
        const s16x4 u = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)(tile + lds_off(row, col >> 3) + ((col & 7) << 1)));
        const s16x4 w = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4*)(tile + lds_off(row + 4, col >> 3) + ((col & 7) << 1)));
        const bf16x4 u4 = __builtin_bit_cast(bf16x4, u), w4 = __builtin_bit_cast(bf16x4, w);
        const bf16x8 a = {u4[0], u4[1], u4[2], u4[3], w4[0], w4[1], w4[2], w4[3]};
        // smallest terms first
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, lo, acc[db], 0, 0, 0);
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, mid, acc[db], 0, 0, 0);
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, hi, acc[db], 0, 0, 0);
      }
    }
  }
}

// Calls f(column, f32x4 of 4 consecutive output columns) for a lane's part of
// an output row (its stationary row n), kNB column blocks from block db0.
template <int kNB, typename F>
__device__ __forceinline__ void for_columns(const f32x16 (&acc)[kNB], int db0, int h, F&& f) {
  if constexpr (kF32 && kNB >= 4) {
#pragma unroll
    for (int vb = 0; vb < kNB / 4; vb++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        f(32 * (db0 + 4 * vb) + 4 * (8 * (r >> 2) + 4 * h + (r & 3)),
          f32x4{acc[4 * vb][r], acc[4 * vb + 1][r], acc[4 * vb + 2][r], acc[4 * vb + 3][r]});
  } else if constexpr (kF32) {
    static_assert(kNB == 2, "fp32 rows of 64 columns or a multiple of 128");
#pragma unroll
    for (int r = 0; r < 16; r += 2)
      f(32 * db0 + 2 * (8 * (r >> 2) + 4 * h + (r & 3)), f32x4{acc[0][r], acc[1][r], acc[0][r + 1], acc[1][r + 1]});
  } else {
#pragma unroll
    for (int db = 0; db < kNB; db++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        f(32 * (db0 + db) + 8 * g + 4 * h,
          f32x4{acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]});
  }
}

__device__ __forceinline__ void store4(float* p, f32x4 v) {
  typedef f32x4 u __attribute__((aligned(4)));
  *reinterpret_cast<u*>(p) = v;
}
__device__ __forceinline__ void store4(bf16* p, f32x4 v) {
  typedef bf16x4 u __attribute__((aligned(2)));
  *reinterpret_cast<u*>(p) = bf16x4{static_cast<bf16>(v[0]), static_cast<bf16>(v[1]), static_cast<bf16>(v[2]),
                                    static_cast<bf16>(v[3])};
}
__device__ __forceinline__ f32x4 load4f(const float* p) {
  typedef f32x4 u __attribute__((aligned(4)));
  return *reinterpret_cast<const u*>(p);
}

// ---- staging --------------------------------------------------------------
// One 32-row tile of a [*, heads, d] tensor, copied by kT threads: rows from
// `base` (head offset applied), `stride` elements apart; rows at or beyond
// `rows` (>= 1) and columns at or beyond d are 0 (a copy of the last row in
// their place would multiply its infinities by a probability of 0).
template <int kT>
struct TileRegs { f32x4 r[kRows * kChunks / kT]; };

// The address of a whole tile's pass is a uniform base plus one 32-bit lane
// offset, the same for every pass (an offset per pass kept the dK/dV kernel's
// tiles from fitting the register file beside its accumulators).
__device__ __forceinline__ const char* uniform_ptr(const void* p) {
  const uint64_t b = reinterpret_cast<uint64_t>(p);
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(b >> 32)));
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(b & 0xffffffffu)));
  return reinterpret_cast<const char*>((static_cast<uint64_t>(hi) << 32) | static_cast<uint64_t>(lo));
}

template <int kT>
__device__ __forceinline__ void fetch_tile(TileRegs<kT>& t, const elem* base, int64_t stride, int rows, int d) {
  static_assert(kT % kChunks == 0, "a lane copies one chunk column");
  constexpr int kStep = kT / kChunks, kPasses = kRows / kStep;
  const int tid = threadIdx.x % kT, row = tid / kChunks, c = tid % kChunks;
  const bool in = kElems * c < d;
  const uint32_t row_bytes = static_cast<uint32_t>(stride) * sizeof(elem);  // at most 32 MiB
  const uint32_t col = in ? 16u * c : 0u;
  const char* src = uniform_ptr(base);
  if (rows >= kRows) {
    const uint32_t off = row * row_bytes + col;
#pragma unroll
    for (int i = 0; i < kPasses; i++) {
      t.r[i] = load_chunk(reinterpret_cast<const elem*>(src + off));
      src += static_cast<uint64_t>(kStep) * row_bytes;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kPasses; i++) {
      const f32x4 x = load_chunk(reinterpret_cast<const elem*>(src + (min(row + kStep * i, rows - 1) * row_bytes + col)));
      t.r[i] = row + kStep * i < rows ? x : f32x4{};
    }
  }
  if (!in) {
#pragma unroll
    for (int i = 0; i < kPasses; i++) t.r[i] = f32x4{};
  }
}
// The same copy straight to LDS, eight passes in flight (where no registers
// are left to hold the tile).
template <int kT>
__device__ __forceinline__ void copy_tile(char* tile, const elem* base, int64_t stride, int rows, int d) {
  constexpr int kStep = kT / kChunks, kPasses = kRows / kStep, kAtOnce = kPasses < 8 ? kPasses : 8;
  const int tid = threadIdx.x % kT, row = tid / kChunks, c = tid % kChunks;
  const bool in = kElems * c < d;
  const uint32_t row_bytes = static_cast<uint32_t>(stride) * sizeof(elem);
  const uint32_t col = in ? 16u * c : 0u;
  const char* src = uniform_ptr(base);
#pragma unroll 1
  for (int i0 = 0; i0 < kPasses; i0 += kAtOnce) {
    f32x4 r[kAtOnce];
#pragma unroll
    for (int i = 0; i < kAtOnce; i++)
      r[i] = load_chunk(reinterpret_cast<const elem*>(src + (min(row + kStep * (i0 + i), rows - 1) * row_bytes + col)));
    if (rows < kRows) {
#pragma unroll
      for (int i = 0; i < kAtOnce; i++) r[i] = row + kStep * (i0 + i) < rows ? r[i] : f32x4{};
    }
#pragma unroll
    for (int i = 0; i < kAtOnce; i++)
      *reinterpret_cast<f32x4*>(tile + lds_off(row + kStep * (i0 + i), c)) = in ? r[i] : f32x4{};
  }
}
template <int kT>
__device__ __forceinline__ void put_tile(const TileRegs<kT>& t, char* tile) {
  const int tid = threadIdx.x % kT;
#pragma unroll
  for (int i = 0; i < kRows * kChunks / kT; i++) {
    const int idx = tid + kT * i, row = idx / kChunks, c = idx % kChunks;
    *reinterpret_cast<f32x4*>(tile + lds_off(row, c)) = t.r[i];
  }
}
// Order one wave's LDS writes before its reads of them, and its reads before
// its next writes (a wave's LDS operations execute in order; this keeps the
// compiler from reordering them and waits for the writes).
__device__ __forceinline__ void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// ---- the key stream of a forward / dQ workgroup ------------------------------
// The leaf's own suffix (its first `suffix_keys` keys, causal), then its key
// runs, in 32-key tiles.
struct KeyTile {
  const elem* k;
  const elem* v;
  int64_t kst, vst;
  int keys;     // keys of the tile, 0 past the end
  int pos;      // position of the first key within its segment
  int col;      // mask column of the first key
  bool causal;
};

struct KeyStream {
  const KernelArgs& a;
  const int32_t* runs;
  int kvh, suffix_col;
  int sg, pos, len, row, run_col;  // current segment: 0 = suffix, 1 + r = run r

  __device__ __forceinline__ KeyStream(const KernelArgs& args, int leaf, int kvh_, int row0, int suffix_keys,
                                       int suffix_col_)
      : a(args), runs(args.plan + args.off_runs + 2 * leaf * args.max_runs), kvh(kvh_), suffix_col(suffix_col_), sg(0),
        pos(0), len(suffix_keys), row(row0), run_col(0) {}

  __device__ __forceinline__ KeyTile tile() const {
    KeyTile t;
    const bool suffix = sg == 0;
    t.keys = min(kRows, len - pos);
    t.pos = pos;
    t.causal = suffix;
    t.col = (suffix ? suffix_col : run_col) + pos;
    const int64_t ks = static_cast<int64_t>(a.hkv) * a.d;
    t.kst = suffix ? a.k_rs : ks;
    t.vst = suffix ? a.v_rs : ks;
    t.k = static_cast<const elem*>(suffix ? a.k : a.pk) + static_cast<int64_t>(row + pos) * t.kst + kvh * a.d;
    t.v = static_cast<const elem*>(suffix ? a.v : a.pv) + static_cast<int64_t>(row + pos) * t.vst + kvh * a.d;
    return t;
  }
  // step over n tiles; past the end the stream stays at an empty segment
  __device__ __forceinline__ void advance(int n) {
    while (true) {
      const int left = (len - pos + kRows - 1) / kRows;
      if (n < left || len == 0) {
        pos = len == 0 ? 0 : pos + n * kRows;
        return;
      }
      n -= left;
      if (sg > 0) run_col += len;
      pos = len = 0;
      if (sg < a.max_runs) {
        row = plan_word(runs + 2 * sg);
        len = plan_word(runs + 2 * sg + 1);  // {0, 0} pads the run list
        sg++;
      }
    }
  }
};

// Mask column of the first key of a segment in a leaf's key sequence: the
// lengths of the leaf's ancestors ahead of node `node` (all of them for
// node < 0, i.e. the leaf's own suffix).
__device__ __forceinline__ int leaf_key_column(const KernelArgs& a, int leaf, int node) {
  const int32_t* anc = a.plan + a.off_anc + static_cast<int64_t>(leaf) * a.max_depth;
  const int32_t* no = a.plan + a.off_node_off;
  int col = 0;
  for (int i = 0; i < a.max_depth; i++) {
    const int n = plan_word(anc + i);
    if (n < 0 || n == node) break;
    col += plan_word(no + n + 1) - plan_word(no + n);
  }
  return col;
}

// A query row's mask bytes of the lane's 16 keys of a tile (keys 16 c + 8 h +
// 0..7); keys at or beyond the tile's end read as hidden.
struct MaskBytes { uint32_t w[4]; };

__device__ __forceinline__ MaskBytes load_mask(const KernelArgs& a, const KeyTile& t, int64_t mask_row, int h) {
  const uint8_t* m = a.mask + mask_row * a.mask_rs + t.col;
  MaskBytes b;
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int k0 = 16 * c + 8 * h;
    if (k0 + 8 <= t.keys) {
      __builtin_memcpy(&b.w[2 * c], m + k0, 8);
    } else {
      b.w[2 * c] = b.w[2 * c + 1] = 0;
#pragma unroll
      for (int e = 0; e < 8; e++)
        b.w[2 * c + e / 4] |= static_cast<uint32_t>(k0 + e < t.keys ? m[k0 + e] : uint8_t{1}) << (8 * (e % 4));
    }
  }
  return b;
}

// Which of a lane's 16 keys of a tile its query row sees (bit r: key
// 16 (r / 8) + 8 h + r % 8).
__device__ __forceinline__ uint32_t visible_bits(const MaskBytes& b) {
  uint32_t vis = 0;
#pragma unroll
  for (int r = 0; r < 16; r++) vis |= (b.w[r / 4] >> (8 * (r % 4)) & 0xffu) == 0 ? 1u << r : 0u;
  return vis;
}
__device__ __forceinline__ uint32_t visible_bits(const KeyTile& t, int tok, int h) {
  uint32_t vis = 0;
  const int lim = min(t.keys - 1, t.causal ? tok - t.pos : kRows);
#pragma unroll
  for (int r = 0; r < 16; r++) vis |= 16 * (r >> 3) + 8 * h + (r & 7) <= lim ? 1u << r : 0u;
  return vis;
}

// How a forward / dQ workgroup runs. kSplit == 1: four waves of 32 rows each
// (heads of one KV head's group first, then tokens) share every K/V tile they
// stage, two tiles per barrier in bf16. kSplit > 1 (few query rows): kSplit
// waves share one row block, each taking every kSplit-th key tile through an
// LDS buffer of its own, without barriers; their partial rows are summed in
// LDS at the end. The next tile is held in registers while one computes.
template <int kSplit>
struct Run {
  static constexpr int kW = kSplit == 1 ? kGenWaves : kSplit;                      // waves
  static constexpr int kT = 64 * kW;                                               // threads
  static constexpr int kCopy = kSplit == 1 ? kT : 64;                              // threads that copy a tile
  static constexpr int kPer = !kF32 && kSplit == 1 && kDP <= 128 ? 2 : 1;          // tiles per step
  static constexpr int kRegs = 2 * kPer * kRows * kChunks / kCopy * 4;             // registers of a step's tiles
  static constexpr bool kAhead = kDP <= 128;
  static constexpr int kStage = 2 * kPer * kTile * (kSplit == 1 ? 1 : kSplit);     // LDS bytes
  static constexpr int kSum = kSplit == 1 ? 0 : kSplit * kRows * (kDP + 4) * 4;
  static constexpr int kLds = kStage > kSum ? kStage : kSum;
  // two workgroups of four waves on a CU (256 registers a wave), or as many
  // waves as the LDS buffers allow
  static constexpr int kMinWaves = kSplit == 1 ? (kDP <= 128 ? 2 : 1) : (kW + 3) / 4;
  // fp32 dQ at head size 128 holds Q, dO, dQ and two score tiles (224
  // registers): the tiles go to LDS as they arrive, and the other workgroup of
  // the CU covers their latency
  static constexpr bool kAheadDq = kAhead && !(kF32 && kDP == 128 && kSplit == 1);
};

// Runs f(tile, mask bytes, K tile, V tile) for this wave's tiles of the stream.
template <bool kMask, int kSplit, bool kAhead, typename F>
__device__ __forceinline__ void stream_keys(KeyStream& ks, int64_t mask_row, int h, int part, char* smem, F&& f) {
  using R = Run<kSplit>;
  constexpr int kPer = R::kPer, kCopy = R::kCopy;
  const KernelArgs& a = ks.a;
  KeyTile cur[kPer];
  TileRegs<kCopy> rk[kPer], rv[kPer];
  MaskBytes mb[kPer] = {};
  char* buf = smem + (kSplit == 1 ? 0 : 2 * kTile * part);
  auto next = [&](int skip) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kPer; u++) {
      ks.advance(u == 0 ? skip : 1);
      cur[u] = ks.tile();
    }
  };
  auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kPer; u++)
      if (cur[u].keys > 0) {
        if constexpr (kAhead) {
          fetch_tile<kCopy>(rk[u], cur[u].k, cur[u].kst, cur[u].keys, a.d);
          fetch_tile<kCopy>(rv[u], cur[u].v, cur[u].vst, cur[u].keys, a.d);
        }
        if constexpr (kMask) mb[u] = load_mask(a, cur[u], mask_row, h);
      }
  };
  next(part);
  fetch();
  while (cur[0].keys > 0) {
    if constexpr (kSplit == 1) __syncthreads();  // the last step's tiles have been read
    else wave_lds_fence();
#pragma unroll
    for (int u = 0; u < kPer; u++)
      if (cur[u].keys > 0) {
        if constexpr (kAhead) {
          put_tile<kCopy>(rk[u], buf + 2 * u * kTile);
          put_tile<kCopy>(rv[u], buf + (2 * u + 1) * kTile);
        } else {
          copy_tile<kCopy>(buf + 2 * u * kTile, cur[u].k, cur[u].kst, cur[u].keys, a.d);
          copy_tile<kCopy>(buf + (2 * u + 1) * kTile, cur[u].v, cur[u].vst, cur[u].keys, a.d);
        }
      }
    if constexpr (kSplit == 1) __syncthreads();
    else wave_lds_fence();
    KeyTile now[kPer];
    MaskBytes mask[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
      now[u] = cur[u];
      mask[u] = mb[u];
    }
    next(kSplit);
    fetch();
#pragma unroll
    for (int u = 0; u < kPer; u++)
      if (now[u].keys > 0) f(now[u], mask[u], buf + 2 * u * kTile, buf + (2 * u + 1) * kTile);
  }
}

struct QueryRows {
  int leaf, kvh, head, tok, row0, len, part, lane, n, h, t;
  int tok_end;  // past the workgroup's last token
  bool any;     // some row of the wave exists
};

template <int kSplit>
__device__ __forceinline__ bool query_rows(const KernelArgs& a, QueryRows& q) {
  const int32_t* item = a.plan + a.off_fwd + 4 * blockIdx.x;
  q.leaf = item[0];
  if (q.leaf < 0) return false;
  const int tok0 = item[1], qh0 = item[2];
  q.kvh = item[3];
  const int32_t* cu = a.plan + a.off_cu;
  q.row0 = cu[q.leaf];
  q.len = cu[q.leaf + 1] - q.row0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = kSplit == 1 ? wave : 0;
  q.part = kSplit == 1 ? 0 : wave;
  q.head = qh0 + slot % a.hpw;
  q.tok = tok0 + kRows * (slot / a.hpw);
  q.tok_end = tok0 + (kSplit == 1 ? kRows * (kGenWaves / a.hpw) : kRows);
  q.lane = threadIdx.x & 63;
  q.n = q.lane & 31;
  q.h = q.lane >> 5;
  q.t = q.tok + q.n;
  q.any = q.tok < q.len;
  return true;
}

// Sums kParts waves' 32-row tiles in LDS, part 0 first: every wave leaves
// acc * f(lane), then the workgroup adds them up and calls out(row, column,
// sum of 4 columns). `smem` holds kParts * 32 rows of kCols + 4 floats.
template <int kParts, int kNB, typename F>
__device__ __forceinline__ void sum_parts(char* smem, const f32x16 (&acc)[kNB], float f, int part, int n, int h, F&& out) {
  constexpr int kPitchF = 32 * kNB + 4, kQuads = 8 * kNB;
  float* buf = reinterpret_cast<float*>(smem);
  __syncthreads();
  for_columns<kNB>(acc, 0, h, [&](int col, f32x4 v) {
    *reinterpret_cast<f32x4*>(buf + (part * kRows + n) * kPitchF + col) = v * f;
  });
  __syncthreads();
  for (int idx = threadIdx.x; idx < kRows * kQuads; idx += 64 * kParts) {
    const int row = idx / kQuads, col = 4 * (idx % kQuads);
    const float* p = buf + row * kPitchF + col;
    f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int s = 1; s < kParts; s++) v += *reinterpret_cast<const f32x4*>(p + s * kRows * kPitchF);
    out(row, col, v);
  }
}

// max over lanes l and l ^ 32 without an LDS round trip
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// ---------------------------------------------------------------------------
// Forward
// O and l are rescaled only when some row's scores exceed the maximum they
// refer to by more than this many log2 units: exact in fp32 (probabilities
// stay below 2^8), and most tiles then need no cross-lane step.
constexpr float kSlack = 8.f;

template <bool kMask, int kSplit>
__global__ __launch_bounds__(Run<kSplit>::kT, Run<kSplit>::kMinWaves) void gen_fwd(KernelArgs a) {
  QueryRows q;
  if (!query_rows<kSplit>(a, q)) return;
  const int d = a.d;
  const int64_t qs = static_cast<int64_t>(a.hq) * d;
  const int trow = min(q.t, q.len - 1);

  __shared__ __attribute__((aligned(1024))) char smem[Run<kSplit>::kLds];
  __shared__ float stat[2][kSplit][kRows];  // m, l of the parts

  const float cs = a.scale * kLog2e;
  Frag qf;
  load_frag(qf, static_cast<const elem*>(a.q) + static_cast<int64_t>(q.row0 + trow) * a.q_rs + q.head * d, d, q.h, cs);
  f32x16 o[kDB];
#pragma unroll
  for (int i = 0; i < kDB; i++) o[i] = f32x16{};
  float m = -INFINITY, l = 0.f;  // m: the row's; l: this lane's keys only, until the end

  // causal: the suffix keys up to the workgroup's last query; masked: all
  const int suffix_keys = kMask ? q.len : min(q.len, q.tok_end);
  KeyStream ks(a, q.leaf, q.kvh, q.row0, suffix_keys, kMask ? leaf_key_column(a, q.leaf, -1) : 0);
  stream_keys<kMask, kSplit, Run<kSplit>::kAhead>(ks, q.row0 + trow, q.h, q.part, smem,
                             [&](const KeyTile& t, const MaskBytes& mb, const char* kt, const char* vt)
                                 __attribute__((always_inline)) {
    if (!q.any || (!kMask && t.causal && t.pos > q.tok + kRows - 1)) return;
    const bool whole = !kMask && t.keys == kRows && (!t.causal || t.pos + kRows - 1 <= q.tok);
    uint32_t vis = 0xffffu;
    if constexpr (kMask) vis = visible_bits(mb);
    else if (!whole) vis = visible_bits(t, q.t, q.h);
    if (kMask && __ballot(vis != 0) == 0) return;
    f32x16 s = row_product(kt, qf, q.n, q.h);
    if constexpr (!kF32) s *= cs;
    if (!whole) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = vis >> r & 1 ? s[r] : -INFINITY;
    }
    float x[8];
#pragma unroll
    for (int r = 0; r < 8; r++) x[r] = fmaxf(s[r], s[r + 8]);
#pragma unroll
    for (int w = 4; w >= 1; w >>= 1)
#pragma unroll
      for (int r = 0; r < w; r++) x[r] = fmaxf(x[r], x[r + w]);
    if (__ballot(x[0] > m + kSlack) != 0) {
      const float mt = fmaxf(m, half_max(x[0]));
      const float alpha = mt == -INFINITY ? 1.f : fast_exp2(m - mt);
      m = mt;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < kDB; i++) o[i] *= alpha;
    }
    // nothing visible yet for this row: every exponent is -inf
    const float mref = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = fast_exp2(s[r] - mref);
#pragma unroll
    for (int r = 0; r < 8; r++) x[r] = s[r] + s[r + 8];
#pragma unroll
    for (int w = 4; w >= 1; w >>= 1)
#pragma unroll
      for (int r = 0; r < w; r++) x[r] += x[r + w];
    l += x[0];
    col_product<false>(vt, s, o, 0, q.lane);
  });
  l = wave_sum32(l);

  // l == 0 only for a row a mask hides every key of: out 0, lse -inf
  elem* out = static_cast<elem*>(a.out);
  float* lse = a.lse + static_cast<int64_t>(q.head) * a.total_q + q.row0;
  if constexpr (kSplit == 1) {
    if (q.t >= q.len) return;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    elem* row = out + static_cast<int64_t>(q.row0 + q.t) * qs + q.head * d;
    for_columns<kDB>(o, 0, q.h, [&](int col, f32x4 v) {
      if (col < d) store4(row + col, v * inv);
    });
    if (q.h == 0) lse[q.t] = l > 0.f ? (m + log2f(l)) * kLn2 : -INFINITY;
  } else {
    if (q.h == 0) {
      stat[0][q.part][q.n] = m;
      stat[1][q.part][q.n] = l;
    }
    __syncthreads();
    float top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int s = 0; s < kSplit; s++) top = fmaxf(top, stat[0][s][q.n]);
    const float ref = top == -INFINITY ? 0.f : top;
#pragma unroll
    for (int s = 0; s < kSplit; s++) sum += fast_exp2(stat[0][s][q.n] - ref) * stat[1][s][q.n];
    const float f = sum > 0.f ? fast_exp2(m - ref) / sum : 0.f;
    if (q.part == 0 && q.h == 0 && q.t < q.len) lse[q.t] = sum > 0.f ? (top + log2f(sum)) * kLn2 : -INFINITY;
    sum_parts<kSplit, kDB>(smem, o, f, q.part, q.n, q.h, [&](int row, int col, f32x4 v) {
      if (q.tok + row < q.len && col < d)
        store4(out + static_cast<int64_t>(q.row0 + q.tok + row) * qs + q.head * d + col, v);
    });
  }
}

// ---------------------------------------------------------------------------
// dQ (the forward's items)
template <bool kMask, int kSplit>
__global__ __launch_bounds__(Run<kSplit>::kT, Run<kSplit>::kMinWaves) void gen_dq(KernelArgs a) {
  QueryRows q;
  if (!query_rows<kSplit>(a, q)) return;
  const int d = a.d;
  const int64_t qs = static_cast<int64_t>(a.hq) * d;
  const int trow = min(q.t, q.len - 1);

  __shared__ __attribute__((aligned(1024))) char smem[Run<kSplit>::kLds];

  const float cs = a.scale * kLog2e;
  Frag qf, gf;
  load_frag(qf, static_cast<const elem*>(a.q) + static_cast<int64_t>(q.row0 + trow) * a.q_rs + q.head * d, d, q.h, cs);
  const elem* grow = static_cast<const elem*>(a.dout) + static_cast<int64_t>(q.row0 + trow) * qs + q.head * d;
  if constexpr (!kReload) load_frag(gf, grow, d, q.h, 1.f);
  f32x16 dq[kDB];
#pragma unroll
  for (int i = 0; i < kDB; i++) dq[i] = f32x16{};
  const int64_t at = static_cast<int64_t>(q.head) * a.total_q + q.row0 + trow;
  const float lse2 = a.lse_in[at] * kLog2e, delta = a.delta[at];

  const int suffix_keys = kMask ? q.len : min(q.len, q.tok_end);
  KeyStream ks(a, q.leaf, q.kvh, q.row0, suffix_keys, kMask ? leaf_key_column(a, q.leaf, -1) : 0);
  stream_keys<kMask, kSplit, Run<kSplit>::kAheadDq>(ks, q.row0 + trow, q.h, q.part, smem,
                             [&](const KeyTile& t, const MaskBytes& mb, const char* kt, const char* vt)
                                 __attribute__((always_inline)) {
    if (!q.any || (!kMask && t.causal && t.pos > q.tok + kRows - 1)) return;
    const bool whole = !kMask && t.keys == kRows && (!t.causal || t.pos + kRows - 1 <= q.tok);
    uint32_t vis = 0xffffu;
    if constexpr (kMask) vis = visible_bits(mb);
    else if (!whole) vis = visible_bits(t, q.t, q.h);
    if (kMask && __ballot(vis != 0) == 0) return;
    f32x16 s = row_product(kt, qf, q.n, q.h);
    f32x16 dp;
    if constexpr (kReload) dp = row_product_reload(vt, grow, d, q.n, q.h);
    else dp = row_product(vt, gf, q.n, q.h);
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float x = kF32 ? s[r] : s[r] * cs;
      s[r] = fast_exp2(x - lse2) * (dp[r] - delta);
    }
    if (!whole) {
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = vis >> r & 1 ? s[r] : 0.f;
    }
    col_product<true>(kt, s, dq, 0, q.lane);
  });

  elem* out = static_cast<elem*>(a.dq);
  if constexpr (kSplit == 1) {
    if (q.t >= q.len) return;
    elem* row = out + static_cast<int64_t>(q.row0 + q.t) * qs + q.head * d;
    for_columns<kDB>(dq, 0, q.h, [&](int col, f32x4 v) {
      if (col < d) store4(row + col, v * a.scale);
    });
  } else {
    sum_parts<kSplit, kDB>(smem, dq, 1.f, q.part, q.n, q.h, [&](int row, int col, f32x4 v) {
      if (q.tok + row < q.len && col < d)
        store4(out + static_cast<int64_t>(q.row0 + q.tok + row) * qs + q.head * d + col, v * a.scale);
    });
  }
}

// ---------------------------------------------------------------------------
// dK/dV: an item is kGenKeys = 64 keys of one KV head of one segment (prefix
// node or leaf suffix), run by two workgroups of 32 keys (grid.y; at head size
// 256 four, each computing 128 columns of dK and dV: the whole rows would not
// fit the register file beside the wave's K and V). Wave w of a workgroup
// takes every kQParts-th 32-query tile (of every head of the group, in the
// plan's order) from tile w on, through LDS buffers of its own and without
// barriers; the parts are added in LDS at the end, so a prefix node's gradient
// is a fixed-order sum over its descendant leaves without atomics. One wave
// per SIMD: the accumulators and the K and V rows take 290 registers at head
// size 128.
constexpr int kOutD = kDP > 128 ? 128 : kDP;
constexpr int kOutB = kOutD / 32;
constexpr int kQParts = kF32 && kDP == 256 ? 2 : 4;
static_assert(kGenKeys == 2 * kRows, "two workgroups per item and column block");

template <bool kMask>
__global__ __launch_bounds__(64 * kQParts) void gen_dkdv(KernelArgs a) {
  const int32_t* item = a.plan + a.off_dkdv + DK_WORDS * blockIdx.x;
  if (item[DK_SRC] < 0) return;
  const bool prefix = item[DK_SRC] == 0;
  const int seg = item[DK_SEG], kvh = item[DK_KVH];
  const int kp0 = item[DK_KEY0] + kRows * (blockIdx.y & 1);  // first key, as a position within the segment
  const int qb_lo = item[DK_QB_LO], qb_hi = item[DK_QB_HI];
  const int32_t* cu = a.plan + a.off_cu;
  const int32_t* no = a.plan + a.off_node_off;
  const int32_t* qblk = a.plan + a.off_qblk;
  const int d = a.d, db0 = kOutB * (blockIdx.y >> 1);
  const int64_t qs = static_cast<int64_t>(a.hq) * d, ks = static_cast<int64_t>(a.hkv) * d;
  const int seg_row0 = prefix ? no[seg] : cu[seg];
  const int seg_len = prefix ? no[seg + 1] - no[seg] : cu[seg + 1] - cu[seg];
  if (kp0 >= seg_len) return;
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const int kp = min(kp0 + n, seg_len - 1);
  const int64_t krow = static_cast<int64_t>(seg_row0 + kp);
  const elem* kbase = static_cast<const elem*>(prefix ? a.pk : a.k);
  const elem* vbase = static_cast<const elem*>(prefix ? a.pv : a.v);

  constexpr int kSum = kQParts * kRows * (kOutD + 4) * 4, kStage = kQParts * 2 * kTile;
  __shared__ __attribute__((aligned(1024))) char smem[kStage > kSum ? kStage : kSum];
  __shared__ __attribute__((aligned(16))) float stats[kQParts][2][kRows];  // lse * log2e, delta

  const float cs = a.scale * kLog2e;
  Frag kf, vf;
  load_frag(kf, kbase + krow * (prefix ? ks : a.k_rs) + kvh * d, d, h, cs);
  load_frag(vf, vbase + krow * (prefix ? ks : a.v_rs) + kvh * d, d, h, 1.f);
  f32x16 dk[kOutB], dv[kOutB];
#pragma unroll
  for (int i = 0; i < kOutB; i++) dk[i] = dv[i] = f32x16{};

  // query tiles: index x of [0, blocks * group), block-major
  struct QTile { int row, toks, tok, col; };
  const int count = (qb_hi - qb_lo) * a.group;
  // The next tile's Q and dO are held in registers while one computes. fp32 at
  // head size 128 has room for one of them: dO is fetched when Q has left for
  // LDS, and lands while the Q product runs (64 MFMAs of 64 cycles). At head
  // size 256 there is room for neither.
  constexpr bool kAhead = kDP <= 128, kBoth = kAhead && !kF32;
  TileRegs<64> rq, rg;
  float st = 0.f;        // lanes 0-31: lse * log2e of the tile's queries, lanes 32-63: delta
  uint8_t mb[16] = {};   // mask bytes of the lane's 16 queries and its key
  int last_leaf = -1, last_col = 0;
  QTile cur = {};
  auto next = [&](int x) __attribute__((always_inline)) {
    const int b = qb_lo + x / a.group;
    const int leaf = plan_word(qblk + 2 * b);
    cur.tok = plan_word(qblk + 2 * b + 1);
    cur.row = plan_word(cu + leaf) + cur.tok;
    cur.toks = min(kRows, plan_word(cu + leaf + 1) - cur.row);
    if (kMask && leaf != last_leaf) {
      last_leaf = leaf;
      last_col = leaf_key_column(a, leaf, prefix ? seg : -1);
    }
    cur.col = last_col;
  };
  auto fetch_g = [&](TileRegs<64>& r, const QTile& t, int x) __attribute__((always_inline)) {
    const int head = kvh * a.group + x % a.group;
    fetch_tile<64>(r, static_cast<const elem*>(a.dout) + static_cast<int64_t>(t.row) * qs + head * d, qs, t.toks, d);
  };
  auto fetch = [&](int x) __attribute__((always_inline)) {
    const int head = kvh * a.group + x % a.group;
    const elem* qp = static_cast<const elem*>(a.q) + static_cast<int64_t>(cur.row) * a.q_rs + head * d;
    if constexpr (kAhead) fetch_tile<64>(rq, qp, a.q_rs, cur.toks, d);
    if constexpr (kBoth) fetch_g(rg, cur, x);
    const int64_t at = static_cast<int64_t>(head) * a.total_q + cur.row + min(n, cur.toks - 1);
    st = h == 0 ? a.lse_in[at] * kLog2e : a.delta[at];
    st = n < cur.toks ? st : 0.f;  // rows past the end: p is 0, and dS = p (dP - delta) with it
    if constexpr (kMask) {
      const uint8_t* mrow = a.mask + static_cast<int64_t>(cur.row) * a.mask_rs + cur.col + kp;
      if (cur.toks == kRows) {
        mrow += 8 * h * a.mask_rs;
#pragma unroll
        for (int r = 0; r < 16; r++) mb[r] = mrow[(16 * (r >> 3) + (r & 7)) * a.mask_rs];
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++) mb[r] = mrow[min(16 * (r >> 3) + 8 * h + (r & 7), cur.toks - 1) * a.mask_rs];
      }
    }
  };
  char* qt = smem + 2 * kTile * part;
  char* gt = qt + kTile;
  if (part < count) {
    next(part);
    fetch(part);
  }
  for (int x = part; x < count; x += kQParts) {
    const QTile t = cur;
    // bit r: query 16 (r / 8) + 8 h + r % 8 of the tile sees this lane's key
    uint32_t vis = 0;
    bool run = true;  // bf16 under a mask: some query of the tile sees some key
    const bool whole = !kMask && t.toks == kRows && (prefix || t.tok >= kp0 + kRows - 1);
    if (!whole) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int i = 16 * (r >> 3) + 8 * h + (r & 7);
        const bool sees = kMask ? mb[r] == 0 : prefix || kp <= t.tok + i;
        vis |= i < t.toks && sees ? 1u << r : 0u;
      }
      if (kMask && !kF32) run = __ballot(vis != 0) != 0;
    }
    wave_lds_fence();
    if (run) {
      if constexpr (kAhead) {
        put_tile<64>(rq, qt);
        if constexpr (kBoth) put_tile<64>(rg, gt);
      } else {
        const int head = kvh * a.group + x % a.group;
        copy_tile<64>(qt, static_cast<const elem*>(a.q) + static_cast<int64_t>(t.row) * a.q_rs + head * d, a.q_rs, t.toks, d);
        copy_tile<64>(gt, static_cast<const elem*>(a.dout) + static_cast<int64_t>(t.row) * qs + head * d, qs, t.toks, d);
      }
      stats[part][h][n] = st;
    }
    wave_lds_fence();
    const bool more = x + kQParts < count;
    if (more) next(x + kQParts);
    if ((kBoth || !kAhead) && more) fetch(x + kQParts);
    if constexpr (kAhead && !kBoth) fetch_g(rg, t, x);
    if (!run) continue;
    f32x16 s = row_product(qt, kf, n, h);
    if constexpr (kAhead && !kBoth) {
      put_tile<64>(rg, gt);
      wave_lds_fence();
      if (more) fetch(x + kQParts);
    }
    f32x16 dp = row_product(gt, vf, n, h);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      f32x4 ls[2], de[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        ls[e] = *reinterpret_cast<const f32x4*>(&stats[part][0][16 * c + 8 * h + 4 * e]);
        de[e] = *reinterpret_cast<const f32x4*>(&stats[part][1][16 * c + 8 * h + 4 * e]);
      }
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int r = 8 * c + e;
        float p = fast_exp2((kF32 ? s[r] : s[r] * cs) - ls[e >> 2][e & 3]);
        if (!whole) p = vis >> r & 1 ? p : 0.f;
        s[r] = p;
        dp[r] = p * (dp[r] - de[e >> 2][e & 3]);
      }
    }
    col_product<false>(gt, s, dv, db0, lane);
    col_product<true>(qt, dp, dk, db0, lane);
  }

  auto finish = [&](const f32x16 (&acc)[kOutB], float mul, void* prefix_out, void* suffix_out) __attribute__((always_inline)) {
    sum_parts<kQParts, kOutB>(smem, acc, 1.f, part, n, h, [&](int row, int col, f32x4 v) {
      const int e = 32 * db0 + col;
      if (kp0 + row >= seg_len || e >= d) return;
      const int64_t at = static_cast<int64_t>(seg_row0 + kp0 + row) * ks + kvh * d + e;
      if (prefix && a.acc_prefix) {
#pragma clang fp contract(off)  // rounded product, then one add
        float* p = static_cast<float*>(prefix_out) + at;
        const f32x4 add = v * mul;
        store4(p, load4f(p) + add);
      } else {
        store4(static_cast<elem*>(prefix ? prefix_out : suffix_out) + at, v * mul);
      }
    });
  };
  finish(dk, a.scale, a.dpk, a.dk);
  finish(dv, 1.f, a.dpv, a.dv);
}

// ---------------------------------------------------------------------------
// delta[h][t] = sum_e dout[t][h][e] * out[t][h][e]: a workgroup takes 64 tokens
// of one head, 16 lanes a row (as mfma_delta), so the reads are whole chunks
// and the sums leave as one run of 64 floats. One thread per row, each
// reading its row alone, took 62 us at 2048 tokens x 32 heads x 128 fp32.
constexpr int kDeltaTokens = 64;

__global__ __launch_bounds__(256) void gen_delta(KernelArgs a) {
  const int head = blockIdx.y, t0 = blockIdx.x * kDeltaTokens;
  const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
  __shared__ float sums[kDeltaTokens];
  float s[4] = {};
  for (int e = kElems * c; e < a.d; e += 16 * kElems) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int t = t0 + 16 * k + r;
      if (t >= a.total_q) continue;
      const int64_t at = (static_cast<int64_t>(t) * a.hq + head) * a.d + e;
      const f32x4 x = load_chunk(static_cast<const elem*>(a.out_in) + at);
      const f32x4 g = load_chunk(static_cast<const elem*>(a.dout) + at);
      if constexpr (kF32) {
#pragma unroll
        for (int i = 0; i < 4; i++) s[k] = fmaf(x[i], g[i], s[k]);
      } else {
        const bf16x8 xb = __builtin_bit_cast(bf16x8, x), gb = __builtin_bit_cast(bf16x8, g);
#pragma unroll
        for (int i = 0; i < 8; i++) s[k] = fmaf(static_cast<float>(xb[i]), static_cast<float>(gb[i]), s[k]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
#pragma unroll
    for (int x = 8; x >= 1; x >>= 1) s[k] += __shfl_xor(s[k], x);
    if (c == 0) sums[16 * k + r] = s[k];
  }
  __syncthreads();
  const int i = threadIdx.x;
  if (i < kDeltaTokens && t0 + i < a.total_q) a.delta[static_cast<int64_t>(head) * a.total_q + t0 + i] = sums[i];
}

template <bool kMask, int kSplit>
void launch_query(const KernelArgs& a, bool dq, hipStream_t s) {
  const dim3 grid(a.n_items), block(Run<kSplit>::kT);
  if (dq) hipLaunchKernelGGL((gen_dq<kMask, kSplit>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((gen_fwd<kMask, kSplit>), grid, block, 0, s, a);
}

}  // namespace

#define TPR_GEN_NAME2(what, t, dp) launch_gen_##what##_##t##_##dp
#define TPR_GEN_NAME1(what, t, dp) TPR_GEN_NAME2(what, t, dp)
#if TPR_GEN_FP32
#define TPR_GEN_NAME(what) TPR_GEN_NAME1(what, f32, TPR_GEN_DP)
#else
#define TPR_GEN_NAME(what) TPR_GEN_NAME1(what, bf16, TPR_GEN_DP)
#endif

// forward (dq = false) or dQ over a.n_items work items
int TPR_GEN_NAME(query)(const KernelArgs& a, bool dq, hipStream_t s) {
  if (a.n_items <= 0) return 0;
  constexpr int kSplit = gen_split(kF32, kDP);
  if (a.split == 1) a.mask ? launch_query<true, 1>(a, dq, s) : launch_query<false, 1>(a, dq, s);
  else a.mask ? launch_query<true, kSplit>(a, dq, s) : launch_query<false, kSplit>(a, dq, s);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

int TPR_GEN_NAME(dkdv)(const KernelArgs& a, int n_dkdv, hipStream_t s) {
  if (n_dkdv <= 0) return 0;
  const dim3 grid(n_dkdv, 2 * kDP / kOutD), block(64 * kQParts);
  if (a.mask) hipLaunchKernelGGL(gen_dkdv<true>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(gen_dkdv<false>, grid, block, 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

int TPR_GEN_NAME(delta)(const KernelArgs& a, hipStream_t s) {
  const int blocks = (a.total_q + kDeltaTokens - 1) / kDeltaTokens;
  if (blocks > 0 && a.hq > 0) hipLaunchKernelGGL(gen_delta, dim3(blocks, a.hq), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 4;
}

}  // namespace tpr
