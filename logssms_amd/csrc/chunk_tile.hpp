// MFMA tile primitives and chunk-local algebra shared by the chunked
// gated-delta-rule kernels (chunk_chain.hip, chunk_scan.hip): operand
// fragments, the gate tables, the decay masks and the blocked inverse.
#pragma once

#include "chunk_common.hpp"

namespace gdn {

constexpr int kC = 64;                    // tokens per chunk
constexpr float kRcpLn2 = 1.4426950216f;  // gated_delta.py:12

typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef short s4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 to_uint4(u4_t v) { return make_uint4(v[0], v[1], v[2], v[3]); }

// LDS row strides (halfs).  The LDS serves a 64-bit access 16 lanes at a
// time over 32 four-byte banks (the layouts below measure zero bank-conflict
// cycles on the K/Q tiles, against 44 % of all LDS-busy cycles with padded
// rows alone).
//
// K and Q tiles: rows of d_k + 16 halfs (a stride of 8 mod 32 dwords), and
// 8-byte chunk q of row r stored at chunk q ^ ((r / 4) mod 4).  The 16 rows of
// a left-operand read (one chunk each) then fall on 4 row phases x 4 chunk
// swizzles = 16 distinct bank pairs, and so do the 4 rows x 4 chunks of a
// transpose read; the swizzle keeps chunks q and q + 4 16 halfs apart.
// Gate table per chunk (floats): G, 2^G, 2^(G_last - G) (0 past the end),
// beta, 2^G_last; then the factors of the off-diagonal 16 x 16 decay tiles:
// 2^(G_t - G_16b) for token t of 16-token block b (G_RF), and for b = 1..3
// 2^(G_16b - G_s) for s < 16 b (G_CF + 64 (b - 1) + s).  For t >= 16 b > s
// their product is 2^(G_t - G_s), so off-diagonal tiles need no exponential;
// with log-decay gates (<= 0, G non-increasing) both factors are <= 1.
constexpr int GTS = 520;
constexpr int G_EXP = 64, G_DEC = 128, G_BETA = 192, G_LAST = 256, G_RF = 264, G_CF = 328;

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ f4_t mma(h8_t a, h8_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t zero4() { return f4_t{0.f, 0.f, 0.f, 0.f}; }

// f16 MFMA operand, round to nearest even (pairs become one v_cvt_pk_f16_f32).
// Magnitudes beyond the f16 range (65504) become +-inf, which then shows in
// the outputs and states rather than passing as a saturated value.
__device__ __forceinline__ _Float16 to_op(float x) { return static_cast<_Float16>(x); }
__device__ __forceinline__ h8_t cat(h4_t lo, h4_t hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
// Left operand, row `row` of a row-major f16 matrix, k block at column k0.
__device__ __forceinline__ h8_t afrag(const _Float16* base, int ld, int row, int k0, int g) {
  const _Float16* p = base + row * ld + k0 + 4 * g;
  return cat(*reinterpret_cast<const h4_t*>(p), *reinterpret_cast<const h4_t*>(p + 16));
}
// afrag of a swizzled K / Q tile: k0 is a multiple of 32 and g < 4, so chunk
// k0 / 4 + g lands on k0 / 4 + (g ^ a), a = (row / 4) mod 4, and chunk + 4 16
// halfs after it.
__device__ __forceinline__ h8_t kqfrag(const _Float16* base, int ld, int row, int k0, int g) {
  const _Float16* p = base + row * ld + k0 + 4 * (g ^ ((row >> 2) & 3));
  return cat(*reinterpret_cast<const h4_t*>(p), *reinterpret_cast<const h4_t*>(p + 16));
}
// Four V values read from the V buffer, which holds them in the io type
// (exact: no operand conversion on the way in).
template <class IOT> __device__ __forceinline__ void v_rows(h4_t raw, float (&x)[4]);
template <> __device__ __forceinline__ void v_rows<f16>(h4_t raw, float (&x)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = static_cast<float>(raw[e]);
}
template <> __device__ __forceinline__ void v_rows<bf16>(h4_t raw, float (&x)[4]) {
  const uint2 w = __builtin_bit_cast(uint2, raw);
  x[0] = __uint_as_float(w.x << 16);
  x[1] = __uint_as_float(w.x & 0xffff0000u);
  x[2] = __uint_as_float(w.y << 16);
  x[3] = __uint_as_float(w.y & 0xffff0000u);
}
// LDS transpose read: the 16 lanes of a group read a 4-row x 16-column block
// (lane r: row r / 4, columns 4 (r % 4)..+3) and lane r receives column r.
__device__ __forceinline__ h4_t tr_read(const _Float16* p) {
  typedef __attribute__((address_space(3))) s4_t lds_s4;
  return __builtin_bit_cast(h4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p)));
}
// Left operand of K^T for a token-major, swizzled K tile: rows of K^T =
// columns c0 + lane % 16 of K (c0 a multiple of 16), k block = tokens
// t0..t0+31 (t0 a multiple of 32) in the k order above.  Lane (lr, lg) reads
// rows r = t0 + 4 lg + lr / 4 and r + 16, whose row phase (r / 4) mod 4 is lg
// for every t0 in {0, 32}: the lane part of the address is the byte offset
// lane_tr_offset(...) from the tile, computed once, and the rest a constant.
__device__ __forceinline__ uint32_t lane_tr_offset(int ld, int lr, int lg) {
  return static_cast<uint32_t>(((4 * lg + (lr >> 2)) * ld + 4 * ((lr & 3) ^ lg)) * 2);
}
template <int LD>
__device__ __forceinline__ h8_t kq_tfrag(const char* lane_tile, int t0, int c0) {
  const char* p = lane_tile + (t0 * LD + c0) * 2;
  return cat(tr_read(reinterpret_cast<const _Float16*>(p)), tr_read(reinterpret_cast<const _Float16*>(p + 16 * LD * 2)));
}
// Right operand from two C-layout accumulator tiles (rows 0-15, rows 16-31).
__device__ __forceinline__ h8_t bfrag(f4_t a, f4_t b) {
  h8_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[e] = to_op(a[e]);
    o[4 + e] = to_op(b[e]);
  }
  return o;
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves (no LDS):
// a scan within each 16-lane row (row_shr 1, 2, 4, 8), then the row totals
// carried upwards (row_bcast 15 into rows 1 and 3, row_bcast 31 into rows 2
// and 3).  Masked-off rows and lanes shifted in from outside a row add 0.
template <int CTRL, int ROW_MASK> __device__ __forceinline__ float dpp_src(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROW_MASK, 0xf, true));
}
__device__ __forceinline__ float wave_prefix_sum(float x) {
  x += dpp_src<0x111, 0xf>(x);
  x += dpp_src<0x112, 0xf>(x);
  x += dpp_src<0x114, 0xf>(x);
  x += dpp_src<0x118, 0xf>(x);
  x += dpp_src<0x142, 0xa>(x);
  x += dpp_src<0x143, 0xc>(x);
  return x;
}

// Block-uniform index read through the scalar data cache (a scalar load: it
// is waited on with the LDS counter, never behind outstanding vector stores).
__device__ __forceinline__ int64_t uniform_index(const void* p, int64_t i, int is64) {
  typedef __attribute__((address_space(4))) const int64_t ci64;
  typedef __attribute__((address_space(4))) const int32_t ci32;
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  return is64 ? reinterpret_cast<ci64*>(a)[i] : static_cast<int64_t>(reinterpret_cast<ci32*>(a)[i]);
}

template <class ST> __device__ __forceinline__ float load_st(const ST* p) { return to_f32(*p); }
template <class ST> __device__ __forceinline__ void store_st(ST* p, float v) { *p = from_f32<ST>(v); }

// ---- 32x32 lower-triangular matrices held as C-layout tiles of X and X^T.
// x[0] = X(0,0), x[1] = X(1,0), x[2] = X(1,1); t[0] = X^T(0,0), t[1] =
// X^T(0,1), t[2] = X^T(1,1) (tile (a, b): rows 16a.., columns 16b..).
struct Tri {
  f4_t x[3], t[3];
};
// A 16 x 16 block X as C-layout tiles of X (x) and of X^T (t).  Fed to a
// 16x16x16 MFMA, the 4 halfs a lane holds of a C-layout tile of Y are the
// A operand Y^T or the B operand Y, so X W comes from (X.t, W.x) and
// (X W)^T from (W.x, X.t) with no data movement between lanes.
struct Sq {
  f4_t x, t;
};
__device__ __forceinline__ h4_t hfrag(f4_t a) {
  h4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = to_op(a[e]);
  return o;
}
__device__ __forceinline__ f4_t mma16(h4_t a, h4_t b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}
// X X for a block in both orientations.
__device__ __forceinline__ Sq sq_square(const Sq& X) {
  const h4_t xt = hfrag(X.t), xx = hfrag(X.x);
  return Sq{mma16(xt, xx, zero4()), mma16(xx, xt, zero4())};
}

// ---------------------------------------------------------------- state slots
// Addresses of one value head's state columns [col_base, ..) in a slot: a
// plain pool, or (EXT) LogState payload frames.
template <class ST, bool EXT>
struct StateSlots {
  const ChunkParams& p;
  int64_t h, col_base;
  static constexpr int64_t kRowBytes = sizeof(ST);
  __device__ __forceinline__ int64_t row_bytes() const { return p.DV * kRowBytes; }
  // Byte address of element (0, col_base) in slot s, or null for a negative
  // slot or an unmapped frame (entry < 0 or past the storage).  Rows follow
  // every row_bytes (plain pools and heads inside one frame).
  __device__ __forceinline__ char* base(int64_t s) const {
    if (s < 0) return nullptr;
    if (!EXT || !p.frames)
      return reinterpret_cast<char*>(static_cast<ST*>(p.state) + s * p.slot_stride +
                                     (p.layer * p.layer_stride + h * p.head_stride + col_base));
    if (s >= p.frame_slots) return nullptr;  // past the frame table: unmapped
    const int64_t logical = (p.layer * p.HV + h) * p.head_bytes;
    const int64_t fr = uniform_index(p.frames, s * p.fps + logical / p.frame_bytes, p.frames_is64);
    if (fr < 0 || fr >= p.num_frames) return nullptr;
    return static_cast<char*>(p.state) + fr * p.frame_bytes + logical % p.frame_bytes + col_base * kRowBytes;
  }
  // Heads spanning several frames (each frame holds whole 16-row tiles): byte
  // address of element (16 ti, col_base) of slot s, or null.
  __device__ __forceinline__ char* frame_tile(int64_t s, int ti) const {
    if (s >= p.frame_slots) return nullptr;
    const int64_t logical = (p.layer * p.HV + h) * p.head_bytes + 16 * ti * row_bytes();
    const int64_t fr = uniform_index(p.frames, s * p.fps + logical / p.frame_bytes, p.frames_is64);
    if (fr < 0 || fr >= p.num_frames) return nullptr;
    return static_cast<char*>(p.state) + fr * p.frame_bytes + logical % p.frame_bytes + col_base * kRowBytes;
  }
  // Row 16 ti in slot s (slice = base(s)), or null.
  __device__ __forceinline__ char* tile(char* slice, int64_t s, int ti) const {
    if (EXT && p.frame_rows) return s >= 0 ? frame_tile(s, ti) : nullptr;
    return slice ? slice + 16 * ti * row_bytes() : nullptr;
  }
  // Rows 16 ti + 4 g + e of every tile, at lane byte offset o (row 4 g, the lane's column).
  template <int HT>
  __device__ __forceinline__ void load(int64_t s, uint32_t o, f4_t (&hT)[HT]) const {
    char* src = EXT && p.frame_rows ? nullptr : base(s);
#pragma unroll
    for (int ti = 0; ti < HT; ++ti) {
      const char* t = tile(src, s, ti);
#pragma unroll
      for (int e = 0; e < 4; ++e) hT[ti][e] = t ? load_st(reinterpret_cast<const ST*>(t + e * row_bytes() + o)) : 0.f;
    }
  }
  template <int HT, class F>
  __device__ __forceinline__ void store(int64_t s, uint32_t o, F&& value) const {
    char* dst = EXT && p.frame_rows ? nullptr : base(s);
    if (!(EXT && p.frame_rows) && !dst) return;
#pragma unroll
    for (int ti = 0; ti < HT; ++ti) {
      const f4_t v = value(ti);
      char* t = tile(dst, s, ti);
      if (t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) store_st(reinterpret_cast<ST*>(t + e * row_bytes() + o), v[e]);
      }
    }
  }
};

// ---------------------------------------------------------------- gate tables
// Gate table of a chunk from per-lane (token) g and beta: the chunk-local
// cumulative gate in log2 units (cumsum.py:19-75) and its exponentials.  nk:
// the chunk's valid tokens.
__device__ __forceinline__ void gate_table(float* gt, int lane, int nk, float x, float bt) {
  const float G = wave_prefix_sum(x) * kRcpLn2;
  const float Gl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), nk > 0 ? nk - 1 : 0));
  gt[lane] = G;
  gt[G_EXP + lane] = fast_exp2(G);
  gt[G_DEC + lane] = lane < nk ? fast_exp2(Gl - G) : 0.f;
  gt[G_BETA + lane] = bt;
  if (lane == 0) gt[G_LAST] = fast_exp2(Gl);
}
// The off-diagonal decay factors of the same chunk.
__device__ __forceinline__ void factor_table(float* gt, int lane, float x) {
  const float G = wave_prefix_sum(x) * kRcpLn2;
  const float G16 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), 16));
  const float G32 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), 32));
  const float G48 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), 48));
  const float G0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), 0));
  gt[G_RF + lane] = fast_exp2(G - (lane < 16 ? G0 : lane < 32 ? G16 : lane < 48 ? G32 : G48));
  gt[G_CF + lane] = lane < 16 ? fast_exp2(G16 - G) : 0.f;
  gt[G_CF + 64 + lane] = lane < 32 ? fast_exp2(G32 - G) : 0.f;
  gt[G_CF + 128 + lane] = lane < 48 ? fast_exp2(G48 - G) : 0.f;
}

// ---------------------------------------------------------------- decay masks
// Entries (t, s0..s0+3) of a row-orientation tile -> masked values.
__device__ __forceinline__ f4_t masked(const float* gt, f4_t s, int t, int s0, bool strict, bool with_beta) {
  const f4_t gs = *reinterpret_cast<const f4_t*>(gt + s0);
  const float gti = gt[t];
  const float bt = with_beta ? gt[G_BETA + t] : 1.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool keep = strict ? t > s0 + e : t >= s0 + e;
    // G is a running sum of log-decays, so kept entries (t >= s) have a
    // non-positive exponent; a dropped entry's exponent may overflow to
    // inf, which the select discards.
    s[e] = keep ? bt * s[e] * fast_exp2(gti - gs[e]) : 0.f;
  }
  return s;
}
// The same for a tile whose rows t lie in 16-token block t / 16 >= 1 and
// whose columns lie in earlier blocks (every entry kept): the decay from
// the gate table's row and boundary factors.
__device__ __forceinline__ f4_t masked_off(const float* gt, f4_t s, int t, int s0, bool with_beta) {
  const f4_t cf = *reinterpret_cast<const f4_t*>(gt + G_CF + 64 * ((t >> 4) - 1) + s0);
  const float r = with_beta ? gt[G_RF + t] * gt[G_BETA + t] : gt[G_RF + t];
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] = r * s[e] * cf[e];
  return s;
}

// ---------------------------------------------------------------- blocked inverse
// A = (I + L)^-1 of the 32-token half whose rows start at r0, blocked into
// 16 x 16 blocks: with L = [D0 0; O D1], A = [A0 0; -A1 O A0  A1], and each
// (I + D)^-1 = (I - D)(I + D^2)(I + D^4)(I + D^8) (D strictly lower
// triangular, so D^16 = 0).  In two parts:
//   first:  L, D^2, D^4, G = (I - D)(I + D^2) for both diagonal blocks
//   second: D^8, A_i = G (I + D^4)(I + D^8), -A1 O A0.
// Block 1 is needed only as A1^T (the output and -A1 O A0 take that form);
// block 0 also as A0 (the right factor of O A0).
struct HalfInverse {
  Sq D4[2], G[2];
  f4_t Ot;  // C-layout tile of O^T
  // K: a swizzled token-major tile; gt: its gate table.
  template <int KS, int LDK>
  __device__ __forceinline__ void first(const _Float16* K, const float* gt, int r0, int lr, int lg) {
    f4_t s00 = zero4(), s11 = zero4(), s01 = zero4();
    h8_t k0[KS], k1[KS];
#pragma unroll
    for (int m = 0; m < KS; ++m) {
      k0[m] = kqfrag(K, LDK, r0 + lr, 32 * m, lg);
      k1[m] = kqfrag(K, LDK, r0 + 16 + lr, 32 * m, lg);
    }
#pragma unroll
    for (int m = 0; m < KS; ++m) {
      s00 = mma(k0[m], k0[m], s00);
      s11 = mma(k1[m], k1[m], s11);
      s01 = mma(k0[m], k1[m], s01);  // C layout: entry (4g + e, 16 + c) of S^T
    }
    // C-layout tiles of L (row 4g + e, col c) and of L^T (row 4g + e, col c
    // of L^T = entry (c, 4g + e) of L); S is symmetric on the diagonal tiles.
    auto lmask_c = [&](f4_t s, int t0, int sc) {  // entries (t0 + 4g + e, sc + c)
      const f4_t gt4 = *reinterpret_cast<const f4_t*>(gt + t0 + 4 * lg);
      const f4_t bt4 = *reinterpret_cast<const f4_t*>(gt + G_BETA + t0 + 4 * lg);
      const float gsc = gt[sc + lr];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        s[e] = (t0 + 4 * lg + e > sc + lr) ? bt4[e] * s[e] * fast_exp2(gt4[e] - gsc) : 0.f;
      return s;
    };
    auto lmask_t = [&](f4_t s, int tc, int s0) {  // entries (tc + c, s0 + 4g + e)
      return masked(gt, s, tc + lr, s0 + 4 * lg, true, true);
    };
    // L.x[1], the off-diagonal block itself, is not needed: O enters only
    // as the left factor of O A0, that is through O^T (L.t[1], from the
    // table's row and boundary factors)
    Tri L;
    L.x[0] = lmask_c(s00, r0, r0);
    L.x[2] = lmask_c(s11, r0 + 16, r0 + 16);
    L.t[0] = lmask_t(s00, r0, r0);
    L.t[1] = masked_off(gt, s01, r0 + 16 + lr, r0 + 4 * lg, true);
    L.t[2] = lmask_t(s11, r0 + 16, r0 + 16);
    const f4_t id = f4_t{4 * lg == lr ? 1.f : 0.f, 4 * lg + 1 == lr ? 1.f : 0.f, 4 * lg + 2 == lr ? 1.f : 0.f,
                         4 * lg + 3 == lr ? 1.f : 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const Sq D{L.x[2 * b], L.t[2 * b]};
      const Sq D2 = sq_square(D);
      D4[b] = sq_square(D2);
      const Sq F{id - D.x, id - D.t};
      const h4_t d2x = hfrag(D2.x), ft = hfrag(F.t);
      G[b].t = mma16(d2x, ft, F.t);
      G[b].x = b == 0 ? mma16(ft, d2x, F.x) : zero4();
    }
    Ot = L.t[1];
  }
  // C-layout tiles of A^T: tile (a, b) holds row 16 b + c, columns 16 a + 4 g..+3
  // of A (a00, a10 = -A1 O A0, a11).
  __device__ __forceinline__ void second(f4_t& a00, f4_t& a10, f4_t& a11) const {
    Sq Ai[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const h4_t d4x = hfrag(D4[b].x), d4t = hfrag(D4[b].t), gt4 = hfrag(G[b].t);
      const h4_t d8x = hfrag(mma16(d4t, d4x, zero4()));
      const Sq H{b == 0 ? mma16(gt4, d4x, G[b].x) : zero4(), mma16(d4x, gt4, G[b].t)};
      const h4_t ht = hfrag(H.t);
      Ai[b].t = mma16(d8x, ht, H.t);
      Ai[b].x = b == 0 ? mma16(ht, d8x, H.x) : zero4();
    }
    // T = O A0, then (-A1 T)^T = -T^T A1^T
    const f4_t Tx = mma16(hfrag(Ot), hfrag(Ai[0].x), zero4());
    a00 = Ai[0].t;
    a10 = -mma16(hfrag(Tx), hfrag(Ai[1].t), zero4());
    a11 = Ai[1].t;
  }
};

}  // namespace gdn
