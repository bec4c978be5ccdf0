// rq_cgemm.hip -- y = x W^T for many activation rows (prefill) on the f16
// matrix cores of gfx950, with the weights as their integer codes.
//
// A quantized weight is a small integer code times a scale shared by a run of
// weights: Q8_0 / Q4_0 / Q5_0 d q, Q6_K d sc (q - 32), Marlin s (q - 8), and
// for Q4_K / Q5_K d (sc q) - dmin m, where sc q <= 63 * 31 = 1953.  All of
// these integers are exact in f16 (below 2048), so the matrix cores take them
// as they are and the scales go onto the f32 sums afterwards.  Against
// decoding every weight to f32 and splitting it into two bf16 limbs, a code
// costs about 1.3 VALU instructions instead of 5, and an f32 activation two
// MFMAs (its two limbs) instead of three.
//
// Activations (k_cg_pack, one pass over x before the product): every row is
// scaled by a power of two so that its largest finite magnitude lies in
// [2^14, 2^15), and split into f16 limbs: hi = f16(x), lo = f16(x - hi), 22
// significant bits, subnormals at 2^-39 of the row's largest value.  bf16
// rows take one limb (8 significant bits), f16 rows one, unscaled.  The limbs
// are stored in the order in which a wave reads them: one MFMA A operand (32
// rows x 16 inputs) is 1 KB of consecutive memory, lane l at byte 16 l.  So
// the product needs no LDS for its operands and no barrier: each wave streams
// its own operands from L2 with contiguous loads, and the waves of a
// workgroup split K and meet once in LDS at the end.
//
// Product (k_cgemm): a wave owns a 64 x 64 tile of y over its share of K (2 x 2
// MFMA tiles of 32 x 32; 32 x 64 for at most 32 rows), KG waves (8 at most) a workgroup.  Per chunk of 64
// inputs and weight row a lane loads its bytes of the row (the two lanes of a
// row take the two 8-input halves of every 16-input step), makes four f16 B
// operands of them, and sums S over a scale's run from zero; S joins the f32
// accumulator with one FMA per output, so a partial sum is at most 64
// products long before it is added up.
//
// Mins (Q4_K / Q5_K): the packer also sums each 32-input sub-block of x in
// f32 and stores the sum as three bf16 limbs; after its chunks a wave adds
// -dmin m (two bf16 limbs, 16 of its 17 bits) times these sums on the bf16
// matrix cores, three MFMAs per 256 inputs.
//
// Bound: the matrix cores (f16 dense 2.5 PFLOP/s, one pass for 16-bit
// activations, two for f32) and the vector loads of the operands (64 bytes a
// clock and CU).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "rq_e4m3.h"
#include "rq_formats.h"
#include "rq_internal.h"

namespace rq {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 cg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// K positions of the eight values that lane half g holds for step s (16
// inputs) of a chunk: 16 s + 8 g .. + 7 in the order 0, 2, 1, 3, 4, 6, 5, 7
// (GGUF formats: a 16-bit mask of a word of quant bytes keeps bytes 0 and 2),
// or, for Marlin records, inputs 32 g + 8 s .. + 7 in the order 0, 4, 1, 5, 2,
// 6, 3, 7 (a mask of a word of nibbles keeps nibbles i and i + 4).
enum { MAP_GGUF = 0, MAP_MARLIN = 1 };

// Flags of a row beside its exponent.
constexpr int kRowNonFinite = 1 << 20;

__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t h2_bits(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 splat_h2(float v) {
  const _Float16 h = (_Float16)v;
  return (f16x2){h, h};
}
// f16 pairs 1024 + q of bytes 0, 2 (1, 3) of a word of codes q < 256.
__device__ __forceinline__ uint32_t code_pair02(uint32_t q) { return __builtin_amdgcn_perm(0x64646464u, q, 0x04020400u); }
__device__ __forceinline__ uint32_t code_pair13(uint32_t q) { return __builtin_amdgcn_perm(0x64646464u, q, 0x04030401u); }

// Eight codes (two words of bytes) minus bias as f16, exact.
__device__ __forceinline__ f16x8 codes_minus(uint32_t a, uint32_t b, float bias) {
  const f16x2 c = splat_h2(-1024.0f - bias);
  const u32x4 r = {h2_bits(as_h2(code_pair02(a)) + c), h2_bits(as_h2(code_pair13(a)) + c),
                   h2_bits(as_h2(code_pair02(b)) + c), h2_bits(as_h2(code_pair13(b)) + c)};
  return __builtin_bit_cast(f16x8, r);
}
// The low (high) nibbles of eight bytes as f16 codes times sc (sc q < 2048),
// exact: one rounding of sc (1024 + q) - 1024 sc, or, with the high nibbles
// left in place, of (sc / 16) (1024 + 16 q) - 64 sc.
__device__ __forceinline__ f16x8 nibbles_times(uint32_t a, uint32_t b, bool high, f16x2 sc) {
  const uint32_t mask = high ? 0x00F000F0u : 0x000F000Fu, magic = 0x64006400u;
  const f16x2 s = high ? sc * splat_h2(0.0625f) : sc, c = sc * splat_h2(high ? -64.0f : -1024.0f);
  const u32x4 r = {h2_bits(__builtin_elementwise_fma(as_h2((a & mask) | magic), s, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2(((a >> 8) & mask) | magic), s, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2((b & mask) | magic), s, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2(((b >> 8) & mask) | magic), s, c))};
  return __builtin_bit_cast(f16x8, r);
}
// Eight codes (bytes) times sc.
__device__ __forceinline__ f16x8 codes_times(uint32_t a, uint32_t b, f16x2 sc) {
  const f16x2 c = sc * splat_h2(-1024.0f);
  const u32x4 r = {h2_bits(__builtin_elementwise_fma(as_h2(code_pair02(a)), sc, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2(code_pair13(a)), sc, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2(code_pair02(b)), sc, c)),
                   h2_bits(__builtin_elementwise_fma(as_h2(code_pair13(b)), sc, c))};
  return __builtin_bit_cast(f16x8, r);
}
// An integer below 64 in byte i of v as an f16 pair of itself.
template <int I>
__device__ __forceinline__ f16x2 splat_byte(uint32_t v) {
  const uint32_t p = __builtin_amdgcn_perm(0x64646464u, v, I ? 0x04010401u : 0x04000400u);
  return as_h2(p) + splat_h2(-1024.0f);
}

// ---- weights --------------------------------------------------------------
//
// A wave takes K in pairs of chunks (128 inputs): the 64 rows' bytes of a pair
// are loaded with neighbouring lanes on neighbouring 16-byte pieces (a lane on
// its own row costs the vector cache one access a lane: 92 accesses an
// instruction measured, against 16), pass through the wave's own LDS region
// (no barrier: a wave's LDS accesses stay in order) and come back a lane a
// row.  The loads of the next pair are in flight while a pair is multiplied.
//
// A decoder gives Stage (a pair's bytes in registers, filled by issue and
// written to LDS by commit), STRIDE (LDS bytes of a row, an odd multiple of
// 16, so that the rows start on different banks), and for one lane (row of
// 32 ni + lane % 32, half g) and chunk c of the pair the four B operands of the
// chunk's 16-input steps and the scales of their sums: GRP steps share one.
// A tile's 64 rows all exist: a ragged last tile starts at row n - 64 (n >= 64)
// and computes some rows a second time, with the same result.

__device__ __forceinline__ u32x4 ld16(const uint8_t *base, uint32_t off) {
  return *reinterpret_cast<const u32x4 *>(base + off);
}
__device__ __forceinline__ u32x2 ld8(const uint8_t *base, uint32_t off) {
  return *reinterpret_cast<const u32x2 *>(base + off);
}
typedef __attribute__((address_space(3))) uint8_t lds_u8;
__device__ __forceinline__ void st16(lds_u8 *p, u32x4 v) {
  *reinterpret_cast<__attribute__((address_space(3))) u32x4 *>(p) = v;
}
__device__ __forceinline__ u32x4 rd16(const lds_u8 *p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4 *>(p);
}
__device__ __forceinline__ u32x2 rd8(const lds_u8 *p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x2 *>(p);
}
__device__ __forceinline__ uint32_t rd4(const lds_u8 *p) {
  return *reinterpret_cast<const __attribute__((address_space(3))) uint32_t *>(p);
}

// The 64 rows of a wave's tile: first row n0, kp pairs (128 inputs) a row.
struct Tile {
  const uint8_t *w, *aux;
  int64_t n0;
  int kp;
};

// Scales and mins of Q4_K / Q5_K sub-blocks 2c, 2c + 1 (scale_min_k4,
// dequant_k.rs:8-16) as integers.
__device__ __forceinline__ void k4_pair(const u32x4 &hd, int c, uint32_t &sc, uint32_t &mn) {
  const int sh = 16 * (c & 1);
  const uint32_t Y = hd.y >> sh, Z = hd.z >> sh, W = hd.w >> sh;
  const uint32_t low = opaque(c < 2 ? 0xFFFFFFFFu : 0u);
  sc = opaque((Y & 0x3F3Fu & low) | (((W & 0x0F0Fu) | ((Y >> 2) & 0x3030u)) & ~low));
  mn = opaque((Z & 0x3F3Fu & low) | ((((W >> 4) & 0x0F0Fu) | ((Z >> 2) & 0x3030u)) & ~low));
}

// Formats of 256-element blocks hold two pairs a block: pair j of row r is
// half P & 1 of block P >> 1, P = r kp + j (rows may start inside a block).
// Rows an even number apart lie a whole number of blocks apart.
template <uint32_t BLOCK>
struct HalfBlocks {
  const uint8_t *base;  // the block that holds row n0's first pair
  uint32_t p0;          // its half
  uint32_t two;         // bytes from a row to the row two below it
  __device__ void init(const uint8_t *w, const Tile &t) {
    const uint64_t P = (uint64_t)t.n0 * (uint64_t)t.kp;
    base = w + (P >> 1) * BLOCK;
    p0 = (uint32_t)(P & 1u);
    two = (uint32_t)t.kp * BLOCK;
  }
  __device__ uint32_t pair(const Tile &t, int row) const { return p0 + (uint32_t)(row * t.kp); }
};

template <bool Q5>
struct CgK4 {
  static constexpr int GRP = 4, MAP = MAP_GGUF, STRIDE = Q5 ? 112 : 80;
  static constexpr bool MINS = true;
  static constexpr uint32_t BLOCK = Q5 ? 176u : 144u, QS = Q5 ? 48u : 16u;
  HalfBlocks<BLOCK> hb;
  uint32_t pq, ph, pr;  // pair 0 of the rows lane / 4 (quants), lane / 2 (high bits) and lane (header)
  struct Stage {
    u32x4 hd, q[4], h[2];
  };
  __device__ void init(const Tile &t, int lane) {
    hb.init(t.w, t);
    pq = hb.pair(t, lane >> 2);
    if constexpr (Q5) ph = hb.pair(t, lane >> 1);
    pr = hb.pair(t, lane);
  }
  __device__ void issue(Stage &s, int j, int lane) const {
    s.hd = ld16(hb.base, ((pr + j) >> 1) * BLOCK);
    const uint32_t P = pq + j, o = (P >> 1) * BLOCK + (P & 1u) * 64u + QS + 16u * (lane & 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) s.q[i] = ld16(hb.base + (uint64_t)(8 * i) * hb.two, o);
    if constexpr (Q5) {
      const uint32_t oh = ((ph + j) >> 1) * BLOCK + 16u + 16u * (lane & 1);
#pragma unroll
      for (int i = 0; i < 2; ++i) s.h[i] = ld16(hb.base + (uint64_t)(16 * i) * hb.two, oh);
    }
  }
  __device__ static void commit(const Stage &s, lds_u8 *L, int lane) {
    st16(L + STRIDE * lane, s.hd);
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(L + STRIDE * (16 * i + (lane >> 2)) + 16 + 16 * (lane & 3), s.q[i]);
    if constexpr (Q5) {
#pragma unroll
      for (int i = 0; i < 2; ++i) st16(L + STRIDE * (32 * i + (lane >> 1)) + 80 + 16 * (lane & 1), s.h[i]);
    }
  }
  // mins: the chunk's two mins as a bf16 pair; dm: -dmin
  __device__ void decode(const lds_u8 *L, int ni, int c, int j, int lane, f16x8 (&b)[4], float (&d)[1], uint32_t &mins,
                         float &dm) const {
    const int g = lane >> 5;
    const lds_u8 *r = L + STRIDE * (32 * ni + (lane & 31));
    const u32x4 hd = rd16(r);
    const u32x2 q0 = rd8(r + 16 + 32 * c + 8 * g), q1 = rd8(r + 32 + 32 * c + 8 * g);
    const int cb = 2 * (int)((pr + j) & 1u) + c;  // chunk of the block (rows 32 apart start in the same half)
    uint32_t sc, mn;
    k4_pair(hd, cb, sc, mn);
    const f16x2 s0 = splat_byte<0>(sc), s1 = splat_byte<1>(sc);
    d[0] = h2f(hd.x);
    dm = -h2f(hd.x >> 16);
    mins = pk_bf16(ub(mn, 0), ub(mn, 1));
    if constexpr (!Q5) {
      b[0] = nibbles_times(q0.x, q0.y, false, s0);
      b[1] = nibbles_times(q1.x, q1.y, false, s0);
      b[2] = nibbles_times(q0.x, q0.y, true, s1);
      b[3] = nibbles_times(q1.x, q1.y, true, s1);
    } else {
      const u32x2 h0 = rd8(r + 80 + 8 * g), h1 = rd8(r + 96 + 8 * g);
      const uint32_t q[4] = {q0.x, q0.y, q1.x, q1.y}, h[4] = {h0.x, h0.y, h1.x, h1.y};
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t t = h[i] >> (2 * cb);
        lo[i] = (q[i] & 0x0F0F0F0Fu) | ((t & 0x01010101u) << 4);
        hi[i] = ((q[i] >> 4) & 0x0F0F0F0Fu) | ((t & 0x02020202u) << 3);
      }
      b[0] = codes_times(lo[0], lo[1], s0);
      b[1] = codes_times(lo[2], lo[3], s0);
      b[2] = codes_times(hi[0], hi[1], s1);
      b[3] = codes_times(hi[2], hi[3], s1);
    }
  }
};

// Q6_K on the split layout: a pair is a half block (ql 64 bytes, qh 32, eight
// scales), chunk c its nibble c; sixteen weights share d sc.
struct CgQ6K {
  static constexpr int GRP = 1, MAP = MAP_GGUF, STRIDE = 112;
  static constexpr bool MINS = false;
  HalfBlocks<208> hb;
  const uint8_t *aux;
  uint32_t pl, ph, pr;
  struct Stage {
    u32x4 q[4], h[2];
    u32x2 sc;
    uint32_t d;
  };
  __device__ void init(const Tile &t, int lane) {
    hb.init(t.w, t);
    aux = t.aux + 2 * (((uint64_t)t.n0 * (uint64_t)t.kp) >> 1);
    pl = hb.pair(t, lane >> 2);
    ph = hb.pair(t, lane >> 1);
    pr = hb.pair(t, lane);
  }
  __device__ void issue(Stage &s, int j, int lane) const {
    const uint32_t R = pr + j;
    s.sc = ld8(hb.base, (R >> 1) * 208u + 192u + 8u * (R & 1u));
    s.d = *reinterpret_cast<const uint16_t *>(aux + (R & ~1u));
    const uint32_t P = pl + j, o = (P >> 1) * 208u + (P & 1u) * 64u + 16u * (lane & 3);
    const uint32_t H = ph + j, oh = (H >> 1) * 208u + 128u + (H & 1u) * 32u + 16u * (lane & 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) s.q[i] = ld16(hb.base + (uint64_t)(8 * i) * hb.two, o);
#pragma unroll
    for (int i = 0; i < 2; ++i) s.h[i] = ld16(hb.base + (uint64_t)(16 * i) * hb.two, oh);
  }
  __device__ static void commit(const Stage &s, lds_u8 *L, int lane) {
    st16(L + STRIDE * lane + 96, (u32x4){s.sc.x, s.sc.y, s.d, 0u});
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(L + STRIDE * (16 * i + (lane >> 2)) + 16 * (lane & 3), s.q[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i) st16(L + STRIDE * (32 * i + (lane >> 1)) + 64 + 16 * (lane & 1), s.h[i]);
  }
  __device__ void decode(const lds_u8 *L, int ni, int c, int, int lane, f16x8 (&b)[4], float (&d)[4], uint32_t &,
                         float &) const {
    const int g = lane >> 5, sh = 4 * c;
    const lds_u8 *r = L + STRIDE * (32 * ni + (lane & 31));
    const u32x2 h0 = rd8(r + 64 + 8 * g), h1 = rd8(r + 80 + 8 * g);
    auto lowc = [&](uint32_t l, uint32_t h) { return ((l >> sh) & 0x0F0F0F0Fu) | (((h >> sh) & 0x03030303u) << 4); };
    auto highc = [&](uint32_t l, uint32_t h) { return ((l >> sh) & 0x0F0F0F0Fu) | (((h >> sh) & 0x0C0C0C0Cu) << 2); };
    static_for<4>([&](auto S) {
      constexpr int s = decltype(S)::value;
      const u32x2 l = rd8(r + 16 * s + 8 * g);
      const u32x2 h = s % 2 ? h1 : h0;
      if constexpr (s < 2) b[s] = codes_minus(lowc(l.x, h.x), lowc(l.y, h.y), 32.0f);
      else b[s] = codes_minus(highc(l.x, h.x), highc(l.y, h.y), 32.0f);
    });
    const uint32_t sc = rd4(r + 96 + 4 * c);
    const float dd = h2f(rd4(r + 104));
#pragma unroll
    for (int s = 0; s < 4; ++s) d[s] = dd * (float)(int8_t)((sc >> (8 * s)) & 0xFFu);
  }
};

// Q8_0 on the split layout: int8 quants in element order, d per 32.
struct CgQ8 {
  static constexpr int GRP = 2, MAP = MAP_GGUF, STRIDE = 144;
  static constexpr bool MINS = false;
  const uint8_t *base, *aux;
  uint32_t oq, oa, step;
  struct Stage {
    u32x4 q[8];
    u32x2 d;
  };
  __device__ void init(const Tile &t, int lane) {
    base = t.w + (uint64_t)t.n0 * (uint64_t)t.kp * 128u;
    aux = t.aux + (uint64_t)t.n0 * (uint64_t)t.kp * 8u;
    oq = (uint32_t)((lane >> 3) * t.kp) * 128u + 16u * (lane & 7);
    oa = (uint32_t)(lane * t.kp) * 8u;
    step = (uint32_t)t.kp * 1024u;
  }
  __device__ void issue(Stage &s, int j, int) const {
    s.d = ld8(aux + 8u * (uint32_t)j, oa);
    const uint8_t *b = base + 128u * (uint32_t)j;
#pragma unroll
    for (int i = 0; i < 8; ++i) s.q[i] = ld16(b + (uint64_t)i * step, oq);
  }
  __device__ static void commit(const Stage &s, lds_u8 *L, int lane) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x2 *>(L + STRIDE * lane + 128) = s.d;
#pragma unroll
    for (int i = 0; i < 8; ++i) st16(L + STRIDE * (8 * i + (lane >> 3)) + 16 * (lane & 7), s.q[i]);
  }
  __device__ void decode(const lds_u8 *L, int ni, int c, int, int lane, f16x8 (&b)[4], float (&d)[2], uint32_t &,
                         float &) const {
    const lds_u8 *r = L + STRIDE * (32 * ni + (lane & 31));
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u32x2 q = rd8(r + 64 * c + 16 * s + 8 * (lane >> 5));
      b[s] = codes_minus(q.x ^ 0x80808080u, q.y ^ 0x80808080u, 128.0f);
    }
    const uint32_t dd = rd4(r + 128 + 4 * c);
    d[0] = h2f(dd);
    d[1] = h2f(dd >> 16);
  }
};

// Q4_0 / Q5_0 on the split layout: element i of a block is nibble i / 16 of
// byte i % 16 (plus qh bit i), d (q - 8) or d (q - 16).
template <bool Q5>
struct CgQx0 {
  static constexpr int GRP = 2, MAP = MAP_GGUF, STRIDE = Q5 ? 112 : 80;
  static constexpr bool MINS = false;
  const uint8_t *base, *aux;
  uint32_t oq, oa, step;
  struct Stage {
    u32x4 q[4], rec[2];  // Q5_0: {qh, d, ..} of two blocks; Q4_0: rec[0].xy the four d
  };
  __device__ void init(const Tile &t, int lane) {
    base = t.w + (uint64_t)t.n0 * (uint64_t)t.kp * 64u;
    aux = t.aux + (uint64_t)t.n0 * (uint64_t)t.kp * (Q5 ? 32u : 8u);
    oq = (uint32_t)((lane >> 2) * t.kp) * 64u + 16u * (lane & 3);
    oa = Q5 ? (uint32_t)((lane >> 1) * t.kp) * 32u + 16u * (lane & 1) : (uint32_t)(lane * t.kp) * 8u;
    step = (uint32_t)t.kp * 1024u;  // 16 rows of quants, 32 rows of Q5_0 records
  }
  __device__ void issue(Stage &s, int j, int) const {
    const uint8_t *a = aux + (Q5 ? 32u : 8u) * (uint32_t)j, *b = base + 64u * (uint32_t)j;
    if constexpr (Q5) {
#pragma unroll
      for (int i = 0; i < 2; ++i) s.rec[i] = ld16(a + (uint64_t)i * step, oa);
    } else {
      const u32x2 v = ld8(a, oa);
      s.rec[0].x = v.x;
      s.rec[0].y = v.y;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s.q[i] = ld16(b + (uint64_t)i * step, oq);
  }
  __device__ static void commit(const Stage &s, lds_u8 *L, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(L + STRIDE * (16 * i + (lane >> 2)) + 16 * (lane & 3), s.q[i]);
    if constexpr (Q5) {
#pragma unroll
      for (int i = 0; i < 2; ++i) st16(L + STRIDE * (32 * i + (lane >> 1)) + 64 + 16 * (lane & 1), s.rec[i]);
    } else {
      *reinterpret_cast<__attribute__((address_space(3))) u32x2 *>(L + STRIDE * lane + 64) =
          (u32x2){s.rec[0].x, s.rec[0].y};
    }
  }
  __device__ void decode(const lds_u8 *L, int ni, int c, int, int lane, f16x8 (&b)[4], float (&d)[2], uint32_t &,
                         float &) const {
    const int g = lane >> 5;
    const lds_u8 *r = L + STRIDE * (32 * ni + (lane & 31));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u32x2 q = rd8(r + 32 * c + 16 * i + 8 * g);
      uint32_t lo0 = q.x & 0x0F0F0F0Fu, lo1 = q.y & 0x0F0F0F0Fu;
      uint32_t hi0 = (q.x >> 4) & 0x0F0F0F0Fu, hi1 = (q.y >> 4) & 0x0F0F0F0Fu;
      if constexpr (Q5) {
        const u32x2 rec = rd8(r + 64 + 16 * c + 8 * i);
        const uint32_t qh = rec.x >> (8 * g);
        // four bits of a nibble to bit 4 of four bytes
        auto spread = [](uint32_t n) { return ((n * 0x00204081u) & 0x01010101u) << 4; };
        lo0 |= spread(qh & 15u);
        lo1 |= spread((qh >> 4) & 15u);
        hi0 |= spread((qh >> 16) & 15u);
        hi1 |= spread((qh >> 20) & 15u);
        d[i] = h2f(rec.y);
      }
      b[2 * i] = codes_minus(lo0, lo1, Q5 ? 16.0f : 8.0f);
      b[2 * i + 1] = codes_minus(hi0, hi1, Q5 ? 16.0f : 8.0f);
    }
    if constexpr (!Q5) {
      const uint32_t dd = rd4(r + 64 + 4 * c);
      d[0] = h2f(dd);
      d[1] = h2f(dd >> 16);
    }
  }
};

// Marlin INT4: a pair is four 32-input records of the row (records of
// neighbouring rows are consecutive), chunk c records 2c and 2c + 1; lane
// half g holds record g, step s its word s; nibbles i and i + 4 of a word
// share a register.
struct CgMarlin {
  static constexpr int GRP = 4, MAP = MAP_MARLIN, STRIDE = 80;
  static constexpr bool MINS = false;
  const uint8_t *base;
  int64_t stride;  // bytes between records of a row
  uint32_t orow;
  int kc;
  struct Stage {
    u32x4 q[4];
  };
  __device__ void init(const Tile &t, int lane) {
    base = t.w + 16 * t.n0;
    orow = 16u * (uint32_t)lane;
  }
  __device__ void issue(Stage &s, int j, int) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * j + i;  // past the end: any record (its activations are zero)
      s.q[i] = ld16(base + (c < kc ? c : kc - 1) * stride, orow);
    }
  }
  __device__ static void commit(const Stage &s, lds_u8 *L, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(L + STRIDE * lane + 16 * i, s.q[i]);
  }
  __device__ void decode(const lds_u8 *L, int ni, int c, int, int lane, f16x8 (&b)[4], float (&d)[1], uint32_t &,
                         float &) const {
    const f16x2 m8 = splat_h2(-1032.0f), m72 = splat_h2(-72.0f), s16 = splat_h2(0.0625f);
    const u32x4 q = rd16(L + STRIDE * (32 * ni + (lane & 31)) + 32 * c + 16 * (lane >> 5));
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint32_t t0 = q[s], t1 = q[s] >> 8;
      const u32x4 r = {h2_bits(as_h2((t0 & 0x000F000Fu) | 0x64006400u) + m8),
                       h2_bits(__builtin_elementwise_fma(as_h2((t0 & 0x00F000F0u) | 0x64006400u), s16, m72)),
                       h2_bits(as_h2((t1 & 0x000F000Fu) | 0x64006400u) + m8),
                       h2_bits(__builtin_elementwise_fma(as_h2((t1 & 0x00F000F0u) | 0x64006400u), s16, m72))};
      b[s] = __builtin_bit_cast(f16x8, r);
    }
    d[0] = 1.0f;
  }
};

// ---- activations ----------------------------------------------------------

// Packed layout of one call, np pairs of chunks a row: limbs [row tile of 32]
// [chunk][limb][step][lane] of 16 bytes, sub-block sums [row tile][pair][lane]
// of 16 bytes (bf16 limbs of the pair's four sums: hi and mid in lanes 0..31,
// lo and zeros in lanes 32..63), and one int per row: its exponent and
// kRowNonFinite.
constexpr int kPackThreads = 512;

// RW rows a workgroup (row = thread % RW, so that the 16-byte pieces of
// neighbouring rows leave as consecutive bytes), eight inputs a piece, B
// pieces a thread and batch.  A row of one batch stays in registers between
// its maximum and its limbs.
template <int XT, int NL, int MAP, bool SUMS, int RW, int B>
__global__ __launch_bounds__(kPackThreads) void k_cg_pack(const void *__restrict__ x, int64_t m, int64_t k, int np,
                                                          bool vec, uint8_t *__restrict__ xp,
                                                          uint8_t *__restrict__ xsum, int *__restrict__ rexp) {
  constexpr int TR = kPackThreads / RW;  // threads of a row
  __shared__ float red[kPackThreads / 64][RW];
  __shared__ int bad[RW];
  const int tid = threadIdx.x, rl = tid % RW, q0 = tid / RW;
  const int64_t row = (int64_t)blockIdx.x * RW + rl;
  const int64_t rowc = row < m ? row : m - 1;
  const int pieces = 16 * np;  // of a row, padding included
  float v[B][8];
  auto load = [&](int base) {
    if (vec) {
      // unconditional loads on clamped pieces, all issued before the first use
      u32x4 raw[B][XT == RQ_F32 ? 2 : 1];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int64_t c0 = 8 * (int64_t)(base + q0 + TR * i), cc = c0 < k ? c0 : k - 8;
        const uint8_t *src = static_cast<const uint8_t *>(x) + (rowc * k + cc) * (XT == RQ_F32 ? 4 : 2);
        raw[i][0] = *reinterpret_cast<const u32x4 *>(src);
        if constexpr (XT == RQ_F32) raw[i][1] = *reinterpret_cast<const u32x4 *>(src + 16);
      }
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const bool live = 8 * (int64_t)(base + q0 + TR * i) < k && row < m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float e0, e1;
          if constexpr (XT == RQ_F32) {
            e0 = __uint_as_float(raw[i][j >> 1][2 * (j & 1)]);
            e1 = __uint_as_float(raw[i][j >> 1][2 * (j & 1) + 1]);
          } else {
            const uint32_t u = raw[i][0][j];
            e0 = XT == RQ_BF16 ? __uint_as_float(u << 16) : h2f(u);
            e1 = XT == RQ_BF16 ? __uint_as_float(u & 0xFFFF0000u) : h2f(u >> 16);
          }
          v[i][2 * j] = live ? e0 : 0.0f;
          v[i][2 * j + 1] = live ? e1 : 0.0f;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int64_t c = 8 * (int64_t)(base + q0 + TR * i) + j;
          v[i][j] = row < m && c < k ? load_x1(x, XT, rowc * k + c) : 0.0f;
        }
    }
  };
  if (tid < RW) bad[tid] = 0;
  float amax = 0.0f;
  bool nonfin = false;
  for (int base = 0; base < pieces; base += TR * B) {
    load(base);
#pragma unroll
    for (int i = 0; i < B; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = fabsf(v[i][j]);
        const bool fin = a <= 3.4028235e38f;
        amax = fmaxf(amax, fin ? a : 0.0f);
        nonfin |= !fin;
      }
  }
#pragma unroll
  for (int off = RW; off < 64; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  if ((tid & 63) < RW) red[tid >> 6][rl] = amax;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPackThreads / 64; ++i) amax = fmaxf(amax, red[i][rl]);
  if (nonfin) bad[rl] = 1;
  // x 2^-e: the largest finite magnitude in [2^14, 2^15) (f16 rows as they are)
  int e = 0;
  if (XT != RQ_F16 && amax > 0.0f) e = __builtin_amdgcn_frexp_expf(amax) - 15;
  __syncthreads();
  if (q0 == 0) rexp[row] = (e & 0xFFFF) | (bad[rl] ? kRowNonFinite : 0);

  const int64_t mt = row >> 5;
  const int r32 = (int)(row & 31);
  for (int base = 0; base < pieces; base += TR * B) {
    if (pieces > TR * B) load(base);
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int p = base + q0 + TR * i;
      float t[8];
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] = __builtin_amdgcn_ldexpf(v[i][j], -e);
      if constexpr (SUMS) {
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += t[j];
        sum += __shfl_xor(sum, RW);  // the four pieces of a sub-block: threads RW apart
        sum += __shfl_xor(sum, 2 * RW);
      }
      if (p < pieces) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // the pair's inputs (MAP_GGUF: 0 2, 1 3, 4 6, 5 7; MAP_MARLIN: i and i + 4)
          const int i0 = MAP == MAP_MARLIN ? j : (j >> 1) * 4 + (j & 1), i1 = i0 + (MAP == MAP_MARLIN ? 4 : 2);
          const float a = t[i0], b = t[i1];
          const f16x2 h = {(_Float16)a, (_Float16)b};
          hi[j] = h2_bits(h);
          if constexpr (NL == 2) {
            const float ra = a - (float)h[0], rb = b - (float)h[1];
            const f16x2 l = {(_Float16)(fabsf(a) <= 3.4028235e38f ? ra : 0.0f),
                             (_Float16)(fabsf(b) <= 3.4028235e38f ? rb : 0.0f)};
            lo[j] = h2_bits(l);
          }
        }
        const int c = p >> 3, pp = p & 7;
        const int s = MAP == MAP_MARLIN ? pp & 3 : pp >> 1, g = MAP == MAP_MARLIN ? pp >> 2 : pp & 1;
        uint8_t *dst = xp + (((mt * 2 * np + c) * NL * 4 + s) * 64 + r32 + 32 * g) * 16;
        *reinterpret_cast<uint4 *>(dst) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        if constexpr (NL == 2) *reinterpret_cast<uint4 *>(dst + 4096) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        if constexpr (SUMS) {
          if ((q0 & 3) == 0) {
            const int sb = p >> 2;  // sub-block of the row
            uint16_t *sd = reinterpret_cast<uint16_t *>(xsum + ((mt * np + (sb >> 2)) * 64 + r32) * 16) + (sb & 3);
            const uint32_t h = f32_to_bf16_bits(sum);
            const float r1 = sum - bf16_bits_to_f32(h);
            const uint32_t md = f32_to_bf16_bits(r1);
            sd[0] = (uint16_t)h;
            sd[4] = (uint16_t)md;
            sd[256] = (uint16_t)f32_to_bf16_bits(r1 - bf16_bits_to_f32(md));
            sd[260] = 0;
          }
        }
      }
    }
  }
}

// ---- the product ----------------------------------------------------------

// Output of a row that holds an infinity or a NaN, for formats with mins: code
// and min parts of such a row would meet as inf - inf where the product with
// the weights themselves has a sign.  One thread an output.
template <bool Q5>
__device__ float cg_plain_dot(const uint8_t *w, const void *x, int xtype, int64_t row, int64_t col, int64_t k) {
  typedef CgK4<Q5> D;
  float v = 0.0f;
  for (int64_t i = 0; i < k; ++i) {
    const uint64_t e = (uint64_t)col * (uint64_t)k + (uint64_t)i;
    const uint8_t *b = w + (e >> 8) * D::BLOCK;
    const int c = (int)((e >> 6) & 3u), r = (int)(e & 63u);
    uint32_t sc, mn;
    const u32x4 hd = *reinterpret_cast<const u32x4 *>(b);
    k4_pair(hd, c, sc, mn);
    const uint32_t byte = b[D::QS + 32 * c + (r & 31)];
    uint32_t q = r < 32 ? byte & 15u : byte >> 4;
    if constexpr (Q5) q |= ((b[16 + (r & 31)] >> (2 * c + (r >> 5))) & 1u) << 4;
    const float wv = h2f(hd.x) * ub(sc, r >> 5) * (float)q - h2f(hd.x >> 16) * ub(mn, r >> 5);
    v = fmaf(load_x1(x, xtype, row * k + i), wv, v);
  }
  return v;
}

// A summed output on its way to y.
template <class D>
__device__ __forceinline__ void cg_finish(float v, const SetEntry &en, const float *rs, const int *rexp, const void *x,
                                          int xtype, int64_t row, int col, int64_t k) {
  const int re = rexp[row];
  v = __builtin_amdgcn_ldexpf(v, (int)(int16_t)(re & 0xFFFF));
  if constexpr (D::MINS) {
    if (re & kRowNonFinite) v = cg_plain_dot<D::BLOCK == 176u>(en.w, x, xtype, row, col, k);
  }
  if constexpr (D::MAP == MAP_MARLIN) v *= rs[col];
  store_linear(en.o, row, en.n, col, v);
}

// VMEM stays where it is written; ALU, LDS and matrix work may move across.
#define CG_PIN_LOADS() __builtin_amdgcn_sched_barrier(0x1 | 0x2 | 0x4 | 0x8 | 0x80 | 0x100 | 0x200)

template <class D, int NL, int MI>
__global__ __launch_bounds__(512) void k_cgemm(const WeightSet set, const float *__restrict__ rs,
                                               const uint8_t *__restrict__ xp, const uint8_t *__restrict__ xsum,
                                               const int *__restrict__ rexp, const void *__restrict__ x, int xtype,
                                               int64_t m, int64_t k, int np, int tm, int S,
                                               float *__restrict__ part) {
  // a staging region of 64 rows a wave, later KG tiles of 32 MI x 64 sums
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KG = (int)(blockDim.x >> 6);
  // XCD x (workgroups x, x + 8, ..) takes a run of consecutive tiles, M
  // fastest, so that the tiles sharing a weight tile share an L2.
  // Split K: the S slices of a tile are consecutive.
  const int T = (int)gridDim.x, xcd = (int)blockIdx.x & 7, qt = T >> 3, rt = T & 7;
  const int unit = xcd * qt + (xcd < rt ? xcd : rt) + ((int)blockIdx.x >> 3);
  const int tile = unit / S, z = unit - tile * S;
  const SetEntry en = pick_entry(set, tile);
  const int lt = tile - en.g0, ntile = lt / tm, mtile = lt - ntile * tm;
  const int n0 = 64 * ntile < en.n - 64 ? 64 * ntile : en.n - 64, m0 = 32 * MI * mtile;
  D dec;
  if constexpr (D::MAP == MAP_MARLIN) {
    dec.stride = 16 * (int64_t)en.n;
    dec.kc = (int)((k + 31) / 32);
  }
  dec.init(Tile{en.w, en.aux, n0, np}, lane);
  const int part_i = z * KG + wave;  // this wave's share of the pairs
  const int lo = np * part_i / (KG * S), hi = np * (part_i + 1) / (KG * S);
  lds_u8 *const L = (lds_u8 *)lds + 64 * D::STRIDE * wave;

  f32x16 acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x16){0};

  if (lo < hi) {
    const uint8_t *xa[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) xa[mi] = xp + (MI * (int64_t)mtile + mi) * (2 * np) * (NL * 4096);
    const uint32_t lo16 = 16u * lane;
    u32x4 a[MI][NL][4];
    typename D::Stage st;
    auto load_a = [&](int mi, int l, int s, int c) __attribute__((always_inline)) {
      a[mi][l][s] = ld16(xa[mi] + (int64_t)c * (NL * 4096) + (l * 4096 + s * 1024), lo16);
    };
    dec.issue(st, lo, lane);
    CG_PIN_LOADS();
#pragma unroll
    for (int l = NL - 1; l >= 0; --l)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) load_a(mi, l, s, 2 * lo);
    CG_PIN_LOADS();
    // A chunk's matrix work; its A operands are reloaded for the chunk after
    // it (not LAST) as soon as the second column tile has used them.
    uint32_t mins[2][2];
    float dm[2];
    auto chunk = [&](int j, auto C, auto Last) __attribute__((always_inline)) {
      constexpr int c = decltype(C)::value;
      constexpr bool LAST = decltype(Last)::value;
      static_for<2>([&](auto NI) __attribute__((always_inline)) {
        constexpr int ni = decltype(NI)::value;
        f16x8 b[4];
        float d[4 / D::GRP];
        dec.decode(L, ni, c, j, lane, b, d, mins[ni][c], dm[ni]);
        static_for<4 / D::GRP>([&](auto GG) __attribute__((always_inline)) {
          constexpr int s0 = decltype(GG)::value * D::GRP;
          f32x16 S[MI];
          static_for<NL>([&](auto LL) __attribute__((always_inline)) {  // the small limb first
            constexpr int l = NL - 1 - decltype(LL)::value;
            static_for<D::GRP>([&](auto SS) __attribute__((always_inline)) {
              constexpr int s = s0 + decltype(SS)::value;
              static_for<MI>([&](auto MM) __attribute__((always_inline)) {
                constexpr int mi = decltype(MM)::value;
                const f32x16 z = {0};
                S[mi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[mi][l][s]), b[s],
                                                               l == NL - 1 && s == s0 ? z : S[mi], 0, 0, 0);
                if constexpr (!LAST && ni == 1) {
                  load_a(mi, l, s, 2 * j + c + 1);
                  CG_PIN_LOADS();
                }
              });
            });
          });
          static_for<MI>([&](auto MM) __attribute__((always_inline)) {
            constexpr int mi = decltype(MM)::value;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              if constexpr (D::MAP == MAP_MARLIN) acc[mi][ni][r] += S[mi][r];
              else acc[mi][ni][r] = fmaf(d[s0 / D::GRP], S[mi][r], acc[mi][ni][r]);
            }
          });
        });
      });
    };
    auto pair = [&](int j, auto Last) __attribute__((always_inline)) {
      constexpr bool LAST = decltype(Last)::value;
      D::commit(st, L, lane);
      __builtin_amdgcn_wave_barrier();
      if constexpr (!LAST) {
        dec.issue(st, j + 1, lane);
        CG_PIN_LOADS();
      }
      u32x4 xs[MI];
      if constexpr (D::MINS) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) xs[mi] = ld16(xsum + ((MI * (int64_t)mtile + mi) * np + j) * 1024, lo16);
        CG_PIN_LOADS();
      }
      chunk(j, std::integral_constant<int, 0>{}, std::false_type{});
      chunk(j, std::integral_constant<int, 1>{}, Last);
      __builtin_amdgcn_wave_barrier();
      if constexpr (D::MINS) {
        // -dmin sum of m X over the pair's four sub-blocks: m exact in bf16
        // against the three limbs of X
        static_for<2>([&](auto NI) __attribute__((always_inline)) {
          constexpr int ni = decltype(NI)::value;
          const bool h0 = lane < 32;
          const u32x4 mb = {mins[ni][0], mins[ni][1], h0 ? mins[ni][0] : 0u, h0 ? mins[ni][1] : 0u};
          static_for<MI>([&](auto MM) __attribute__((always_inline)) {
            constexpr int mi = decltype(MM)::value;
            const f32x16 z = {0};
            const f32x16 M = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(cg_bf16x8, xs[mi]),
                                                                     __builtin_bit_cast(cg_bf16x8, mb), z, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mi][ni][r] = fmaf(dm[ni], M[r], acc[mi][ni][r]);
          });
        });
      }
    };
    for (int j = lo; j < hi - 1; ++j) pair(j, std::false_type{});
    pair(hi - 1, std::true_type{});
  }

  // The waves' tiles summed in wave order.  Slot q of a tile: MFMA tile
  // q / 16 (32 x 32: row half q / 32, column half (q / 16) % 2), register
  // q % 16; a wave takes every KG-th slot, two rows of 32 outputs each.
  constexpr int TS = 2048 * MI;  // sums of a tile
  float *const red = reinterpret_cast<float *>(lds);
  __syncthreads();  // every wave's staging reads are done
  float *mine = red + TS * wave + lane;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[((2 * mi + ni) * 16 + r) * 64] = acc[mi][ni][r];
  __syncthreads();
  for (int q = wave; q < 32 * MI; q += KG) {
    float v = red[64 * q + lane];
    for (int w = 1; w < KG; ++w) v += red[TS * w + 64 * q + lane];
    const int64_t row = m0 + 32 * (q >> 5) + 8 * ((q & 15) >> 2) + (q & 3) + 4 * (lane >> 5);
    const int col = n0 + 32 * ((q >> 4) & 1) + (lane & 31);
    if (row < m) {
      if (part) part[((int64_t)tile * S + z) * TS + 64 * q + lane] = v;
      else cg_finish<D>(v, en, rs, rexp, x, xtype, row, col, k);
    }
  }
}

// Split K: the S slices of every tile added in order, one thread an output.
template <class D, int MI>
__global__ __launch_bounds__(256) void k_cg_sum(const WeightSet set, const float *__restrict__ rs,
                                                const float *__restrict__ part, const int *__restrict__ rexp,
                                                const void *__restrict__ x, int xtype, int64_t m, int64_t k, int tm,
                                                int S) {
  constexpr int WG = 8 * MI, TS = 2048 * MI;  // workgroups a tile, sums of a tile
  const int tile = (int)blockIdx.x / WG, q = 4 * ((int)blockIdx.x % WG) + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const SetEntry en = pick_entry(set, tile);
  const int lt = tile - en.g0, ntile = lt / tm, mtile = lt - ntile * tm;
  const int64_t row = 32 * MI * (int64_t)mtile + 32 * (q >> 5) + 8 * ((q & 15) >> 2) + (q & 3) + 4 * (lane >> 5);
  const int n0 = 64 * ntile < en.n - 64 ? 64 * ntile : en.n - 64;
  const int col = n0 + 32 * ((q >> 4) & 1) + (lane & 31);
  if (row >= m) return;
  const float *p = part + (int64_t)tile * S * TS + 64 * q + lane;
  float v = p[0];
  for (int z = 1; z < S; ++z) v += p[TS * z];
  cg_finish<D>(v, en, rs, rexp, x, xtype, row, col, k);
}

int last_launch(const char *what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? RQ_OK : set_error(RQ_E_DEVICE, "%s launch: %s", what, hipGetErrorString(e));
}

template <auto KERNEL>
bool lds_allow(size_t bytes) {
  if (bytes <= 65536) return true;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, 8 * 16384);
  if (attr != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}

// Waves a workgroup (kg, each a share of K) and workgroups a tile (S, summed
// by a second kernel): the cheapest of all by a model fitted to this card.  A
// CU holds eight waves of this kernel (two a SIMD); with w of them at work a
// pair takes about 1 + w / 8 half-units (measured, eight waves: 3.3 - 4.9 us a
// pair with one limb, 3.6 - 6.6 with two), a round of workgroups about 4 us
// beside its pairs (first loads, sum over the waves, stores), the second
// kernel 3 us and its reads (16 KB a tile and slice at 3.5 TB/s).  On
// tiles of 32 rows a pair waits on its loads rather than on the matrix cores:
// 1.5 + w / 4 us (m = 5, with the pack: 2 x
// 8192 x 2048 16.7 us on eight waves a tile, 2 x 14336 x 4096 38.3 on four and
// 42.3 on eight, 2048 x 8192 20.3 / 22.6 / 28.3 / 38.7 on 8 / 4 / 2 / 1 slices).
struct Plan {
  int kg, S;
};
Plan cg_plan(int64_t tiles, int np, int nl, int mi) {
  Plan best{1, 1};
  double cost = 1e30;
  for (int S = 1; S <= 8; S *= 2) {
    for (int kg = 1; kg <= 8; ++kg) {
      if (kg * S > np && kg * S > 1) continue;
      const int res = 8 / kg;  // workgroups a CU holds
      const int64_t slots = 256 * res, wgs = tiles * S, rounds = (wgs + slots - 1) / slots;
      const int64_t per_cu = (wgs + 255) / 256 < res ? (wgs + 255) / 256 : res;
      const double unit = mi == 1 ? (nl == 2 ? 1.0 : 0.85) * (1.5 + 0.25 * (double)(per_cu * kg))
                                  : (nl == 2 ? 2.5 : 2.0) * (1.0 + (double)(per_cu * kg) / 8.0);
      const double c = (double)rounds * (4.0 + unit * (double)((np + kg * S - 1) / (kg * S))) +
                       (S > 1 ? 3.0 + (double)wgs * 8192.0 * mi / 3.5e6 : 0.0);
      if (c <= cost) cost = c, best = Plan{kg, S};
    }
  }
  return best;
}

constexpr size_t cg_lds(int kg, int mi, int stride) {
  const size_t a = (size_t)kg * 8192 * mi, b = (size_t)kg * 64 * stride;
  return a > b ? a : b;
}

template <class D, int NL, int MI>
int go(const WeightSet &set, int64_t tiles, const float *rs, const uint8_t *xp, const uint8_t *xsum, const int *rexp,
       const void *x, int xtype, int64_t m, int64_t k, int np, hipStream_t s, WsLease &ws) {
  const Plan plan = cg_plan(tiles, np, NL, MI);
  const int kg = plan.kg;
  int S = plan.S;
  float *part = nullptr;
  if (S > 1) {
    int rc = RQ_OK;
    part = static_cast<float *>(ws.get((size_t)tiles * S * 8192 * MI, &rc, true));
    if (!part) S = 1;
  }
  const size_t lds = cg_lds(kg, MI, D::STRIDE);
  if (!lds_allow<&k_cgemm<D, NL, MI>>(lds)) return RQ_E_UNSUPPORTED;
  const int tm = (int)((m + 32 * MI - 1) / (32 * MI));
  hipLaunchKernelGGL((k_cgemm<D, NL, MI>), dim3((unsigned)(tiles * S)), dim3(64 * kg), lds, s, set, rs, xp, xsum, rexp, x,
                     xtype, m, k, np, tm, S, part);
  int rc = last_launch("codes gemm");
  if (!rc && S > 1) {
    hipLaunchKernelGGL((k_cg_sum<D, MI>), dim3((unsigned)(tiles * 8 * MI)), dim3(256), 0, s, set, rs, part, rexp, x,
                       xtype, m, k, tm, S);
    rc = last_launch("codes gemm sum");
  }
  return rc;
}

// Rows packed for m rows of x: whole tiles of 32 (m <= 32) or 64.
int64_t cg_rows(int64_t m) { return m <= 32 ? 32 : (m + 63) / 64 * 64; }

// One or two rows a workgroup where that many workgroups are needed to fill
// the chip, else four (wider consecutive stores).
template <int XT, int NL, int MAP, bool SUMS>
int pack(const void *x, int64_t m, int64_t k, int np, uint8_t *xp, uint8_t *xsum, int *rexp, hipStream_t s) {
  const bool vec = k % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const int64_t rows = cg_rows(m);
#define RQ_PACK(RW, B)                                                                                            \
  hipLaunchKernelGGL((k_cg_pack<XT, NL, MAP, SUMS, RW, B>), dim3((unsigned)(rows / RW)), dim3(kPackThreads), 0, s, \
                     x, m, k, np, vec, xp, xsum, rexp)
  if (rows <= 128) {  // 512 threads a row
    if (np <= 32) RQ_PACK(1, 1);
    else RQ_PACK(1, 4);
  } else if (np <= 16) {
    RQ_PACK(4, 2);
  } else if (np <= 32) {
    RQ_PACK(2, 2);
  } else {
    RQ_PACK(2, 4);
  }
#undef RQ_PACK
  return last_launch("activation pack");
}

template <int NL, int MI>
int by_type(int qtype, const WeightSet &set, int64_t tiles, const uint8_t *xp, const uint8_t *xsum, const int *rexp,
            const void *x, int xtype, int64_t m, int64_t k, int np, hipStream_t s, WsLease &ws) {
  switch (qtype) {
    case RQ_Q4_K: return go<CgK4<false>, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    case RQ_Q5_K: return go<CgK4<true>, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    case RQ_Q6_K: return go<CgQ6K, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    case RQ_Q8_0: return go<CgQ8, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    case RQ_Q4_0: return go<CgQx0<false>, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    case RQ_Q5_0: return go<CgQx0<true>, NL, MI>(set, tiles, nullptr, xp, xsum, rexp, x, xtype, m, k, np, s, ws);
    default: return RQ_E_UNSUPPORTED;
  }
}

// Scratch of a slice of `rows` (a multiple of 64) activation rows.
struct Pack {
  size_t limbs, sums, rows;
  size_t total() const { return limbs + sums + rows; }
};
Pack pack_bytes(int64_t rows, int np, int nl) {
  return {(size_t)rows * np * 256 * nl, (size_t)(rows / 32) * np * 1024, (size_t)rows * 4};
}
// At most this much scratch a call: more rows go in slices.
constexpr size_t kPackMax = 128u << 20;

int64_t slice_rows(int64_t m, int np, int nl) {
  int64_t rows = cg_rows(m);
  while (rows > 64 && pack_bytes(rows, np, nl).total() > kPackMax) rows = (rows / 2 + 63) / 64 * 64;
  return rows;
}

}  // namespace

int launch_linear_codes(const rq_weight *const *w, int count, const void *x, int xtype, int64_t m, const Out *o,
                        hipStream_t s, WsLease &ws, CodesPack *shared) {
  const int64_t k = w[0]->k;
  if (count < 1 || count > kMultiMax || m < 1 || k % 128 != 0 || k > (1 << 20) ||
      reinterpret_cast<uintptr_t>(x) % 16 != 0)
    return RQ_E_UNSUPPORTED;
  for (int j = 1; j < count; ++j)
    if (w[j]->qtype != w[0]->qtype || w[j]->k != k) return RQ_E_UNSUPPORTED;
  for (int j = 0; j < count; ++j)
    if (w[j]->n < 64) return RQ_E_UNSUPPORTED;
  const int np = (int)(k / 128), nl = xtype == RQ_F32 ? 2 : 1;
  const size_t xb = xtype == RQ_F32 ? 4 : 2;
  const int64_t rows = slice_rows(m, np, nl);
  const Pack pb = pack_bytes(rows, np, nl);
  int rc = RQ_OK;
  const bool mins = w[0]->qtype == RQ_Q4_K || w[0]->qtype == RQ_Q5_K;
  // One slice only: a later slice overwrites the pack.
  if (rows < m) shared = nullptr;
  const bool packed = shared && shared->xp && (shared->sums || !mins);
  const bool sums = mins || (shared && shared->sums);
  uint8_t *xp = packed ? const_cast<uint8_t *>(shared->xp) : static_cast<uint8_t *>(ws.get(pb.total(), &rc, true));
  if (!xp) return RQ_E_UNSUPPORTED;
  uint8_t *xsum = xp + pb.limbs;
  int *rexp = reinterpret_cast<int *>(xsum + pb.sums);
  for (int64_t r0 = 0; r0 < m; r0 += rows) {
    const int64_t mm = m - r0 < rows ? m - r0 : rows;
    const void *xs = static_cast<const uint8_t *>(x) + (size_t)r0 * (size_t)k * xb;
    Out os[kMultiMax];
    for (int j = 0; j < count; ++j) {
      os[j] = o[j];
      os[j].y = static_cast<uint8_t *>(o[j].y) + (size_t)r0 * (size_t)w[j]->n * (o[j].ytype == RQ_F32 ? 4 : 2);
    }
    const bool few = mm <= 32;
    const int64_t tm = few ? 1 : (mm + 63) / 64;
    WeightSet set;
    int64_t tiles = 0;
    rc = fill_set(set, w, count, os, [&](const rq_weight *wj) { return tm * ((wj->n + 63) / 64); }, &tiles);
    if (rc) return rc;
#define RQ_CG_PACK(XT, NL)                                                                          \
  rc = sums ? pack<XT, NL, MAP_GGUF, true>(xs, mm, k, np, xp, xsum, rexp, s)                        \
            : pack<XT, NL, MAP_GGUF, false>(xs, mm, k, np, xp, xsum, rexp, s)
    if (packed) rc = RQ_OK;
    else if (xtype == RQ_F32) RQ_CG_PACK(RQ_F32, 2);
    else if (xtype == RQ_BF16) RQ_CG_PACK(RQ_BF16, 1);
    else RQ_CG_PACK(RQ_F16, 1);
#undef RQ_CG_PACK
    if (rc) return rc;
    if (shared && !packed) {
      shared->xp = xp;
      shared->sums = sums;
    }
#define RQ_CG_GO(NL, MI) by_type<NL, MI>(w[0]->qtype, set, tiles, xp, xsum, rexp, xs, xtype, mm, k, np, s, ws)
    if (few) rc = nl == 2 ? RQ_CG_GO(2, 1) : RQ_CG_GO(1, 1);
    else rc = nl == 2 ? RQ_CG_GO(2, 2) : RQ_CG_GO(1, 2);
#undef RQ_CG_GO
    if (rc) return rc;
  }
  return RQ_OK;
}

int launch_marlin_codes(const uint32_t *packed, const float *scales, int64_t n, int64_t k, const void *x, int xtype,
                        int64_t m, void *y, int ytype, hipStream_t s, WsLease &ws) {
  if (m < 1 || k > (1 << 20) || n < 64 || n > 0x7FFFFFFF) return RQ_E_UNSUPPORTED;
  const int np = (int)((k + 127) / 128), nl = xtype == RQ_F32 ? 2 : 1;
  const size_t xb = xtype == RQ_F32 ? 4 : 2, yb = ytype == RQ_F32 ? 4 : 2;
  const int64_t rows = slice_rows(m, np, nl);
  const Pack pb = pack_bytes(rows, np, nl);
  int rc = RQ_OK;
  uint8_t *xp = static_cast<uint8_t *>(ws.get(pb.total(), &rc, true));
  if (!xp) return RQ_E_UNSUPPORTED;
  int *rexp = reinterpret_cast<int *>(xp + pb.limbs + pb.sums);
  for (int64_t r0 = 0; r0 < m; r0 += rows) {
    const int64_t mm = m - r0 < rows ? m - r0 : rows;
    const void *xs = static_cast<const uint8_t *>(x) + (size_t)r0 * (size_t)k * xb;
    const bool few = mm <= 32;
    const int64_t tiles = (few ? 1 : (mm + 63) / 64) * ((n + 63) / 64);
    if (tiles > 0x3FFFFFF) return RQ_E_UNSUPPORTED;
    WeightSet set = {};
    set.w[0] = reinterpret_cast<const uint8_t *>(packed);
    set.y[0] = static_cast<uint8_t *>(y) + (size_t)r0 * (size_t)n * yb;
    set.n[0] = (int32_t)n;
    set.g_end[0] = (int32_t)tiles;
    for (int j = 1; j < kMultiMax; ++j) set.g_end[j] = 0x7FFFFFFF;
    set.count = 1;
    set.ytype = ytype;
    if (xtype == RQ_F32) rc = pack<RQ_F32, 2, MAP_MARLIN, false>(xs, mm, k, np, xp, nullptr, rexp, s);
    else if (xtype == RQ_BF16) rc = pack<RQ_BF16, 1, MAP_MARLIN, false>(xs, mm, k, np, xp, nullptr, rexp, s);
    else rc = pack<RQ_F16, 1, MAP_MARLIN, false>(xs, mm, k, np, xp, nullptr, rexp, s);
    if (rc) return rc;
#define RQ_CG_GO(NL, MI) go<CgMarlin, NL, MI>(set, tiles, scales, xp, nullptr, rexp, xs, xtype, mm, k, np, s, ws)
    if (few) rc = nl == 2 ? RQ_CG_GO(2, 1) : RQ_CG_GO(1, 1);
    else rc = nl == 2 ? RQ_CG_GO(2, 2) : RQ_CG_GO(1, 2);
#undef RQ_CG_GO
    if (rc) return rc;
  }
  return RQ_OK;
}

}  // namespace rq
