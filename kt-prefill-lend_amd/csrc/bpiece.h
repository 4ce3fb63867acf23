// B pieces for the grouped MFMA GEMMs: one lane's 32 dequantised weights of one row for
// one 64-value K step, as 16 packed bf16 words.
//
// Each format is split into load_head() (the bytes a super-block column shares over its
// four steps: scales, d), load<SUB>() (the step's quant bytes) and decode() (ALU only), so
// a kernel can keep the loads two steps ahead of their use, load the shared bytes once per
// super-block, and decode after the MFMAs of the previous step. The values are the exact
// dequantisation of formats.h rounded once to bf16 (Q4_K uses an FMA: d*sc*q is exact in
// fp32, so fma(d*sc, q, -dmin*m) rounds the same value as the separate multiply and
// subtract).
//
// K steps: a 256-value super-block column sb is 4 steps SUB = 0..3 of 64 values (SUB is a
// template parameter: every field position is then a compile-time constant). 256 sb +
// ksub<SUB>() + coff(q) is the row offset of the step's 8-value chunk q (q = 0..7, step
// positions 8q..8q+7); the activation tile uses the same map, so any permutation of K
// inside a super-block is fine for the product. Natural order (ksub = 64 SUB, coff = 8 q)
// except Q6_K, whose step SUB = 2 h + c covers the two 32-runs of half h that share their
// ql/qh bytes: 128 h + 32 c + [0, 32) and the same + 64.
// Piece h (0 or 1) of a step covers:
//   Q4_K : positions [16h, 16h+16) and [32+16h, +16): the two nibbles of qs bytes
//          [32g+16h, +16), g = SUB (sub-blocks 2g and 2g+1)
//   Q6_K : positions [16h, +16) (run c, low nibbles of ql and bits 2c of qh) and
//          [32+16h, +16) (run c+2, high nibbles and bits 2c+4 of the same bytes)
//   Q8_0, IQ3_S: positions [32h, 32h+32) (one Q8_0 block, one IQ3_S 32-group)
// `off0`/`off1` give the step positions of out[0..7] and out[8..15] (16 values each).
//
// Infinite scales give what a plain product gives (+-inf) in every kernel; so do zero codes (d * -0)
// in the GEMMs and in the dequant entry point, whose bytes are its result and which runs the same
// bodies. Where a kernel takes the other form (decode_hp<S2, PLAIN = false>) a zero's sign may
// differ, which no sum of products sees.
//
// Every SUB-dependent member also exists with the step parity as a run-time value: the
// `_hp<S2>(..., p)` forms take SUB = 2 S2 + p with S2 a compile-time constant and p a
// per-lane value (the decode-sized layer's 16x16x32 MFMA operands hold pieces of both
// parities in one wave); the `<SUB>` forms are those with p constant. One body per format
// serves both, so the values are the same.
//
// The fields of 2-byte aligned blocks are read from global memory where they lie (Q6_K 210 B,
// IQ3_S 110 B: the hardware takes unaligned addresses), from LDS with dword reads of the
// dword-aligned address below and v_alignbyte (words()); Q8_0's 34 B see its Raw.
#pragma once
#include "formats.h"

namespace ktmi {

__device__ __forceinline__ uint32_t alignbyte(uint32_t hi, uint32_t lo, uint32_t shift) {
  return __builtin_amdgcn_alignbyte(hi, lo, shift);
}
__device__ __forceinline__ const uint32_t* dword_floor(const uint8_t* p) {
  return (const uint32_t*)((uintptr_t)p & ~(uintptr_t)3);
}
__device__ __forceinline__ uint32_t byte_shift(const uint8_t* p) { return (uint32_t)((uintptr_t)p & 3); }

// a & m where the compiler cannot see the mask, so byte extracts of the result stay
// single v_cvt_f32_ubyteN conversions instead of folding into bit-field extracts
__device__ __forceinline__ uint32_t and_opaque(uint32_t a, uint32_t m) {
  uint32_t r;
  asm("v_and_b32 %0, %1, %2" : "=v"(r) : "s"(m), "v"(a));
  return r;
}

// (a & m) | (b & ~m) as one v_bfi_b32 (the compiler otherwise spends an AND, an AND and an OR)
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(m), "v"(a), "v"(b));
  return r;
}

// (a & m) | b as one v_and_or_b32 (opaque to the compiler, which would otherwise split the
// mask per 16-bit half of a result used as two halves)
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t b) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(m), "v"(b));
  return r;
}

// d * q + c in one rounding, q the fp16 number in the low (HI = 0) or high half of w: one
// v_fma_mix_f32. A code of up to 10 bits left as it is in a half-word is the fp16 denormal
// code * 2^-24, so with d scaled by 2^24 (exact) this is the fp32 FMA of the code itself, and
// no conversion instruction is needed. With a v_cvt a value the grouped K loop held 890 / 842 /
// 1088 VALU a super-block column (Q4_K / Q8_0 / Q6_K, the last two with run-time realignment),
// so 710 / 810 / 924; a 128-route block of one wave a SIMD spends half of its time issuing them
// (2048 x 512 Q4_K/Q6_K layer, 77 tokens, in the GEMMs: 67 -> 64 us; 7168 x 2048, 300 tokens: 340 -> 322).
constexpr float kCodeScale = 16777216.0f;  // 2^24
template <int HI>
__device__ __forceinline__ float fma_code(float d, uint32_t w, float c) {
  const _Float16 q = __builtin_bit_cast(_Float16, (uint16_t)(HI ? w >> 16 : w & 0xFFFFu));
  return __builtin_fmaf(d, (float)q, c);
}
// unsigned codes less MID in both half-words of w, as signed fp16 denormals: one v_pk_add_f16,
// exact
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
template <int MID>
__device__ __forceinline__ uint32_t code_sub(uint32_t w) {
  constexpr uint32_t m = 0x8000u | MID;
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2_t, w) + __builtin_bit_cast(f16x2_t, m | m << 16));
}
// -0, opaque to the compiler: an FMA with it is the plain product, signed zeros and infinities
// included, and stays one v_fma_mix (a multiply would need a conversion)
__device__ __forceinline__ float minus_zero() {
  float z = -0.0f;
  asm("" : "+s"(z));
  return z;
}
// the bf16 pairs of four codes: bytes 0 and 2 of a word as the halves of e, bytes 1 and 3 of o
__device__ __forceinline__ void codes4(float d, float c, uint32_t e, uint32_t o, uint32_t* out) {
  out[0] = f2bf2(fma_code<0>(d, e, c), fma_code<0>(d, o, c));
  out[1] = f2bf2(fma_code<1>(d, e, c), fma_code<1>(d, o, c));
}

// the same of codes that hold q + MID: the plain product (PLAIN; d * -0 and +-inf as they are) or,
// for finite d only, its value by taking MID d from the FMA (+0 for every zero; inf - inf where d is
// infinite), 2 of 11 VALU less. The GEMMs, within 1 % of the same time either way, and the dequant
// entry point take the first, the decode-sized kernels the second where `unbounded` finds no
// infinite or NaN scale
template <int MID, bool PLAIN>
__device__ __forceinline__ void biased4(float d, float c, uint32_t e, uint32_t o, uint32_t* out) {
  if constexpr (PLAIN) codes4(d, minus_zero(), code_sub<MID>(e), code_sub<MID>(o), out);
  else codes4(d, c, e, o, out);
}

// Where a piece's bytes are read from: global memory (through the caches) or LDS (rows a
// kernel has staged there, at the same offsets as in the row). words<N>: N = 1, 2 or 4 dwords
// from a 2-byte aligned address.
struct GMem {
  template <typename T>
  __device__ __forceinline__ static T ld(const void* p) { return gload<T>(p); }
  template <int N>
  __device__ __forceinline__ static void words(const uint8_t* p, uint32_t* w) {
    if constexpr (N == 4) {
      const u32x4_a2_t v = gload<u32x4_a2_t>(p);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = v[i];
    } else if constexpr (N == 2) {
      const u32x2_a2_t v = gload<u32x2_a2_t>(p);
      w[0] = v[0];
      w[1] = v[1];
    } else {
      w[0] = gload<u32_a2_t>(p);
    }
  }
};
struct LMem {
  // the LDS offset is the generic address's low 32 bits (an address-space cast of a generic
  // pointer would add a null check that the compiler here lowers wrongly)
  template <typename T>
  __device__ __forceinline__ static T ld(const void* p) {
    return *(const __attribute__((address_space(3))) T*)(uintptr_t)(uint32_t)(uintptr_t)p;
  }
  // the last dword read holds the field's last bytes, or (p dword aligned) the two after it:
  // a staged row is followed by the next one, or by the rest of its own 16-byte chunk
  template <int N>
  __device__ __forceinline__ static void words(const uint8_t* p, uint32_t* w) {
    const uint32_t* a = dword_floor(p);
    const uint32_t s = byte_shift(p);
    uint32_t v[N + 1];
    if constexpr (N == 4) {
      const u32x4_t q = ld<u32x4_a4_t>(a);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = q[i];
    } else if constexpr (N == 2) {
      const u32x2_t q = ld<u32x2_a4_t>(a);
      v[0] = q[0];
      v[1] = q[1];
    } else {
      v[0] = ld<uint32_t>(a);
    }
    v[N] = ld<uint32_t>(a + N);
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = alignbyte(v[i + 1], v[i], s);
  }
};

template <int TYPE>
struct BPiece;

// lookup<SUB>() issues a piece's codebook reads, convert<SUB>() does the rest of decode<SUB>()
// with them (a kernel can put the reads ahead of other LDS traffic). Formats without a
// codebook read nothing there.
template <class P>
struct NoLookup {
  struct Look {};
  template <int SUB, class Head, class Raw>
  __device__ static void lookup(const Head&, const Raw&, const uint32_t*, Look&) {}
  template <int SUB, class Head, class Raw>
  __device__ static void convert(const Head& hd, const Raw& r, const uint32_t* grid, const Look&, uint32_t out[16]) {
    P::template decode<SUB>(hd, r, grid, out);
  }
  template <int S2, class Head, class Raw>
  __device__ static void lookup_hp(const Head&, const Raw&, const uint32_t*, int, Look&) {}
  template <int S2, class Head, class Raw>
  __device__ static void convert_hp(const Head& hd, const Raw& r, const uint32_t* grid, int p, const Look&,
                                    uint32_t out[16]) {
    P::template decode_hp<S2>(hd, r, grid, p, out);
  }
  // the <SUB> forms through the run-time parity bodies
  template <int SUB, class Raw>
  __device__ static void load(const uint8_t* row, int sb, int h, const uint32_t* grid, Raw& r) {
    P::template load_hp<SUB / 2>(row, sb, h, SUB & 1, grid, r);
  }
  template <int SUB, class Head, class Raw>
  __device__ static void decode(const Head& hd, const Raw& r, const uint32_t* grid, uint32_t out[16]) {
    P::template decode_hp<SUB / 2>(hd, r, grid, SUB & 1, out);
  }
  // load<SUB> for a kernel that holds the raw bytes of step SUB - 1 of the same super-block
  // in `prev` (a format whose step pairs share bytes takes them from there)
  template <int SUB, class Raw>
  __device__ static void load_next(const uint8_t* row, int sb, int h, const uint32_t* grid, Raw& r, const Raw&) {
    P::template load_hp<SUB / 2>(row, sb, h, SUB & 1, grid, r);
  }
};

template <>
struct BPiece<GGML_Q4_K> : NoLookup<BPiece<GGML_Q4_K>> {
  static constexpr int NLOAD = 1;  // VMEM instructions per load<SUB>, at least
  static constexpr int NLOAD2 = 2;  // VMEM instructions of load_next over two consecutive steps
  static constexpr int VPM = 4;    // VALU instructions the GEMM schedule places after each MFMA
  struct Head { u32x4_t hdr; };  // d, dmin, scales[12]
  struct Raw { u32x4_t q; };
  template <int SUB>
  __device__ static int ksub() { return 64 * SUB; }
  template <int S2>
  __device__ static int ksub_hp(int p) { return 128 * S2 + 64 * p; }
  __device__ static int coff(int q) { return 8 * q; }
  template <class M = GMem>
  __device__ static void load_head(const uint8_t* row, int sb, int, Head& hd) { hd.hdr = M::template ld<u32x4_t>(row + sb * QB4_K); }
  template <int S2, class M = GMem>
  __device__ __forceinline__ static void load_hp(const uint8_t* row, int sb, int h, int p, const uint32_t*, Raw& r) {
    r.q = M::template ld<u32x4_t>(row + sb * QB4_K + 16 + 64 * S2 + 32 * p + 16 * h);
  }
  __device__ static bool unbounded(const Head&, const Raw&) { return false; }
  template <int S2, bool PLAIN = true>
  __device__ __forceinline__ static void decode_hp(const Head& hd, const Raw& r, const uint32_t*, int p,
                                                   uint32_t out[16]) {
    const float d = half_bits_to_float(hd.hdr[0] & 0xFFFF);
    const float dmin = half_bits_to_float(hd.hdr[0] >> 16);
    // sub-blocks 2g, 2g+1 (g = SUB = 2 S2 + p): for g < 2 the 6-bit fields sit in
    // scales[0..7]; for g >= 2 the low 4 bits are in scales[8..11] and the high 2 bits in
    // bits 6-7 of scales[0..7]
    const int sh = 16 * p;
    const uint32_t ws = hd.hdr[1] >> sh, wm = hd.hdr[2] >> sh, lo = hd.hdr[3] >> sh;
    constexpr bool hi = S2 == 1;
    const int sc0 = hi ? (int)((lo & 15) | (((ws >> 6) & 3) << 4)) : (int)(ws & 63);
    const int sc1 = hi ? (int)(((lo >> 8) & 15) | (((ws >> 14) & 3) << 4)) : (int)((ws >> 8) & 63);
    const int m0 = hi ? (int)(((lo >> 4) & 15) | (((wm >> 6) & 3) << 4)) : (int)(wm & 63);
    const int m1 = hi ? (int)(((lo >> 12) & 15) | (((wm >> 14) & 3) << 4)) : (int)((wm >> 8) & 63);
    // nibbles left in place: low ones (positions off0..) at bit 0 of a half-word, high ones
    // (off1..) at bit 4, the code times 16
    const float dn = d * kCodeScale;
    const float d1a = dn * (float)sc0, m1a = dmin * (float)m0;
    const float d1b = 0.0625f * (dn * (float)sc1), m1b = dmin * (float)m1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = r.q[i], v = w >> 8;
      codes4(d1a, -m1a, and_opaque(w, 0x000F000Fu), and_opaque(v, 0x000F000Fu), out + 2 * i);
      codes4(d1b, -m1b, and_opaque(w, 0x00F000F0u), and_opaque(v, 0x00F000F0u), out + 8 + 2 * i);
    }
  }
  __device__ static int off0(int h) { return 16 * h; }
  __device__ static int off1(int h) { return 32 + 16 * h; }
};

template <>
struct BPiece<GGML_Q8_0> : NoLookup<BPiece<GGML_Q8_0>> {
  static constexpr int NLOAD = 3;  // VMEM instructions per load<SUB>, at least
  static constexpr int NLOAD2 = 6;  // VMEM instructions of load_next over two consecutive steps
  static constexpr int VPM = 4;    // VALU instructions the GEMM schedule places after each MFMA
  struct Head {};
  // the 9 dwords from the dword at or below the block, s = byte shift (0 or 2). Read dword
  // aligned: two unaligned 16-byte loads cost the address unit more than the ninth dword does
  // (2048 x 768 layer, 512 tokens: 87 against 70 us)
  struct Raw { uint32_t w[9]; uint32_t s; };
  template <int SUB>
  __device__ static int ksub() { return 64 * SUB; }
  template <int S2>
  __device__ static int ksub_hp(int p) { return 128 * S2 + 64 * p; }
  __device__ static int coff(int q) { return 8 * q; }
  template <class M = GMem>
  __device__ static void load_head(const uint8_t*, int, int, Head&) {}
  template <int S2, class M = GMem>
  __device__ __forceinline__ static void load_hp(const uint8_t* row, int sb, int h, int p, const uint32_t*, Raw& r) {
    const uint8_t* b = row + (8 * sb + 4 * S2 + 2 * p + h) * QB8_0;
    const uint32_t* a = dword_floor(b);
    r.s = byte_shift(b);
    const u32x4_t w0 = M::template ld<u32x4_a4_t>(a), w1 = M::template ld<u32x4_a4_t>(a + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r.w[i] = w0[i];
      r.w[4 + i] = w1[i];
    }
    r.w[8] = M::template ld<uint32_t>(a + 8);
  }
  __device__ static bool unbounded(const Head&, const Raw& r) {
    return ((r.s ? r.w[0] >> 16 : r.w[0]) & 0x7C00u) == 0x7C00u;
  }
  template <int S2, bool PLAIN = true>
  __device__ __forceinline__ static void decode_hp(const Head&, const Raw& r, const uint32_t*, int, uint32_t out[16]) {
    const float d = half_bits_to_float((uint16_t)(r.s ? r.w[0] >> 16 : r.w[0] & 0xFFFFu));
    // the block's codes start 2 bytes past its d: bytes 0 and 2 of word i are bytes 2 and 4
    // (s = 0) or 4 and 6 (s = 2) of the dword pair i, i + 1
    const float dn = d * kCodeScale;
    const uint32_t even = r.s ? 0x0C060C04u : 0x0C040C02u, odd = even + 0x00010001u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t lo = r.w[i] ^ 0x80808080u, hi = r.w[i + 1] ^ 0x80808080u;
      biased4<128, PLAIN>(dn, -128.0f * d, __builtin_amdgcn_perm(hi, lo, even), __builtin_amdgcn_perm(hi, lo, odd), out + 2 * i);
    }
  }
  __device__ static int off0(int h) { return 32 * h; }
  __device__ static int off1(int h) { return 32 * h + 16; }
};

template <>
struct BPiece<GGML_Q6_K> : NoLookup<BPiece<GGML_Q6_K>> {
  static constexpr int NLOAD = 2;  // VMEM instructions per load<SUB>, at least
  // VMEM instructions of load_next over two consecutive steps: the odd step of a pair loads
  // only its ql bytes (the pair's qh bytes are the same)
  static constexpr int NLOAD2 = 3;
  // VALU instructions the GEMM schedule places after each MFMA
  static constexpr int VPM = 4;
  struct Head { uint32_t sc[4]; uint32_t d; };  // scales[16] and d
  struct Raw { uint32_t ql[4], qh[4]; };
  template <int SUB>
  __device__ static int ksub() { return 128 * (SUB >> 1) + 32 * (SUB & 1); }
  template <int S2>
  __device__ static int ksub_hp(int p) { return 128 * S2 + 32 * p; }
  __device__ static int coff(int q) { return q < 4 ? 8 * q : 64 + 8 * (q - 4); }
  template <class M = GMem>
  __device__ static void load_head(const uint8_t* row, int sb, int, Head& hd) {
    const uint8_t* sc = row + sb * QB6_K + 192;
    M::template words<4>(sc, hd.sc);
    hd.d = M::template ld<uint16_t>(sc + 16);
  }
  template <int S2, class M = GMem>
  __device__ __forceinline__ static void load_hp(const uint8_t* row, int sb, int h, int p, const uint32_t*, Raw& r) {
    const uint8_t* b = row + sb * QB6_K;
    M::template words<4>(b + 64 * S2 + 32 * p + 16 * h, r.ql);
    M::template words<4>(b + 128 + 32 * S2 + 16 * h, r.qh);
  }
  // steps 2 hh and 2 hh + 1 read the same 16 qh bytes (bits 2c.. of run c, c = SUB & 1): the
  // odd step takes them from the even one's raw bytes and loads only its ql bytes
  template <int SUB>
  __device__ __forceinline__ static void load_next(const uint8_t* row, int sb, int h, const uint32_t* grid, Raw& r,
                                                   const Raw& prev) {
    if constexpr ((SUB & 1) == 0) {
      load_hp<SUB / 2>(row, sb, h, 0, grid, r);
    } else {
      GMem::words<4>(row + sb * QB6_K + 64 * (SUB / 2) + 32 + 16 * h, r.ql);
#pragma unroll
      for (int i = 0; i < 4; ++i) r.qh[i] = prev.qh[i];
    }
  }
  __device__ static bool unbounded(const Head& hd, const Raw&) { return (hd.d & 0x7C00u) == 0x7C00u; }
  template <int S2, bool PLAIN = true>
  __device__ __forceinline__ static void decode_hp(const Head& hd, const Raw& r, const uint32_t*, int p,
                                                   uint32_t out[16]) {
    constexpr int hh = S2;
    const int c = p;
    // scales[8hh + 2c + h] (run c) and scales[8hh + 2c + h + 4] (run c+2): bytes 2c + h of
    // scale words 2hh and 2hh + 1
    const uint32_t h8 = 8 * ((threadIdx.x >> 5) & 1);
    const uint32_t sa = hd.sc[2 * hh], sbw = hd.sc[2 * hh + 1];
    const float d = half_bits_to_float((uint16_t)hd.d);
    const float fa = d * (float)(int8_t)((sa >> (16 * c + h8)) & 0xFF);
    const float fb = d * (float)(int8_t)((sbw >> (16 * c + h8)) & 0xFF);
    const int hsh = 2 * c;
    // run c: low nibbles and qh bits hsh, hsh+1; run c+2: high nibbles and bits hsh+4, hsh+5
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lw = r.ql[i], hw = r.qh[i];
      // bits 6 and 7 of the bytes are others' and masked off with the split into half-words
      const uint32_t va = bfi(0x0F0F0F0Fu, lw, hw << (4 - hsh)), vb = bfi(0x0F0F0F0Fu, lw >> 4, hw >> hsh);
      biased4<32, PLAIN>(fa * kCodeScale, -32.0f * fa, and_opaque(va, 0x003F003Fu), and_opaque(va >> 8, 0x003F003Fu), out + 2 * i);
      biased4<32, PLAIN>(fb * kCodeScale, -32.0f * fb, and_opaque(vb, 0x003F003Fu), and_opaque(vb >> 8, 0x003F003Fu), out + 8 + 2 * i);
    }
  }
  __device__ static int off0(int h) { return 16 * h; }
  __device__ static int off1(int h) { return 32 + 16 * h; }
};

template <>
struct BPiece<GGML_IQ3_S> {
  // `grid` is the codebook as byte selectors, staged in LDS by stage_iq3s_sel (formats.h).
  static constexpr int NLOAD = 2;  // VMEM instructions per load<SUB>: qs and the signs
  static constexpr int NLOAD2 = 4;  // VMEM instructions of load_next over two consecutive steps
  static constexpr int VPM = 4;    // VALU instructions the GEMM schedule places after each MFMA
  // d, the 4 scale bytes and the 8 qh bytes of the block
  struct Head { uint32_t d, sc, qh[2]; };
  // qs[8] and signs[4] of group ib
  struct Raw { uint32_t qs[2], sg; };
  template <int SUB>
  __device__ static int ksub() { return 64 * SUB; }
  template <int S2>
  __device__ static int ksub_hp(int p) { return 128 * S2 + 64 * p; }
  __device__ static int coff(int q) { return 8 * q; }
  template <class M = GMem>
  __device__ static void load_head(const uint8_t* row, int sb, int, Head& hd) {
    const uint8_t* b = row + sb * QBIQ3_S;
    hd.d = M::template ld<uint16_t>(b);
    M::template words<2>(b + 66, hd.qh);
    M::template words<1>(b + 106, &hd.sc);
  }
  template <int S2, class M = GMem>
  __device__ __forceinline__ static void load_hp(const uint8_t* row, int sb, int h, int p, const uint32_t*, Raw& r) {
    const uint8_t* b = row + sb * QBIQ3_S;
    const int ib = 4 * S2 + 2 * p + h;
    M::template words<2>(b + 2 + 8 * ib, r.qs);
    M::template words<1>(b + 74 + 4 * ib, &r.sg);
  }
  // the 8 codebook entries of the piece's 4-value groups
  struct Look { uint32_t g[8]; };
  template <int S2>
  __device__ __forceinline__ static void lookup_hp(const Head& hd, const Raw& r, const uint32_t* grid, int p,
                                                   Look& lk) {
    const uint32_t h = (threadIdx.x >> 5) & 1;
    const uint32_t qs0 = r.qs[0], qs1 = r.qs[1];
    const uint32_t qh = __builtin_amdgcn_ubfe(hd.qh[S2], 8 * (2 * (uint32_t)p + h), 8);  // qh byte 4 S2 + 2p + h
    const uint32_t qh2 = qh | (qh << 16);
    // the 9-bit indices of groups 2j and 2j + 1 as the two 16-bit halves of one word: their
    // qs bytes moved to bits 0 and 16 by one v_perm, qh bits 2j and 2j + 1 to bits 8 and 24
    // by one packed 16-bit shift of qh2 and merged with one v_and_or; each half then becomes
    // an LDS address with one v_lshlrev_b32_sdwa (2.5 VALU an index instead of 4)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t qsw = j < 2 ? qs0 : qs1;
      const uint32_t b0 = (2 * j) & 3, b1 = (2 * j + 1) & 3;
      const uint32_t lo = __builtin_amdgcn_perm(0u, qsw, b0 | 0x0C00u | (b1 << 16) | 0x0C000000u);
      const u16x2_t hv = __builtin_bit_cast(u16x2_t, qh2) << u16x2_t{(uint16_t)(8 - 2 * j), (uint16_t)(7 - 2 * j)};
      const uint32_t w = and_or(__builtin_bit_cast(uint32_t, hv), 0x01000100u, lo);
      lk.g[2 * j] = grid[w & 0xFFFF];
      lk.g[2 * j + 1] = grid[w >> 16];
    }
  }
  template <int S2>
  __device__ __forceinline__ static void convert_hp(const Head& hd, const Raw& r, const uint32_t*, int p,
                                                    const Look& lk, uint32_t out[16]) {
    const uint32_t h = (threadIdx.x >> 5) & 1;
    const uint32_t sg = r.sg;
    const uint32_t nib = (hd.sc >> (8 * (2 * S2 + p) + 4 * h)) & 15;  // group 4 S2 + 2p + h
    const uint32_t dbits = hd.d;
    const float db = half_bits_to_float((uint16_t)dbits) * (float)(1 + 2 * (int)nib);
    // A group has only eight magnitudes m = 2e + 1: bf16(db * m) of each (the same rounding
    // of the same exact product as a value-by-value decode) goes into a table of two byte
    // planes, byte e of {tl1:tl0} the low byte of entry e, of {th1:th0} its high byte. The
    // codebook entries are staged as selectors e (stage_iq3s_sel), so one v_perm per plane
    // gathers the four values of a codebook entry and two more interleave them into bf16
    // pairs: 8 VALU per four values with the signs, against 14 for convert, scale and pack.
    uint32_t pw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pw[i] = f2bf2(db * (float)(4 * i + 1), db * (float)(4 * i + 3));
    const uint32_t tl0 = __builtin_amdgcn_perm(pw[1], pw[0], 0x06040200u);
    const uint32_t th0 = __builtin_amdgcn_perm(pw[1], pw[0], 0x07050301u);
    const uint32_t tl1 = __builtin_amdgcn_perm(pw[3], pw[2], 0x06040200u);
    const uint32_t th1 = __builtin_amdgcn_perm(pw[3], pw[2], 0x07050301u);
    // value 4k + j takes sign bit 4k + j of sg. (sign ? -v : v) of v = db * m flips the sign
    // bit of v, and so of its bf16 rounding: bits 2p and 2p + 1 of sg are moved to bits 15
    // and 31 of the packed pair of values 2p, 2p + 1 by one packed 16-bit shift of sg's
    // half-word (in both halves) and xored in
    const uint32_t sgw[2] = {(sg & 0xFFFFu) | (sg << 16), (sg >> 16) | (sg & 0xFFFF0000u)};
    auto pair_signs = [&](int pr) {
      const int q = (2 * pr) & 15;
      const u16x2_t v = __builtin_bit_cast(u16x2_t, sgw[pr >> 3]) << u16x2_t{(uint16_t)(15 - q), (uint16_t)(14 - q)};
      return __builtin_bit_cast(uint32_t, v) & 0x80008000u;
    };
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t lo = __builtin_amdgcn_perm(tl1, tl0, lk.g[k]);  // low bytes of values 0..3
      const uint32_t hi = __builtin_amdgcn_perm(th1, th0, lk.g[k]);  // their high bytes
      out[2 * k] = __builtin_amdgcn_perm(hi, lo, 0x05010400u) ^ pair_signs(2 * k);
      out[2 * k + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u) ^ pair_signs(2 * k + 1);
    }
  }
  __device__ static bool unbounded(const Head&, const Raw&) { return false; }
  template <int S2, bool PLAIN = true>
  __device__ __forceinline__ static void decode_hp(const Head& hd, const Raw& r, const uint32_t* grid, int p,
                                                   uint32_t out[16]) {
    Look lk;
    lookup_hp<S2>(hd, r, grid, p, lk);
    convert_hp<S2>(hd, r, grid, p, lk, out);
  }
  // the <SUB> forms through the run-time parity bodies
  template <int SUB>
  __device__ static void load(const uint8_t* row, int sb, int h, const uint32_t* grid, Raw& r) {
    load_hp<SUB / 2>(row, sb, h, SUB & 1, grid, r);
  }
  template <int SUB>
  __device__ static void load_next(const uint8_t* row, int sb, int h, const uint32_t* grid, Raw& r, const Raw&) {
    load_hp<SUB / 2>(row, sb, h, SUB & 1, grid, r);
  }
  template <int SUB>
  __device__ static void lookup(const Head& hd, const Raw& r, const uint32_t* grid, Look& lk) {
    lookup_hp<SUB / 2>(hd, r, grid, SUB & 1, lk);
  }
  template <int SUB>
  __device__ static void convert(const Head& hd, const Raw& r, const uint32_t* grid, const Look& lk, uint32_t out[16]) {
    convert_hp<SUB / 2>(hd, r, grid, SUB & 1, lk, out);
  }
  template <int SUB>
  __device__ static void decode(const Head& hd, const Raw& r, const uint32_t* grid, uint32_t out[16]) {
    decode_hp<SUB / 2>(hd, r, grid, SUB & 1, out);
  }
  __device__ static int off0(int h) { return 32 * h; }
  __device__ static int off1(int h) { return 32 * h + 16; }
};

}  // namespace ktmi
