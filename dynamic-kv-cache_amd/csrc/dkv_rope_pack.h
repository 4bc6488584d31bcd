// RoPE and the pack of one projection row held by 8 lanes, shared by dkv_rope_pack (dkv_pack.hip) and
// the Q/K/V projection that ends in it (dkv_linear.hip), and the quantizer they share with dkv_pack.
#pragma once
#include "dkv_common.h"

namespace dkv {

constexpr float TIE_GUARD = 0.5f - 0x1p-13f;

struct RowDst {
  uint8_t* payload;  // start of the row's payload
  float2* meta;      // the row's (offset, scale)
};

__device__ __forceinline__ RowDst row_dst(const dkv_pack_job& j, int kv, int head, int tok, uint8_t* arena,
                                          int layers, int heads) {
  const int r_seg = j.row0 + tok;
  const int ti = r_seg / TILE;
  const int rt = r_seg - ti * TILE;
  const int rows_i = min(TILE, j.seg_rows - ti * TILE);
  const int64_t sb = subblock_bytes(rows_i, j.bits);
  uint8_t* sub = arena + j.seg_offset + (int64_t)ti * slab_bytes(TILE, j.bits, layers, heads) +
                 ((int64_t)(j.layer * 2 + kv) * heads + head) * sb;
  RowDst d;
  d.payload = sub + (int64_t)rt * row_bytes(j.bits);
  d.meta = reinterpret_cast<float2*>(sub + (int64_t)rows_i * row_bytes(j.bits)) + rt;
  return d;
}

// The offset of a row whose minimum is zero: -0 when the row holds a -0, else
// +0, the sign IEEE 754-2019 minimum() gives. (v_min_f32 and torch's amin,
// src/kv_quantization.py:63, leave it to the order of the reduction; codes,
// scales and dequantized values do not depend on it.)
__device__ __forceinline__ float zero_min_sign(uint32_t has_neg_zero) { return has_neg_zero ? -0.0f : 0.0f; }

// Codes of 8 elements of a row whose (offset, scale) is (a, s), with r ~ 1/s,
// packed: BITS 4 -> out[0] (element e in bits 4e..4e+3), BITS 8 -> out[0..1]
// (element e in byte e). `fast` says r and every t below are finite.
//
// rint(t) comes from m = t + 2^23, which for 0 <= t < 2^22 rounds t to an
// integer (round to nearest even, as rintf) and leaves it in the low mantissa
// bits: byte 0 of m's bit pattern is the code. The group takes the exact
// division when any t is within 2^-13 of a half-integer.
template <int BITS>
__device__ __forceinline__ void quantize8(const float* x, float a, float s, float r, bool fast, uint32_t* out) {
  constexpr float LEVELS = BITS == 4 ? 15.0f : 255.0f;
  constexpr float MAGIC = 0x1p23f;
  uint32_t y[8];
  float dev = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float t = __fmul_rn(x[e] - a, r);
    const float m = __fadd_rn(t, MAGIC);
    dev = fmaxf(dev, fabsf(t - (m - MAGIC)));
    y[e] = __float_as_uint(m);
  }
  if (!(fast && dev < TIE_GUARD)) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      y[e] = (uint32_t)__builtin_amdgcn_fmed3f(rintf(__fdiv_rn(x[e] - a, s)), 0.0f, LEVELS);
  }
  if (BITS == 4) {
    uint32_t p[4];  // byte 0 of p[i] = element 2i + 1 in the high nibble, 2i in the low one
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = (y[2 * i + 1] << 4) | y[2 * i];
    const uint32_t lo = __builtin_amdgcn_perm(p[1], p[0], 0x07060400u);
    const uint32_t hi = __builtin_amdgcn_perm(p[3], p[2], 0x07060400u);
    out[0] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
  } else {
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t lo = __builtin_amdgcn_perm(y[4 * w + 1], y[4 * w], 0x07060400u);
      const uint32_t hi = __builtin_amdgcn_perm(y[4 * w + 3], y[4 * w + 2], 0x07060400u);
      out[w] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
  }
}

__device__ __forceinline__ void write_segment_tiles(const dkv_pack_job& j, int layers, int heads,
                                                    dkv_tile* tiles) {
  write_tile_descriptors(j.seg_offset, j.seg_rows, j.seg_token_start, j.bits, j.tile_index0, layers, heads,
                         tiles);
}

// Eight elements of one row after RoPE: y = bf16(bf16(x * cos) + bf16(sign *
// partner * sin)), where partner is the element 32 columns away (rotate_half)
// and sign is -1 on the first half of the row. Products of two bf16 values are
// exact in fp32, so this is transformers' apply_rotary_pos_emb in bf16
// operation by operation (q * cos + rotate_half(q) * sin, each op rounded).
__device__ __forceinline__ u32x4 rope8(const u32x4& x, const u32x4& partner, const u32x4& cs, const u32x4& sn,
                                       bool first_half) {
  const float sg = first_half ? -1.0f : 1.0f;
  u32x4 y;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float lo = round_bf16(round_bf16(bf16_lo(x[k]) * bf16_lo(cs[k])) +
                                round_bf16(sg * bf16_lo(partner[k]) * bf16_lo(sn[k])));
    const float hi = round_bf16(round_bf16(bf16_hi(x[k]) * bf16_hi(cs[k])) +
                                round_bf16(sg * bf16_hi(partner[k]) * bf16_hi(sn[k])));
    y[k] = pack_bf16(lo, hi);
  }
  return y;
}

// Packs one row held by 8 lanes (lane c of the row holds columns [8c, 8c + 8)
// in w): min/max over the row through the 8 lanes, then the arithmetic of
// pack_loaded (every lane of the row forms the same a, s and 1/s) and quantize8
// on the lane's 8 elements. Lanes of rows r >= nrows still take part in the
// exchanges but store nothing.
template <int BITS>
__device__ __forceinline__ void pack_row8(const dkv_pack_job& j, int kv, int head, int tok, bool valid, int c,
                                          const u32x4& w, uint8_t* arena, int layers, int heads) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = bf16_lo(w[e]);
    x[2 * e + 1] = bf16_hi(w[e]);
  }
  if (BITS == 16) {
    if (valid) *reinterpret_cast<u32x4*>(row_dst(j, kv, head, tok, arena, layers, heads).payload + 16 * c) = w;
    return;
  }
  float lo = x[0], hi = x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) {
    lo = fminf(lo, x[e]);
    hi = fmaxf(hi, x[e]);
  }
  uint32_t nz = 0;  // the row holds a -0 (the sign of a zero minimum, see zero_min_sign)
#pragma unroll
  for (int e = 0; e < 8; ++e) nz |= __float_as_uint(x[e]) == 0x80000000u;
#pragma unroll
  for (int o = 1; o < 8; o <<= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
    nz |= __shfl_xor(nz, o);
  }
  const float a = lo == 0.0f ? zero_min_sign(nz) : lo;
  const float span = hi - a;
  const float s = span > 0.0f ? __fdiv_rn(span, BITS == 4 ? 15.0f : 255.0f) : 1.0f;
  const float rs = __builtin_amdgcn_rcpf(s);
  const bool fast = s >= 0x1p-126f && s <= 0x1p125f;
  uint32_t out[2];
  quantize8<BITS>(x, a, s, rs, fast, out);
  if (!valid) return;
  const RowDst d = row_dst(j, kv, head, tok, arena, layers, heads);
  if (BITS == 4) *reinterpret_cast<uint32_t*>(d.payload + 4 * c) = out[0];
  else *reinterpret_cast<uint2*>(d.payload + 8 * c) = make_uint2(out[0], out[1]);
  if (c == 0) *d.meta = make_float2(a, s);
}

// One row of one projection head, held by 8 lanes (lane c: columns [8c, 8c + 8) in x, its cos and sin in
// cs and sn): RoPE (Q and K heads; V rows are rotated too and keep their input: a select, not a branch
// that loads could be moved into), the row of q_out, k_out or v_out ([heads, n, 64] each), and for K and V
// heads the row packed into job j's segment. Heads [0, q_heads) are Q, then `heads` K, then `heads` V.
__device__ __forceinline__ void rope_pack_row(const u32x4& x, const u32x4& cs, const u32x4& sn, int hh, int tok,
                                              bool valid, int c, int n, int q_heads, uint16_t* __restrict__ q_out,
                                              uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out,
                                              const dkv_pack_job& j, uint8_t* arena, int layers, int heads) {
  const bool is_v = hh >= q_heads + heads;
  // rotate_half pairs column d with d +- 32: lane c with lane c ^ 4 of the same row
  u32x4 p;
#pragma unroll
  for (int e = 0; e < 4; ++e) p[e] = __shfl_xor(x[e], 4);
  const u32x4 rot = rope8(x, p, cs, sn, c < 4);
  const u32x4 w = is_v ? x : rot;
  uint16_t* dst = hh < q_heads ? q_out + (int64_t)hh * n * D
                               : (is_v ? v_out + (int64_t)(hh - q_heads - heads) * n * D
                                       : k_out + (int64_t)(hh - q_heads) * n * D);
  if (valid) *reinterpret_cast<u32x4*>(dst + (int64_t)tok * D + 8 * c) = w;

  if (hh < q_heads) return;
  const bool packs = valid && tok < j.n;  // rows the job packs
  const int kv = is_v ? 1 : 0;
  const int head = hh - q_heads - kv * heads;
  const int bits = __builtin_amdgcn_readfirstlane(j.bits);
  if (bits == 4) pack_row8<4>(j, kv, head, tok, packs, c, w, arena, layers, heads);
  else if (bits == 8) pack_row8<8>(j, kv, head, tok, packs, c, w, arena, layers, heads);
  else pack_row8<16>(j, kv, head, tok, packs, c, w, arena, layers, heads);
}

// Host: whether a pack job is well formed and lies in the arena (DKV_EINVAL and a message if not).
int check_job(const dkv_pack_job& j, int64_t arena_bytes, int layers, int heads);

}  // namespace dkv
