// Attention of long chunks (prompts, several hundred query rows per KV head) over the packed
// history, gfx950. Three launches instead of the frame-chunk kernel's two:
//
//   1. prompt_tiles_kernel unpacks every key once per KV head: history tokens and the chunk's own
//      K/V become one stream of keys, cut into units of 64, each a 16 KB image (K and V^T, bf16; at
//      precision 1 another 16 KB of their low parts) in the order the lanes of the MFMA operands
//      read them. The frame-chunk kernel dequantizes a tile again for every 192 query rows, and a
//      tile of few tokens (one decode step's) costs it a whole unit.
//   2. prompt_kernel: a workgroup of 8 waves takes 256 query rows of one KV head (wave = one Q head's
//      32 tokens, so all of a workgroup's rows end at nearly the same token) over a range of the
//      units that some row of it sees: units past its last token are not touched. Images go straight
//      to LDS (global_load_lds) PROMPT_RING - 1 units ahead.
//   3. prompt_merge_kernel merges the ranges of one row, where a group of rows has several.
//
// Ranges: every group of 256 rows sees another number of units, up to the whole chunk's, so a fixed
// number of ranges per group would leave the last groups the longest. All ranges are about
// unit_len units, chosen so that they come to one or two workgroups per CU.
//
// What bounds it: the softmax's VALU work (about 130 instructions and 32 exponentials per wave and
// unit beside 32 MFMAs), then the two small launches around it (4 to 5 us each). Frame-chunk kernel ->
// these, us per call, 15 Q / 5 KV heads, bf16 (fp32 precision):
//    512 tokens past 1024   23.7 ->  19.6   (29.1 -> 24.6)
//   1000 tokens past  640   36.8 ->  22.8   (46.0 -> 30.7)
//   2048 tokens past 1000   88.5 ->  45.3  (104.5 -> 65.1)
//   2048 tokens past 8128  266.5 -> 113.0  (338.6 -> 190.5)
//   8192 tokens            648.0 -> 187.0  (785.0 -> 286.0)   690 TFLOP/s of causal work
// Precision 0 rounds K, V and p to bf16, precision 1 splits each in two bf16 parts, as the
// frame-chunk kernel does (dkv_attn_mfma.hip).
#include "dkv_attn_common.h"
#include "dkv_attn_prompt.h"

namespace dkv {

typedef __bf16 pbf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 pbf16x2 __attribute__((ext_vector_type(2)));
typedef float pf32x2 __attribute__((ext_vector_type(2)));
typedef float pf32x4 __attribute__((ext_vector_type(4)));
typedef float pf32x8 __attribute__((ext_vector_type(8)));
typedef _Float16 pf16x8 __attribute__((ext_vector_type(8)));

union POp {
  pbf16x8 v;
  u32x4 u;
};

constexpr int PROMPT_RING = 3;  // LDS buffers of one unit's image
constexpr int PIECE = 1024;     // bytes of one MFMA operand: 64 lanes x 16 bytes

__device__ __forceinline__ uint32_t pk2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((pf32x2{lo, hi}), pbf16x2));
}

// ---------------------------------------------------------------------------
// 1. Unit images. One workgroup per (unit, KV head). Image of 64 keys: 8 pieces of K, piece
// (kg, j, ks) holding for lane 16 g + col the 8 columns 32 ks + 8 g of key 32 kg + 8 (col / 4) + 4 j
// + col % 4 (the order in which the scores of a lane come out as the operand of P V), then 8 pieces
// of V^T, piece (kg, db) holding for lane 16 g + col the keys 32 kg + 8 g .. + 7 of column
// 16 db + col; at precision 1 the low parts follow in the same order. Keys past the stream are zero.

// 16 elements of a row from its raw bytes (bits 16: 32 bytes in w0, w1; 8: 16 in w0; 4: 8 in w0;
// 0: no such key, zeros).
__device__ __forceinline__ void expand16(int bits, const u32x4& w0, const u32x4& w1, const float2& as, float* x) {
  if (bits == 16 || bits == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = bf16_lo(w0[i]);
      x[2 * i + 1] = bf16_hi(w0[i]);
      x[8 + 2 * i] = bf16_lo(w1[i]);
      x[8 + 2 * i + 1] = bf16_hi(w1[i]);
    }
    return;
  }
  uint32_t code[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    code[i] = bits == 4 ? (w0[i >> 3] >> (4 * (i & 7))) & 15u : (w0[i >> 2] >> (8 * (i & 3))) & 255u;
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = __fadd_rn(__fmul_rn((float)code[i], as.y), as.x);
}

template <int PREC>
__global__ void __launch_bounds__(256)
prompt_tiles_kernel(dkv_attn_args a, uint8_t* __restrict__ images) {
  constexpr int VS = 72;  // LDS row of V, in bf16 elements
  __shared__ uint32_t starts[2];
  __shared__ int first_tile;
  __shared__ dkv_tile desc[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t vt[PREC ? 2 : 1][TILE * VS];
  const int u = blockIdx.x, h = blockIdx.y;
  const int t = threadIdx.x, lane = t & 63;
  const int tok0 = u * TILE;
  const int hist = min(max(a.past - tok0, 0), TILE);  // keys of this unit that are history
  if (hist > 0 && t < 64) {
    // 64 descriptors around where the unit's tiles are if most tiles are full, in one load; if they do
    // not hold the unit's tokens, the last tile that starts at or before tok0 is searched for, 64
    // evenly spaced candidates per step, and the 64 from it on hold them (every tile has a row).
    int lo = max(min(u - 16, a.n_tiles - 64), 0);
    dkv_tile d = a.tiles[min(lo + lane, a.n_tiles - 1)];
    const int reach = min(64, a.n_tiles - lo) - 1;  // the last lane with a tile of its own
    const int from = __builtin_amdgcn_readlane(d.token_start, 0);
    const int to = __builtin_amdgcn_readlane(d.token_start + (int)d.rows, reach);
    if (from > tok0 || to < tok0 + hist) {
      int n = a.n_tiles;  // it is one of [lo, lo + n)
      lo = 0;
      while (n > 1) {
        const int step = (n + 63) >> 6, at = lo + min(lane * step, n - 1);
        const uint64_t ok = __builtin_amdgcn_ballot_w64(a.tiles[at].token_start <= tok0);
        // ok is a run of ones from lane 0 (lanes past the last candidate repeat the last tile)
        const int k = min(63 - __builtin_clzll(ok | 1), (n - 1) / step);
        n = min(step, n - k * step);
        lo += k * step;
      }
      d = a.tiles[min(lo + lane, a.n_tiles - 1)];
    }
    // Key r is in the tile after the unit's first by as many tile starts as lie in (tok0, tok0 + r].
    desc[lane] = d;
    const int at = d.token_start - tok0;
    const bool mine = lo + lane < a.n_tiles;
    const int upto = __builtin_popcountll(__builtin_amdgcn_ballot_w64(mine && at <= 0));
    if (lane == 0) {
      starts[0] = starts[1] = 0;
      first_tile = upto - 1;
    }
    if (mine && at > 0 && at < TILE) atomicOr(&starts[at >> 5], 1u << (at & 31));
  }
  __syncthreads();
  const int r = t >> 2, c = t & 3;  // key of the unit; a quarter of its columns
  // Everything a row needs (its bytes of K and of V, their (offset, scale)) in one round of loads: row
  // by kind, both of them in each branch.
  int bits = 0;
  const uint8_t *kp = nullptr, *vp = nullptr;
  u32x4 k0 = {0, 0, 0, 0}, k1 = k0, v0 = k0, v1 = k0;
  float2 ka = make_float2(0.f, 0.f), va = ka;
  if (r < hist) {
    const uint64_t before = ((uint64_t)starts[1] << 32 | starts[0]) & ((2ull << r) - 1);
    const int at = first_tile + __builtin_popcountll(before);  // (-1: no tile starts at or before the unit)
    const dkv_tile d = desc[max(at, 0)];
    const int row = tok0 + r - d.token_start;
    // The host saw a table that covers the history. A replay of a captured launch reads the device table of
    // that time: a key it does not hold stays zero and is not read from past its tile.
    if (at >= 0 && row >= 0 && row < (int)d.rows) {
      bits = d.bits;
      const int64_t sb = subblock_bytes(d.rows, bits);
      const uint8_t* ks = static_cast<const uint8_t*>(a.arena) + d.offset + ((int64_t)a.layer * 2 * a.heads + h) * sb;
      const uint8_t* vs = ks + a.heads * sb;
      const int rb = (int)row_bytes(bits);
      if (bits != 16) {
        ka = reinterpret_cast<const float2*>(ks + d.rows * rb)[row];
        va = reinterpret_cast<const float2*>(vs + d.rows * rb)[row];
      }
      kp = ks + row * rb + c * (rb >> 2);
      vp = vs + row * rb + c * (rb >> 2);
    }
  } else if (tok0 + r < a.past + a.nq) {
    const int64_t j = tok0 + r - a.past;
    bits = 16;
    kp = static_cast<const uint8_t*>(a.k_new) + 2 * (h * a.kn_head_stride + j * a.kn_tok_stride) + 32 * c;
    vp = static_cast<const uint8_t*>(a.v_new) + 2 * (h * a.vn_head_stride + j * a.vn_tok_stride) + 32 * c;
  }
  if (bits == 16) {
    k0 = reinterpret_cast<const u32x4*>(kp)[0];
    v0 = reinterpret_cast<const u32x4*>(vp)[0];
    k1 = reinterpret_cast<const u32x4*>(kp)[1];
    v1 = reinterpret_cast<const u32x4*>(vp)[1];
  } else if (bits == 8) {
    k0 = *reinterpret_cast<const u32x4*>(kp);
    v0 = *reinterpret_cast<const u32x4*>(vp);
  } else if (bits == 4) {
    const uint2 kw = *reinterpret_cast<const uint2*>(kp), vw = *reinterpret_cast<const uint2*>(vp);
    k0[0] = kw.x;
    k0[1] = kw.y;
    v0[0] = vw.x;
    v0[1] = vw.y;
  }
  float xk[16], xv[16];
  expand16(bits, k0, k1, ka, xk);
  expand16(bits, v0, v1, va, xv);
  uint8_t* img = images + ((int64_t)h * gridDim.x + u) * prompt_image_bytes(PREC);
  // K: key r is row (a, j, b) of key group kg
  const int kg = r >> 5, j = (r >> 2) & 1, col = 4 * ((r >> 3) & 3) + (r & 3);
#pragma unroll
  for (int q = 0; q < 2; ++q) {  // columns 16 c + 8 q .. + 7
    const int ks = c >> 1, g = 2 * (c & 1) + q;
    const float* x = xk + 8 * q;
    const u32x4 hi = {pk2(x[0], x[1]), pk2(x[2], x[3]), pk2(x[4], x[5]), pk2(x[6], x[7])};
    uint8_t* dst = img + (kg * 4 + j * 2 + ks) * PIECE + (16 * g + col) * 16;
    *reinterpret_cast<u32x4*>(dst) = hi;
    if (PREC) {
      u32x4 lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = pk2(x[2 * i] - bf16_lo(hi[i]), x[2 * i + 1] - bf16_hi(hi[i]));
      *reinterpret_cast<u32x4*>(dst + 16 * PIECE) = lo;
    }
  }
  // V^T through LDS
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float* x = xv + 8 * q;
    const u32x4 hi = {pk2(x[0], x[1]), pk2(x[2], x[3]), pk2(x[4], x[5]), pk2(x[6], x[7])};
    *reinterpret_cast<u32x4*>(&vt[0][r * VS + 16 * c + 8 * q]) = hi;
    if (PREC) {
      u32x4 lo;
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = pk2(x[2 * i] - bf16_lo(hi[i]), x[2 * i + 1] - bf16_hi(hi[i]));
      *reinterpret_cast<u32x4*>(&vt[PREC ? 1 : 0][r * VS + 16 * c + 8 * q]) = lo;
    }
  }
  __syncthreads();
#pragma unroll
  for (int part = 0; part < (PREC ? 2 : 1); ++part)
#pragma unroll
    for (int q = 0; q < 2; ++q) {  // lane of piece `piece` (kg, db)
      const int piece = (t >> 6) + 4 * q, pcol = lane & 15, pg = lane >> 4;
      const uint16_t* src = &vt[part][(32 * (piece >> 2) + 8 * pg) * VS + 16 * (piece & 3) + pcol];
      u32x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = src[2 * i * VS] | (uint32_t)src[(2 * i + 1) * VS] << 16;
      *reinterpret_cast<u32x4*>(img + (16 * part + 8 + piece) * PIECE + lane * 16) = w;
    }
}

// ---------------------------------------------------------------------------
// 2. The attention.

// max(a, b, c) of values that are never NaN, one instruction (see max_nn).
__device__ __forceinline__ float max3_nn(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// Over the four lanes 16 apart that hold one query column.
__device__ __forceinline__ float col_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = max_nn(__uint_as_float(r[0]), __uint_as_float(r[1]));
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return max_nn(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float col_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// HALF: the partials of groups with several ranges, see PromptPlan::half.
template <int PREC, bool HALF>
__global__ void __launch_bounds__(64 * PROMPT_WAVES, 4)
prompt_kernel(dkv_attn_args a, int units, int unit_len, int max_splits, int groups, const uint8_t* __restrict__ images,
              float* __restrict__ part_o, float2* __restrict__ part_ml) {
  constexpr int PIECES = PREC ? 32 : 16, PW = PIECES / PROMPT_WAVES;  // pieces of an image; per wave
  __shared__ __attribute__((aligned(1024))) u32x4 lds[PROMPT_RING * PIECES][64];
  const int G = a.q_heads / a.heads;
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  // Workgroup -> (KV head, group, range): the k-th range of head h, counted over the groups 64 at a
  // time. (A grid of max_splits x groups, the rest returning at once, left the XCDs uneven numbers
  // of real workgroups, and one round became two.)
  const int h = blockIdx.x % a.heads;
  int k = blockIdx.x / a.heads, grp = 0, n_units = 0, splits = 1;
  for (int g0 = 0; g0 < groups; g0 += 64) {
    const int nu = g0 + lane < groups ? prompt_group_units(g0 + lane, G, a.nq, a.past) : 0;
    const int ns = prompt_splits(nu, unit_len);
    int upto = ns;  // ranges of groups g0 .. g0 + lane
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o);
      if (lane >= o) upto += v;
    }
    const uint64_t past_k = __builtin_amdgcn_ballot_w64(upto > k);
    if (past_k) {
      const int at = __builtin_ctzll(past_k);
      grp = g0 + at;
      n_units = __builtin_amdgcn_readlane(nu, at);
      splits = __builtin_amdgcn_readlane(ns, at);
      k -= __builtin_amdgcn_readlane(upto, at) - splits;
      break;
    }
    k -= __builtin_amdgcn_readlane(upto, 63);
  }
  const int split = k;
  const int u0 = (uint32_t)n_units * split / splits, u1 = (uint32_t)n_units * (split + 1) / splits;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float xs = a.scale * LOG2E;

  const int task = grp * PROMPT_WAVES + wave;
  const int tb = task / G, gq = task - tb * G;
  const int m0 = tb * 32;            // first token of this wave
  const bool wave_on = m0 < a.nq;    // (the last group may have waves without rows)
  const int m_last = min(m0 + 31, a.nq - 1);

  const uint8_t* img = images + ((int64_t)h * units + u0) * prompt_image_bytes(PREC) + PIECE * wave + 16 * lane;
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  uint32_t fill = base + PIECE * wave;
  int ahead = u0;  // unit loaded next (past the last one, the last again, never used)
  auto load_next = [&]() {
#pragma unroll
    for (int q = 0; q < PW; ++q) load_piece(img + q * PROMPT_WAVES * PIECE, fill + q * PROMPT_WAVES * PIECE);
    fill = fill + PIECES * PIECE >= base + PROMPT_RING * PIECES * PIECE ? base + PIECE * wave : fill + PIECES * PIECE;
    if (++ahead < u1) img += prompt_image_bytes(PREC);
  };

  // Query operands and the mask of this lane's column in each block of 16 tokens.
  POp qop[2][2];
  int qhi[2], qlo[2];  // last and first visible chunk row
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int m = min(m0 + 16 * nb + col, a.nq - 1);
    const uint16_t* src = static_cast<const uint16_t*>(a.q) + (int64_t)(h * G + gq) * a.q_head_stride +
                          (int64_t)m * a.q_tok_stride + 8 * g;
    qop[nb][0].u = *reinterpret_cast<const u32x4*>(src);
    qop[nb][1].u = *reinterpret_cast<const u32x4*>(src + 32);
    qhi[nb] = m;
    qlo[nb] = chunk_seg_start(a, m);
  }
#pragma unroll
  for (int k = 0; k < PROMPT_RING - 1; ++k) load_next();
  // The query operands arrive here, with the first units: a wait for them inside the unit loop would
  // drain the loads in flight in every iteration.
  asm volatile("" ::"v"(qop[0][0].u), "v"(qop[0][1].u), "v"(qop[1][0].u), "v"(qop[1][1].u));
  pf32x4 acc[2][4];
  float m_run[2], l_part[2];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    m_run[nb] = -INFINITY;
    l_part[nb] = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db) acc[nb][db] = pf32x4{0.f, 0.f, 0.f, 0.f};
  }

  auto compute = [&](int u, const u32x4 (*st)[64]) {
    // Masks: units with a chunk row after this wave's first token, or any chunk row where the chunk has
    // segments. A low part only where packed keys are.
    const int rows_end = (u + 1) * TILE - a.past;  // chunk rows of the unit end before this one
    const bool masked = rows_end - 1 > m0 || (a.n_segs > 1 && rows_end > 0), lo_on = PREC && u * TILE < a.past;
    pf32x4 s[2][4];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int b = 0; b < 4; ++b) s[nb][b] = pf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int pass = 0; pass < (PREC ? 2 : 1); ++pass) {
      if (pass && !lo_on) break;
#pragma unroll
      for (int b = 0; b < 4; ++b)  // key block (kg, j) = (b / 2, b % 2)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          POp ka;
          ka.u = st[16 * pass + 2 * b + ks][lane];
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            s[nb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka.v, qop[nb][ks].v, s[nb][b], 0, 0, 0);
        }
    }
    POp p[2][2], pl[2][PREC ? 2 : 1];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      if (masked) {  // keys of this lane are chunk rows first + off, off = 32 kg + 4 j + i
        const int first = u * TILE + 8 * g - a.past;
        const int hi = qhi[nb] - first;
        if (a.n_segs > 1) {  // history, and the rows of the query's segment up to its own
          const int lo = qlo[nb] - first;
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int off = 32 * (b >> 1) + 4 * (b & 1) + i;
              s[nb][b][i] = off <= hi && (off >= lo || off < -first) ? s[nb][b][i] : -INFINITY;
            }
        } else {
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[nb][b][i] = 32 * (b >> 1) + 4 * (b & 1) + i <= hi ? s[nb][b][i] : -INFINITY;
        }
      }
      const pf32x4 *v = s[nb];
      const float t0 = max3_nn(v[0][0], v[0][1], v[0][2]), t1 = max3_nn(v[0][3], v[1][0], v[1][1]);
      const float t2 = max3_nn(v[1][2], v[1][3], v[2][0]), t3 = max3_nn(v[2][1], v[2][2], v[2][3]);
      const float t4 = max3_nn(v[3][0], v[3][1], v[3][2]);
      const float t5 = max_nn(max3_nn(t0, t1, t2), max3_nn(t3, t4, v[3][3]));
      // The running maximum moves when some lane's scores pass it; only then do the four lanes of a
      // column exchange theirs. Precision 0 keeps the exact maximum, so that the largest p is 1 and
      // rounds to bf16 without error (moved only past 2^8, 2048 tokens past 8128 took 99.4 us instead
      // of 101.8, but outputs were 7% further from exact ones); precision 1 moves it past 2^6. (The
      // frame-chunk kernel's two key groups each have a maximum and move it past 2^8. With 2^8 here 2048
      // tokens past 1000 took 65.3 us instead of 65.7, but at 4.280e-6 from float64 where that kernel is
      // at 4.218e-6; with 2^6 4.190e-6, and below that kernel at every size measured.)
      if (__builtin_amdgcn_ballot_w64(t5 * xs > m_run[nb] + (PREC ? 6.f : 0.f))) {
        const float mnew = max_nn(m_run[nb], col_max(t5) * xs);
        const float alpha = mnew == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run[nb] - mnew);
        m_run[nb] = mnew;
        l_part[nb] *= alpha;
#pragma unroll
        for (int db = 0; db < 4; ++db) acc[nb][db] *= alpha;
      }
      const float mref = m_run[nb] == -INFINITY ? 0.f : m_run[nb];
      float sum = 0.f;
#pragma unroll
      for (int kg = 0; kg < 2; ++kg) {
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          e[i] = __builtin_amdgcn_exp2f(__fmaf_rn(s[nb][2 * kg + (i >> 2)][i & 3], xs, -mref));
          sum += e[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[nb][kg].u[i] = pk2(e[2 * i], e[2 * i + 1]);
          if (PREC)
            pl[nb][PREC ? kg : 0].u[i] = pk2(e[2 * i] - bf16_lo(p[nb][kg].u[i]), e[2 * i + 1] - bf16_hi(p[nb][kg].u[i]));
        }
      }
      l_part[nb] += sum;
    }
#pragma unroll
    for (int kg = 0; kg < 2; ++kg)
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        POp va;
        va.u = st[8 + 4 * kg + db][lane];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          acc[nb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va.v, p[nb][kg].v, acc[nb][db], 0, 0, 0);
          if (PREC)
            acc[nb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va.v, pl[nb][PREC ? kg : 0].v, acc[nb][db], 0, 0, 0);
        }
        if (PREC && lo_on) {
          va.u = st[(PREC ? 24 : 8) + 4 * kg + db][lane];
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            acc[nb][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va.v, p[nb][kg].v, acc[nb][db], 0, 0, 0);
        }
      }
  };
  int buf = 0;
  for (int u = u0; u < u1; ++u) {
    // The unit has landed (this wave's pieces: at most those of the PROMPT_RING - 2 units after it are
    // under way; the other waves': the barrier), and every wave is past the unit before it, whose
    // buffer the next loads overwrite.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((PROMPT_RING - 2) * PW) : "memory");
    __builtin_amdgcn_s_barrier();
    load_next();
    if (wave_on && u * TILE <= a.past + m_last) compute(u, lds + buf * PIECES);  // (else: past this wave's last token)
    buf = buf + 1 == PROMPT_RING ? 0 : buf + 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads are done before the next barrier
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the last unit still write this workgroup's LDS
  if (!wave_on) return;

#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    float l = col_sum(l_part[nb]);
    const int lr = 16 * nb + col, m = m0 + lr;
    if (m >= a.nq) continue;
    if (splits == 1) {
      const float inv = 1.f / l;
      const int64_t off = (int64_t)m * a.out_tok_stride + (int64_t)(h * G + gq) * a.out_head_stride + 4 * g;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const pf32x4 o = acc[nb][db] * inv;
        if (a.out_dtype == 1)
          *reinterpret_cast<pf32x4*>(static_cast<float*>(a.out) + off + 16 * db) = o;
        else
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + off + 16 * db) =
              make_uint2(pk2(o[0], o[1]), pk2(o[2], o[3]));
      }
      continue;
    }
    const int64_t row = ((int64_t)h * max_splits + split) * ((int64_t)groups * PROMPT_ROWS) + grp * PROMPT_ROWS +
                        32 * wave + lr;
    if (!HALF) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
        __builtin_nontemporal_store(acc[nb][db], reinterpret_cast<pf32x4*>(part_o + row * D + 16 * db + 4 * g));
    } else {  // O / l in fp16, in half_slot() order, scaled where |V| is near the fp16 range
      const float inv = l > 0.f ? 1.f / l : 0.f;
      pf32x4 o[4];
      float amax = 0.f;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        o[db] = acc[nb][db] * inv;
#pragma unroll
        for (int e = 0; e < 4; ++e) amax = fmaxf(amax, fabsf(o[db][e]));
      }
      if (__builtin_amdgcn_ballot_w64(amax >= 32768.f)) {
        const int ex = half_partial_exponent(col_max(amax));
        if (ex) {
          const float sc = __builtin_amdgcn_ldexpf(1.f, -ex);
#pragma unroll
          for (int db = 0; db < 4; ++db) o[db] *= sc;
          l = half_partial_sum(l, ex);
        }
      }
      _Float16* ph = reinterpret_cast<_Float16*>(part_o) + row * D + 8 * g;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        __builtin_nontemporal_store(
            __builtin_convertvector((pf32x8{o[2 * k][0], o[2 * k][1], o[2 * k][2], o[2 * k][3], o[2 * k + 1][0],
                                            o[2 * k + 1][1], o[2 * k + 1][2], o[2 * k + 1][3]}), pf16x8),
            reinterpret_cast<pf16x8*>(ph + 32 * k));
    }
    if (g == 0) __builtin_nontemporal_store((pf32x2{m_run[nb], l}), reinterpret_cast<pf32x2*>(part_ml + row));
  }
}

// ---------------------------------------------------------------------------
// 3. The merge. A lane holds one 16-byte chunk of one row and walks the row's splits, four loads at a
// time: no exchange between lanes. (The frame-chunk merge spreads a row's splits, up to 51, over the
// lanes of a wave; here a row has two to about ten.)
template <bool HALF>
__global__ void __launch_bounds__(256)
prompt_merge_kernel(dkv_attn_args a, int unit_len, int max_splits, int groups, const float* __restrict__ part_o,
                    const float2* __restrict__ part_ml) {
  constexpr int CH = HALF ? 8 : 16;  // 16-byte chunks per row
  const int h = blockIdx.y;
  const int64_t rows = (int64_t)groups * PROMPT_ROWS;
  const int64_t rp = ((int64_t)blockIdx.x * 256 + threadIdx.x) / CH;
  const int c = threadIdx.x % CH;
  const int grp = (int)(rp / PROMPT_ROWS), lr = (int)(rp % PROMPT_ROWS);
  if (grp >= groups) return;
  const int G = a.q_heads / a.heads;
  const int splits = prompt_splits(prompt_group_units(grp, G, a.nq, a.past), unit_len);
  if (splits == 1) return;  // stored by the attention
  const int task = grp * PROMPT_WAVES + (lr >> 5), tb = task / G, gq = task - tb * G;
  const int m = 32 * tb + (lr & 31);
  if (m >= a.nq) return;
  const u32x4* po = reinterpret_cast<const u32x4*>(part_o);
  const pf32x2* pml = reinterpret_cast<const pf32x2*>(part_ml);
  const int64_t first = (int64_t)h * max_splits * rows + rp;
  constexpr int V = HALF ? 8 : 4;
  float M = -INFINITY, L = 0.f, o[V];
#pragma unroll
  for (int e = 0; e < V; ++e) o[e] = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 4) {
    pf32x2 ml[4];
    u32x4 raw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t at = first + min(s0 + i, splits - 1) * rows;
      ml[i] = __builtin_nontemporal_load(pml + at);
      raw[i] = __builtin_nontemporal_load(po + at * CH + c);
    }
    float bm = M;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (s0 + i >= splits) ml[i][0] = -INFINITY;
      bm = fmaxf(bm, ml[i][0]);
    }
    const float f0 = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - bm);
    L *= f0;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] *= f0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float w = ml[i][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[i][0] - bm);
      if constexpr (!HALF) {
        L = fmaf(ml[i][1], w, L);
        const float4 v = __builtin_bit_cast(float4, raw[i]);
        o[0] = fmaf(v.x, w, o[0]);
        o[1] = fmaf(v.y, w, o[1]);
        o[2] = fmaf(v.z, w, o[2]);
        o[3] = fmaf(v.w, w, o[3]);
      } else {
        int ex;
        const float ls = half_partial_decode(ml[i][1], ex) * w;
        L += ls;
        w = ex ? __builtin_amdgcn_ldexpf(ls, ex) : ls;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[2 * e] = fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(raw[i][e] & 0xffffu)), w, o[2 * e]);
          o[2 * e + 1] = fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(raw[i][e] >> 16)), w, o[2 * e + 1]);
        }
      }
    }
    M = bm;
  }
  const float inv = 1.f / L;
  const int64_t off = (int64_t)m * a.out_tok_stride + (int64_t)(h * G + gq) * a.out_head_stride;
#pragma unroll
  for (int k = 0; k < V / 4; ++k) {
    const int at = HALF ? half_column(8 * c + 4 * k) : 4 * c;
    const pf32x4 v = {o[4 * k] * inv, o[4 * k + 1] * inv, o[4 * k + 2] * inv, o[4 * k + 3] * inv};
    if (a.out_dtype == 1) *reinterpret_cast<pf32x4*>(static_cast<float*>(a.out) + off + at) = v;
    else *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + off + at) = make_uint2(pk2(v[0], v[1]), pk2(v[2], v[3]));
  }
}

// ---------------------------------------------------------------------------
// Host side.

PromptPlan prompt_plan(const dkv_attn_args& a, int cus, bool half) {
  PromptPlan p;
  p.half = half;
  const int G = a.q_heads / a.heads;
  p.groups = prompt_groups(G, a.nq);
  p.units = (int)(((int64_t)a.past + a.nq + TILE - 1) / TILE);
  int64_t total = 0;
  for (int i = 0; i < p.groups; ++i) total += prompt_group_units(i, G, a.nq, a.past);
  // One round of workgroups, all resident at once (two rounds at precision 1 from PROMPT_TWO_FROM on): the
  // shortest ranges of which there are no more than slots (a few more would take another round as long). Chunks of more groups than
  // that take as many rounds as it needs for several ranges per slot.
  int64_t slots = (int64_t)(total * a.heads >= (int64_t)PROMPT_TWO_FROM * cus ? 2 : 1) * cus;
  if ((int64_t)p.groups * a.heads * 4 > slots * 3) slots *= ((int64_t)p.groups * a.heads * 2 + slots - 1) / slots;
  p.unit_len = (int)((total * a.heads + slots - 1) / slots);
  if (p.unit_len < PROMPT_MIN_LEN) p.unit_len = PROMPT_MIN_LEN;
  for (;; ++p.unit_len) {
    int64_t items = 0;
    for (int i = 0; i < p.groups; ++i) items += prompt_splits(prompt_group_units(i, G, a.nq, a.past), p.unit_len);
    p.ranges = (int)items;
    if (items * a.heads <= slots || items == p.groups) break;
  }
  p.max_splits = prompt_splits(prompt_group_units(p.groups - 1, G, a.nq, a.past), p.unit_len);
  p.image_bytes = (int64_t)a.heads * p.units * prompt_image_bytes(a.precision);
  const int64_t rows = p.max_splits > 1 ? (int64_t)a.heads * p.max_splits * p.groups * PROMPT_ROWS : 0;
  p.part_o_bytes = rows * D * (half ? 2 : 4);
  p.part_ml_bytes = rows * 8;
  return p;
}

template <int PREC, bool HALF>
static void launch_prec(const dkv_attn_args& a, const PromptPlan& p, uint8_t* ws, hipStream_t s) {
  float* part_o = reinterpret_cast<float*>(ws + p.image_bytes);
  float2* part_ml = reinterpret_cast<float2*>(ws + p.image_bytes + p.part_o_bytes);
  hipLaunchKernelGGL(prompt_tiles_kernel<PREC>, dim3(p.units, a.heads), dim3(256), 0, s, a, ws);
  hipLaunchKernelGGL((prompt_kernel<PREC, HALF>), dim3(p.ranges * a.heads), dim3(64 * PROMPT_WAVES), 0, s, a, p.units,
                     p.unit_len, p.max_splits, p.groups, ws, part_o, part_ml);
  if (p.max_splits > 1) {
    const int64_t threads = (int64_t)p.groups * PROMPT_ROWS * (HALF ? 8 : 16);
    hipLaunchKernelGGL(prompt_merge_kernel<HALF>, dim3((unsigned)(threads / 256), a.heads), dim3(256), 0, s, a,
                       p.unit_len, p.max_splits, p.groups, part_o, part_ml);
  }
}

int launch_attn_prompt(const dkv_attn_args& a, const PromptPlan& p, void* ws, hipStream_t s) {
  uint8_t* w = static_cast<uint8_t*>(ws);
  if (a.precision == 1) launch_prec<1, false>(a, p, w, s);
  else if (p.half) launch_prec<0, true>(a, p, w, s);
  else launch_prec<0, false>(a, p, w, s);
  return (int)hipGetLastError();
}

}  // namespace dkv
