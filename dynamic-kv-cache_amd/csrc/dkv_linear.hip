// Decoder projections for short chunks: out = epilogue(prologue(x) w^T) with
// x [rows, k] and w [n, k] bf16 (both row-major, k contiguous), fp32
// accumulation on v_mfma_f32_16x16x32_bf16, bf16 out.
//
//   prologue  none, or RMSNorm of the x rows with the torch composition's two
//             bf16 roundings (bf16(bf16(x * rsqrt(mean(x^2) + eps)) * g),
//             src/gpu_ops.py:9-12) applied in registers;
//   epilogue  plain: bf16(acc);
//             residual: bf16(r + bf16(acc)), the decoder's residual add after
//             o_proj and down_proj;
//             silu_mul: w holds [gate | up] rows (2 * inter of them) and
//             out[:, c] = bf16(bf16(silu(bf16(g_c))) * bf16(u_c))
//             (src/gpu_ops.py:14-17, 23-25);
//             rope: w holds the joined [q | k | v] heads of 64 rows; RoPE on q and k, the q, k and v
//             blocks, and K and V packed into a segment (dkv_rope_pack's work and bytes).
//
// The chunks are 1-100 rows, so the weights (1.8-9.8 MB per projection of the
// 960-wide decoder) dominate the traffic: the kernel is a weight stream. A
// workgroup owns NB column blocks of 16 weight rows and RB blocks of 16 x
// rows; its waves split k in 64-element pairs of MFMA steps (wave w takes
// pairs w, w + WAVES, ...), issue every load of their share before the first
// MFMA, and meet in LDS, where one wave per output tile sums the partials in
// wave order (deterministic). With Y^T = W X^T on the MFMA (weights on the M
// axis), lane (col, g) ends with 4 consecutive output columns of one row: 8
// byte stores. Consecutive workgroups go to different XCDs; the RB = 1 layout
// numbers its tiles so that the row blocks sharing a weight tile land on one
// XCD (one L2).
#include "dkv_common.h"
#include "dkv_rope_pack.h"

namespace dkv {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

union Op8 {
  bf16x8_t v;
  u32x4 u;
};

enum { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SILU_MUL = 2, EPI_ROPE = 3 };

struct LinearArgs {  // passed by value and never written (a written copy would go to scratch)
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* w;
  int64_t ldw;
  const uint16_t* norm;  // RMSNorm weight [k] (prologue only)
  const uint16_t* res;   // residual [rows, n] (EPI_RESIDUAL only)
  int64_t ldr;
  uint16_t* out;
  int64_t ldo;
  float eps;
  int rows, k, kp;  // kp = k / 64
  int n_tiles;      // column tiles of 16 * NT output columns
  int row_groups;   // ceil(rows / (16 * RB))
  int up;           // n_out (EPI_SILU_MUL: the first weight row of the up half)
  int layout;       // LAYOUT_* bits: which of w, x and out are MFMA-tiled
};

struct NoRope {};
struct RopeArgs {  // EPI_ROPE: what dkv_rope_pack takes after the projection
  const uint16_t* cosv;
  const uint16_t* sinv;
  int64_t cs_stride;
  uint16_t* q_out;
  uint16_t* k_out;
  uint16_t* v_out;
  dkv_pack_job hjob;
  const dkv_pack_job* djob;  // read in place of hjob unless null
  uint8_t* arena;
  dkv_tile* tiles;
  int q_heads, heads, layers;
};

// Operand layouts. Rows of k contiguous elements, or MFMA-tiled: the 16 rows x 64 k of one pair
// of MFMA steps are 2 KB in the order the lanes read them, one 1 KB half per step (element (r, c)
// at ((r / 16) * kp + c / 64) * 1024 + (c / 32 % 2) * 512 + ((c / 8 % 4) * 16 + r % 16) * 8 + c % 8),
// so that each 16-byte-per-lane load instruction reads 1 KB of consecutive bytes (8 full cache
// lines instead of 64-byte halves of 16). A tiled x or out has its rows rounded up to 16.
enum {
  LAYOUT_W_TILED = DKV_LINEAR_W_TILED,
  LAYOUT_X_TILED = DKV_LINEAR_X_TILED,
  LAYOUT_OUT_TILED = DKV_LINEAR_OUT_TILED,
  LAYOUT_RES_TILED = DKV_LINEAR_RES_TILED
};

// Offset of element (r, c) of a tiled matrix with kp pairs of 64 columns per row.
__device__ __forceinline__ int64_t tiled_offset(int r, int c, int kp) {
  return ((int64_t)(r >> 4) * kp + (c >> 6)) * 1024 + ((c >> 5) & 1) * 512 + (((c >> 3) & 3) * 16 + (r & 15)) * 8 + (c & 7);
}

__device__ __forceinline__ float lane_group_sum(float x) {
  // sum over lanes col, col + 16, col + 32, col + 48 (gfx950 lane swaps)
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

template <int CH, int NT, int WAVES, int RB, int EPI, bool NORM, int OPS, typename Rope>
__device__ __forceinline__ void linear_body(const LinearArgs& a, const Rope& rope) {
  constexpr int NB = EPI == EPI_SILU_MUL ? 2 * NT : NT;  // column blocks multiplied
  // The arguments the first loads depend on, read together (placed by their uses, the compiler
  // read them in two dependent rounds of scalar loads, each a round trip to the cache hierarchy).
  asm volatile("" ::"s"(a.x), "s"(a.ldx), "s"(a.w), "s"(a.ldw), "s"(a.rows), "s"(a.kp), "s"(a.n_tiles),
               "s"(a.row_groups), "s"(a.up), "s"(a.layout));
  if constexpr (NORM) asm volatile("" ::"s"(a.norm));
  if constexpr (EPI == EPI_RESIDUAL) asm volatile("" ::"s"(a.res), "s"(a.ldr));
  const int b = blockIdx.x;
  const int xcd = b & 7, j = b >> 3;
  const int rg = j % a.row_groups;
  const int ct = (j / a.row_groups) * 8 + xcd;
  if (ct >= a.n_tiles) return;  // uniform over the workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int n0 = ct * 16 * NT;

  // A lane's operand pointers for pair 0, half 0, and the element steps to pair p and half h
  // (k = 64 p + 32 h): rows of k elements, or the MFMA-tiled layout (OPS = the layout bits of w
  // and x, compile-time so that the steps are immediate offsets of the loads).
  constexpr bool w_tiled = OPS & LAYOUT_W_TILED, x_tiled = OPS & LAYOUT_X_TILED;
  constexpr int wsp = w_tiled ? 1024 : 64, wsh = w_tiled ? 512 : 32;
  constexpr int xsp = x_tiled ? 1024 : 64, xsh = x_tiled ? 512 : 32;
  const uint16_t* wrow[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int r = (EPI == EPI_SILU_MUL && nb >= NT) ? a.up + n0 + 16 * (nb - NT) : n0 + 16 * nb;
    wrow[nb] = w_tiled ? a.w + (int64_t)(r >> 4) * a.kp * 1024 + 8 * lane : a.w + (int64_t)(r + col) * a.ldw + 8 * g;
  }
  // Rows past the end read the last row (or a tiled x's padding rows): x row j only reaches
  // output row j, which is not stored.
  const uint16_t* xrow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = min((rg * RB + rb) * 16 + col, a.rows - 1);
    // a tiled x ends with the block of its last row (the second block of a pair may be past it)
    const int block = min(rg * RB + rb, (a.rows - 1) >> 4);
    xrow[rb] = x_tiled ? a.x + (int64_t)block * a.kp * 1024 + 8 * lane : a.x + (int64_t)row * a.ldx + 8 * g;
  }

  constexpr int TILES = RB * NB, OUT = RB * NT;
  // The residual of the output tiles this wave finishes (tile o belongs to wave o % WAVES), loaded
  // first, so that it arrives with the operands: loaded in the epilogue it was one more memory
  // round trip after the reduction. Rows past the end read the last row (never stored).
  uint2 resv[EPI == EPI_RESIDUAL ? OUT : 1];
  if constexpr (EPI == EPI_RESIDUAL) {
#pragma unroll
    for (int o = 0; o < OUT; ++o) {
      if (o % WAVES != wave) continue;
      const int row = min((rg * RB + o / NT) * 16 + col, a.rows - 1), c = n0 + 16 * (o % NT) + 4 * g;
      // a tiled residual has its rows rounded up to 16: row (rg * RB + o / NT) * 16 + col is there
      resv[o] = *reinterpret_cast<const uint2*>(
          a.res + ((a.layout & LAYOUT_RES_TILED) ? tiled_offset((rg * RB + o / NT) * 16 + col, c, a.up >> 6)
                                                 : (int64_t)row * a.ldr + c));
    }
  }

  // EPI_ROPE: cos, sin and the job of the 8 rows that waves 0 and 1 finish each, 8 lanes per row.
  // (Read here, the job arrives with the operands; read where it is used it was one more round trip.)
  u32x4 cs = {0, 0, 0, 0}, sn = cs;
  dkv_pack_job job = {};
  if constexpr (EPI == EPI_ROPE) {
    job = rope.djob ? *rope.djob : rope.hjob;
    asm volatile("" ::: "memory");
    if (wave < 2) {
      const int64_t o = (int64_t)min(rg * 16 + 8 * wave + (lane >> 3), a.rows - 1) * rope.cs_stride + 8 * (lane & 7);
      cs = *reinterpret_cast<const u32x4*>(rope.cosv + o);
      sn = *reinterpret_cast<const u32x4*>(rope.sinv + o);
    }
  }

  // Every load of this wave's pairs (the host guarantees CH * WAVES >= kp) is
  // issued before the first MFMA. With the RMSNorm prologue the x rows and
  // the norm weight go first, unconditionally (a pair past kp loads pair
  // kp - 1 and is skipped below, so the loads form one straight-line block
  // whose uses wait for exactly what they need), and the weight tiles, which
  // come from HBM, only once x has arrived (load_weights below): the prologue
  // normalizes while they are in flight. Without it the first MFMA needs both,
  // and pairs past kp (p < kp is uniform over the wave) load nothing.
  Op8 xa[CH][2][RB], wa[CH][2][NB], gn[NORM ? CH : 1][2];
  auto load_weights = [&]() {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int p = min(wave + WAVES * i, a.kp - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 64 * p + 32 * h;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) wa[i][h][nb].u = *reinterpret_cast<const u32x4*>(wrow[nb] + p * wsp + h * wsh);
      }
    }
  };
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int p = min(wave + WAVES * i, a.kp - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = 64 * p + 32 * h;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) xa[i][h][rb].u = *reinterpret_cast<const u32x4*>(xrow[rb] + p * xsp + h * xsh);
        gn[i][h].u = *reinterpret_cast<const u32x4*>(a.norm + k + 8 * g);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int p = wave + WAVES * i;
      if (p < a.kp) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) wa[i][h][nb].u = *reinterpret_cast<const u32x4*>(wrow[nb] + p * wsp + h * wsh);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) xa[i][h][rb].u = *reinterpret_cast<const u32x4*>(xrow[rb] + p * xsp + h * xsh);
        }
      }
    }
  }
  if constexpr (NORM) {
    __shared__ float ssum[WAVES][RB][16];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (wave + WAVES * i < a.kp)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float lo = bf16_lo(xa[i][h][rb].u[e]), hi = bf16_hi(xa[i][h][rb].u[e]);
              ss = __fmaf_rn(lo, lo, ss);
              ss = __fmaf_rn(hi, hi, ss);
            }
      }
      ss = lane_group_sum(ss);
      if (g == 0) ssum[wave][rb][col] = ss;
    }
    // The weight tiles go out once x is in: issued with x, the CU took the waves' loads in issue
    // order and the later waves' x rows queued behind the first waves' weight tiles, so the
    // normalization barrier waited 1-2 us longer for them. A wave issues its weights when its own
    // x has arrived, or, with 32 x rows per workgroup (the SiLU*up shape), when every wave's has
    // (after the barrier): in a chain of 32 dependent launches Q/K/V took 6.32 us per launch with
    // the weights issued with x, 5.24 with them after a barrier that waits for no memory, 5.13
    // after the wave's own x, 5.44 after every wave's; gate/up 10.66, 10.12, 9.85 and 9.70 us.
    constexpr bool AFTER_BARRIER = RB > 1;
    if constexpr (!AFTER_BARRIER) load_weights();
    __syncthreads();
    if constexpr (AFTER_BARRIER) load_weights();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) tot += ssum[w][rb][col];
      const float rstd = 1.f / sqrtf(tot / (float)a.k + a.eps);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (wave + WAVES * i < a.kp)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t xv = xa[i][h][rb].u[e], gv = gn[i][h].u[e];
              xa[i][h][rb].u[e] = pack_bf16(round_bf16(bf16_lo(xv) * rstd) * bf16_lo(gv),
                                            round_bf16(bf16_hi(xv) * rstd) * bf16_hi(gv));
            }
      }
    }
  }
  f32x4_t acc[RB][NB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[rb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (wave + WAVES * i < a.kp)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            acc[rb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[i][h][nb].v, xa[i][h][rb].v, acc[rb][nb], 0, 0, 0);
  }

  // The waves' partials are summed in wave order through LDS, TP tiles per
  // phase (at most 32 KB of partials). Output tile o = (rb, nt) belongs to
  // wave o % WAVES, which sums its gate (and up) partial tiles and runs the
  // epilogue.
  constexpr int TP = TILES < 32 / WAVES ? TILES : 32 / WAVES;
  __shared__ f32x4_t red[WAVES][TP][64];
  f32x4_t gsum[OUT], usum[OUT];
#pragma unroll
  for (int ph = 0; ph < (TILES + TP - 1) / TP; ++ph) {
    if (ph) __syncthreads();  // the previous phase's partials have been read
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      const int t = ph * TP + j;
      if (t < TILES) red[wave][j][lane] = acc[t / NB][t % NB];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      const int t = ph * TP + j;
      if (t >= TILES) continue;
      const int rb = t / NB, nb = t % NB;
      const int o = rb * NT + nb % NT;  // output tile of this partial tile
      if (o % WAVES != wave) continue;
      f32x4_t s = red[0][j][lane];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) {
        const f32x4_t v = red[w][j][lane];
        s[0] += v[0];
        s[1] += v[1];
        s[2] += v[2];
        s[3] += v[3];
      }
      if (nb < NT) gsum[o] = s;
      else usum[o] = s;
    }
  }
  if constexpr (EPI == EPI_ROPE) {
    // The workgroup holds 16 whole rows of one 64-wide head: rounded to bf16 they meet in LDS, and
    // two waves rotate and pack 8 rows each.
    static_assert(NT == 4 && RB == 1, "one head per workgroup");
    constexpr int RS = D + 8;  // LDS row, in elements
    __shared__ __attribute__((aligned(16))) uint16_t head_rows[16 * RS];
#pragma unroll
    for (int o = 0; o < OUT; ++o) {
      if (o % WAVES != wave) continue;
      *reinterpret_cast<uint2*>(head_rows + col * RS + 16 * o + 4 * g) =
          make_uint2(pack_bf16(gsum[o][0], gsum[o][1]), pack_bf16(gsum[o][2], gsum[o][3]));
    }
    __syncthreads();
    if (wave >= 2) return;
    const int r = 8 * wave + (lane >> 3), c = lane & 7, tok = rg * 16 + r;
    if (ct == 0 && rg == 0 && wave == 0 && job.write_tiles) write_segment_tiles(job, rope.layers, rope.heads, rope.tiles);
    rope_pack_row(*reinterpret_cast<const u32x4*>(head_rows + r * RS + 8 * c), cs, sn, ct, tok, tok < a.rows, c, a.rows,
                  rope.q_heads, rope.q_out, rope.k_out, rope.v_out, job, rope.arena, rope.layers, rope.heads);
    return;
  }
#pragma unroll
  for (int o = 0; o < OUT; ++o) {
    if (o % WAVES != wave) continue;
    const int rb = o / NT, nt = o % NT;
    const int row = (rg * RB + rb) * 16 + col;
    if (row >= a.rows) continue;
    const int c = n0 + 16 * nt + 4 * g;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = round_bf16(gsum[o][e]);
    if (EPI == EPI_RESIDUAL) {
      const uint2 r = resv[o];
      y[0] += bf16_lo(r.x);
      y[1] += bf16_hi(r.x);
      y[2] += bf16_lo(r.y);
      y[3] += bf16_hi(r.y);
    } else if (EPI == EPI_SILU_MUL) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = round_bf16(y[e] / (1.f + expf(-y[e]))) * round_bf16(usum[o][e]);
    }
    // a tiled out is the next projection's tiled x (k = n_out = a.up)
    uint16_t* dst = a.out + ((a.layout & LAYOUT_OUT_TILED) ? tiled_offset(row, c, a.up >> 6) : (int64_t)row * a.ldo + c);
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
  }
}

template <int CH, int NT, int WAVES, int RB, int EPI, bool NORM, int OPS>
__global__ void __launch_bounds__(64 * WAVES) linear_kernel(const LinearArgs a) {
  linear_body<CH, NT, WAVES, RB, EPI, NORM, OPS>(a, NoRope{});
}

// Q/K/V with the RMSNorm prologue that ends in dkv_rope_pack's work: a workgroup computes 16 rows of one
// 64-wide head, so the rows it rotates and quantizes are its own. Half as many workgroups as the plain
// projection, each with twice the weight bytes (123 KB at k 960, which bounds it), but one launch and one
// round trip of q | k | v through memory less: the 960-wide decoder's launch 7.2 us instead of 5.6 + 3.5
// at 64 rows. A whole layer past 640 in graph replays, two launches -> one: 1 row 25.6 -> 25.0 us,
// 16 rows 28.2 -> 27.1, 64 rows 32.4 -> 31.1, 128 rows 42.6 -> 39.5, 256 rows 56.5 -> 54.0, 340 rows
// 64.0 -> 62.1: better at every size that keeps the few-row kernel.
template <int CH, int OPS>
__global__ void __launch_bounds__(512) linear_rope_kernel(const LinearArgs a, const RopeArgs rope) {
  linear_body<CH, 4, 8, 1, EPI_ROPE, true, OPS>(a, rope);
}

// The same projections for many rows (prompts, several frames at once), where linear_kernel reads
// every weight tile again for each 16 or 32 rows. A workgroup of 4 waves (2 x 2) computes 64 x rows
// by 64 weight rows. Per pair of MFMA steps (64 k) 64 + 64 rows go to LDS, 1 KB per 16 rows and step
// in the order the lanes read them, so every LDS access is 1 KB of consecutive bytes.
//
// The arithmetic is linear_kernel's, operation for operation, so that a row's result does not
// depend on how many rows its call has: that kernel's wave w accumulates the pairs w, w + 8, ... (a
// chain) from zero, and the chains are added in wave order. Here a wave walks chain after chain.
//
// Loads go straight to LDS (global_load_lds), into one of TILE_RING buffers, TILE_RING - 1 pairs
// ahead; one barrier per pair. (Through registers, the ds_writes took longer than the loads: gate/up
// at 1000 rows 29.4 us, 17.8 with the writes left out.) What bounds it now is the rate at which a CU
// takes bytes from L2, about 60 KB/us each however many CUs load: 245 KB per 64 x 64 tile of k 960.
// The 960-wide decoder's projections, linear_kernel -> this (with the norm launch), us per launch:
//   rows   Q/K/V            o_proj           gate/up          down_proj
//    256   10.1 -> 11.1      6.4 ->  7.4     16.7 -> 12.6      8.1 -> 13.6
//    512   16.4 -> 11.9     10.8 ->  7.6     26.5 -> 16.1     13.7 -> 13.9
//   1000   29.4 -> 15.0     19.5 ->  8.2     50.6 -> 24.1     40.9 -> 14.5
//   2048   60.4 -> 24.4     36.3 -> 14.1    103.6 -> 42.9     94.3 -> 21.5
// Tiles of 128 x 64 and 128 x 128 (4 or 8 waves) were slower below 2048 rows (fewer workgroups, and
// prologues and epilogues that nothing overlaps); a ring of 4 buffers changed nothing.
constexpr int TILE_M = 64, TILE_N = 64, TILE_RING = 3;

// A wave's operands of one MFMA step, out of LDS: two pieces from x and two from w on, the second 2 KB
// after the first (the up piece of SiLU*up WSTEP bytes after the gate's). One asm block with its own
// wait: as ordinary LDS loads they waited for every global_load_lds in flight at the head of the
// pair loop.
template <int WSTEP>
__device__ __forceinline__ void lds_operands(uint32_t x, uint32_t w, Op8 (&xa)[2], Op8 (&wa)[2]) {
  asm volatile(
      "ds_read_b128 %0, %4\n ds_read_b128 %1, %4 offset:2048\n"
      "ds_read_b128 %2, %5\n ds_read_b128 %3, %5 offset:%6\n s_waitcnt lgkmcnt(0)"
      : "=&v"(xa[0].u), "=&v"(xa[1].u), "=&v"(wa[0].u), "=&v"(wa[1].u)
      : "v"(x), "v"(w), "n"(WSTEP)
      : "memory");
}

// A pair's eight pieces of x: (step, block of 16 rows).
__device__ __forceinline__ void lds_pair(uint32_t x, Op8 (&xa)[2][4]) {
  asm volatile(
      "ds_read_b128 %0, %8\n ds_read_b128 %1, %8 offset:2048\n"
      "ds_read_b128 %2, %8 offset:4096\n ds_read_b128 %3, %8 offset:6144\n"
      "ds_read_b128 %4, %8 offset:1024\n ds_read_b128 %5, %8 offset:3072\n"
      "ds_read_b128 %6, %8 offset:5120\n ds_read_b128 %7, %8 offset:7168\n s_waitcnt lgkmcnt(0)"
      : "=&v"(xa[0][0].u), "=&v"(xa[0][1].u), "=&v"(xa[0][2].u), "=&v"(xa[0][3].u), "=&v"(xa[1][0].u),
        "=&v"(xa[1][1].u), "=&v"(xa[1][2].u), "=&v"(xa[1][3].u)
      : "v"(x)
      : "memory");
}

template <int EPI, int OPS, typename Rope>
__device__ __forceinline__ void tile_body(const LinearArgs& a, const Rope& rope) {
  constexpr int NT = EPI == EPI_SILU_MUL ? TILE_N / 2 : TILE_N;  // output columns of the workgroup
  constexpr int NH = EPI == EPI_SILU_MUL ? 1 : 2;                // 16-column blocks of them per wave
  constexpr int XF = TILE_M / 8, F = XF + TILE_N / 8, FW = F / 4;  // 1 KB pieces of a pair: of x, in all, per wave
  __shared__ __attribute__((aligned(1024))) u32x4 lds[TILE_RING * F][64];
  const int b = blockIdx.x;
  const int xcd = b & 7, j = b >> 3;
  const int rg = j % a.row_groups;
  const int ct = (j / a.row_groups) * 8 + xcd;
  if (ct >= a.n_tiles) return;  // uniform over the workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  const int n0 = ct * NT, m0 = rg * TILE_M;
  constexpr bool w_tiled = OPS & LAYOUT_W_TILED, x_tiled = OPS & LAYOUT_X_TILED;
  const int last_block = (a.rows - 1) >> 4;

  // Piece f of a pair: block f / 2 of x (then of w), MFMA step f % 2. A wave loads pieces wave,
  // wave + 4, ...
  const uint16_t* src[FW];
#pragma unroll
  for (int q = 0; q < FW; ++q) {
    const int f = wave + 4 * q, h = f & 1;
    if (4 * q < XF) {  // rows past the end read the last row (block) and are not stored
      const int row = m0 + 16 * (f >> 1);
      src[q] = x_tiled ? a.x + (int64_t)min(row >> 4, last_block) * a.kp * 1024 + 512 * h + 8 * lane
                       : a.x + (int64_t)min(row + col, a.rows - 1) * a.ldx + 32 * h + 8 * g;
    } else {
      const int cb = (f - XF) >> 1;
      const int r = EPI == EPI_SILU_MUL && cb >= NT / 16 ? a.up + n0 + 16 * (cb - NT / 16) : n0 + 16 * cb;
      src[q] = w_tiled ? a.w + (int64_t)(r >> 4) * a.kp * 1024 + 512 * h + 8 * lane
                       : a.w + (int64_t)(r + col) * a.ldw + 32 * h + 8 * g;
    }
  }
  auto next = [&](int p) {  // the pair after p: the next of its chain, or the next chain's first
    const int q = p + 8;
    return q < a.kp ? q : (p & 7) + 1;
  };
  // Past the last pair the last one is loaded again (never used), so that every pair has FW loads
  // after it.
  int pl = 0, loaded = 0;  // pair loaded next and its place in the order
  int fill = 0;  // the buffer loaded next
  auto load_next = [&]() {
#pragma unroll
    for (int q = 0; q < FW; ++q) {
      const uint16_t* from = src[q] + ((4 * q < XF ? x_tiled : w_tiled) ? 1024 * pl : 64 * pl);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                       (__attribute__((address_space(3))) void*)lds[fill * F + wave + 4 * q], 16, 0, 0);
    }
    fill = fill + 1 == TILE_RING ? 0 : fill + 1;
    if (++loaded < a.kp) pl = next(pl);
  };

  f32x4_t acc[2][2], sum[2][2];  // the chain in progress; the chains done
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      acc[mb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      sum[mb][nb] = f32x4_t{-0.f, -0.f, -0.f, -0.f};  // -0 + x is x, for every x
    }
  // LDS byte addresses of this wave's first x and w piece in buffer 0
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds + 16 * lane;
  const uint32_t xl = base + 4096 * wm, wl = base + 1024 * XF + 2048 * wn * NH;
  constexpr int WSTEP = EPI == EPI_SILU_MUL ? 2048 * (NT / 16) : 2048;
  auto compute = [&](uint32_t at) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      Op8 xa[2], wa[2];
      lds_operands<WSTEP>(xl + at + 1024 * h, wl + at + 1024 * h, xa, wa);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[nb].v, xa[mb].v, acc[mb][nb], 0, 0, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < TILE_RING - 1; ++k) load_next();
  int p = 0;        // pair being computed
  uint32_t at = 0;  // its buffer, in bytes
  for (int s = 0; s < a.kp; ++s) {
    // The pair's pieces have landed (this wave's: at most the loads of the TILE_RING - 2 pairs after it
    // are under way; the other waves': the barrier), and every wave is past the pair before it,
    // whose buffer the next loads overwrite.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((TILE_RING - 2) * FW) : "memory");
    __builtin_amdgcn_s_barrier();
    load_next();
    compute(at);
    at = at + 1024 * F == 1024 * F * TILE_RING ? 0 : at + 1024 * F;
    if (p + 8 >= a.kp) {  // the chain's last pair
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            sum[mb][nb][e] += acc[mb][nb][e];
            acc[mb][nb][e] = 0.f;
          }
    }
    p = next(p);
  }

  // The loads past the last pair still write this workgroup's LDS.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  if constexpr (EPI == EPI_ROPE) {
    // A tile is 64 rows of one 64-wide head: rounded to bf16 they meet in LDS (over the operand
    // buffers, once every wave's last loads have landed), and a wave rotates and packs 16 of them.
    constexpr int RS = D + 8;  // LDS row, in elements
    static_assert(TILE_N == D && TILE_M * RS * 2 <= (int)sizeof(lds), "one head per workgroup");
    uint16_t* head_rows = reinterpret_cast<uint16_t*>(lds);
    const dkv_pack_job job = rope.djob ? *rope.djob : rope.hjob;
    const int c = lane & 7;
    u32x4 cs[2], sn[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t o = (int64_t)min(m0 + 16 * wave + 8 * i + (lane >> 3), a.rows - 1) * rope.cs_stride + 8 * c;
      cs[i] = *reinterpret_cast<const u32x4*>(rope.cosv + o);
      sn[i] = *reinterpret_cast<const u32x4*>(rope.sinv + o);
    }
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
        *reinterpret_cast<uint2*>(head_rows + (16 * (wm * 2 + mb) + col) * RS + 16 * (wn * 2 + nb) + 4 * g) =
            make_uint2(pack_bf16(sum[mb][nb][0], sum[mb][nb][1]), pack_bf16(sum[mb][nb][2], sum[mb][nb][3]));
    __syncthreads();
    if (ct == 0 && rg == 0 && wave == 0 && job.write_tiles) write_segment_tiles(job, rope.layers, rope.heads, rope.tiles);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = 16 * wave + 8 * i + (lane >> 3), tok = m0 + r;
      rope_pack_row(*reinterpret_cast<const u32x4*>(head_rows + r * RS + 8 * c), cs[i], sn[i], ct, tok, tok < a.rows, c,
                    a.rows, rope.q_heads, rope.q_out, rope.k_out, rope.v_out, job, rope.arena, rope.layers, rope.heads);
    }
    return;
  }

  uint2 resv[2][2];
  if constexpr (EPI == EPI_RESIDUAL) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const int row = min(m0 + 16 * (wm * 2 + mb) + col, a.rows - 1), c = n0 + 16 * (wn * 2 + nb) + 4 * g;
        resv[mb][nb] = *reinterpret_cast<const uint2*>(
            a.res + ((a.layout & LAYOUT_RES_TILED) ? tiled_offset(row, c, a.up >> 6) : (int64_t)row * a.ldr + c));
      }
  }
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int row = m0 + 16 * (wm * 2 + mb) + col;
    if (row >= a.rows) continue;
#pragma unroll
    for (int nb = 0; nb < NH; ++nb) {
      const int c = n0 + 16 * (wn * NH + nb) + 4 * g;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = round_bf16(sum[mb][nb][e]);
      if constexpr (EPI == EPI_RESIDUAL) {
        const uint2 r = resv[mb][nb];
        y[0] += bf16_lo(r.x);
        y[1] += bf16_hi(r.x);
        y[2] += bf16_lo(r.y);
        y[3] += bf16_hi(r.y);
      } else if constexpr (EPI == EPI_SILU_MUL) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          y[e] = round_bf16(y[e] / (1.f + expf(-y[e]))) * round_bf16(sum[mb][NH + nb][e]);
      }
      uint16_t* dst = a.out + ((a.layout & LAYOUT_OUT_TILED) ? tiled_offset(row, c, a.up >> 6) : (int64_t)row * a.ldo + c);
      *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
    }
  }
}

template <int EPI, int OPS>
__global__ void __launch_bounds__(256, 3) linear_tile_kernel(const LinearArgs a) {
  tile_body<EPI, OPS>(a, NoRope{});
}

// Q/K/V of many rows, ending in dkv_rope_pack's work as linear_rope_kernel does: the 960-wide decoder's
// launch at 1000 rows 12.6 us instead of 10.4 + 4.3. A whole eager layer past 640, recorded in a HIP graph to
// time it, two launches -> one: 380 rows 64.6 -> 63.4 us, 512 rows 71.1 -> 69.9, 700 rows 77.5 -> 75.5, 1000
// rows 81.7 -> 79.0. (Layers of so many rows under graph steps keep the two launches.)
template <int OPS>
__global__ void __launch_bounds__(256, 3) linear_tile_rope_kernel(const LinearArgs a, const RopeArgs rope) {
  tile_body<EPI_ROPE, OPS>(a, rope);
}

// SiLU*up over [gate | up] weights for many rows, linear_tile_kernel's arithmetic. A wave owns 64 x rows by
// 16 gate and 16 up columns, so no weight tile is shared between waves: each goes straight from memory to
// the registers of the one wave that multiplies it, two pairs ahead, and only x passes through LDS: 24 KB of
// loads per 64 x 128 weight rows and pair instead of 32, and 40 KB of LDS traffic instead of 96. It needs
// the chip full, since a workgroup covers twice the columns (GLU_FROM): gate/up of the 960-wide decoder,
// 64 x 64 tiles -> this, us per launch: 256 rows (160 workgroups) 8.9 -> 9.7, 512 rows (320) 12.0 -> 12.2,
// 1000 rows (640) 19.6 -> 17.6, 2048 rows (1280) 37.1 -> 28.8. It is bound as the tiles are, by the
// bytes a CU takes from L2. (A ring of 4 spilled; reading x a step at a time changed nothing.)
constexpr int GLU_RING = 3;
constexpr int GLU_N = 64;      // output columns of a workgroup: 4 waves of 16
constexpr int GLU_FROM = 512;  // workgroups from which it runs (two per CU)

template <int OPS>
__global__ void __launch_bounds__(256, 3) linear_glu_kernel(const LinearArgs a) {
  constexpr int XF = TILE_M / 8, XW = XF / 4;  // 1 KB pieces of x per pair, and per wave
  __shared__ __attribute__((aligned(1024))) u32x4 lds[GLU_RING * XF][64];
  const int b = blockIdx.x;
  const int xcd = b & 7, j = b >> 3;
  const int rg = j % a.row_groups;
  const int ct = (j / a.row_groups) * 8 + xcd;
  if (ct >= a.n_tiles) return;  // uniform over the workgroup
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int n0 = ct * GLU_N + 16 * wave, m0 = rg * TILE_M;
  const int nl = min(n0, a.up - 16);  // a wave past the last column loads the last columns and stores nothing
  constexpr bool w_tiled = OPS & LAYOUT_W_TILED, x_tiled = OPS & LAYOUT_X_TILED;
  constexpr int wsp = w_tiled ? 1024 : 64, wsh = w_tiled ? 512 : 32;

  const uint16_t* xsrc[XW];  // this wave's pieces: block f / 2 of x, MFMA step f % 2
#pragma unroll
  for (int q = 0; q < XW; ++q) {  // rows past the end read the last row (block) and are not stored
    const int f = wave + 4 * q, h = f & 1, row = m0 + 16 * (f >> 1);
    xsrc[q] = x_tiled ? a.x + (int64_t)min(row >> 4, (a.rows - 1) >> 4) * a.kp * 1024 + 512 * h + 8 * lane
                      : a.x + (int64_t)min(row + col, a.rows - 1) * a.ldx + 32 * h + 8 * g;
  }
  const uint16_t* wsrc[2];  // gate, up
#pragma unroll
  for (int nb = 0; nb < 2; ++nb) {
    const int r = nl + nb * a.up;
    wsrc[nb] = w_tiled ? a.w + (int64_t)(r >> 4) * a.kp * 1024 + 8 * lane : a.w + (int64_t)(r + col) * a.ldw + 8 * g;
  }
  auto next = [&](int p) {  // the pair after p: the next of its chain, or the next chain's first
    const int q = p + 8;
    return q < a.kp ? q : (p & 7) + 1;
  };
  // Past the last pair the last one is loaded again (never used), so that every pair has as many loads
  // after it.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  Op8 w[GLU_RING][2][2];
  int pl = 0, loaded = 0, fill = 0;  // pair loaded next, its place in the order, its buffer
  auto load_next = [&](Op8 (&to)[2][2]) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int h = 0; h < 2; ++h) to[nb][h].u = *reinterpret_cast<const u32x4*>(wsrc[nb] + wsp * pl + wsh * h);
#pragma unroll
    for (int q = 0; q < XW; ++q)
      load_piece(xsrc[q] + (x_tiled ? 1024 : 64) * pl, lds0 + 1024 * (fill * XF + wave + 4 * q));
    fill = fill + 1 == GLU_RING ? 0 : fill + 1;
    if (++loaded < a.kp) pl = next(pl);
  };
  f32x4_t acc[4][2], sum[4][2];  // the chain in progress; the chains done
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      acc[mb][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      sum[mb][nb] = f32x4_t{-0.f, -0.f, -0.f, -0.f};  // -0 + x is x, for every x
    }
  const uint32_t base = lds0 + 16 * lane;
#pragma unroll
  for (int k = 0; k < GLU_RING - 1; ++k) load_next(w[k]);
  int p = 0;  // pair being computed
  for (int s0 = 0; s0 < a.kp; s0 += GLU_RING) {
#pragma unroll
    for (int i = 0; i < GLU_RING; ++i) {  // pair s0 + i, in buffer i
      if (s0 + i >= a.kp) break;
      // The pair's pieces have landed (this wave's: only the GLU_RING - 2 pairs after it are under way;
      // the other waves': the barrier), and every wave is past the pair before it.
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((GLU_RING - 2) * (XW + 4)) : "memory");
      // the wait above is for this pair's weights too; the compiler places its own here, not after the
      // loads below
      asm volatile("" : "+v"(w[i][0][0].u), "+v"(w[i][0][1].u), "+v"(w[i][1][0].u), "+v"(w[i][1][1].u));
      __builtin_amdgcn_s_barrier();
      load_next(w[(i + GLU_RING - 1) % GLU_RING]);
      const uint32_t at = base + 1024 * XF * i;
      Op8 xa[2][4];
      lds_pair(at, xa);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][nb][h].v, xa[h][mb].v, acc[mb][nb], 0, 0, 0);
      if (p + 8 >= a.kp) {  // the chain's last pair
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              sum[mb][nb][e] += acc[mb][nb][e];
              acc[mb][nb][e] = 0.f;
            }
      }
      p = next(p);
    }
  }
  // The loads past the last pair still write this workgroup's LDS.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (n0 >= a.up) return;
  const int c = n0 + 4 * g;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    const int row = m0 + 16 * mb + col;
    if (row >= a.rows) continue;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = round_bf16(sum[mb][0][e]);
      y[e] = round_bf16(x / (1.f + expf(-x))) * round_bf16(sum[mb][1][e]);
    }
    uint16_t* dst = a.out + ((a.layout & LAYOUT_OUT_TILED) ? tiled_offset(row, c, a.up >> 6) : (int64_t)row * a.ldo + c);
    *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
  }
}

// RMSNorm of x rows into the MFMA-tiled layout, for linear_tile_kernel: linear_kernel's prologue as
// a launch of its own (there every workgroup normalizes its x rows again; with 16 times the rows per
// weight tile that work is worth doing once). One workgroup per 16 rows; wave w sums and normalizes
// pairs w, w + 8, ..., in linear_kernel's order.
template <int CH, bool XT>
__global__ void __launch_bounds__(512)
rms_tiled_kernel(const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ norm,
                 uint16_t* __restrict__ out, int rows, int k, int kp, float eps) {
  constexpr int WAVES = 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int64_t tile = (int64_t)blockIdx.x * kp * 1024 + 8 * lane;
  const uint16_t* xr = XT ? x + tile : x + (int64_t)min((int)blockIdx.x * 16 + col, rows - 1) * ldx + 8 * g;
  Op8 xa[CH][2], gn[CH][2];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int p = min(wave + WAVES * i, kp - 1);  // a pair past kp is loaded and skipped
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xa[i][h].u = *reinterpret_cast<const u32x4*>(xr + (XT ? 1024 * p + 512 * h : 64 * p + 32 * h));
      gn[i][h].u = *reinterpret_cast<const u32x4*>(norm + 64 * p + 32 * h + 8 * g);
    }
  }
  __shared__ float ssum[WAVES][16];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    if (wave + WAVES * i < kp)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = bf16_lo(xa[i][h].u[e]), hi = bf16_hi(xa[i][h].u[e]);
          ss = __fmaf_rn(lo, lo, ss);
          ss = __fmaf_rn(hi, hi, ss);
        }
  }
  ss = lane_group_sum(ss);
  if (g == 0) ssum[wave][col] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) tot += ssum[w][col];
  const float rstd = 1.f / sqrtf(tot / (float)k + eps);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int p = wave + WAVES * i;
    if (p >= kp) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t xv = xa[i][h].u[e], gv = gn[i][h].u[e];
        y[e] = pack_bf16(round_bf16(bf16_lo(xv) * rstd) * bf16_lo(gv), round_bf16(bf16_hi(xv) * rstd) * bf16_hi(gv));
      }
      *reinterpret_cast<u32x4*>(out + tile + 1024 * p + 512 * h) = y;  // padding rows repeat the last row
    }
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Launch shapes, from graph-replay timings of the 960-wide decoder's projections at 64 rows
// (weights streamed from HBM): narrow outputs use one 16-row block per workgroup (more
// workgroups); the joined gate/up projection 32 x rows and 32 output columns per workgroup
// (160 workgroups at 64 rows, all resident at once). With the RMSNorm prologue every
// workgroup normalizes its own x rows, so fewer rows per workgroup cost less VALU time than
// the second read of each weight tile they bring (64 rows per workgroup: 13.3 us, 32: 11.4 us).
struct Shape {
  int ch, nt, waves, rb;
  bool tile;  // linear_tile_kernel
};

constexpr int MAX_CH = 5;       // pairs per wave: k <= 5 * 8 * 64 = 2560
constexpr int MAX_NORM_CH = 2;  // with the RMSNorm prologue (k <= 1024), which keeps those
                                // variants out of scratch

Shape pick(int rows, int n_out, int kp, bool norm, int epilogue) {
  Shape s;
  s.waves = 8;
  s.ch = (kp + s.waves - 1) / s.waves;  // every pair of a wave in registers at once
  s.tile = false;
  if (epilogue == EPI_SILU_MUL) {  // 32 gate and 32 up weight rows, 32 x rows
    s.nt = 2;
    s.rb = 2;
  } else {
    s.nt = (n_out % 32 == 0 && n_out / 16 > 64) ? 2 : 1;
    s.rb = 1;
  }
  // Many rows: linear_tile_kernel, from the number of linear_kernel workgroups on at which it was
  // faster (table above; 256 CUs). SiLU*up: as soon as they are more than one per CU (rows 96 -> 128:
  // 7.2 -> 11.9 us, tiles 10.7 with the norm launch). Other projections: k 960 at 1000 to 1200
  // workgroups (o_proj 256 rows 6.4 against 7.4 us, 384 rows 8.6 against 7.5; Q/K/V 256 rows 10.1
  // against 11.1, 384 rows 13.9 against 11.5), k 2560 at 1920 (512 rows 13.7 against 13.9, 768 rows
  // 20.7 against 14.3).
  const int cols = 16 * s.nt, per = epilogue == EPI_SILU_MUL ? 2 : 1;
  const int64_t groups = (int64_t)((rows + 16 * s.rb - 1) / (16 * s.rb)) * (n_out / cols);
  const int64_t most = epilogue == EPI_SILU_MUL ? 256 : (kp > 16 ? 2000 : 1100);
  if (!norm && n_out * per % TILE_N == 0 && groups > most) {
    s.tile = true;
    s.nt = TILE_N / per / 16;
    s.rb = TILE_M / 16;
  }
  return s;
}

template <int CH, int NT, int WAVES, int RB, int EPI, bool NORM, int OPS>
void launch_one(const LinearArgs& a, hipStream_t st) {
  const int groups = (a.n_tiles + 7) / 8;
  const unsigned blocks = (unsigned)groups * 8u * (unsigned)a.row_groups;
  hipLaunchKernelGGL((linear_kernel<CH, NT, WAVES, RB, EPI, NORM, OPS>), dim3(blocks), dim3(64 * WAVES), 0, st, a);
}

template <int EPI, int OPS>
void launch_tile(LinearArgs a, hipStream_t st) {
  if constexpr (EPI == EPI_SILU_MUL) {
    const int wide = (a.up + GLU_N - 1) / GLU_N;
    if ((int64_t)wide * a.row_groups >= GLU_FROM) {
      a.n_tiles = wide;
      hipLaunchKernelGGL((linear_glu_kernel<OPS>), dim3((unsigned)((wide + 7) / 8) * 8u * (unsigned)a.row_groups), dim3(256), 0,
                         st, a);
      return;
    }
  }
  const unsigned blocks = (unsigned)((a.n_tiles + 7) / 8) * 8u * (unsigned)a.row_groups;
  hipLaunchKernelGGL((linear_tile_kernel<EPI, OPS>), dim3(blocks), dim3(256), 0, st, a);
}

template <int NT, int WAVES, int RB, int EPI, bool NORM, int OPS>
void launch_ch(int ch, const LinearArgs& a, hipStream_t st) {
  if constexpr (NORM) {
    if (ch == 1) launch_one<1, NT, WAVES, RB, EPI, NORM, OPS>(a, st);
    else launch_one<MAX_NORM_CH, NT, WAVES, RB, EPI, NORM, OPS>(a, st);
  } else {
    switch (ch) {
      case 1: launch_one<1, NT, WAVES, RB, EPI, NORM, OPS>(a, st); break;
      case 2: launch_one<2, NT, WAVES, RB, EPI, NORM, OPS>(a, st); break;
      case 3: launch_one<3, NT, WAVES, RB, EPI, NORM, OPS>(a, st); break;
      case 4: launch_one<4, NT, WAVES, RB, EPI, NORM, OPS>(a, st); break;
      default:
        if constexpr (EPI != EPI_SILU_MUL) launch_one<MAX_CH, NT, WAVES, RB, EPI, NORM, OPS>(a, st);
        break;  // dkv_linear_supported rules out the rest
    }
  }
}

template <int EPI, bool NORM, int OPS>
void launch_ops(const Shape& s, const LinearArgs& a, hipStream_t st) {
  if constexpr (!NORM)
    if (s.tile) return launch_tile<EPI, OPS>(a, st);
  if constexpr (EPI == EPI_SILU_MUL) {
    launch_ch<2, 8, 2, EPI, NORM, OPS>(s.ch, a, st);
  } else {
    if (s.nt == 2) launch_ch<2, 8, 1, EPI, NORM, OPS>(s.ch, a, st);
    else launch_ch<1, 8, 1, EPI, NORM, OPS>(s.ch, a, st);
  }
}

template <int EPI, bool NORM>
void launch_epi(const Shape& s, const LinearArgs& a, hipStream_t st) {
  switch (a.layout & (LAYOUT_W_TILED | LAYOUT_X_TILED)) {
    case 0: launch_ops<EPI, NORM, 0>(s, a, st); break;
    case LAYOUT_W_TILED: launch_ops<EPI, NORM, LAYOUT_W_TILED>(s, a, st); break;
    case LAYOUT_X_TILED: launch_ops<EPI, NORM, LAYOUT_X_TILED>(s, a, st); break;
    default: launch_ops<EPI, NORM, LAYOUT_W_TILED | LAYOUT_X_TILED>(s, a, st); break;
  }
}

}  // namespace
}  // namespace dkv

using namespace dkv;

extern "C" {

int dkv_linear_supported(int32_t rows, int32_t n, int32_t k, int32_t has_norm, int32_t epilogue) {
  if (rows < 0 || n <= 0 || k <= 0 || (k & 63) || epilogue < 0 || epilogue > 2) return 0;
  const int n_out = epilogue == EPI_SILU_MUL ? n / 2 : n;
  if (epilogue == EPI_SILU_MUL && (n & 1)) return 0;
  if (n_out % 16) return 0;
  const Shape s = pick(rows, n_out, k / 64, has_norm, epilogue);
  const int max_ch = has_norm ? MAX_NORM_CH : (epilogue == EPI_SILU_MUL ? 4 : MAX_CH);  // register budget
  if (s.ch > max_ch) return 0;
  if (n_out % (16 * s.nt)) return 0;
  return 1;
}

int dkv_linear_tiled(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int32_t rows,
                     int32_t n, int32_t k, const void* norm_weight, float eps, int32_t epilogue, const void* residual,
                     int64_t residual_row_stride, void* out, int64_t out_row_stride, int32_t layout, void* stream) {
  clear_error();
  const bool norm = norm_weight != nullptr;
  const int n_out = epilogue == EPI_SILU_MUL ? n / 2 : n;
  // row strides of tiled operands are not used (their layout fixes every offset)
  const bool wt = layout & LAYOUT_W_TILED, xt = layout & LAYOUT_X_TILED, ot = layout & LAYOUT_OUT_TILED;
  const bool rt = layout & LAYOUT_RES_TILED;
  if (!x || !w || !out || !dkv_linear_supported(rows, n, k, norm, epilogue) || !al16(x) || !al16(w) ||
      !al16(out) || (norm && !al16(norm_weight)) || (layout & ~15) || ((ot || rt) && (n_out & 63)) ||
      (rt && epilogue != EPI_RESIDUAL) ||
      (!xt && ((x_row_stride & 7) || x_row_stride < k)) || (!wt && ((w_row_stride & 7) || w_row_stride < k)) ||
      (!ot && ((out_row_stride & 3) || out_row_stride < n_out)) ||
      (epilogue == EPI_RESIDUAL &&
       (!residual || ((uintptr_t)residual & 7) || (!rt && ((residual_row_stride & 3) || residual_row_stride < n_out))))) {
    set_error("dkv_linear: unsupported or bad arguments (rows %d, n %d, k %d, epilogue %d, layout %d; k a multiple "
              "of 64, 16-byte aligned bf16 rows, a tiled out or residual n_out a multiple of 64)", rows, n, k,
              epilogue, layout);
    return DKV_EINVAL;
  }
  if (rows == 0) return 0;
  const Shape s = pick(rows, n_out, k / 64, norm, epilogue);
  LinearArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = x_row_stride;
  a.w = static_cast<const uint16_t*>(w);
  a.ldw = w_row_stride;
  a.norm = static_cast<const uint16_t*>(norm_weight);
  a.res = static_cast<const uint16_t*>(residual);
  a.ldr = residual_row_stride;
  a.out = static_cast<uint16_t*>(out);
  a.ldo = out_row_stride;
  a.eps = eps;
  a.rows = rows;
  a.k = k;
  a.kp = k / 64;
  a.n_tiles = n_out / (16 * s.nt);
  a.row_groups = (rows + 16 * s.rb - 1) / (16 * s.rb);
  a.up = n_out;
  a.layout = layout;
  hipStream_t st = (hipStream_t)stream;
  if (epilogue == EPI_PLAIN) norm ? launch_epi<EPI_PLAIN, true>(s, a, st) : launch_epi<EPI_PLAIN, false>(s, a, st);
  else if (epilogue == EPI_RESIDUAL)
    norm ? launch_epi<EPI_RESIDUAL, true>(s, a, st) : launch_epi<EPI_RESIDUAL, false>(s, a, st);
  else norm ? launch_epi<EPI_SILU_MUL, true>(s, a, st) : launch_epi<EPI_SILU_MUL, false>(s, a, st);
  return (int)hipGetLastError();
}

int dkv_linear_rope_pack(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int32_t n, int32_t k,
                         const void* norm_weight, float eps, int32_t layout, const void* cos, const void* sin,
                         int64_t cs_row_stride, int32_t q_heads, void* q_out, void* k_out, void* v_out,
                         const dkv_pack_job* job, int32_t job_on_device, void* arena, int64_t arena_bytes,
                         dkv_tile* tiles, int32_t layers, int32_t heads, void* stream) {
  clear_error();
  const bool wt = layout & LAYOUT_W_TILED, xt = layout & LAYOUT_X_TILED;
  if (!x || !w || (norm_weight == nullptr) != xt || !cos || !sin || !q_out || !k_out || !v_out || !job || !arena || !tiles ||
      n < 1 || k <= 0 || (k & 63) || k > 64 * 8 * MAX_NORM_CH || q_heads <= 0 || heads <= 0 || layers <= 0 ||
      (layout & ~(LAYOUT_W_TILED | LAYOUT_X_TILED)) || !al16(x) || !al16(w) || !al16(norm_weight) || !al16(cos) ||
      !al16(sin) || !al16(q_out) || !al16(k_out) || !al16(v_out) || (!xt && ((x_row_stride & 7) || x_row_stride < k)) ||
      (!wt && ((w_row_stride & 7) || w_row_stride < k)) || (cs_row_stride & 7) || cs_row_stride < D) {
    set_error("dkv_linear_rope_pack: bad arguments (%d rows of %d; at least one row, k a multiple of 64 up to %d, 16-byte "
              "aligned bf16 buffers, strides multiples of 8 elements)", n, k, 64 * 8 * MAX_NORM_CH);
    return DKV_EINVAL;
  }
  if (!job_on_device) {
    if (int rc = check_job(*job, arena_bytes, layers, heads)) return rc;
    if (job->n != n || (job->write_tiles && job->tile_index0 < 0)) {
      set_error("dkv_linear_rope_pack: the job appends %d tokens, the projection has %d (or a negative tile index)",
                job->n, n);
      return DKV_EINVAL;
    }
  }
  LinearArgs a = {};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = x_row_stride;
  a.w = static_cast<const uint16_t*>(w);
  a.ldw = w_row_stride;
  a.norm = static_cast<const uint16_t*>(norm_weight);
  a.eps = eps;
  a.rows = n;
  a.k = k;
  a.kp = k / 64;
  a.n_tiles = q_heads + 2 * heads;
  a.row_groups = (n + 15) / 16;
  a.up = a.n_tiles * D;
  a.layout = layout;
  RopeArgs r;
  r.cosv = static_cast<const uint16_t*>(cos);
  r.sinv = static_cast<const uint16_t*>(sin);
  r.cs_stride = cs_row_stride;
  r.q_out = static_cast<uint16_t*>(q_out);
  r.k_out = static_cast<uint16_t*>(k_out);
  r.v_out = static_cast<uint16_t*>(v_out);
  r.hjob = job_on_device ? dkv_pack_job{} : *job;
  r.djob = job_on_device ? job : nullptr;
  r.arena = static_cast<uint8_t*>(arena);
  r.tiles = tiles;
  r.q_heads = q_heads;
  r.heads = heads;
  r.layers = layers;
  hipStream_t st = (hipStream_t)stream;
  if (xt) a.row_groups = (n + TILE_M - 1) / TILE_M;
  const dim3 grid((unsigned)((a.n_tiles + 7) / 8) * 8u * (unsigned)a.row_groups);
  if (xt) {
    if (wt) hipLaunchKernelGGL((linear_tile_rope_kernel<LAYOUT_X_TILED | LAYOUT_W_TILED>), grid, dim3(256), 0, st, a, r);
    else hipLaunchKernelGGL((linear_tile_rope_kernel<LAYOUT_X_TILED>), grid, dim3(256), 0, st, a, r);
  } else if (a.kp <= 8) {
    if (wt) hipLaunchKernelGGL((linear_rope_kernel<1, LAYOUT_W_TILED>), grid, dim3(512), 0, st, a, r);
    else hipLaunchKernelGGL((linear_rope_kernel<1, 0>), grid, dim3(512), 0, st, a, r);
  } else {
    if (wt) hipLaunchKernelGGL((linear_rope_kernel<2, LAYOUT_W_TILED>), grid, dim3(512), 0, st, a, r);
    else hipLaunchKernelGGL((linear_rope_kernel<2, 0>), grid, dim3(512), 0, st, a, r);
  }
  return (int)hipGetLastError();
}

int dkv_linear_prenorm(int32_t rows, int32_t n, int32_t k, int32_t epilogue) {
  if (!dkv_linear_supported(rows, n, k, 1, epilogue) || !dkv_linear_supported(rows, n, k, 0, epilogue)) return 0;
  return pick(rows, epilogue == EPI_SILU_MUL ? n / 2 : n, k / 64, false, epilogue).tile;
}

int dkv_rms_norm_tiled(const void* x, int64_t x_row_stride, const void* weight, void* out, int32_t rows, int32_t k,
                       float eps, int32_t layout, void* stream) {
  clear_error();
  const bool xt = layout & LAYOUT_X_TILED;
  if (!x || !weight || !out || rows < 0 || k <= 0 || (k & 63) || k > 64 * 8 * MAX_NORM_CH || !al16(x) || !al16(weight) ||
      !al16(out) || (layout & ~LAYOUT_X_TILED) || (!xt && ((x_row_stride & 7) || x_row_stride < k))) {
    set_error("dkv_rms_norm_tiled: bad arguments (rows %d, k %d, layout %d; k a multiple of 64, at most %d, 16-byte "
              "aligned bf16 rows)", rows, k, layout, 64 * 8 * MAX_NORM_CH);
    return DKV_EINVAL;
  }
  if (rows == 0) return 0;
  const dim3 grid((rows + 15) / 16);
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* wp = static_cast<const uint16_t*>(weight);
  auto* op = static_cast<uint16_t*>(out);
  hipStream_t st = (hipStream_t)stream;
  const int kp = k / 64;
  if (kp <= 8) {
    if (xt) hipLaunchKernelGGL((rms_tiled_kernel<1, true>), grid, dim3(512), 0, st, xp, x_row_stride, wp, op, rows, k, kp, eps);
    else hipLaunchKernelGGL((rms_tiled_kernel<1, false>), grid, dim3(512), 0, st, xp, x_row_stride, wp, op, rows, k, kp, eps);
  } else {
    if (xt) hipLaunchKernelGGL((rms_tiled_kernel<2, true>), grid, dim3(512), 0, st, xp, x_row_stride, wp, op, rows, k, kp, eps);
    else hipLaunchKernelGGL((rms_tiled_kernel<2, false>), grid, dim3(512), 0, st, xp, x_row_stride, wp, op, rows, k, kp, eps);
  }
  return (int)hipGetLastError();
}

int dkv_linear(const void* x, int64_t x_row_stride, const void* w, int64_t w_row_stride, int32_t rows, int32_t n,
               int32_t k, const void* norm_weight, float eps, int32_t epilogue, const void* residual,
               int64_t residual_row_stride, void* out, int64_t out_row_stride, void* stream) {
  return dkv_linear_tiled(x, x_row_stride, w, w_row_stride, rows, n, k, norm_weight, eps, epilogue, residual,
                          residual_row_stride, out, out_row_stride, 0, stream);
}

}  // extern "C"
