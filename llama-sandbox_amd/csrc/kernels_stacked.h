// kernels_stacked.h -- grouped gate/up and down on items of up to 32 or 64
// rows, the two Q8_0 digit planes stacked along K of one MFMA, in fp6.
//
// v_mfma_scale_f32_32x32x64_f8f6f4 reduces 64 K per output value.  Here A is
// the weight tile (A row r = weight row r, fp4 with its E8M0 exponent) and B
// the item's tokens (B column n = token n), and the 64 K are one MXFP4 block
// twice: K 0-31 carry the block's hi digits (B scale 2^4), K 32-63 its lo
// digits (2^0), and both A lane halves hold the same weight block.  D[r][n]
// is then 2^(e_w - 127) times the exact integer block dot of row r and token
// n (16*hi + lo = q), scaled by the token's d and added in f32, block by
// block.
//
// The digits (hi in [-8, 7], lo in [0, 15]) are e2m3 codes (fp6: digit / 8,
// the code of a magnitude is the magnitude itself, the sign bit 32), not e4m3:
// with fp6 an MFMA keeps the matrix core busy for 32 cycles instead of 64
// (counters), and a token's block takes 48 bytes instead of 64.
//
// Staged activations ("quad records"): per row and quad of 4 blocks 208 bytes
//   [0, 96)    hi digits of blocks 0..3, 24 bytes each (6 bits per K offset)
//   [96, 192)  lo digits, likewise
//   [192, 208) d of the 4 blocks, f32
// x row by row (a chunk of 4 quads of a row is one run of 832 bytes), h quad by
// quad (an item's rows of a quad are one run).  The direct global-to-LDS loads
// of a chunk (1 KiB each) read such runs in order, about 10 cache lines per
// load; with one 16-byte piece per (token, block) and load, 64 lines, the load
// path bounds the kernel (a build that staged 96 bytes per block that way:
// gate/up of 2048 tokens on the V3 layer 2003 us, 1353 us with the same bytes
// contiguous).
//
// Items of up to 16 rows, of which small batches and the remainders of long
// chunks are made, run the MFMA with its operands swapped (skf_loop): tokens on
// D's elements, and only the elements of tokens that the item holds are scaled.
// Items of 33-64 rows share each weight pair between two token tiles (sk_loop2).
//
// What bounds them (V3 layer, profiles/prefill_stacked_counters.md): at 512
// tokens, uniform, the weight stream (vector issue 43% of the cycles, matrix
// cores 17%; the bare stream of gate/up's bytes takes 560 us); at 2048 tokens
// the vector issue, 19 instructions per MFMA in 66% of the cycles at the 1.7 GHz
// that the chip holds.  Timed on one box against the kernels before them (e4m3
// digits staged in pieces): 512 tokens uniform 1171 -> 1101 us, Zipf 829 -> 686,
// 2048 tokens 2831 -> 2140, the V4-Pro layer 933 -> 764; 300 tokens on a 5120 x
// 1536 layer, octets before, 553 -> 421 (sums in f64, sk_scale).
//
// Operand lanes.  A lane r + 32*g holds weight row r, K [32g, 32g + 32): the
// record layout gives lane (r, g) block 2j + g of a quad in one load, and
// v_permlane32_swap turns that pair into [block 2j | block 2j] and [block
// 2j+1 | block 2j+1].  B lane n + 32*g holds token n's hi (g = 0) or lo (g = 1)
// digits, 24 bytes.  D lane n + 32*g holds token n, rows 8i + 4g + j at element
// 4i + j: a lane has one d, and the epilogues need no exchange (a lane holds
// gate and up of the same values).
#pragma once

#include <type_traits>

#include "grouped_plan.h"
#include "kernels_grouped.h"

typedef double f64x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

#define MOE_SQ_DW 52    // dwords of a quad record
#define MOE_SQ_U4 13    // its 16-byte units (odd: the operand reads of 8 tokens hit 8 bank groups)
#define MOE_SK_ROWS MOE_PLAN_ROWS  // tokens of an MFMA; items of up to MOE_PLAN_ROWS2 rows take two (sk_loop2)
#define MOE_SK_CH 4       // quads per staged chunk of 32 rows (of 64 rows: 2)
#define MOE_SK_BUF_DW (MOE_SK_CH * MOE_SK_ROWS * MOE_SQ_DW)  // 26 KiB
#define MOE_SK_DMA (MOE_SK_BUF_DW / 256)                     // 1 KiB loads per chunk (26)
#define MOE_SK_NBUF 2
#define MOE_SK_LDS_BYTES (MOE_SK_NBUF * MOE_SK_BUF_DW * 4)
#define MOE_SK_WAVES 4
#define MOE_SK_WDMA ((MOE_SK_DMA + MOE_SK_WAVES - 1) / MOE_SK_WAVES)  // loads per wave and chunk (7; waves 2, 3: 6)
#define MOE_SK_OOB 0xffffff00u  // a lane offset past any staged buffer: the load returns 0

// ---------------------------------------------------------------------------
// Q8_0 into quad records

// Eight digits (K order) of one plane as 48 bits, from digits packed one per byte.
__device__ __forceinline__ uint32_t pack6x4(uint32_t b) {  // 4 bytes of 6 bits -> 24 bits
  const uint32_t x = (b & 0x003f003fu) | ((b >> 2) & 0x0fc00fc0u);
  return (x & 0xfffu) | ((x >> 4) & 0xfff000u);
}

// The fp6 codes of q's digits: lo in byte 0, hi in byte 1.
__device__ __forceinline__ uint32_t digit_codes(int q) {
  const int hi = q >> 4;
  return (uint32_t)(q & 15) | (uint32_t)(hi < 0 ? 32 - hi : hi) << 8;
}

// Codes of 8 values in K order -> 48 bits of lo digits and of hi digits.
struct half48 {
  uint32_t lo, hi;  // low 32 and high 16 bits
};

__device__ __forceinline__ void pack_digits8(const uint32_t (&c)[8], half48 &l, half48 &h) {
  uint32_t yl[2], yh[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t *a = c + 4 * i;
    // v_perm selects bytes 0-3 from the second operand, 4-7 from the first
    const uint32_t t0 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u);  // lo0 lo1 hi0 hi1
    const uint32_t t1 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u);
    yl[i] = pack6x4(__builtin_amdgcn_perm(t1, t0, 0x05040100u));
    yh[i] = pack6x4(__builtin_amdgcn_perm(t1, t0, 0x07060302u));
  }
  l.lo = yl[0] | (yl[1] << 24);
  l.hi = yl[1] >> 8;
  h.lo = yh[0] | (yh[1] << 24);
  h.hi = yh[1] >> 8;
}

// 48 + 48 bits: half a block's digits of one plane.
__device__ __forceinline__ void join48(const half48 &a, const half48 &b, uint32_t *dst) {
  dst[0] = a.lo;
  dst[1] = a.hi | (b.lo << 16);
  dst[2] = (b.lo >> 16) | (b.hi << 16);
}

// Q8_0 of nb blocks (whole rows of a multiple of 4 blocks, from a quad's first
// block on) into quad records; two lanes per block, lane half h the K offsets
// 16h .. 16h + 15 (offset 2i: element 8h + i, 2i + 1: element 16 + 8h + i).
__device__ __forceinline__ void stage_quant_quads(const float *__restrict__ x, int nb, uint32_t *xs, int tid, int nthr) {
  const int h = tid & 1;
  for (int b = tid >> 1; b < nb; b += nthr >> 1) {
    const float4 *xb = reinterpret_cast<const float4 *>(x + (size_t)b * MOE_QK + 8 * h);
    const float4 a0 = xb[0], a1 = xb[1], c0 = xb[4], c1 = xb[5];
    const float v[16] = {a0.x, c0.x, a0.y, c0.y, a0.z, c0.z, a0.w, c0.w,
                         a1.x, c1.x, a1.y, c1.y, a1.z, c1.z, a1.w, c1.w};
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, dpp_f<0xB1>(amax));  // partner lane (lane ^ 1) holds the other half
    half48 l[2], u[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      uint32_t code[8];
#pragma unroll
      for (int i = 0; i < 8; i++) code[i] = digit_codes((int)q8_code(v[8 * c + i], amax));
      pack_digits8(code, l[c], u[c]);
    }
    uint32_t *rec = xs + (size_t)(b >> 2) * MOE_SQ_DW;
    join48(u[0], u[1], rec + (b & 3) * 6 + 3 * h);
    join48(l[0], l[1], rec + 24 + (b & 3) * 6 + 3 * h);
    if (!h) rec[48 + (b & 3)] = __builtin_bit_cast(uint32_t, (float)q8_scale_f16(amax));
  }
}

// The 32 h values of a token's unit, 16 in each of the lanes n and n + 32
// (h[4i + j] = row 8i + 4g + j), as Q8_0 into block b of quad record rec.
__device__ __forceinline__ void h_quad_store(const float (&h)[16], uint32_t *rec, int b, int lane) {
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) amax = fmaxf(amax, fabsf(h[i]));
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  // rows 8c + 4g + (0..3) and the same + 16: K offsets 16c + 8g + (0..7)
  half48 l[2], u[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    uint32_t code[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      code[2 * j] = digit_codes((int)q8_code(h[4 * c + j], amax));
      code[2 * j + 1] = digit_codes((int)q8_code(h[8 + 4 * c + j], amax));
    }
    pack_digits8(code, l[c], u[c]);
  }
  // lane n collects the hi digits of both lanes, lane n + 32 the lo digits,
  // of K offsets 0-15 (c = 0) and 16-31 (c = 1)
  uint32_t o[6];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const auto a = __builtin_amdgcn_permlane32_swap(u[c].lo, l[c].lo, false, false);
    const auto e = __builtin_amdgcn_permlane32_swap(u[c].hi, l[c].hi, false, false);
    join48(half48{a[0], e[0]}, half48{a[1], e[1]}, o + 3 * c);
  }
  const int g = lane >> 5;
#pragma unroll
  for (int i = 0; i < 6; i++) rec[24 * g + 6 * b + i] = o[i];
  if (!g) rec[48 + b] = __builtin_bit_cast(uint32_t, (float)q8_scale_f16(amax));
}

// ---------------------------------------------------------------------------
// Staging of a chunk: 1 KiB load i = wave, wave + 4, ... fills the units [64i,
// 64i + 64) of [quad][token][unit].
struct sdma {
  const uint32_t *src;
  uint32_t bytes;
  uint32_t chunk;            // from one chunk to the next
  uint32_t vo[MOE_SK_WDMA];  // this lane's offsets at chunk 0
  int wave, chunks;
};

// row: the staged row of token lane % 32 (< 0: absent), of `rows` rows of NQ
// quads (quad_major: all rows of a quad, then the next quad).  NT == 64: row2 is
// that of token 32 + lane % 32.
template <int NT>
__device__ __forceinline__ sdma make_sdma(const uint32_t *src, int rows, int NQ, bool quad_major, int row, int row2,
                                          int lane, int wave) {
  constexpr int CH = MOE_SK_CH * MOE_SK_ROWS / NT;  // quads per chunk
  sdma s;
  const uint32_t rs = quad_major ? 1u : (uint32_t)NQ, qs = quad_major ? (uint32_t)rows : 1u;
  s.src = src;
  s.bytes = (uint32_t)rows * (uint32_t)NQ * (MOE_SQ_DW * 4);
  s.chunk = CH * qs * (MOE_SQ_DW * 4);
  s.wave = wave;
  s.chunks = (NQ + CH - 1) / CH;
#pragma unroll
  for (int i = 0; i < MOE_SK_WDMA; i++) {
    const int u = 64 * (wave + MOE_SK_WAVES * i) + lane;
    const int q = u / (NT * MOE_SQ_U4), v = u % (NT * MOE_SQ_U4), t = v / MOE_SQ_U4;
    int r = __shfl(row, t & 31);
    if (NT == 64) {
      const int r2 = __shfl(row2, t & 31);
      r = t < 32 ? r : r2;
    }
    s.vo[i] = r >= 0 ? ((uint32_t)r * rs + (uint32_t)q * qs) * (MOE_SQ_DW * 4) + (v % MOE_SQ_U4) * 16 : MOE_SK_OOB;
  }
  return s;
}

// Chunk C into buf.  The quads past the end (NQ % 4 != 0) read on into the next
// row, or past the buffer: the K loop does not use them.  A chunk past the
// end issues its loads out of range, since the waits count them; its scalar
// offset stays 0, as the bounds check compares the lane offset with the
// buffer's size less the scalar offset.
__device__ __forceinline__ void sdma_issue(const sdma &s, uint32_t *buf, int C) {
  typedef __attribute__((address_space(3))) void *lds_t;
  const bool in = C < s.chunks;
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)s.src, 0, (int)s.bytes, MOE_RSRC_FLAGS);
  const uint32_t so = in ? (uint32_t)C * s.chunk : 0u;
#pragma unroll
  for (int i = 0; i < MOE_SK_WDMA; i++) {
    if (MOE_SK_WAVES * i + s.wave >= MOE_SK_DMA) break;  // uniform over the wave
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_t)(buf + (s.wave + MOE_SK_WAVES * i) * 256), 16,
                                             in ? s.vo[i] : MOE_SK_OOB, so, 0, 0);
  }
}

// ---------------------------------------------------------------------------
// A block pair (K step) of this lane's B operands: the digits (hi or lo by lane half) of its two blocks.
struct skb {
  i32x8_t x[2];  // the two blocks' MFMA operands (6 dwords of 8)
};

__device__ __forceinline__ const u32x4_t *sk_units(const uint32_t *buf, int lane) {
  return reinterpret_cast<const u32x4_t *>(buf) + (lane & 31) * MOE_SQ_U4;
}

// Pair j of quad q of a chunk (tile: its second 32 tokens of 64).
template <int NT = 32>
__device__ __forceinline__ skb load_skb(const uint32_t *buf, int lane, int q, int j, int tile = 0) {
  const u32x4_t *p = sk_units(buf, lane) + 6 * (lane >> 5) + (q * NT + 32 * tile) * MOE_SQ_U4 + 3 * j;
  const u32x2_t *t = reinterpret_cast<const u32x2_t *>(p + 1);
  const u32x4_t w0 = p[0];
  const u32x2_t t0 = t[0];
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");  // t0 and t1 as one load would cost the operands 4 moves a pair
  const u32x2_t t1 = t[1];
  const u32x4_t w1 = p[2];
  skb b;
  b.x[0] = i32x8_t{(int)w0.x, (int)w0.y, (int)w0.z, (int)w0.w, (int)t0.x, (int)t0.y, 0, 0};
  b.x[1] = i32x8_t{(int)t1.x, (int)t1.y, (int)w1.x, (int)w1.y, (int)w1.z, (int)w1.w, 0, 0};
  return b;
}

// d of the quad's 4 blocks for this lane's token.
template <int NT = 32>
__device__ __forceinline__ f32x4_t load_skd(const uint32_t *buf, int lane, int q, int tile = 0) {
  return __builtin_bit_cast(f32x4_t, sk_units(buf, lane)[(q * NT + 32 * tile) * MOE_SQ_U4 + 12]);
}

// [x | x] and [y | y] from a register holding x in lanes 0-31, y in 32-63.
__device__ __forceinline__ void dup_halves(const u32x4_t &w, u32x4_t &a0, u32x4_t &a1) {
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const auto p = __builtin_amdgcn_permlane32_swap(w[c], w[c], false, false);
    a0[c] = p[0];
    a1[c] = p[1];
  }
}

__device__ __forceinline__ void dup_halves1(uint32_t w, uint32_t &a0, uint32_t &a1) {
  const auto p = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  a0 = p[0];
  a1 = p[1];
}

// Two weight streams of 32 rows (gate and up, or two tiles of down).
struct skw {
  const uint8_t *w[2];
  uint32_t bytes, vo, so;  // of a 32-row tile; lane offsets of the data and of the exponents
  int pairs, NG;
};

__device__ __forceinline__ skw make_skw(const uint8_t *w0, const uint8_t *w1, int NQ, int lane) {
  skw p;
  p.w[0] = w0;
  p.w[1] = w1;
  p.NG = moe_nq4(NQ);
  p.pairs = 2 * NQ;
  p.bytes = 2u * p.NG * MOE_REC_BYTES;
  const aoff32 ao = make_aoff32(lane, p.NG);
  p.vo = ao.v;
  p.so = ao.s;
  return p;
}

// Block pair S (past the end: no records and scalar offset 0, nothing read).
template <int CPOL>
__device__ __forceinline__ void load_skw(u32x4_t (&w)[2], const skw &p, int S) {
  const bool in = S < p.pairs;
  const int q = S >> 1, so = in ? (q >> 2) * (int)MOE_REC_BYTES + (q & 3) * 1024 : 0;
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void *)p.w[s], 0, in ? (int)p.bytes : 0, MOE_RSRC_FLAGS);
    w[s] = __builtin_amdgcn_raw_buffer_load_b128(r, p.vo + (S & 1) * 512, so, CPOL);
  }
}

// Exponent dwords of group G: lane (r, g) holds block position 2j + g, byte q = quad q.
__device__ __forceinline__ void load_sksc(uint32_t (&sc)[2][2], const skw &p, int G) {
  const bool in = G < p.NG;
#pragma unroll
  for (int s = 0; s < 2; s++) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc((void *)p.w[s], 0, in ? (int)p.bytes : 0, MOE_RSRC_FLAGS);
#pragma unroll
    for (int j = 0; j < 2; j++)
      sc[s][j] = __builtin_amdgcn_raw_buffer_load_b32(r, p.so + j * 128, in ? G * (int)MOE_REC_BYTES : 0, 0);
  }
}

#define MOE_SK_RP 4  // weight ring, in block pairs: 3 ahead, 6 KiB in flight per wave (7 ahead measured the same)

struct skring {
  u32x4_t w[MOE_SK_RP][2];
  uint32_t e[2][4];    // this group's exponents by block position, the same in both lane halves
  uint32_t scn[2][2];  // the next group's, as loaded
  skb b[2];            // B of this pair and the next
  f32x4_t d[2];        // d of this quad and the next
  f32x16_t r[2];       // the block sums last multiplied
  float du;            // d of stream 1's pending block
};

// acc += d * r, in f64 if WIDE.
template <bool WIDE>
__device__ __forceinline__ void sk_scale(f32x16_t &acc, f64x16_t &wide, float d, const f32x16_t &r) {
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if constexpr (WIDE) wide[i] = __builtin_fma((double)d, (double)r[i], wide[i]);
    else acc[i] = __builtin_fmaf(d, r[i], acc[i]);
  }
  if constexpr (WIDE) asm volatile("" : "+v"(wide));
  else asm volatile("" : "+v"(acc));
}

// One block against both streams.  Stream 0's MFMA runs while stream 1's last
// result is scaled, and the other way round; stream 1's result stays pending.
// WIDE: the sums in f64 (an f64 FMA issues like an f32 one; each result is
// converted first).
template <int SEL, int J, int JD, bool WIDE>
__device__ __forceinline__ void sk_block(skring &g, const u32x4_t &w0, const u32x4_t &w1, const skb &b, float d, int sb,
                                         f32x16_t (&acc)[2], f64x16_t (&wide)[2]) {
  const i32x8_t x = b.x[J];
  const i32x8_t a0 = {(int)w0.x, (int)w0.y, (int)w0.z, (int)w0.w, 0, 0, 0, 0};
  const i32x8_t a1 = {(int)w1.x, (int)w1.y, (int)w1.z, (int)w1.w, 0, 0, 0, 0};
  const f32x16_t z = {};
  g.r[0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a0, x, z, 4, 2, SEL, (int)g.e[0][JD], 0, sb);
  __builtin_amdgcn_sched_barrier(0);
  sk_scale<WIDE>(acc[1], wide[1], g.du, g.r[1]);
  __builtin_amdgcn_sched_barrier(0);
  g.r[1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a1, x, z, 4, 2, SEL, (int)g.e[1][JD], 0, sb);
  __builtin_amdgcn_sched_barrier(0);
  sk_scale<WIDE>(acc[0], wide[0], d, g.r[0]);
  g.du = d;
  __builtin_amdgcn_sched_barrier(0);
}

// Pair SG of group G (its chunk in buffer cur).  The barrier of a chunk sits
// before its last pair: every wave has then read its operands of that pair, so
// the buffer is free for the chunk MOE_SK_NBUF ahead, and the next chunk,
// loaded MOE_SK_NBUF - 1 chunks ago, is visible to all.
template <int CPOL, bool WIDE, int SG>
__device__ __forceinline__ void sk_pair(skring &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane, int sb,
                                        int G, f32x16_t (&acc)[2], f64x16_t (&wide)[2]) {
  static_assert(MOE_SK_CH == 4 && 8 % MOE_SK_RP == 0 && MOE_SK_NBUF == 2, "a chunk is one group; two buffers");
  load_skw<CPOL>(g.w[(SG + MOE_SK_RP - 1) % MOE_SK_RP], w, G * 8 + SG + MOE_SK_RP - 1);
  if constexpr (SG == 0) load_sksc(g.scn, w, G + 1);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (SG == 7) {
    // younger than the next chunk's staging: a chunk's weights (8 pairs of two loads) and exponents
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(8 * 2 + 4));
    lds_barrier();
    sdma_issue(st, lds + cur * MOE_SK_BUF_DW, G + MOE_SK_NBUF);
    cur ^= 1;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  const uint32_t *buf = lds + cur * MOE_SK_BUF_DW;
  g.b[(SG + 1) & 1] = load_skb(buf, lane, ((SG + 1) & 7) >> 1, (SG + 1) & 1);
  if constexpr (SG & 1) g.d[((SG >> 1) + 1) & 1] = load_skd(buf, lane, ((SG + 1) & 7) >> 1);
  u32x4_t a[2][2];
#pragma unroll
  for (int s = 0; s < 2; s++) dup_halves(g.w[SG % MOE_SK_RP][s], a[s][0], a[s][1]);
  __builtin_amdgcn_sched_barrier(0);
  const f32x4_t d = g.d[(SG >> 1) & 1];
  constexpr int j = SG & 1;
  sk_block<(SG >> 1), 0, 2 * j, WIDE>(g, a[0][0], a[1][0], g.b[j], d[2 * j], sb, acc, wide);
  sk_block<(SG >> 1), 1, 2 * j + 1, WIDE>(g, a[0][1], a[1][1], g.b[j], d[2 * j + 1], sb, acc, wide);
}

template <int CPOL, bool WIDE, int SG>
__device__ __forceinline__ void sk_group(skring &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane, int sb,
                                         int G, int quads, f32x16_t (&acc)[2], f64x16_t (&wide)[2]) {
  if constexpr (SG < 8) {
    if (quads <= (SG >> 1)) return;  // the last group of a K that is no multiple of 512
    sk_pair<CPOL, WIDE, SG>(g, w, st, lds, cur, lane, sb, G, acc, wide);
    sk_group<CPOL, WIDE, SG + 1>(g, w, st, lds, cur, lane, sb, G, quads, acc, wide);
  }
}

// The K loop of one wave: its two weight streams over NQ quads against the
// staged tokens.  acc[s]: lane n + 32*g, element 4i + j = row 8i + 4g + j of
// stream s, token n, summed block by block; WIDE: in f64,
// rounded once.  CPOL: the weights' cache policy.
template <int CPOL, bool WIDE, bool QUAD_MAJOR, class ROW>
__device__ __forceinline__ void sk_loop(const skw &w, const uint32_t *src, int n_src, int NQ, ROW row, uint32_t *lds, int lane,
                                        int wave, f32x16_t (&acc)[2]) {
  skring g;
  uint32_t sc[2][2];
  f64x16_t wide[2];
  // the first weights go out before the rows are known (for gate/up a load and a division away)
  load_sksc(sc, w, 0);
#pragma unroll
  for (int i = 0; i + 1 < MOE_SK_RP; i++) load_skw<CPOL>(g.w[i], w, i);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  const sdma st = make_sdma<32>(src, n_src, NQ, QUAD_MAJOR, row(0), 0, lane, wave);
#pragma unroll
  for (int c = 0; c < MOE_SK_NBUF; c++) sdma_issue(st, lds + c * MOE_SK_BUF_DW, c);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(MOE_SK_WDMA - 1));  // chunk 0 has landed, the second may be on its way
  lds_barrier();
  int cur = 0;
  g.b[0] = load_skb(lds, lane, 0, 0);
  g.d[0] = load_skd(lds, lane, 0);
#pragma unroll
  for (int s = 0; s < 2; s++) {
    acc[s] = f32x16_t{};
    wide[s] = f64x16_t{};
  }
  g.r[1] = f32x16_t{};  // the first block scales a zero result: acc stays +0
  g.du = 0.0f;
  const int sb = (lane >> 5) ? 130 : 134;  // lo digits x 2^3 (fp6 codes are eighths), hi digits x 2^7
  auto group = [&](int G, int quads) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      dup_halves1(sc[s][0], g.e[s][0], g.e[s][1]);
      dup_halves1(sc[s][1], g.e[s][2], g.e[s][3]);
    }
    sk_group<CPOL, WIDE, 0>(g, w, st, lds, cur, lane, sb, G, quads, acc, wide);
  };
  int G = 0;
  // whole groups in a loop of their own: with the last group's exits in it,
  // the waits at its head would cover the loads in flight
#pragma unroll 1
  for (; 4 * G + 4 <= NQ; G++) {
    group(G, 4);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int j = 0; j < 2; j++) sc[s][j] = g.scn[s][j];
  }
  if constexpr (WIDE)
    if (4 * G < NQ) group(G, NQ - 4 * G);
  sk_scale<WIDE>(acc[1], wide[1], g.du, g.r[1]);
  if constexpr (WIDE) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 16; i++) acc[s][i] = (float)wide[s][i];
  }
}

// ---------------------------------------------------------------------------
// The same for items of 33-64 rows: two token tiles share each weight pair, so
// the weights of a large expert are read (mostly from L2) and duplicated
// across the lane halves half as often.  A chunk is 2 quads of 64 rows.  V3
// layer: 512 tokens Zipf 682 -> 658 us, 2048 tokens 2298 -> 2115 us; V4-Pro
// layer 768 -> 746 us.
struct skring2 {
  u32x4_t w[MOE_SK_RP][2];
  uint32_t e[2][4];
  uint32_t scn[2][2];
  skb b[2];       // B of this pair, per token tile (loaded again as soon as its last MFMA is out)
  f32x4_t d[2];   // d of this quad, per token tile
  f32x16_t r[2];  // the last two MFMAs' results
  float du;       // d of the pending one (token tile 1, stream 1)
};

template <int SEL, int J, int JD>
__device__ __forceinline__ void sk_mma2(skring2 &g, f32x16_t &r, const u32x4_t &w, uint32_t e, const skb &b, int sb) {
  const i32x8_t x = b.x[J];
  const i32x8_t a = {(int)w.x, (int)w.y, (int)w.z, (int)w.w, 0, 0, 0, 0};
  const f32x16_t z = {};
  __builtin_amdgcn_sched_barrier(0);
  r = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, x, z, 4, 2, SEL, (int)e, 0, sb);
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void sk_fma2(f32x16_t &acc, float d, const f32x16_t &r) {
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = __builtin_fmaf(d, r[i], acc[i]);
  asm volatile("" : "+v"(acc));
  __builtin_amdgcn_sched_barrier(0);
}

// Pair SG of group G.  acc[tile][stream]; each MFMA runs while the result
// before it is scaled.  The barrier of a chunk sits at the end of its last pair
// (SG 3 and 7).
template <int CPOL, int SG>
__device__ __forceinline__ void sk_pair2(skring2 &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane, int sb,
                                         int G, f32x16_t (&acc)[2][2]) {
  load_skw<CPOL>(g.w[(SG + MOE_SK_RP - 1) % MOE_SK_RP], w, G * 8 + SG + MOE_SK_RP - 1);
  if constexpr (SG == 0) load_sksc(g.scn, w, G + 1);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  u32x4_t a[2][2];  // [stream][block]
#pragma unroll
  for (int s = 0; s < 2; s++) dup_halves(g.w[SG % MOE_SK_RP][s], a[s][0], a[s][1]);
  constexpr int SEL = SG >> 1, j = SG & 1;
  const float d00 = g.d[0][2 * j], d10 = g.d[1][2 * j], d01 = g.d[0][2 * j + 1], d11 = g.d[1][2 * j + 1];
  sk_mma2<SEL, 0, 0>(g, g.r[0], a[0][0], g.e[0][2 * j], g.b[0], sb);
  sk_fma2(acc[1][1], g.du, g.r[1]);
  sk_mma2<SEL, 0, 0>(g, g.r[1], a[1][0], g.e[1][2 * j], g.b[0], sb);
  sk_fma2(acc[0][0], d00, g.r[0]);
  sk_mma2<SEL, 0, 0>(g, g.r[0], a[0][0], g.e[0][2 * j], g.b[1], sb);
  sk_fma2(acc[0][1], d00, g.r[1]);
  sk_mma2<SEL, 0, 0>(g, g.r[1], a[1][0], g.e[1][2 * j], g.b[1], sb);
  sk_fma2(acc[1][0], d10, g.r[0]);
  sk_mma2<SEL, 1, 0>(g, g.r[0], a[0][1], g.e[0][2 * j + 1], g.b[0], sb);
  sk_fma2(acc[1][1], d10, g.r[1]);
  sk_mma2<SEL, 1, 0>(g, g.r[1], a[1][1], g.e[1][2 * j + 1], g.b[0], sb);
  sk_fma2(acc[0][0], d01, g.r[0]);
  sk_mma2<SEL, 1, 0>(g, g.r[0], a[0][1], g.e[0][2 * j + 1], g.b[1], sb);
  sk_fma2(acc[0][1], d01, g.r[1]);
  sk_mma2<SEL, 1, 0>(g, g.r[1], a[1][1], g.e[1][2 * j + 1], g.b[1], sb);
  if constexpr ((SG & 3) == 3) {
    // younger than the next chunk's staging: 4 pairs of two loads, and in a group's first half its exponents
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(4 * 2 + (SG == 3 ? 4 : 0)));
    lds_barrier();
    sdma_issue(st, lds + cur * MOE_SK_BUF_DW, 2 * G + (SG >> 2) + MOE_SK_NBUF);
    cur ^= 1;
    asm volatile("" ::: "memory");
  }
  const uint32_t *buf = lds + cur * MOE_SK_BUF_DW;
  constexpr int nq = ((SG + 1) & 3) >> 1, nj = (SG + 1) & 1;  // the next pair's quad of its chunk
#pragma unroll
  for (int t = 0; t < 2; t++) {
    g.b[t] = load_skb<64>(buf, lane, nq, nj, t);
    if constexpr (nj == 0) g.d[t] = load_skd<64>(buf, lane, nq, t);
  }
  __builtin_amdgcn_sched_barrier(0);
  sk_fma2(acc[1][0], d11, g.r[0]);
  g.du = d11;
}

template <int CPOL, int SG>
__device__ __forceinline__ void sk_group2(skring2 &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane,
                                          int sb, int G, f32x16_t (&acc)[2][2]) {
  if constexpr (SG < 8) {
    sk_pair2<CPOL, SG>(g, w, st, lds, cur, lane, sb, G, acc);
    sk_group2<CPOL, SG + 1>(g, w, st, lds, cur, lane, sb, G, acc);
  }
}

// acc[tile][stream], block by block in order; NQ % 4 == 0.
template <int CPOL, bool QUAD_MAJOR, class ROW>
__device__ __forceinline__ void sk_loop2(const skw &w, const uint32_t *src, int n_src, int NQ, ROW row, uint32_t *lds,
                                         int lane, int wave, f32x16_t (&acc)[2][2]) {
  skring2 g;
  uint32_t sc[2][2];
  load_sksc(sc, w, 0);
#pragma unroll
  for (int i = 0; i + 1 < MOE_SK_RP; i++) load_skw<CPOL>(g.w[i], w, i);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  const sdma st = make_sdma<64>(src, n_src, NQ, QUAD_MAJOR, row(0), row(32), lane, wave);
#pragma unroll
  for (int c = 0; c < MOE_SK_NBUF; c++) sdma_issue(st, lds + c * MOE_SK_BUF_DW, c);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(MOE_SK_WDMA - 1));  // chunk 0 has landed, the second may be on its way
  lds_barrier();
  int cur = 0;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    g.b[t] = load_skb<64>(lds, lane, 0, 0, t);
    g.d[t] = load_skd<64>(lds, lane, 0, t);
    acc[t][0] = acc[t][1] = f32x16_t{};
  }
  g.r[1] = f32x16_t{};  // the first block scales a zero result: acc stays +0
  g.du = 0.0f;
  const int sb = (lane >> 5) ? 130 : 134;
#pragma unroll 1
  for (int G = 0; 4 * G < NQ; G++) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      dup_halves1(sc[s][0], g.e[s][0], g.e[s][1]);
      dup_halves1(sc[s][1], g.e[s][2], g.e[s][3]);
    }
    sk_group2<CPOL, 0>(g, w, st, lds, cur, lane, sb, G, acc);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int j = 0; j < 2; j++) sc[s][j] = g.scn[s][j];
  }
  sk_fma2(acc[1][1], g.du, g.r[1]);
}

// ---------------------------------------------------------------------------
// The same for items of at most 8 * NG rows, with the MFMA's operands swapped
// (their lane layouts are alike): tokens are the A rows and weight rows the B
// columns, so D lane n + 32*g holds weight row n, tokens 8i + 4g + j at element
// 4i + j, and only the 4 * NG elements of tokens that the item can hold are
// scaled, each by its own token's d (broadcast reads from LDS, a pair ahead):
// 4 or 8 scaling FMAs per MFMA instead of 16, in f64 10 or 20 instructions
// instead of 32.  The block sums and their order are those of sk_loop: the same
// bits.  us per layer, cold weights, 2, 4, 8 rows per expert: 5120 x 1536 (f64),
// 128 experts, 292 -> 251, 315 -> 283, 348 -> 313; 7168 x 2048, 32 experts, 137
// -> 132, 168 -> 160, 172 -> 163.  NG = 3 does not fit the registers of two
// waves per SIMD (spills; 2-14% slower than scaling all 16 elements).
template <int NG>
struct skringf {
  u32x4_t w[MOE_SK_RP][2];
  uint32_t e[2][4];
  uint32_t scn[2][2];
  skb b[2];
  f32x2_t d[2][4 * NG];  // d of this pair's two blocks and of the next pair's
  f32x16_t r[2];
  float du[4 * NG];      // d of stream 1's pending block
};

template <int NG>
__device__ __forceinline__ void load_skfd(f32x2_t (&d)[4 * NG], const uint32_t *buf, int lane, int q, int j) {
  const uint32_t *p = buf + (4 * (lane >> 5) + q * MOE_SK_ROWS) * MOE_SQ_DW + 48 + 2 * j;
#pragma unroll
  for (int i = 0; i < 4 * NG; i++)
    d[i] = *reinterpret_cast<const f32x2_t *>(p + (8 * (i >> 2) + (i & 3)) * MOE_SQ_DW);
}

template <bool WIDE, int NG>
__device__ __forceinline__ void skf_scale(f32x4_t (&acc)[NG], f64x4_t (&wide)[NG], const float (&d)[4 * NG],
                                          const f32x16_t &r) {
#pragma unroll
  for (int i = 0; i < 4 * NG; i++) {
    if constexpr (WIDE) wide[i >> 2][i & 3] = __builtin_fma((double)d[i], (double)r[i], wide[i >> 2][i & 3]);
    else acc[i >> 2][i & 3] = __builtin_fmaf(d[i], r[i], acc[i >> 2][i & 3]);
  }
#pragma unroll
  for (int i = 0; i < NG; i++) {
    if constexpr (WIDE) asm volatile("" : "+v"(wide[i]));
    else asm volatile("" : "+v"(acc[i]));
  }
}

template <int SEL, int J, int JD, bool WIDE, int NG>
__device__ __forceinline__ void skf_block(skringf<NG> &g, const u32x4_t &w0, const u32x4_t &w1, const skb &b,
                                          const f32x2_t (&dp)[4 * NG], int sb, f32x4_t (&acc)[2][NG],
                                          f64x4_t (&wide)[2][NG]) {
  const i32x8_t x = b.x[J];
  const i32x8_t a0 = {(int)w0.x, (int)w0.y, (int)w0.z, (int)w0.w, 0, 0, 0, 0};
  const i32x8_t a1 = {(int)w1.x, (int)w1.y, (int)w1.z, (int)w1.w, 0, 0, 0, 0};
  const f32x16_t z = {};
  float d[4 * NG];
#pragma unroll
  for (int i = 0; i < 4 * NG; i++) d[i] = dp[i][J];
  g.r[0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, a0, z, 2, 4, 0, sb, SEL, (int)g.e[0][JD]);
  __builtin_amdgcn_sched_barrier(0);
  skf_scale<WIDE, NG>(acc[1], wide[1], g.du, g.r[1]);
  __builtin_amdgcn_sched_barrier(0);
  g.r[1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, a1, z, 2, 4, 0, sb, SEL, (int)g.e[1][JD]);
  __builtin_amdgcn_sched_barrier(0);
  skf_scale<WIDE, NG>(acc[0], wide[0], d, g.r[0]);
#pragma unroll
  for (int i = 0; i < 4 * NG; i++) g.du[i] = d[i];
  __builtin_amdgcn_sched_barrier(0);
}

// Pair SG of group G: waits and barrier as in sk_pair.
template <int CPOL, bool WIDE, int NG, int SG>
__device__ __forceinline__ void skf_pair(skringf<NG> &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane,
                                         int sb, int G, f32x4_t (&acc)[2][NG], f64x4_t (&wide)[2][NG]) {
  load_skw<CPOL>(g.w[(SG + MOE_SK_RP - 1) % MOE_SK_RP], w, G * 8 + SG + MOE_SK_RP - 1);
  if constexpr (SG == 0) load_sksc(g.scn, w, G + 1);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (SG == 7) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(8 * 2 + 4));
    lds_barrier();
    sdma_issue(st, lds + cur * MOE_SK_BUF_DW, G + MOE_SK_NBUF);
    cur ^= 1;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  const uint32_t *buf = lds + cur * MOE_SK_BUF_DW;
  constexpr int nq = ((SG + 1) & 7) >> 1, nj = (SG + 1) & 1;  // the next pair's quad of its chunk
  g.b[nj] = load_skb(buf, lane, nq, nj);
  load_skfd<NG>(g.d[nj], buf, lane, nq, nj);
  u32x4_t a[2][2];
#pragma unroll
  for (int s = 0; s < 2; s++) dup_halves(g.w[SG % MOE_SK_RP][s], a[s][0], a[s][1]);
  __builtin_amdgcn_sched_barrier(0);
  constexpr int j = SG & 1;
  skf_block<(SG >> 1), 0, 2 * j, WIDE, NG>(g, a[0][0], a[1][0], g.b[j], g.d[j], sb, acc, wide);
  skf_block<(SG >> 1), 1, 2 * j + 1, WIDE, NG>(g, a[0][1], a[1][1], g.b[j], g.d[j], sb, acc, wide);
}

template <int CPOL, bool WIDE, int NG, int SG>
__device__ __forceinline__ void skf_group(skringf<NG> &g, const skw &w, const sdma &st, uint32_t *lds, int &cur, int lane,
                                          int sb, int G, int quads, f32x4_t (&acc)[2][NG], f64x4_t (&wide)[2][NG]) {
  if constexpr (SG < 8) {
    if (quads <= (SG >> 1)) return;
    skf_pair<CPOL, WIDE, NG, SG>(g, w, st, lds, cur, lane, sb, G, acc, wide);
    skf_group<CPOL, WIDE, NG, SG + 1>(g, w, st, lds, cur, lane, sb, G, quads, acc, wide);
  }
}

// acc[s][i]: lane n + 32*g, element j = row n of stream s, token 8i + 4g + j.
template <int CPOL, bool WIDE, int NG, bool QUAD_MAJOR, class ROW>
__device__ __forceinline__ void skf_loop(const skw &w, const uint32_t *src, int n_src, int NQ, ROW row, uint32_t *lds,
                                         int lane, int wave, f32x4_t (&acc)[2][NG]) {
  skringf<NG> g;
  uint32_t sc[2][2];
  f64x4_t wide[2][NG];
  load_sksc(sc, w, 0);
#pragma unroll
  for (int i = 0; i + 1 < MOE_SK_RP; i++) load_skw<CPOL>(g.w[i], w, i);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  const sdma st = make_sdma<32>(src, n_src, NQ, QUAD_MAJOR, row(0), 0, lane, wave);
#pragma unroll
  for (int c = 0; c < MOE_SK_NBUF; c++) sdma_issue(st, lds + c * MOE_SK_BUF_DW, c);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(MOE_SK_WDMA - 1));  // chunk 0 has landed, the second may be on its way
  lds_barrier();
  int cur = 0;
  g.b[0] = load_skb(lds, lane, 0, 0);
  load_skfd<NG>(g.d[0], lds, lane, 0, 0);
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int i = 0; i < NG; i++) {
      acc[s][i] = f32x4_t{};
      wide[s][i] = f64x4_t{};
    }
  g.r[1] = f32x16_t{};  // the first block scales a zero result: acc stays +0
#pragma unroll
  for (int i = 0; i < 4 * NG; i++) g.du[i] = 0.0f;
  const int sb = (lane >> 5) ? 130 : 134;
  auto group = [&](int G, int quads) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      dup_halves1(sc[s][0], g.e[s][0], g.e[s][1]);
      dup_halves1(sc[s][1], g.e[s][2], g.e[s][3]);
    }
    skf_group<CPOL, WIDE, NG, 0>(g, w, st, lds, cur, lane, sb, G, quads, acc, wide);
  };
  int G = 0;
#pragma unroll 1
  for (; 4 * G + 4 <= NQ; G++) {
    group(G, 4);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int j = 0; j < 2; j++) sc[s][j] = g.scn[s][j];
  }
  if constexpr (WIDE)
    if (4 * G < NQ) group(G, NQ - 4 * G);
  skf_scale<WIDE, NG>(acc[1], wide[1], g.du, g.r[1]);
  if constexpr (WIDE) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 4 * NG; i++) acc[s][i >> 2][i & 3] = (float)wide[s][i >> 2][i & 3];
  }
}

// The chunk buffers are free for an epilogue: the chunks issued past the end
// (zeros) have landed, and every wave has read its last operands.
__device__ __forceinline__ void sk_lds_free() {
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  lds_barrier();
}

#define MOE_SK_YST 260  // floats from a token's row to the next in k_down_sk's LDS

// gate/up -> clamp -> SwiGLU -> Q8_0(h) on items of up to 64 rows: one
// workgroup of 4 waves per (quad of F, item), wave = the gate and the up tile
// of one 32-row unit over all of K.  h quad-major in quad records.  grid (F/128,
// item capacity), 256 threads, LDS MOE_SK_LDS_BYTES.
template <bool WIDE>
__global__ __launch_bounds__(64 * MOE_SK_WAVES) __attribute__((amdgpu_waves_per_eu(2)))
void k_gate_up_sk(const uint8_t *__restrict__ w_g, const uint8_t *__restrict__ w_u, const uint32_t *__restrict__ xs,
                  const int32_t *__restrict__ items, const int32_t *__restrict__ perm, int k, int T, int F, int H,
                  float clamp, uint32_t *__restrict__ hs, float *__restrict__ htap) {
  extern __shared__ __align__(16) uint32_t lds[];
  const int4 it = item_of(items, blockIdx.y);  // beside the count (the list holds a record for every grid row)
  if ((int)blockIdx.y >= items[0]) return;
  const int NQ = H / 128, NG = moe_nq4(NQ), tiles = F / MOE_TILE;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int P = T * k, row0 = it.y, nt = it.z;
  const bool shared = (it.w & MOE_ITEM_SHARED) != 0, split = (it.w & MOE_ITEM_SPLIT) != 0;
  const int u = MOE_SK_WAVES * blockIdx.x + wave, n = lane & 31, gb = lane >> 5;
  const size_t rec = ((size_t)it.x * tiles + 2 * u) * NG * MOE_REC_BYTES;
  auto row = [&](int t0) { return t0 + n < nt ? (shared ? row0 + t0 + n - P : perm[row0 + t0 + n] / k) : -1; };
  const skw w = make_skw(w_g + rec, w_u + rec, NQ, lane);
  // SwiGLU and Q8_0 of 32 tokens into the records of LDS rows t0 ..
  auto finish = [&](const f32x16_t &g, const f32x16_t &up, int t0) {
    float h[16];
#pragma unroll
    for (int i = 0; i < 16; i++) h[i] = swiglu(g[i], up[i], clamp);  // an absent token's sums are 0
    h_quad_store(h, lds + (t0 + n) * MOE_SQ_DW, wave, lane);
    if (htap && t0 + n < nt) {
#pragma unroll
      for (int i = 0; i < 16; i++)
        htap[(size_t)(row0 + t0 + n) * F + (size_t)u * MOE_UNIT + 8 * (i >> 2) + 4 * gb + (i & 3)] = h[i];
    }
  };
  // the same after skf_loop, lanes = rows of F: h by token in LDS, quantized
  // from there
  auto finish_few = [&](auto &acc, auto ng) {
    constexpr int NG_ = decltype(ng)::value;
    float *hb = reinterpret_cast<float *>(lds + MOE_SK_ROWS * MOE_SQ_DW);  // [token][128], behind the records
#pragma unroll
    for (int i = 0; i < 4 * NG_; i++) {
      const int t = 8 * (i >> 2) + 4 * gb + (i & 3);
      const float h = swiglu(acc[0][i >> 2][i & 3], acc[1][i >> 2][i & 3], clamp);
      hb[t * 128 + MOE_UNIT * wave + n] = h;
      if (htap && t < nt) htap[(size_t)(row0 + t) * F + (size_t)u * MOE_UNIT + n] = h;
    }
    __syncthreads();
    stage_quant_quads(hb, 4 * nt, lds, threadIdx.x, 64 * MOE_SK_WAVES);
  };
  auto few = [&](auto ng) {
    constexpr int NG_ = decltype(ng)::value;
    f32x4_t acc[2][NG_];
    if (split) skf_loop<0, WIDE, NG_, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    else skf_loop<MOE_CPOL_NT, WIDE, NG_, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    sk_lds_free();
    finish_few(acc, ng);
  };
  // an expert of one item reads its tiles once: non-temporal, as in decode;
  // the items of a larger expert share them through L2
  // the 4 waves' blocks meet as whole records in LDS, and the item's records
  // of this quad leave as one run (stored from the waves in 24-byte pieces they
  // cost the weight stream 27 of 730 us at 512 tokens)
  if (!WIDE && nt > MOE_SK_ROWS) {
    f32x16_t acc[2][2];
    if (split) sk_loop2<0, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    else sk_loop2<MOE_CPOL_NT, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    sk_lds_free();
    finish(acc[0][0], acc[0][1], 0);
    finish(acc[1][0], acc[1][1], 32);
  } else if (nt <= 8) {
    few(std::integral_constant<int, 1>{});
  } else if (nt <= 16) {
    few(std::integral_constant<int, 2>{});
  } else {
    f32x16_t acc[2];
    if (split) sk_loop<0, WIDE, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    else sk_loop<MOE_CPOL_NT, WIDE, false>(w, xs, T, NQ, row, lds, lane, wave, acc);
    sk_lds_free();
    finish(acc[0], acc[1], 0);
  }
  __syncthreads();
  uint4 *dst = reinterpret_cast<uint4 *>(hs + ((size_t)blockIdx.x * (P + T) + row0) * MOE_SQ_DW);
  for (int i = threadIdx.x; i < nt * MOE_SQ_U4; i += 64 * MOE_SK_WAVES) dst[i] = reinterpret_cast<const uint4 *>(lds)[i];
}

// down x router weight on items of up to 64 rows: one workgroup of 4 waves
// per (256 rows of H, item), wave = two 32-row tiles over all of F against the
// item's h rows; y[row] = the tiles' rows x the pair's router weight (the
// shared expert's rows unweighted).  grid (ceil(H/256), item capacity), 256
// threads, LDS MOE_SK_LDS_BYTES.
template <bool WIDE>
__global__ __launch_bounds__(64 * MOE_SK_WAVES) __attribute__((amdgpu_waves_per_eu(2)))
void k_down_sk(const uint8_t *__restrict__ w_d, const uint32_t *__restrict__ hs, int n_rows,
               const int32_t *__restrict__ items, const int32_t *__restrict__ perm, const float *__restrict__ wts, int F,
               int H, float *__restrict__ y) {
  extern __shared__ __align__(16) uint32_t lds[];
  const int4 it = item_of(items, blockIdx.y);  // beside the count (the list holds a record for every grid row)
  if ((int)blockIdx.y >= items[0]) return;
  const int NQ = F / 128, NG = moe_nq4(NQ), tiles = H / MOE_TILE;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = it.y, nt = it.z;
  const bool shared = (it.w & MOE_ITEM_SHARED) != 0;
  const int n = lane & 31, gb = lane >> 5;
  const int t64 = MOE_SK_WAVES * blockIdx.x + wave;  // 64 rows of H
  const bool rows = t64 < H / 64;                    // H % 256 == 128: the last workgroup's upper waves only stage
  const uint8_t *w0 = w_d + ((size_t)it.x * tiles + 4 * (rows ? t64 : 0)) * NG * MOE_REC_BYTES;
  auto row = [&](int t0) { return t0 + n < nt ? row0 + t0 + n : -1; };
  const skw w = make_skw(w0, w0 + (size_t)2 * NG * MOE_REC_BYTES, NQ, lane);
  const int col = 256 * blockIdx.x + 4 * lane;
  // the rows of tokens t0 .. t0 + 31, 256 columns each, meet in LDS and leave as runs of 1 KiB
  auto store_rows = [&](int t0) {
    __syncthreads();
    const float *red = reinterpret_cast<const float *>(lds);
    if (col < H)
      for (int t = wave; t < 32 && t0 + t < nt; t += MOE_SK_WAVES)
        *reinterpret_cast<f32x4_t *>(y + (size_t)(row0 + t0 + t) * H + col) =
            *reinterpret_cast<const f32x4_t *>(red + t * MOE_SK_YST + 4 * lane);
  };
  auto finish = [&](const f32x16_t &a0, const f32x16_t &a1, int t0) {
    const bool live = t0 + n < nt;
    const float wt = live && !shared ? wts[perm[row0 + t0 + n]] : 1.0f;
    sk_lds_free();
    float *red = reinterpret_cast<float *>(lds);  // [token][256 columns, 4 of padding]
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const f32x16_t &a = s ? a1 : a0;
        f32x4_t v;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = shared ? a[4 * i + j] : __fmul_rn(a[4 * i + j], wt);
        *reinterpret_cast<f32x4_t *>(red + n * MOE_SK_YST + 64 * wave + 32 * s + 8 * i + 4 * gb) = v;
      }
    store_rows(t0);
  };
  const bool split = (it.w & MOE_ITEM_SPLIT) != 0;
  // items of up to 16 tokens, lanes = rows of H
  auto few = [&](auto ng) {
    constexpr int NG_ = decltype(ng)::value;
    f32x4_t acc[2][NG_];
    if (split) skf_loop<0, WIDE, NG_, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    else skf_loop<MOE_CPOL_NT, WIDE, NG_, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    float wt[4 * NG_];
#pragma unroll
    for (int i = 0; i < 4 * NG_; i++) {
      const int t = 8 * (i >> 2) + 4 * gb + (i & 3);
      wt[i] = t < nt && !shared ? wts[perm[row0 + t]] : 1.0f;
    }
    sk_lds_free();
    float *red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int i = 0; i < 4 * NG_; i++) {
        const float a = acc[s][i >> 2][i & 3];
        red[(8 * (i >> 2) + 4 * gb + (i & 3)) * MOE_SK_YST + 64 * wave + 32 * s + n] = shared ? a : __fmul_rn(a, wt[i]);
      }
    store_rows(0);
  };
  if (!WIDE && nt > MOE_SK_ROWS) {
    f32x16_t acc[2][2];
    if (split) sk_loop2<0, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    else sk_loop2<MOE_CPOL_NT, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    finish(acc[0][0], acc[0][1], 0);
    finish(acc[1][0], acc[1][1], 32);
  } else if (nt <= 8) {
    few(std::integral_constant<int, 1>{});
  } else if (nt <= 16) {
    few(std::integral_constant<int, 2>{});
  } else {
    f32x16_t acc[2];
    if (split) sk_loop<0, WIDE, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    else sk_loop<MOE_CPOL_NT, WIDE, true>(w, hs, n_rows, NQ, row, lds, lane, wave, acc);
    finish(acc[0], acc[1], 0);
  }
}
