// x3gemm.hip -- batches (2 and more tokens) through quantized weights with fp32 accuracy on the
// matrix cores: grouped gate/up and down over every expert of a call, one expert, or one matrix.
//
// The reference's s > 1 products (kernels.rs:233 matmul_mxfp4, :276 matmul_i4_grouped) read a weight
// row once for all tokens. Here a workgroup takes a tile of up to X3Args::tch tokens and a block of rows, so
// a weight byte comes from HBM once per tile of its expert. tch is 16, or 32 where an expert has more than
// 16 tokens on average (x3_tch; one expert's batch: from 49 tokens on); the shared expert of S tokens has
// S / tch tiles. Both operands are exact in bf16 parts:
//   activations  x = hi + mid + lo, three truncated bf16 parts (8 significant bits each: exact);
//   MXFP4        e2m1 * 2^(b-127), exact in bf16 (v_cvt_scalef32_pk_bf16_fp4);
//   grouped int4 the value -8..7 as sign and magnitude in an e4m3 byte (magnitudes 0..8 are m * 2^-9:
//                e4m3's subnormals and first binade), v_cvt_scalef32_pk_bf16_fp8 times 2^9; the group's
//                scale multiplies the group's fp32 sum.
// Each product is exact and the sums are fp32: partial sums of 32 columns (int4, the group) or 256
// (MXFP4) in the MFMA accumulator, then added to the row's sum. Error against 64 bits (2048-8192 columns,
// 2-norm): MXFP4 0.6-0.9e-7 (the decode GEMV 1.2e-7), int4 1.0-1.4e-7 (2.6-2.9e-7).
//
// MFMA operands (v_mfma_f32_16x16x32_bf16): A's 16 rows are activation rows, B's 16 columns weight
// rows, so that a lane's column, and with it a group's scale, is one weight row. MFMA j of a
// 128-column step covers block j of 32 columns: lane (r, g) holds columns 32 j + 8 g .. +7 of weight
// row r (one dword of codes) and of activation row r. int4 codes decode as even columns then odd ones
// (x3_pos); an int4 product's activation parts are written in that order.
//
// How a tile's tokens map to activation rows depends on their number (X3_SMALL, X3_MID, X3_BIG):
// up to 5 tokens put their three parts in rows of one block (one MFMA per block of weights); 6-16
// tokens chain the three parts into one accumulator (three MFMAs, but one scaling of the sums); 17-32
// tokens take two such blocks, so that the decode of a weight serves 32 tokens.
//
// A wave owns two 16-row weight tiles. Its codes stream as 8 rows x 128 bytes per load instruction, a
// 256-column group ahead, through a wave-private LDS area that is read back in the MFMA layout; its
// scales come in whole lines. The activations, loaded a group ahead too, go through an LDS double buffer
// shared by the four waves. Three workgroups per CU for tiles of 16 tokens, two for 32.
//
// What bounds it, hidden 6144, 256 int4 experts of 2048, 301 tokens (283 tiles): gate/up 1.19 ms for
// 4.5 GB of tiles (3.8 TB/s), against 7.77 ms for a GEMV per token and expert. VALU 61%, LDS 45% and
// MFMA 27% busy, waves waiting a quarter of their cycles; without activation loads 1.03 ms, with a third
// of the MFMAs 1.06. Tried: the MFMA layout loaded straight from memory (16 rows x 64 bytes) and
// transposed by permlane swaps 2.16 ms; 512-column groups at two workgroups per CU 1.37; units in
// contiguous runs over all XCDs 1.27 (6.6 GB fetched); static dealing 1.29; the stored code with the -8
// folded into the MFMA's start 1.18 (38% fewer VALU instructions); each product scaled one block later
// 1.21.
#include <algorithm>

#include "rbt_device.h"
#include "rbt_internal.h"

namespace rbt {

typedef __bf16 xb8 __attribute__((ext_vector_type(8)));
typedef __bf16 xb2 __attribute__((ext_vector_type(2)));
typedef float xf4 __attribute__((ext_vector_type(4)));

constexpr int X3_BS = 128 + 16;  // bf16 per staged activation row (288 B: 16-byte reads of 16 rows conflict-free)
constexpr int X3_KG = 256;       // columns per group (two 128-column steps)
constexpr int X3_WS = 128 + 16;  // bytes per staged weight row (a group's codes)
constexpr int X3_WT = 16 * X3_WS;
constexpr int X3_SS = 48;        // bytes per staged row of int4 scales (a group's 8 floats, padded)
constexpr int X3_ST = 16 * X3_SS;
enum { X3_SMALL, X3_MID, X3_BIG };  // up to 5, 16, 32 tokens
constexpr int x3_arows(int mode) { return mode == X3_SMALL ? 1 : mode == X3_MID ? 3 : 6; }  // 16-row blocks staged
// LDS of a workgroup: the activation double buffer, each wave's two weight tiles and their scales.
constexpr int x3_lds_bytes(bool i4, int mode) {
  return 2 * x3_arows(mode) * 16 * X3_BS * 2 + 4 * 2 * X3_WT + (i4 ? 4 * 2 * X3_ST : 0);
}

// Position of column e (0..7) among the 8 codes of a dword as x3_b decodes them.
__device__ __forceinline__ int x3_pos(bool i4, int e) { return i4 ? (e >> 1) + 4 * (e & 1) : e; }

// One dword of codes -> 8 bf16 weights (MXFP4: times the block's E8M0 value; int4: -8..7).
template <bool I4>
__device__ __forceinline__ xb8 x3_b(uint32_t w, float sc) {
  xb2 a, b, c, d;
  if (I4) {
    // per nibble q: n = 8 where q < 8 (negative), z = |q - 8|; then bytes sign | magnitude
    const uint32_t n = ~w & 0x88888888u, k = n >> 3;
    const uint32_t z = ((w & 0x77777777u) ^ (n - k)) + k;
    const uint32_t ev = (z & 0x0F0F0F0Fu) | ((n << 4) & 0x80808080u);
    const uint32_t od = ((z >> 4) & 0x0F0F0F0Fu) | (n & 0x80808080u);
    a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(ev, 512.0f, false);
    b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(ev, 512.0f, true);
    c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(od, 512.0f, false);
    d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(od, 512.0f, true);
  } else {
    a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 0);
    b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 1);
    c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 2);
    d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 3);
  }
  return xb8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// x = p[0] + p[1] + p[2] exactly: each part the leading 8 significant bits of what is left. An
// infinite or NaN x is all three parts. MXFP4 weights may be infinite (E8M0 253 and 254), and a part that is
// zero would make NaN of a product that is infinite: from 2^-95 on such a part is 2^-126 with the sign of x,
// which adds 2^-30 of the exact product at most and is rounded away from every sum that is not itself as small
// (parts dealt out evenly stay exact but cost precision: bf16 activations 6.8e-8 -> 7.2e-8 from 64 bits).
template <bool I4>
__device__ __forceinline__ void x3_split(float x, __bf16 (&p)[3]) {
  const uint32_t b = __float_as_uint(x);
  if ((b & 0x7F800000u) == 0x7F800000u) {
    p[0] = p[1] = p[2] = (__bf16)x;
    return;
  }
  const float h = __uint_as_float(b & 0xFFFF0000u);
  const float r = __fsub_rn(x, h);
  float m = __uint_as_float(__float_as_uint(r) & 0xFFFF0000u);
  float l = __fsub_rn(r, m);
  if (!I4 && (b & 0x7F800000u) >= (32u << 23)) {
    const float tiny = __uint_as_float((b & 0x80000000u) | (1u << 23));
    m = m == 0.0f ? tiny : m;
    l = l == 0.0f ? tiny : l;
  }
  p[0] = (__bf16)h;
  p[1] = (__bf16)m;
  p[2] = (__bf16)l;
}

// 8 consecutive columns of one row: the parts (in x3_pos order), part_stride apart.
template <bool I4>
__device__ __forceinline__ void x3_write8(const float (&v)[8], __bf16 *__restrict__ dst, long part_stride) {
  xb8 o[3];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    __bf16 p[3];
    x3_split<I4>(v[e], p);
#pragma unroll
    for (int q = 0; q < 3; q++) o[q][x3_pos(I4, e)] = p[q];
  }
#pragma unroll
  for (int q = 0; q < 3; q++) *reinterpret_cast<xb8 *>(dst + q * part_stride) = o[q];
}

// x [S, K] fp32 -> xb3 [3 S, K] (row 3 t + part); clears the unit queues of the products that follow.
// With pick, the last workgroup lists one expert's tokens instead.
template <bool I4>
__global__ __launch_bounds__(256) void k_x3split(const float *__restrict__ x, long n8, int k8,
                                                 __bf16 *__restrict__ xb3, unsigned *__restrict__ queue,
                                                 const X3Pick pick) {
  if (pick.ids && blockIdx.x == gridDim.x - 1) {  // (uniform) a workgroup of its own
    rbt_single_rows(pick.ids, pick.w, pick.S, pick.k, pick.eid, pick.pair_tok, pick.pair_w, pick.nr);
    return;
  }
  if (queue && blockIdx.x == 0 && threadIdx.x < X3_QN) queue[threadIdx.x] = 0u;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const long t = i / k8, K = 8L * k8;
  float v[8];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const float4 f = *reinterpret_cast<const float4 *>(x + 8 * i + 4 * q);
    v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
  }
  x3_write8<I4>(v, xb3 + 2 * t * K + 8 * i, K);
}

// One tile through one row block of BR = 64 TILES rows, columns 256 g0 .. 256 (g0 + ng) - 1.
// Wave w owns TILES 16-row tiles of each of NM matrices per row block. src: the activation parts at the
// tile's base row, so[q]: this thread's byte offset of staged row tid / 16 of block q, columns
// 8 (tid % 16) ... acc[t][q]: the sums of weight tile t (matrix t / TILES), accumulator block q. Uniform bases and 32-bit lane offsets keep the addresses
// in scalar registers.
//
// A row's scales are fetched in lines (int4: 128 bytes, four groups; MXFP4: 64 bytes, eight), lane l
// holding 1/4 of row l / 4's line: fetched a group's bytes at a time, the lines left the L2 between
// their groups (0.5 GB more fetched at the shape above).
template <bool I4, int NM, int TILES, int MODE>
__device__ __forceinline__ void x3_run(const uint8_t *src, const uint32_t (&so)[x3_arows(MODE)],
                                       const uint8_t *const (&a)[NM], const uint8_t *const (&sc)[NM], int K, int rb,
                                       int g0, int ng, uint8_t *lds, xf4 (&acc)[NM * TILES][MODE == X3_BIG ? 2 : 1]) {
  constexpr int NT = NM * TILES, BR = 64 * TILES, AR = x3_arows(MODE), NQ = MODE == X3_BIG ? 2 : 1;
  constexpr int NP = MODE == X3_SMALL ? 1 : 3;  // MFMAs chained per accumulator block
  constexpr int LG = I4 ? 4 : 8, GB = I4 ? 32 : 8, NL = I4 ? 2 : 1;  // groups per line, bytes per group, u4 per lane
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int rowb = K >> 1, rows = I4 ? K >> 3 : K >> 5;  // bytes per row: codes, scales
  typedef __bf16 Buf[AR][16][X3_BS];
  Buf *bs = reinterpret_cast<Buf *>(lds);
  uint8_t *const wl = lds + 2 * sizeof(Buf) + w * (NT * X3_WT);
  uint8_t *const sl = lds + 2 * sizeof(Buf) + 4 * (NT * X3_WT) + w * (NT * X3_ST);
  const uint8_t *pa[NT], *ps[NT];  // uniform
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const long row = (long)rb * BR + 16 * TILES * w + 16 * (t % TILES);
    pa[t] = a[t / TILES] + row * rowb + 128L * g0;
    ps[t] = sc[t / TILES] + row * rows + (long)GB * g0;
  }
  // codes: 8 rows x 128 bytes per instruction
  const uint32_t oc = (uint32_t)(lane >> 3) * rowb + 16 * (lane & 7);
  int f_g = 0;  // next group to fetch (past the end: the last one again, never used)
  rbt_u4 nw[NT][2], ln[NT][NL];
  auto fetch = [&]() {
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int t = 0; t < NT; t++) nw[t][q] = __builtin_nontemporal_load((const rbt_gu4 *)(pa[t] + 128L * f_g + 8L * q * rowb + oc));
    f_g = min(f_g + 1, ng - 1);
  };
  // line l (groups LG l ..): the lane's quarter, clamped to the last quarter in range
  auto line = [&](int l) {
    const int q0 = LG / 4 * (4 * l + (lane & 3));  // first group of the quarter
    const uint32_t off = (uint32_t)(lane >> 2) * rows + GB * min(q0, ng - LG / 4);
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int u = 0; u < NL; u++) ln[t][u] = *(const rbt_gu4 *)(ps[t] + off + 16 * u);
  };
  // activations: st[d] holds the next step of parity d, loaded a group ahead
  rbt_u4 st[2][AR];
  const int nst = 2 * ng;
  int a_s = 0;
  auto stage_load = [&](int slot) {
#pragma unroll
    for (int q = 0; q < AR; q++) st[slot][q] = *(const rbt_gu4 *)(src + 256L * (2 * g0 + a_s) + so[q]);
    a_s = min(a_s + 1, nst - 1);
  };
  const int tl = threadIdx.x >> 4, tc = threadIdx.x & 15;
  auto stage_store = [&](int slot) {
#pragma unroll
    for (int q = 0; q < AR; q++) *reinterpret_cast<rbt_u4 *>(&bs[slot][q][tl][8 * tc]) = st[slot][q];
  };
  stage_load(0);
  stage_load(1);
  line(0);
  fetch();
  stage_store(0);
  stage_load(0);
  __syncthreads();
  // ch: the chained products; cl (MXFP4, three chained parts): those of the two small parts, so that the
  // full-size sum rounds once per block and not three times
  xf4 ch[NT][NQ], cl[NT][NQ];
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int q = 0; q < NQ; q++) acc[t][q] = ch[t][q] = cl[t][q] = xf4{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < ng; it++) {
    // the group's codes -> the wave's LDS area; its scales: int4 from the lanes holding this quarter of
    // the line to LDS, MXFP4 by shuffles; then the next group's codes and, after a line's last group, the
    // next line
    const int lq = it & (LG - 1);
    uint2 cs[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      uint8_t *wt = wl + t * X3_WT + (lane >> 3) * X3_WS + 16 * (lane & 7);
#pragma unroll
      for (int q = 0; q < 2; q++) *reinterpret_cast<rbt_u4 *>(wt + 8 * q * X3_WS) = nw[t][q];
      if (I4) {
        if ((lane & 3) == lq) {
          rbt_u4 *st = reinterpret_cast<rbt_u4 *>(sl + t * X3_ST + (lane >> 2) * X3_SS);
          st[0] = ln[t][0];
          st[1] = ln[t][NL - 1];
        }
      } else {
        const int from = 4 * r + (lq >> 1);
        const rbt_u4 v = ln[t][0];
        cs[t].x = (uint32_t)__shfl((int)(lq & 1 ? v.z : v.x), from, 64);
        cs[t].y = (uint32_t)__shfl((int)(lq & 1 ? v.w : v.y), from, 64);
      }
    }
    if (lq == LG - 1 && it + 1 < ng) line((it + 1) / LG);
    fetch();
#pragma unroll
    for (int d = 0; d < 2; d++) {
      stage_store(d ^ 1);  // the next step's activations
      stage_load(d ^ 1);
      xf4 s4[NT];
      if (I4) {
#pragma unroll
        for (int t = 0; t < NT; t++) s4[t] = *reinterpret_cast<const xf4 *>(sl + t * X3_ST + r * X3_SS + 16 * d);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        xb8 av[AR];
#pragma unroll
        for (int q = 0; q < AR; q++) av[q] = *reinterpret_cast<const xb8 *>(&bs[d][q][r][32 * j + 8 * g]);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const uint32_t code = *reinterpret_cast<const uint32_t *>(wl + t * X3_WT + r * X3_WS + 16 * (4 * d + j) + 4 * g);
          const xb8 bv = x3_b<I4>(code, I4 ? 0.0f : rbt_e8m0(((d ? cs[t].y : cs[t].x) >> (8 * j)) & 0xffu));
#pragma unroll
          for (int q = 0; q < NQ; q++) {
            xf4 dd = I4 ? xf4{0.f, 0.f, 0.f, 0.f} : NP == 3 ? cl[t][q] : ch[t][q];
#pragma unroll
            for (int p = NP - 1; p >= (I4 ? 0 : NP == 3); p--)
              dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[NP * q + p], bv, dd, 0, 0, 0);
            if (!I4 && NP == 3) {
              cl[t][q] = dd;
              dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[NP * q], bv, ch[t][q], 0, 0, 0);
            }
            if (I4) {
#pragma unroll
              for (int i = 0; i < 4; i++) acc[t][q][i] = __builtin_fmaf(s4[t][j], dd[i], acc[t][q][i]);
            } else {
              ch[t][q] = dd;
            }
          }
        }
      }
      if (I4) {
        // keep the step's multiply-adds in the step: sunk towards the sums' use, every group's product
        // and scales stay live to the end of the loop body
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
          for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int i = 0; i < 4; i++) asm volatile("" : "+v"(acc[t][q][i]));
      }
      __syncthreads();
    }
    if (!I4) {
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < NQ; q++) {
#pragma unroll
          for (int i = 0; i < 4; i++) acc[t][q][i] += NP == 3 ? ch[t][q][i] + cl[t][q][i] : ch[t][q][i];
          ch[t][q] = cl[t][q] = xf4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
}

// The tile of index ti: its expert, first pair and token count (0: nothing to do).
struct X3Tile {
  RbtExpertDev J;
  int pbase, M;
  int n;  // single: the rows there are
};
__device__ __forceinline__ int x3_rows(const X3Args &A) { return A.nrows_dev ? min(A.nrows, *A.nrows_dev) : A.nrows; }

__device__ __forceinline__ X3Tile x3_tile(const X3Args &A, int ti) {
  X3Tile T;
  if (A.tiles) {
    const PTile t = A.tiles[ti];
    const PSeg s = A.segs[t.seg];
    T.J = s.eid >= 0 ? A.table[s.eid] : *A.shared_dev;
    T.pbase = s.off + t.c0;
    T.M = min(A.tch, s.cnt - t.c0);
    if (T.J.gd == nullptr || T.J.ud == nullptr || T.J.dd == nullptr) T.M = 0;  // reported by k_pgroup
    T.n = 0;
  } else {
    T.n = x3_rows(A);
    T.J = A.single;
    T.pbase = ti * A.tch;
    T.M = min(A.tch, T.n - T.pbase);
  }
  return T;
}

// Token (within the tile) and part of activation row m of staged block q. X3_SMALL: lane group m / 4
// holds token m / 4's parts in rows 4 g + 0..2, and part g of the fifth token in row 4 g + 3 (row 15
// repeats part 0, never read); else block 3 b + p is part p of tokens 16 b .. 16 b + 15.
template <int MODE>
__device__ __forceinline__ void x3_row(int q, int m, int &tok, int &part) {
  if (MODE == X3_SMALL) {
    const int g = m >> 2, i = m & 3;
    tok = i < 3 ? g : 4;
    part = i < 3 ? i : g < 3 ? g : 0;
  } else {
    tok = 16 * (q / 3) + m;
    part = q % 3;
  }
}

template <bool I4, bool GATEUP, int MODE>
__device__ __forceinline__ void x3_unit(const X3Args &A, const X3Tile &T, int KS, int ks, int rb, uint8_t *lds) {
  constexpr int NM = GATEUP ? 2 : 1, TILES = GATEUP ? 1 : 2, NT = NM * TILES, BR = 64 * TILES;
  constexpr int AR = x3_arows(MODE), NQ = MODE == X3_BIG ? 2 : 1;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, w = threadIdx.x >> 6;
  const int K = A.K, O = A.O, n2 = K / (2 * X3_KG);
  const int g0 = ks * n2 / KS * 2, g1 = (ks + 1) * n2 / KS * 2;  // K parts of whole 512 columns
  // activation rows: a token's through row_tok from the call's first row, else from the tile's first
  const long row0 = A.row_tok ? 0 : T.pbase;
  const uint8_t *src = reinterpret_cast<const uint8_t *>(A.xb3 + 3 * row0 * K);
  uint32_t so[AR];
#pragma unroll
  for (int q = 0; q < AR; q++) {
    int tok, part;
    x3_row<MODE>(q, threadIdx.x >> 4, tok, part);
    tok = min(tok, T.M - 1);
    const int row = A.row_tok ? min(max(A.row_tok[T.pbase + tok], 0), A.S - 1) : tok;
    so[q] = ((uint32_t)(3 * row + part) * K + (threadIdx.x & 15) * 8) * 2;
  }
  const uint8_t *wa[NM], *ws[NM];
  if (GATEUP) {
    wa[0] = T.J.gd, ws[0] = (const uint8_t *)T.J.gs;
    wa[NM - 1] = T.J.ud, ws[NM - 1] = (const uint8_t *)T.J.us;
  } else {
    wa[0] = T.J.dd, ws[0] = (const uint8_t *)T.J.ds;
  }
  xf4 acc[NT][NQ];
  x3_run<I4, NM, TILES, MODE>(src, so, wa, ws, K, rb, g0, g1 - g0, lds, acc);
  const int o0 = rb * BR + 16 * TILES * w + r;
  // v[t]: token tok's sum of weight tile t, row o0 + 16 (t % TILES)
  auto put = [&](int tok, const float(&v)[NT]) {
    if (tok >= T.M) return;
    const long pr = T.pbase + tok;
    if (A.part) {
#pragma unroll
      for (int t = 0; t < NT; t++)
        A.y[((long)(ks * NM + t / TILES) * T.n + pr) * O + o0 + 16 * (t % TILES)] = v[t];
    } else if (GATEUP) {
      __bf16 p[3];
      x3_split<I4>(rbt_act(A.act, v[0], v[NT - 1]), p);
      __bf16 *d = A.hb3 + 3 * pr * O + (o0 & ~7) + x3_pos(I4, o0 & 7);
#pragma unroll
      for (int q = 0; q < 3; q++) d[(long)q * O] = p[q];
    } else {
#pragma unroll
      for (int t = 0; t < NT; t++) A.y[pr * O + o0 + 16 * t] = v[t];
    }
  };
  if (MODE == X3_SMALL) {
    float v[NT], v4[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
      v[t] = (acc[t][0][0] + acc[t][0][1]) + acc[t][0][2];
      const float l = acc[t][0][3];
      v4[t] = (__shfl(l, r, 64) + __shfl(l, 16 + r, 64)) + __shfl(l, 32 + r, 64);
    }
    put(g, v);
    if (g == 0) put(4, v4);
  } else {
#pragma unroll
    for (int q = 0; q < NQ; q++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float v[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) v[t] = acc[t][q][i];
        put(16 * q + 4 * g + i, v);
      }
  }
}

// Units (tile, row block, K part): XCD x (workgroups x, x + 8, ..) takes [x U / 8, (x + 1) U / 8), its
// workgroups dealt over them in turn, so that at any time an XCD works on a few tiles and their
// activations (590 KB per tile of 16 at 6144 columns, more than a row block's weights) stay in its L2.
// The tile count is on the device for a grouped call, so the grid is fixed. With A.queue (grouped calls,
// whose tiles cost between one and three MFMAs per weight block) a workgroup takes its next unit from its
// XCD's counter, read a unit ahead.
// TOP: the largest mode the launch can meet (tiles of up to 16 tokens: three workgroups per CU, 32: two).
template <bool I4, bool GATEUP, int TOP>
__global__ __launch_bounds__(256, TOP == X3_BIG ? 2 : 3) void k_x3(const X3Args A) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[x3_lds_bytes(I4, TOP)];
  const int RB = x3_row_blocks(A.O, GATEUP), rows = A.tiles ? 0 : x3_rows(A);
  const int KS = A.part ? x3_ks(rows, A.tch, A.K, RB, A.wgs) : 1;
  const int nt = A.tiles ? *A.ntiles : (rows + A.tch - 1) / A.tch;
  const long U = (long)nt * RB * KS;
  const int xcd = blockIdx.x & 7, nx = gridDim.x >> 3;
  __shared__ int next_s;
  const int u0 = (int)(xcd * U / 8), n = (int)((xcd + 1) * U / 8) - u0;
  for (int i = blockIdx.x >> 3; i < n;) {
    const int u = u0 + i;
    unsigned taken = 0;
    if (A.queue && threadIdx.x == 0) taken = atomicAdd(A.queue + xcd, 1u);
    const int ks = u % KS;
    const int ub = u / KS;
    const int ti = ub / RB, rb0 = ub - ti * RB;
    const X3Tile T = x3_tile(A, ti);
    if (T.M <= 0) {
    } else if (T.M <= 5)
      x3_unit<I4, GATEUP, X3_SMALL>(A, T, KS, ks, rb0, lds);
    else if (TOP == X3_MID || T.M <= 16)
      x3_unit<I4, GATEUP, X3_MID>(A, T, KS, ks, rb0, lds);
    else
      x3_unit<I4, GATEUP, X3_BIG>(A, T, KS, ks, rb0, lds);
    if (A.queue) {
      __syncthreads();
      if (threadIdx.x == 0) next_s = nx + (int)taken;
      __syncthreads();
      i = next_s;
    } else {
      i += nx;
    }
  }
}

// Sums of K parts. Matrix: y[i] = sum over the parts of part[p][i], in part order (n4 float4s).
__global__ __launch_bounds__(256) void k_x3sum(const xf4 *__restrict__ part, long n4, int KS, xf4 *__restrict__ y) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  xf4 v = part[i];
  for (int p = 1; p < KS; p++) {
    const xf4 q = part[p * n4 + i];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] += q[e];
  }
  y[i] = v;
}

// Gate/up: h = act(sum of gate parts, sum of up parts), as the down product's activation parts. Four
// threads per 8 columns of a row, each summing every fourth part (one thread summing them all waits for
// memory once per part, of which there are up to X3_KSMAX); rows past *nrows_dev are left alone.
template <bool I4>
__global__ __launch_bounds__(256) void k_x3act(const X3Args A) {
  const int o8 = A.O >> 3, q4 = threadIdx.x & 3;
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) >> 2;
  const int n = x3_rows(A), KS = x3_ks(n, A.tch, A.K, x3_row_blocks(A.O, true), A.wgs);
  const long pr = i / o8;
  if (pr >= n) return;  // the four threads together
  const long c = 8 * (i - pr * o8);
  float gu[2][8] = {};
  for (int p = q4; p < KS; p += 4)
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const xf4 v = *reinterpret_cast<const xf4 *>(A.y + ((long)(p * 2 + m) * n + pr) * A.O + c + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; e++) gu[m][4 * q + e] += v[e];
      }
#pragma unroll
  for (int m = 0; m < 2; m++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      gu[m][e] = rbt_dpp_add<0xB1>(gu[m][e]);  // quad_perm: xor 1, xor 2
      gu[m][e] = rbt_dpp_add<0x4E>(gu[m][e]);
    }
  if (q4) return;
  float h[8];
#pragma unroll
  for (int e = 0; e < 8; e++) h[e] = rbt_act(A.act, gu[0][e], gu[1][e]);
  x3_write8<I4>(h, A.hb3 + 3 * pr * A.O + c, A.O);
}

// One expert's weighted rows into the tokens' (glm52/moe.rs:508-512); a token appears at most once.
__global__ __launch_bounds__(256) void k_x3acc(const X3Args A, const int *__restrict__ tok,
                                               const float *__restrict__ w, float *__restrict__ out) {
  const int o4 = A.O >> 2;
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int n = x3_rows(A), KS = x3_ks(n, A.tch, A.K, x3_row_blocks(A.O, false), A.wgs);
  const long r = i / o4;
  if (r >= n) return;
  const xf4 *part = reinterpret_cast<const xf4 *>(A.y);
  xf4 v = part[i];
  for (int p = 1; p < KS; p++) {
    const xf4 q = part[(long)p * n * o4 + i];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] += q[e];
  }
  float *o = out + (long)tok[r] * A.O + 4 * (i - r * o4);
  const float wr = w[r];
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = __fadd_rn(o[e], __fmul_rn(wr, v[e]));
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
bool x3_ok(int kind, size_t gs, size_t cols, size_t rows, bool gateup) {
  // pairs of groups (the MXFP4 scale lines stay 16-byte aligned); whole row blocks (64 rows of gate and of up, or 128 rows)
  return (kind == RBT_QT_MXFP4 || (kind == RBT_QT_I4_GROUPED && gs == 32)) && cols % (2 * X3_KG) == 0 &&
         rows % (gateup ? 64 : 128) == 0 && cols <= (1u << 20) && rows <= (1u << 20);
}

long x3_max_tiles(int S, int k, int E, int has_shared, int tch) {
  const long P = (long)S * k;
  const long nseg = std::min<long>(E, P) + (has_shared ? 1 : 0);
  return nseg + (P + (has_shared ? S : 0) + tch - 1) / tch;
}

// workgroups, a multiple of 8
int x3_wgs(const Ctx &c, int tch) { return ((tch > 16 ? 2 : 3) * c.num_cu + 7) / 8 * 8; }

hipError_t launch_x3split(const Ctx &c, int kind, const float *x, size_t S, size_t K, __bf16 *xb3, unsigned *queue,
                          const X3Pick *pick) {
  const long n8 = (long)(S * K / 8);
  if (n8 <= 0) return hipSuccess;
  const dim3 grid((unsigned)((n8 + 255) / 256 + (pick ? 1 : 0)));
  const X3Pick p = pick ? *pick : X3Pick{};
  if (kind == RBT_QT_I4_GROUPED)
    launch_k(c, k_x3split<true>, grid, dim3(256), x, n8, (int)(K / 8), xb3, queue, p);
  else
    launch_k(c, k_x3split<false>, grid, dim3(256), x, n8, (int)(K / 8), xb3, queue, p);
  return hipGetLastError();
}

hipError_t launch_x3(const Ctx &c, int kind, bool gateup, const X3Args &A) {
  if (A.K % (2 * X3_KG) || A.O % (gateup ? 64 : 128) || (A.tch != 16 && A.tch != 32)) return hipErrorInvalidValue;
  // a lane's 32-bit offset reaches over all S rows' parts through row_tok, else over one tile's
  if (6L * (A.row_tok ? A.S : A.tch) * A.K >= (1L << 32)) return hipErrorInvalidValue;
  const dim3 grid(x3_wgs(c, A.tch)), blk(256);
#define RBT_X3(I4_, GU_)                                                                   \
  {                                                                                        \
    if (A.tch > 16)                                                                        \
      launch_k(c, (k_x3<I4_, GU_, X3_BIG>), grid, blk, A);                                  \
    else                                                                                   \
      launch_k(c, (k_x3<I4_, GU_, X3_MID>), grid, blk, A);                                  \
  }
  if (kind == RBT_QT_I4_GROUPED) {
    if (gateup) RBT_X3(true, true) else RBT_X3(true, false)
  } else {
    if (gateup) RBT_X3(false, true) else RBT_X3(false, false)
  }
#undef RBT_X3
  return hipGetLastError();
}

hipError_t launch_x3sum(const Ctx &c, const float *part, size_t n, int KS, float *y) {
  const long n4 = (long)(n / 4);
  launch_k(c, k_x3sum, dim3((unsigned)((n4 + 255) / 256)), dim3(256), reinterpret_cast<const xf4 *>(part), n4, KS,
           reinterpret_cast<xf4 *>(y));
  return hipGetLastError();
}

hipError_t launch_x3acc(const Ctx &c, const X3Args &A, const int *tok, const float *w, float *out) {
  const long n = (long)A.nrows * (A.O / 4);
  launch_k(c, k_x3acc, dim3((unsigned)((n + 255) / 256)), dim3(256), A, tok, w, out);
  return hipGetLastError();
}

hipError_t launch_x3act(const Ctx &c, int kind, const X3Args &A) {
  const long n = (long)A.nrows * (A.O / 8) * 4;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (kind == RBT_QT_I4_GROUPED)
    launch_k(c, k_x3act<true>, grid, dim3(256), A);
  else
    launch_k(c, k_x3act<false>, grid, dim3(256), A);
  return hipGetLastError();
}

}  // namespace rbt
