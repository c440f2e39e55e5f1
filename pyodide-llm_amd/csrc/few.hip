// few.hip — a few tokens on the matrix cores: the products of matmul_q8r_tile, matmul_q6r, matmul_t2r_tile and
// matmul_b1r_tile for the token counts between the token kernels' (gemv.hip: the weights read once a 4 tokens) and the
// prompt tiles' (gemm.hip: tiles of 64 tokens and 32 rows or more, too few to fill the GPU with).
//
// A block of 4 waves computes 16 RT rows x 16 NT tokens; wave k is the reference's chain k, as in gemm.hip: the groups
// 4 j + k of int8 / int6 (relaxed/int8.ts:26-47), part k of every group of 128 of ternary / binary
// (relaxed/signs.ts:28-55), in order, so every (row, token) is the token kernel's number to the bit.  A step of a chain
// (one group or part of 32) of a 16 x 16 sub-tile is one v_mfma_i32_16x16x32_i8, exact, the correction its accumulator
// input (the caller's wc; -64 sum(w) by an MFMA of the weights against -64; interleave()'s sums), then the
// reference's float32 operations on 4 values a lane.
//
// Why so: the smallest tile of rows that the matrix cores take, so that 4096 rows are 256 blocks; every byte goes from
// HBM / L2 to LDS by buffer-to-LDS loads into a ring of stages (SG steps of the four chains each: 512 or 256 values of
// every row and token), 16-byte chunks swizzled so that 16 rows (or tokens) reading one chunk hit 16 different bank
// quads.  The loads are written in assembly because the compiler, which cannot tell which stage buffer they write, would
// wait for all of them before every LDS read; it sees only the LDS reads, and orders and overlaps those itself.  A
// load into LDS costs about the same whatever its width (the scales as 4-byte loads: 7 us of a 29 us gate/up launch), so
// scales come 16 bytes a lane where they are aligned.
//
// Measured (through hq_matmuls, us, before: 4 tokens a gemv launch below 16 tokens, gemm.hip's tiles from 16): an 8B
// layer of int8 without / with wc, 11 tokens 137 / 148 -> 78 / 80, 16 tokens 174 / 201 -> 80 / 83, 32 tokens 183 / 217 ->
// 110 / 115; the 27B MLP of int6, 16 tokens 199 -> 96; of ternary, 4 tokens 96 -> 66, 16 tokens 212 -> 69, 64 tokens 233 ->
// 152, 128 tokens 321 -> 230.
// What bounds it (an 8B gate/up of 16 tokens, 30 us; copies with a part left out): the loads alone 28 us (the weights and
// scales at HBM's rate are 20), the arithmetic alone 19, neither 10: a block's life has ~2 us of addresses, first loads
// and sums that other blocks hide in part.  More tokens: the arithmetic (16 VALU instructions, 16 to 32 matrix-core
// cycles a sub-tile's step, which add on this part).
#include "common.hpp"
#include "launch.hpp"
#include "stage.hpp"

namespace hq {

namespace {

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

// The ring's LDS where three stages leave room in it (binary, and two token sub-tiles of ternary and of int6 without wc: 34 to 39
// KB, four blocks a CU by LDS); the others' three stages take 42 to 72 KB, two or three blocks.  Rings of 78 KB measured no
// faster for 16 tokens and 4-7 % slower for 17..32
constexpr int kFewLds = 39 * 1024;
struct FewBatch {
  Job job[kMaxJobs];
  int32_t block0[kMaxJobs];  // the first block of each job (INT32_MAX past the last)
  int32_t blocks[kMaxJobs];
};

// ---- buffer-to-LDS loads the compiler does not track ----------------------------------------------------------------
typedef int32_t rsrc4 __attribute__((ext_vector_type(4)));
HQ_DEV rsrc4 few_resource(const char *base, int64_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  const int64_t n = bytes < 0 ? 0 : bytes > 0xFFFFFFFFLL ? 0xFFFFFFFFLL : bytes;
  rsrc4 r;
  r[0] = __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)(a >> 32) & 0xffff);
  r[2] = __builtin_amdgcn_readfirstlane((int32_t)(uint32_t)n);
  r[3] = 0x00020000;
  return r;
}
// Lane l's SIZE bytes at r + vo + so land at LDS address dst + max(SIZE, 4) l (2 bytes zero-extended); past r's size: 0.
// M0, which the loads take their LDS address from, is declared as written (a reserved register: the compiler warns that it
// does not allocate it).  A vector memory instruction may read a scalar register five wait states after a vector
// instruction (v_readfirstlane) wrote it, and the compiler, which would insert these, does not look into the assembly:
// FewLoads::settle() waits them once, and what the loads read later comes from scalar instructions.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int SIZE>
HQ_DEV void dma(rsrc4 r, uint32_t dst, uint32_t vo, uint32_t so) {
  if (SIZE == 16)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(dst), "v"(vo), "s"(r), "s"(so) : "m0", "memory");
  else if (SIZE == 4)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :: "s"(dst), "v"(vo), "s"(r), "s"(so) : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds"
                 :: "s"(dst), "v"(vo), "s"(r), "s"(so) : "m0", "memory");
}
#pragma clang diagnostic pop

// ---- a stage's layout ------------------------------------------------------------------------------------------------
// PACK: bits of a weight as stored (8 int8, 6 int6, 2 ternary, 1 binary).  WIDE: the int8 / int6 rows' and every token's
// scales read 16 bytes at a time: the group count a multiple of 4, their bases and token stride 16-byte aligned
// (few_wide); else 4 bytes a lane.  (Ternary's and binary's token scales and sums: 4 bytes a lane, landing transposed,
// [step][chain][token], so that a lane's four tokens' are one 16-byte read.)
enum FewKind { kFewW, kFewX, kFewS, kFewC, kFewXS, kFewSums };
template <int PACK_, bool WC_, bool WIDE_, int RT_, int NT_>
struct Few {
  static constexpr int PACK = PACK_, RT = RT_, NT = NT_;
  static constexpr bool WC = WC_, WIDE = WIDE_, SIGNS = PACK <= 2;
  static constexpr int SG = RT + NT <= 2 || (SIGNS && NT == 1) ? 4 : 2;  // steps a stage
  // whether a stage's operands are read while the stage before is folded (int8's 8B layer at 11 tokens 85 -> 78 us,
  // at 32 tokens 120 -> 111); ternary and binary, whose operands would take 206 registers, gain more from the waves
  static constexpr bool PIPE = !SIGNS;
  static constexpr int KS = 128 * SG;                    // values of a row (or token) a stage
  static constexpr int WROW = KS * PACK / 8;             // bytes of a row of weights a stage
  static constexpr int CH = WROW / 16;                   // its 16-byte chunks
  static constexpr int CHX = KS / 16;                    // a token's
  // a stage's LDS: 1 KB pieces of weights and activations; the scales (corrections, sums) of a row or token as SG
  // 16-byte pieces of a step's four groups, places swizzled; ternary's and binary's float16 scales [rt][step][16], a
  // word each
  static constexpr int PWT = (16 * RT * WROW + 1023) / 1024;
  static constexpr int PX = 16 * NT * KS / 1024;
  static constexpr int SB = SIGNS ? (16 * RT * SG + 63) / 64 * 256 : 16 * RT * SG * 16, XSB = 16 * NT * SG * 16;  // (the tokens')
  static constexpr int up(int bytes) { return (bytes + 1023) / 1024 * 1024; }  // (a load writes 64 lanes whole)
  static constexpr int W = 0;
  static constexpr int X = W + 1024 * PWT;
  static constexpr int S = X + 1024 * PX;
  static constexpr int C = S + (SIGNS ? SB : up(SB));
  static constexpr int XS = C + (WC ? up(SB) : 0);
  static constexpr int SUMS = XS + up(XSB);
  static constexpr int STAGE = SUMS + (SIGNS ? up(XSB) : 0);
  // the loads: pieces of 64 lanes in this order, dealt to the four waves in turn
  static constexpr int SLANE = SIGNS ? 4 : WIDE ? 16 : 4, XLANE = WIDE && !SIGNS ? 16 : 4;  // LDS bytes a lane
  static constexpr int PS = (SB + 64 * SLANE - 1) / (64 * SLANE), PXS = (XSB + 64 * XLANE - 1) / (64 * XLANE);
  static constexpr int END[6] = {PWT, PWT + PX, PWT + PX + PS, PWT + PX + PS * (WC ? 2 : 1),
                                 PWT + PX + PS * (WC ? 2 : 1) + PXS,
                                 PWT + PX + PS * (WC ? 2 : 1) + PXS * (SIGNS ? 2 : 1)};
  static constexpr int P = END[5], LOADS = (P + 3) / 4;
  static constexpr FewKind kind(int p) {
    return p < END[0] ? kFewW : p < END[1] ? kFewX : p < END[2] ? kFewS : p < END[3] ? kFewC : p < END[4] ? kFewXS : kFewSums;
  }
  static constexpr int nth(int p) { return kind(p) == kFewW ? p : p - END[kind(p) - 1]; }  // its place in its kind
  // the ring: as many stages as kFewLds holds, 3 at least
  static constexpr int RING = 3 * STAGE > kFewLds ? 3 : kFewLds / STAGE < 8 ? kFewLds / STAGE : 8;
  static constexpr int LDS = RING * STAGE;
  static_assert(4 * RT * NT * 4 * 64 * 4 * (SIGNS ? 1 : 2) <= LDS, "the chains' sums and tails fit");
};

// chunk c of row r (its place in 16) is stored at place few_place(c, r) of the row's CH chunks, so that the 16 rows'
// places times 16 bytes cover the 64 banks; few_chunk is its inverse
template <int CH>
HQ_DEV int few_place(int c, int r) {
  if (CH >= 16 && CH != 24) return c ^ r;             // int8, the activations
  if (CH == 24) return (c + (r >> 1)) % 24;           // int6, 512 values
  if (CH == 12) return (c + (r >> 2)) % 12;           // int6, 256
  if (CH == 8) return c ^ ((r >> 1) & 7);             // ternary, 512
  if (CH == 4) return c ^ ((r >> 2) & 3);             // ternary, 256; binary, 512; scales of 4 steps
  return c ^ ((r >> 3) & 1);                          // binary, 256; scales of 2 steps
}
template <int CH>
HQ_DEV int few_chunk(int place, int r) {
  if (CH == 24) return (place + 24 - (r >> 1)) % 24;
  if (CH == 12) return (place + 12 - (r >> 2)) % 12;
  return few_place<CH>(place, r);
}

// a block's loads: the resources, and the lane's offset of each of the wave's pieces (wave w: pieces w, w + 4, ...; past
// the last piece it loads the last again, the same bytes to the same place, so that every wave issues LOADS loads a
// stage and one wait count serves them all).  A slot of four pieces of one kind is straight-line code; a mixed one a
// branch on the wave's number.
template <class L>
struct FewLoads {
  rsrc4 rw, rx, rs, rc, rxs;
  uint32_t off[L::LOADS];
  uint32_t sums;  // the tokens' sums after their scales
  int wave;

  static constexpr int piece(int i, int w) { return 4 * i + w < L::P ? 4 * i + w : L::P - 1; }
  static constexpr bool alike(int i) { return L::kind(piece(i, 0)) == L::kind(piece(i, 3)) && 4 * i + 3 < L::P; }
  // f(the wave's piece of slot i: its number in its kind, and the kind)
  template <typename F>
  HQ_DEV void slot(int i, F f) const {
    if (alike(i)) f(L::nth(4 * i) + wave, L::kind(4 * i));
    else if (wave == 0) f(L::nth(piece(i, 0)), L::kind(piece(i, 0)));
    else if (wave == 1) f(L::nth(piece(i, 1)), L::kind(piece(i, 1)));
    else if (wave == 2) f(L::nth(piece(i, 2)), L::kind(piece(i, 2)));
    else f(L::nth(piece(i, 3)), L::kind(piece(i, 3)));
  }

  HQ_DEV FewLoads(const Job &J, int row0, int tok0, int w) : wave(w) {
    const int lane = threadIdx.x & 63, ng = J.n >> 5;
    const int64_t rb = (int64_t)ng * 4 * L::PACK, rows = J.r1 - row0, toks = J.count - 1 - tok0;
    const int64_t sb = L::SIGNS ? (int64_t)(ng >> 2) * 2 : (int64_t)ng * 4;
    rw = few_resource(J.wq + row0 * rb, rows * rb);
    rs = few_resource(J.ws + row0 * sb, rows * sb);
    rc = few_resource(J.wc + row0 * sb, L::WC ? rows * sb : 0);
    rx = few_resource(J.xq + tok0 * J.frame, toks * J.frame + J.n);
    rxs = few_resource(J.xs + tok0 * J.sframe, toks * J.sframe + (L::SIGNS ? 8 : 4) * ng);
    sums = 4 * ng;
    // a lane's scales: the 16-byte place (WIDE) or word `at` of the rows' (tokens') places, row by row
    const auto scales = [&](int at, int lane_bytes, uint32_t stride) {
      const int place = lane_bytes == 16 ? at : at >> 2, row = place / L::SG;
      return row * stride + 16 * few_chunk<L::SG>(place % L::SG, row & 15) + (lane_bytes == 16 ? 0 : 4 * (at & 3));
    };
#pragma unroll
    for (int i = 0; i < L::LOADS; i++)
      slot(i, [&](int p, FewKind kind) {
        const int at = 64 * p + lane;
        if (kind == kFewW) {
          const int row = at / L::CH;
          off[i] = row * (uint32_t)rb + few_chunk<L::CH>(at % L::CH, row & 15) * 16;
        } else if (kind == kFewX) {
          const int tok = at / L::CHX;
          off[i] = tok * (uint32_t)J.frame + few_chunk<L::CHX>(at % L::CHX, tok & 15) * 16;
        } else if (kind == kFewXS || kind == kFewSums) {
          // (SIGNS: token at % 16 of sub-tile at / (64 SG), group at / 16 of the stage's)
          off[i] = L::SIGNS ? (16 * (at / (64 * L::SG)) + at % 16) * (uint32_t)J.sframe + 4 * (at / 16 % (4 * L::SG))
                            : scales(at, L::XLANE, (uint32_t)J.sframe);
        } else if (L::SIGNS) {
          off[i] = (16 * (at / (16 * L::SG)) + at % 16) * (uint32_t)sb + 2 * (at / 16 % L::SG);
        } else {
          off[i] = scales(at, L::SLANE, (uint32_t)sb);
        }
      });
  }

  // the resources and the wave's number are in scalar registers, and a load may read them (dma)
  HQ_DEV void settle() const {
    asm volatile("s_nop 4" :: "s"(wave), "s"(rw), "s"(rx), "s"(rs), "s"(rxs));
    if (L::WC) asm volatile("s_nop 4" :: "s"(rc));
  }

  // the wave's loads of a stage into the stage buffer at `base`; past the last stage they read nothing (sizes and
  // offsets 0; a stage's own scalar offsets are always below the sizes)
  HQ_DEV void load(uint32_t base, int stage, int stages) const {
    const int s = stage < stages ? stage : 0;
    const auto sized = [&](rsrc4 r) {
      r[2] = stage < stages ? r[2] : 0;
      return r;
    };
#pragma unroll
    for (int i = 0; i < L::LOADS; i++)
      slot(i, [&](int p, FewKind kind) {
        if (kind == kFewW) dma<16>(sized(rw), base + L::W + 1024 * p, off[i], s * L::WROW);
        else if (kind == kFewX) dma<16>(sized(rx), base + L::X + 1024 * p, off[i], s * L::KS);
        else if (kind == kFewXS) dma<L::XLANE>(sized(rxs), base + L::XS + 64 * L::XLANE * p, off[i], s * L::SG * 16);
        else if (kind == kFewSums)
          dma<L::XLANE>(sized(rxs), base + L::SUMS + 64 * L::XLANE * p, off[i], stage < stages ? s * L::SG * 16 + sums : 0);
        else if (L::SIGNS) dma<2>(sized(rs), base + L::S + 256 * p, off[i], s * L::SG * 2);
        else if (kind == kFewS) dma<L::SLANE>(sized(rs), base + L::S + 64 * L::SLANE * p, off[i], s * L::SG * 16);
        else dma<L::SLANE>(sized(rc), base + L::C + 64 * L::SLANE * p, off[i], s * L::SG * 16);
      });
  }
};

HQ_DEV long few_pair(uint32_t a, uint32_t b) { return (long)(((uint64_t)b << 32) | a); }

// LDS at a byte address
template <typename T>
HQ_DEV T few_lds(uint32_t at) { return *(const __attribute__((address_space(3))) T *)(uintptr_t)at; }

// The lane's offsets in a stage buffer, step by step, made once (opaque to the compiler, which would otherwise make
// them again every stage): its 8 bytes of the weights' row r (int6: its 8 bytes of nibbles, then of top bits), of the
// activations of token r, its row's scale and the scale of token 4 q.  Sub-tiles and the tokens 4 q + i lie at constant
// distances from these.
template <class L>
struct FewLane {
  static constexpr int NW = L::PACK == 6 ? 2 : 1;
  uint32_t w[L::SG][NW], x[L::SG], s[L::SG], xs[L::SG];
  HQ_DEV FewLane(int k, int lane) {
    const int q = lane >> 4, r = lane & 15;
    const auto weights = [&](int piece) {  // the 8-byte piece of the stage's row
      return (uint32_t)(L::W + r * L::WROW + 16 * few_place<L::CH>(piece >> 1, r) + 8 * (piece & 1));
    };
#pragma unroll
    for (int j = 0; j < L::SG; j++) {
      if (L::PACK == 8) w[j][0] = weights(16 * j + 4 * k + q);
      else if (L::PACK == 2) w[j][0] = weights(4 * j + k);               // part k's 8 code bytes (every quarter's)
      else if (L::PACK == 1) w[j][0] = weights(2 * j + (k & 1));         // bytes 8 (k & 1) .. of the group
      else w[j][0] = weights(12 * j + 3 * k + (q & 1)), w[j][NW - 1] = weights(12 * j + 3 * k + 2);
      // int8 / int6: bytes 8 q .. of the group; ternary / binary: 8 bytes of plane q of the part's half of its block
      const int c = L::SIGNS ? 8 * j + 4 * (k >> 1) + q : 8 * j + 2 * k + (q >> 1), half = L::SIGNS ? k & 1 : q & 1;
      x[j] = (uint32_t)(L::X + r * L::KS + 16 * few_place<L::CHX>(c, r) + 8 * half);
      s[j] = (uint32_t)(L::S + (L::SIGNS ? (j * 16 + r) * 4 : (r * L::SG + few_place<L::SG>(j, r)) * 16 + 4 * k));
      xs[j] = (uint32_t)(L::XS + (L::SIGNS ? (4 * j + k) * 64 + 16 * q : (4 * q * L::SG + few_place<L::SG>(j, 4 * q)) * 16 + 4 * k));
#pragma unroll
      for (int e = 0; e < NW; e++) asm volatile("" : "+v"(w[j][e]));
      asm volatile("" : "+v"(x[j]), "+v"(s[j]), "+v"(xs[j]));
    }
  }
};

// a stage's operands of a wave
template <class L>
struct FewOps {
  v2u w[L::SG][L::RT][2];
  uint32_t ws[L::SG][L::RT];
  int32_t wc[L::SG][L::RT];
  v2u x[L::SG][L::NT];
  v4f xs[L::SG][L::NT];
  v4i sum[L::SG][L::NT];
  HQ_DEV void read(const FewLane<L> &at, uint32_t st) {
#pragma unroll
    for (int j = 0; j < L::SG; j++) {
#pragma unroll
      for (int rt = 0; rt < L::RT; rt++)
#pragma unroll
        for (int e = 0; e < FewLane<L>::NW; e++) w[j][rt][e] = few_lds<v2u>(at.w[j][e] + st + 16 * rt * L::WROW);
#pragma unroll
      for (int nt = 0; nt < L::NT; nt++) x[j][nt] = few_lds<v2u>(at.x[j] + st + 16 * nt * L::KS);
#pragma unroll
      for (int rt = 0; rt < L::RT; rt++) {
        const uint32_t row = at.s[j] + st + (L::SIGNS ? rt * L::SG * 64 : 16 * rt * L::SG * 16);
        ws[j][rt] = few_lds<uint32_t>(row);
        if (L::WC) wc[j][rt] = few_lds<int32_t>(row + (L::C - L::S));
      }
#pragma unroll
      for (int nt = 0; nt < L::NT; nt++) {
        if (L::SIGNS) {
          const uint32_t toks = at.xs[j] + st + nt * L::SG * 256;
          xs[j][nt] = few_lds<v4f>(toks);
          sum[j][nt] = few_lds<v4i>(toks + (L::SUMS - L::XS));
          continue;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) xs[j][nt][i] = few_lds<float>(at.xs[j] + st + (16 * nt + i) * L::SG * 16);
      }
    }
  }
};

// those 8 values: the MFMA's K order is the group's own (int8, int6), or plane q of the part's 8 bytes (ternary,
// binary), against the activations' bytes in the same order
template <class L>
HQ_DEV long few_values(const v2u v[2], int k, int q) {
  if (L::PACK == 8) return few_pair(v[0].x, v[0].y);
  if (L::PACK == 6) {
    const int sl = 4 * (q >> 1), su = 2 * q;
    return few_pair((((v[0].x >> sl) & 0x0f0f0f0fu) << 2) | (((v[1].x >> su) & 0x03030303u) << 6),
                    (((v[0].y >> sl) & 0x0f0f0f0fu) << 2) | (((v[1].y >> su) & 0x03030303u) << 6));
  }
  if (L::PACK == 2) return few_pair((v[0].x >> (2 * q)) & 0x03030303u, (v[0].y >> (2 * q)) & 0x03030303u);
  const int b = 4 * (k >> 1) + q;
  return few_pair(((v[0].x >> b) & 0x01010101u) << 1, ((v[0].y >> b) & 0x01010101u) << 1);
}

// chain k's SG steps of a stage: the MFMAs, then term(j, rt, nt, i, value) of each step j's float32 terms (row r of
// sub-tile rt, token 4 q + i of token sub-tile nt)
template <class L, typename Term>
HQ_DEV void few_terms(const FewOps<L> &o, int k, int q, Term term) {
  constexpr int RT = L::RT, NT = L::NT, SG = L::SG;
  const v4i zero = {0, 0, 0, 0};
  v4i d[SG][RT][NT];
#pragma unroll
  for (int j = 0; j < SG; j++)
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      const long w = few_values<L>(o.w[j][rt], k, q);
      v4i cin = zero;
      if (L::WC) cin = (v4i){o.wc[j][rt], o.wc[j][rt], o.wc[j][rt], o.wc[j][rt]};
      else if (!L::SIGNS) cin = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)0xc0c0c0c0c0c0c0c0ull, w, zero, 0, 0, 0);
#pragma unroll
      for (int nt = 0; nt < NT; nt++) {
        if (L::SIGNS) cin = o.sum[j][nt];
        d[j][rt][nt] = __builtin_amdgcn_mfma_i32_16x16x32_i8(few_pair(o.x[j][nt].x, o.x[j][nt].y), w, cin, 0, 0, 0);
      }
    }
#pragma unroll
  for (int j = 0; j < SG; j++)
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
      const float ws = L::SIGNS ? half_to_float(o.ws[j][rt]) : __uint_as_float(o.ws[j][rt]);
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float f = (float)d[j][rt][nt][i], xs = o.xs[j][nt][i];
          term(j, rt, nt, i, L::SIGNS ? fmul(fmul(f, xs), ws) : fmul(f, fmul(ws, xs)));
        }
    }
}

constexpr int kFewThreads = 256;
template <class L>
__global__ __launch_bounds__(kFewThreads, 2) void gemm_few(FewBatch batch) {
  constexpr int RT = L::RT, NT = L::NT;
  __shared__ __attribute__((aligned(1024))) char lds[L::LDS];
  int jb = 0;
#pragma unroll
  for (int i = 1; i < kMaxJobs; i++) jb += (int)blockIdx.x >= batch.block0[i] ? 1 : 0;
  const Job &J = batch.job[jb];
  const int M = J.count, ng = J.n >> 5;
  // the blocks of one XCD (every eighth) take consecutive tiles, the token tiles of a row tile one after the other, so
  // that they read its weights from that XCD's L2
  const int blk = (int)blockIdx.x - batch.block0[jb], nb = batch.blocks[jb], x8 = blk % kXcds;
  const int tile = x8 * (nb / kXcds) + min(x8, nb % kXcds) + blk / kXcds;
  const int ntt = (M + 16 * NT - 1) / (16 * NT);
  const int row0 = J.r0 + tile / ntt * 16 * RT, tok0 = tile % ntt * 16 * NT;
  const int lane = threadIdx.x & 63, k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int steps = ng >> 2, tail = L::SIGNS ? 0 : ng & 3;  // whole steps; the groups past the fours
  const int stages = (steps + (tail ? 1 : 0) + L::SG - 1) / L::SG;

  const uint32_t lds0 = lds_addr(lds);
  const FewLoads<L> loads(J, row0, tok0, k);
  loads.settle();
#pragma unroll
  for (int s = 0; s < L::RING - 1; s++) loads.load(lds0 + s * L::STAGE, s, stages);
  float acc[RT][NT][4], last[RT][NT][4];  // the chain's sums; the term of the group past the fours (chains k < tail)
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int i = 0; i < 4; i++) acc[rt][nt][i] = last[rt][nt][i] = 0.0f;
  // a stage's operands are read while the stage before it is folded
  const FewLane<L> at(k, lane);
  const int q = lane >> 4;
  uint32_t cur = lds0;
  uint32_t next = lds0 + (L::RING - 1) * L::STAGE;
  const auto read = [&](FewOps<L> &o, int s) {
    // stage s landed everywhere, and every wave has read stage s - 1, whose buffer takes stage s + RING - 1
    stage_ready<(L::RING - 2) * L::LOADS>();
    loads.load(next, s + L::RING - 1, stages);
    next = cur;
    o.read(at, cur);
    cur = cur + L::STAGE == lds0 + L::LDS ? lds0 : cur + L::STAGE;
    if (L::PIPE) __builtin_amdgcn_sched_barrier(0);
  };
  const auto fold = [&](const FewOps<L> &o) {
    few_terms<L>(o, k, q, [&](int j, int rt, int nt, int i, float t) { acc[rt][nt][i] = fadd(acc[rt][nt][i], t); });
  };
  const auto finish = [&](const FewOps<L> &o, int s) {  // the last stage: its steps may end early, and hold the tail
    few_terms<L>(o, k, q, [&](int j, int rt, int nt, int i, float t) {
      if (s * L::SG + j < steps) acc[rt][nt][i] = fadd(acc[rt][nt][i], t);
      else if (s * L::SG + j == steps) last[rt][nt][i] = t;
    });
  };
  FewOps<L> a, b;
  if (!L::PIPE) {
    for (int s = 0; s < stages; s++) {
      read(a, s);
      if (s + 1 < stages) fold(a);
      else finish(a, s);
    }
  } else {
    read(a, 0);
    for (int s = 0;; s += 2) {
      if (s + 1 == stages) {
        finish(a, s);
        break;
      }
      read(b, s + 1);
      fold(a);
      if (s + 2 == stages) {
        finish(b, s + 1);
        break;
      }
      read(a, s + 2);
      fold(b);
    }
  }
  // ((l0 + l1) + l2) + l3, then the groups past the fours one at a time (math.ts:7-9, relaxed/int8.ts:40-47): the
  // chains' values through LDS, wave i adding and storing the tokens 4 q + i of every sub-tile
  stage_ready<0>();
  float *sums = (float *)lds, *tails = sums + 4 * RT * NT * 4 * 64;  // [chain][value][lane]
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int at = ((k * RT + rt) * NT + nt) * 4 + i;
        sums[at * 64 + lane] = acc[rt][nt][i];
        if (k < tail) tails[at * 64 + lane] = last[rt][nt][i];
      }
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      const auto value = [&](const float *of, int chain) { return of[(((chain * RT + rt) * NT + nt) * 4 + k) * 64 + lane]; };
      float v = fadd(fadd(fadd(value(sums, 0), value(sums, 1)), value(sums, 2)), value(sums, 3));
      for (int t = 0; t < tail; t++) v = fadd(v, value(tails, t));
      const int row = row0 + 16 * rt + (lane & 15), tok = tok0 + 16 * nt + 4 * (lane >> 4) + k;
      if (row < J.r1 && tok < M) ((float *)(J.out + tok * J.os))[row] = v;
    }
}

template <class L>
hipError_t launch_few_of(const Job *jobs, int32_t njobs, hipStream_t s) {
  FewBatch b{};
  int64_t blocks = 0;
  for (int j = 0; j < kMaxJobs; j++) b.block0[j] = INT32_MAX;
  for (int j = 0; j < njobs; j++) {
    b.job[j] = jobs[j];
    b.block0[j] = (int32_t)blocks;
    const int64_t rows = (jobs[j].r1 - jobs[j].r0 + 16 * L::RT - 1) / (16 * L::RT);
    b.blocks[j] = (int32_t)(rows * ((jobs[j].count + 16 * L::NT - 1) / (16 * L::NT)));
    blocks += b.blocks[j];
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((gemm_few<L>), dim3((uint32_t)blocks), dim3(kFewThreads), 0, s, b);
  return hipGetLastError();
}

// The tile of a pack: 16 rows of int8 / int6; 32 of ternary / binary, whose activations are four to eight times their
// weights' bytes (the 27B ternary MLP at 64 tokens 217 -> 153 us; int8's 8B layer with 32 rows 80 -> 99 us at 16 tokens).
// Token sub-tiles: at most what keeps two waves a SIMD without spills.
constexpr int few_rows(int pack) { return pack <= 2 ? 2 : 1; }
constexpr int few_most(int pack) { return pack <= 2 ? 2 : pack == 6 ? 3 : 4; }

template <int PACK, bool WC, bool WIDE>
hipError_t launch_few_tile(const Job *jobs, int32_t njobs, hipStream_t s) {
  constexpr int RT = few_rows(PACK), MOST = few_most(PACK);
  const int subs = (jobs[0].count + 15) / 16, tiles = (subs + MOST - 1) / MOST, nt = (subs + tiles - 1) / tiles;
  if constexpr (MOST >= 4)
    if (nt == 4) return launch_few_of<Few<PACK, WC, WIDE, RT, 4>>(jobs, njobs, s);
  if constexpr (MOST >= 3)
    if (nt == 3) return launch_few_of<Few<PACK, WC, WIDE, RT, 3>>(jobs, njobs, s);
  return nt == 2 ? launch_few_of<Few<PACK, WC, WIDE, RT, 2>>(jobs, njobs, s) : launch_few_of<Few<PACK, WC, WIDE, RT, 1>>(jobs, njobs, s);
}

// Row steps of few tiles, measured: us per 1000 values of a row with 1, 2 (, 3) blocks of the tile on a compute unit, as many
// as its LDS and registers let in, by token sub-tiles (further blocks wait their turn); and what a launch takes besides,
// and for each block on a unit
struct FewCost {
  double start, block;
  double step[4][3];
};
constexpr FewCost kFewInt8{4.5, 1.2, {{1.05, 1.95}, {1.9, 2.95}, {2.45, 3.8}, {3.05, 4.65}}};
constexpr FewCost kFewInt6{4.5, 1.8, {{1.42, 1.92}, {2.6, 3.2, 4.6}, {3.15, 4.0}}};
constexpr FewCost kFewSigns{2.5, 0.0, {{1.85, 2.4, 3.5}, {4.25, 5.05, 6.45}}};

// every job's scales in 16-byte runs a step (Few's WIDE)
bool few_wide(const Job *jobs, int32_t njobs) {
  uintptr_t bits = 0;
  for (int j = 0; j < njobs; j++) {
    const Job &q = jobs[j];
    bits |= (uintptr_t)q.xs | (uintptr_t)(q.count > 1 ? q.sframe : 0) | (uintptr_t)q.ws | (uintptr_t)q.wc | (uintptr_t)(q.n >> 3);
  }
  return bits % 16 == 0;
}

template <int PACK, bool WC>
hipError_t launch_few_pack(const Job *jobs, int32_t njobs, hipStream_t s) {
  if constexpr (PACK > 2)
    if (!few_wide(jobs, njobs)) return launch_few_tile<PACK, WC, false>(jobs, njobs, s);
  return launch_few_tile<PACK, WC, true>(jobs, njobs, s);
}

}  // namespace

double few_us(Kind kind, const Job *jobs, int32_t njobs) {
  const bool signs = signs_kind(kind);
  const int pack = signs ? 2 : kind == Q8R ? 8 : 6, rt = few_rows(pack), most = few_most(pack);
  const int subs = (jobs[0].count + 15) / 16, tiles = (subs + most - 1) / most, nt = (subs + tiles - 1) / tiles;
  int64_t blocks = 0, n = 0;
  for (int j = 0; j < njobs; j++) {
    blocks += (int64_t)((jobs[j].r1 - jobs[j].r0 + 16 * rt - 1) / (16 * rt)) * tiles;
    if (jobs[j].n > n) n = jobs[j].n;
  }
  const FewCost &c = signs ? kFewSigns : pack == 8 ? kFewInt8 : kFewInt6;
  const double *step = c.step[nt - 1];
  const int64_t each = (blocks + cu_count() - 1) / cu_count(), in = step[2] > 0 ? 3 : 2;
  const double rest = c.block * (double)each +
                      0.001 * (double)n * ((double)(each / in) * step[in - 1] + (each % in ? step[each % in - 1] : 0.0));
  // (scales loaded 4 bytes a lane cost these tiles 9 % more, the prompt tiles nothing: int8 with wc, 17740 rows of 288 values at 76
  // tokens 23 us here, 13 there; the token kernel's rows of such lengths are slower too)
  return c.start + (!signs && jobs[0].count >= 16 && !few_wide(jobs, njobs) ? 1.09 : 1.0) * rest;
}

hipError_t launch_few(Kind kind, const Job *jobs, int32_t njobs, hipStream_t s) {
  if (njobs < 1 || njobs > kMaxJobs) return hipErrorInvalidValue;
  const bool wc = jobs[0].wc != nullptr;
  switch (kind) {
  case Q8R: return wc ? launch_few_pack<8, true>(jobs, njobs, s) : launch_few_pack<8, false>(jobs, njobs, s);
  case Q6R: return wc ? launch_few_pack<6, true>(jobs, njobs, s) : launch_few_pack<6, false>(jobs, njobs, s);
  case T2R:
  case T2: return launch_few_pack<2, false>(jobs, njobs, s);
  case B1R:
  case B1: return launch_few_pack<1, false>(jobs, njobs, s);
  default: return hipErrorNotSupported;
  }
}

}  // namespace hq
