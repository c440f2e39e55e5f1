// q4k.hip — a few tokens or a prompt of Q4_K blocks on the matrix cores (matmul_sbr_tile, kernels/blocks/tile.ts:144-147):
// every (row, token) the token kernel's number to the bit, as blocks.hip's tile.
//
// A block of 4 waves computes R rows x NT tokens; wave k is the reference's lane k, which adds for every block of 256
// weights in order f(f(f(f(G_k xs_k) + f(G_{k+4} xs_{k+4})) F) - f(f(f(M_k V_k xs_k) + f(M_{k+4} V_{k+4} xs_{k+4})) Fm))
// (kernels/blocks/types.ts:48-57), G the group's S times its exact integer (an MFMA of T x T outputs, T 32 or 16: A
// the tokens, B the rows, K the group's 32), V the sum of its 32 activations (M V is exact in float32: below 2^18).  The
// lanes meet in LDS at the end, ((l0 + l1) + l2) + l3.
//
// Unlike the other types' tile, which decodes the rows' blocks into int8 tiles in LDS between two barriers, a wave
// takes its groups' nibbles straight from the raw blocks into the matrix core's operand: 8 VALU operations a group and
// 32 rows, for 16 VALU operations an output and pair of groups.  So a step has no decode, one barrier, and the next
// block's bytes (in registers while this one is multiplied) go into the other of two buffers.
//
// Measured (the 8B gate/up and down through hq_matmuls, us, before: 4 tokens a launch of the token kernel below 16
// tokens, blocks.hip's tile from 16): 4 tokens 108 -> 63, 15 tokens 353 -> 64, 16 tokens 187 -> 64, 32 tokens 190 -> 85,
// 64 tokens 254 -> 111, 333 tokens 916 -> 459, 512 tokens 1127 -> 644 (160 -> 280 TOPS), passes back to back (a few after an idle
// second: 720 to 795).  Of that, S times the integer as a float32 product instead of v_mul_i32_i24, which issues slower: 333
// tokens 521 -> 477, 512 tokens 728 -> 672 when it was brought in.
// What bounds a prompt: those 16 operations, 563 of a SIMD's cycles a pair and 32 x 32 outputs, beside 64 of the matrix
// cores' (which add on this part: 459 TOPS at 2.2 GHz), and per step of a wave ~60 operations of scales and operands.
// A few tokens: the steps' latency, one after the other down a row (56 steps of the down projection, 0.6 us each).
// Tried: two to four blocks ahead in registers (as fast at few tokens, 3-25 % slower for prompts), 64 rows a block (15-20 %
// slower), 64 tokens (2 % faster at 512 tokens, 2-60 % slower below).
#include "common.hpp"
#include "launch.hpp"
#include "stage.hpp"

namespace hq {

namespace {

typedef int32_t v2i __attribute__((ext_vector_type(2)));
typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t v16i __attribute__((ext_vector_type(16)));

struct Q4kBatch {
  Job job[kMaxJobs];
  int32_t block0[kMaxJobs];  // the first block of each job (INT32_MAX past the last)
  int32_t blocks[kMaxJobs];
};

constexpr int kQ4kBytes = 144;
template <int R, int NT>
struct Q4k {
  static constexpr int PITCH = 256 + 16;         // a token's 256 bytes (16 tokens' 16-byte reads in different banks)
  static constexpr int RAW = 0;                  // [R][144]
  static constexpr int X = R * kQ4kBytes;        // int8 [NT][PITCH]
  static constexpr int XS = X + NT * PITCH;      // float [8][NT]
  static constexpr int V = XS + 8 * NT * 4;      // float [8][NT]
  static constexpr int SIZE = V + 8 * NT * 4;
  // 16-byte loads a thread: the tokens' bytes, the rows' blocks (and one of the tokens' scales and sums of 16)
  static constexpr int XU = NT * 16 / 256, RU = (R * 9 + 255) / 256;
  static_assert(4 * NT * 32 * 4 <= 2 * SIZE, "the lanes' sums of T rows fit");
};

template <int R, int NT>
struct Q4kLoads {
  using L = Q4k<R, NT>;
  v4i x[L::XU], aux, raw[L::RU];
  // block b's bytes
  HQ_DEV void load(const Job &J, __amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rw, int b) {
    const int tid = threadIdx.x, n = J.n;
    const int frame = (int)J.frame, sframe = (int)J.sframe, row_bytes = (n >> 8) * kQ4kBytes;
#pragma unroll
    for (int u = 0; u < L::XU; u++) {
      const int i = tid + 256 * u;
      x[u] = __builtin_amdgcn_raw_buffer_load_b128(rx, (i >> 4) * frame + 16 * (i & 15), 256 * b, 0);
    }
    const int a = tid < 4 * NT ? tid : 0, part = a & 3;  // a token's scales (parts 0, 1), sums of 16 (2, 3)
    aux = __builtin_amdgcn_raw_buffer_load_b128(ra, (a >> 2) * sframe + 16 * (part & 1) + (part & 2 ? n >> 3 : 0), 32 * b, 0);
#pragma unroll
    for (int u = 0; u < L::RU; u++) {
      const int i = tid + 256 * u, r = i / 9;
      raw[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, (r < R ? r : 0) * row_bytes + 16 * (i - 9 * r), kQ4kBytes * b, 0);
    }
  }
  HQ_DEV void store(char *lds) const {
    const int tid = threadIdx.x;
#pragma unroll
    for (int u = 0; u < L::XU; u++) {
      const int i = tid + 256 * u;
      *(v4i *)(lds + L::X + (i >> 4) * L::PITCH + 16 * (i & 15)) = x[u];
    }
    if (tid < 4 * NT) {
      const int tok = tid >> 2, part = tid & 3;
      uint32_t *to = (uint32_t *)(lds + (part & 2 ? L::V : L::XS)) + 4 * (part & 1) * NT + tok;
      const uint32_t sums = 0u - (uint32_t)(part >> 1);  // (a mask, not a branch an element)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        // two int16 sums of 16: the group's sum of 32
        const int32_t sum = (int32_t)(int16_t)(aux[i] & 0xffff) + (aux[i] >> 16);
        to[i * NT] = (__float_as_uint((float)sum) & sums) | ((uint32_t)aux[i] & ~sums);
      }
    }
#pragma unroll
    for (int u = 0; u < L::RU; u++) {
      const int i = tid + 256 * u;
      if (i < 9 * R) *(v4i *)(lds + L::RAW + 16 * i) = raw[u];
    }
  }
};

template <int T> struct Q4kMfma;
template <> struct Q4kMfma<32> {
  typedef v4i op;  // a lane's 16 values: K half lane / 32 of row (token) lane % 32
  typedef v16i out;  // register r: token 8 (r / 4) + 4 (lane / 32) + r % 4, row lane % 32
  static HQ_DEV out dot(op a, op b) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, (out){}, 0, 0, 0); }
};
template <> struct Q4kMfma<16> {
  typedef v2i op;  // a lane's 8 values: K quarter lane / 16 of row (token) lane % 16
  typedef v4i out;  // register r: token 4 (lane / 16) + r, row lane % 16
  static HQ_DEV out dot(op a, op b) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), (out){}, 0, 0, 0);
  }
};

template <int T, int R, int NT>
__global__ __launch_bounds__(256, 2) void gemm_q4k(Q4kBatch batch) {
  using L = Q4k<R, NT>;
  using X = Q4kMfma<T>;
  using Op = typename X::op;
  constexpr int RS = R / T, TS = NT / T, REGS = T * T / 64, W = T / 8;  // W: an operand's dwords
  __shared__ __attribute__((aligned(16))) char lds[2 * L::SIZE];
  int jb = 0;
#pragma unroll
  for (int i = 1; i < kMaxJobs; i++) jb += (int)blockIdx.x >= batch.block0[i] ? 1 : 0;
  const Job &J = batch.job[jb];
  // the blocks of one XCD (every eighth) take consecutive tiles, a row tile's token tiles one after the other
  const int blk = (int)blockIdx.x - batch.block0[jb], nb = batch.blocks[jb], x8 = blk % kXcds;
  const int tile = x8 * (nb / kXcds) + min(x8, nb % kXcds) + blk / kXcds;
  const int ntt = (J.count + NT - 1) / NT;
  const int r0 = J.r0 + tile / ntt * R, t0 = tile % ntt * NT;
  const int blocks = J.n >> 8;
  const int64_t row_bytes = (int64_t)blocks * kQ4kBytes, toks = (int64_t)J.count - 1 - t0;
  // (rows and tokens past the job's read zeros and are not stored)
  const __amdgpu_buffer_rsrc_t rx = resource(J.xq + t0 * J.frame, toks * J.frame + J.n);
  const __amdgpu_buffer_rsrc_t ra = resource(J.xs + t0 * J.sframe, toks * J.sframe + (J.n >> 2));
  const __amdgpu_buffer_rsrc_t rw = resource(J.wq + r0 * row_bytes, (J.r1 - r0) * row_bytes);
  const int lane = threadIdx.x & 63, sub = lane / T, at = lane % T;
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  float acc[RS][TS][REGS];
#pragma unroll
  for (int sp = 0; sp < RS; sp++)
#pragma unroll
    for (int h = 0; h < TS; h++)
#pragma unroll
      for (int r = 0; r < REGS; r++) acc[sp][h][r] = 0.0f;
  Q4kLoads<R, NT> loads;
  loads.load(J, rx, ra, rw, 0);
  loads.store(lds);
  __syncthreads();
  for (int b = 0; b < blocks; b++) {
    const char *st = lds + (b & 1) * L::SIZE;
    const bool more = b + 1 < blocks;
    if (more) loads.load(J, rx, ra, rw, b + 1);
    // the rows' operands of groups k and k + 4: the nibbles, S, M, and the blocks' F and Fm
    Op B[RS][2];
    float S[RS][2], M[RS][2], F[RS], Fm[RS];
#pragma unroll
    for (int sp = 0; sp < RS; sp++) {
      const char *row = st + L::RAW + (T * sp + at) * kQ4kBytes;
      const uint4 head = *(const uint4 *)row;
      const char *nibbles = row + 16 + 32 * (k >> 1) + T / 2 * sub;
      const Op w0 = *(const Op *)nibbles, w1 = *(const Op *)(nibbles + 64);
      const int sh = 4 * (k & 1);
#pragma unroll
      for (int i = 0; i < W; i++) {
        B[sp][0][i] = (int32_t)(((uint32_t)w0[i] >> sh) & 0x0f0f0f0fu);
        B[sp][1][i] = (int32_t)(((uint32_t)w1[i] >> sh) & 0x0f0f0f0fu);
      }
      // bytes 4 + k, 8 + k, 12 + k: group k's S and M in the low six bits of the first two, group k + 4's low four bits
      // in the third's halves and their top two above those (types.ts:230-232)
      const uint32_t s = head.y >> (8 * k), m = head.z >> (8 * k), hi = head.w >> (8 * k);
      S[sp][0] = (float)(s & 63);
      S[sp][1] = (float)((hi & 15) | ((s >> 2) & 48));
      M[sp][0] = (float)(m & 63);
      M[sp][1] = (float)(((hi >> 4) & 15) | ((m >> 2) & 48));
      F[sp] = half_to_float(head.x & 0xffff);
      Fm[sp] = half_to_float(head.x >> 16);
    }
#pragma unroll
    for (int h = 0; h < TS; h++) {
      const char *tok = st + L::X + (T * h + at) * L::PITCH + 32 * k + T / 2 * sub;
      const Op A0 = *(const Op *)tok, A1 = *(const Op *)(tok + 128);
      const float *xs = (const float *)(st + L::XS) + T * h + 4 * sub, *v = (const float *)(st + L::V) + T * h + 4 * sub;
      typename X::out C[RS][2];
#pragma unroll
      for (int sp = 0; sp < RS; sp++) {
        C[sp][0] = X::dot(A0, B[sp][0]);
        C[sp][1] = X::dot(A1, B[sp][1]);
      }
#pragma unroll
      for (int m = 0; m < REGS / 4; m++) {
        const float4 x0 = *(const float4 *)(xs + k * NT + 8 * m), x1 = *(const float4 *)(xs + (k + 4) * NT + 8 * m);
        const float4 v0 = *(const float4 *)(v + k * NT + 8 * m), v1 = *(const float4 *)(v + (k + 4) * NT + 8 * m);
        const float xa[4] = {x0.x, x0.y, x0.z, x0.w}, xb[4] = {x1.x, x1.y, x1.z, x1.w};
        const float va[4] = {v0.x, v0.y, v0.z, v0.w}, vb[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int sp = 0; sp < RS; sp++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int r = 4 * m + i;
            // (S times the integer is exact in float32: below 2^22)
            const float g = fadd(fmul(fmul(S[sp][0], (float)C[sp][0][r]), xa[i]), fmul(fmul(S[sp][1], (float)C[sp][1][r]), xb[i]));
            const float least = fadd(fmul(fmul(M[sp][0], va[i]), xa[i]), fmul(fmul(M[sp][1], vb[i]), xb[i]));
            acc[sp][h][r] = fadd(acc[sp][h][r], fsub(fmul(g, F[sp]), fmul(least, Fm[sp])));
            // (kept here: the compiler would sink the folds of every token half past the next block's stores, and spill)
            asm volatile("" : "+v"(acc[sp][h][r]));
          }
      }
    }
    if (more) loads.store(lds + ((b + 1) & 1) * L::SIZE);
    __syncthreads();
  }
  // ((l0 + l1) + l2) + l3 (math.ts:7-9), T rows at a time: wave w adds and stores a quarter of each lane's values
  float *sums = (float *)lds;
  constexpr int VALUES = TS * REGS;
#pragma unroll
  for (int sp = 0; sp < RS; sp++) {
#pragma unroll
    for (int h = 0; h < TS; h++)
#pragma unroll
      for (int r = 0; r < REGS; r++) sums[(k * VALUES + REGS * h + r) * 64 + lane] = acc[sp][h][r];
    __syncthreads();
    const int row = r0 + T * sp + at;
#pragma unroll
    for (int e = 0; e < VALUES / 4; e++) {
      const int which = VALUES / 4 * k + e, r = which % REGS;
      const auto of = [&](int c) { return sums[(c * VALUES + which) * 64 + lane]; };
      const int t = t0 + T * (which / REGS) + 8 * (r >> 2) + 4 * sub + (r & 3);
      const float v = fadd(fadd(fadd(of(0), of(1)), of(2)), of(3));
      if (row < J.r1 && t < J.count) ((float *)(J.out + t * J.os))[row] = v;
    }
    __syncthreads();
  }
}

template <int T, int R, int NT>
hipError_t launch_q4k_of(const Job *jobs, int32_t njobs, hipStream_t s) {
  Q4kBatch b{};
  int64_t blocks = 0;
  for (int j = 0; j < kMaxJobs; j++) b.block0[j] = INT32_MAX;
  for (int j = 0; j < njobs; j++) {
    b.job[j] = jobs[j];
    b.block0[j] = (int32_t)blocks;
    b.blocks[j] = (int32_t)((int64_t)((jobs[j].r1 - jobs[j].r0 + R - 1) / R) * ((jobs[j].count + NT - 1) / NT));
    blocks += b.blocks[j];
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL((gemm_q4k<T, R, NT>), dim3((uint32_t)blocks), dim3(256), 0, s, b);
  return hipGetLastError();
}

}  // namespace

// The jobs these tiles take: Q4_K whose blocks start on 16 bytes, three tokens or more (two: 63 us in the token kernel
// against 68 for the 8B gate/up and down), offsets within a tile in 32 bits.
bool q4k_tile(const Job &j) {
  return j.type == 12 && j.count >= 3 && ((uintptr_t)j.wq & 15) == 0 && j.frame > 0 && j.sframe > 0 &&
         j.frame < kSbTileFrameMax && j.sframe < kSbTileFrameMax && (int64_t)32 * (j.n >> 8) * kQ4kBytes < INT32_MAX;
}

// us per 1000 values of a row with one block of 16 rows x 16 tokens on a compute unit; another on it adds a fifth of that, and
// past four (resident together) they take 0.8 each
double q4k_us(int64_t n, int64_t blocks) {
  const int64_t cus = cu_count(), each = (blocks + cus - 1) / cus;
  const double some = 2.48 + 0.55 * (double)(each - 1), many = 0.8 * (double)each;
  return 0.001 * (double)n * (some > many ? some : many);
}

// 16 x 16 tiles up to 32 tokens and for launches whose 32 x 32 tiles are fewer than one and a half a compute unit (a step
// is a quarter as long, and four times the blocks share the chip: the 8B gate/up and down at 16 tokens 107 -> 67 us, at
// 64 the down projection 64 -> 58, a 1024-wide model's at 64 28 -> 23); 32 x 32 otherwise (64 tokens of the 8B gate/up 87 ->
// 70 us, 512 tokens 640 -> 466)
hipError_t launch_q4k(const Job *jobs, int32_t njobs, hipStream_t s) {
  if (njobs < 1 || njobs > kMaxJobs) return hipErrorInvalidValue;
  int64_t tiles = 0;
  for (int j = 0; j < njobs; j++) tiles += (int64_t)((jobs[j].r1 - jobs[j].r0 + 31) / 32) * ((jobs[j].count + 31) / 32);
  return jobs[0].count <= 32 || 2 * tiles < 3 * (int64_t)cu_count() ? launch_q4k_of<16, 16, 16>(jobs, njobs, s)
                                                                   : launch_q4k_of<32, 32, 32>(jobs, njobs, s);
}

}  // namespace hq
