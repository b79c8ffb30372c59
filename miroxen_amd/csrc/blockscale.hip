// MXFP8 block-scaled GEMM for gfx950: quantizer + GEMM on the MX-scaled MFMA.
// Reference: src/kernels/blockscale.{h,cu} (quantize_blockscaled :113-131,
// quant_kernel MXFP8 branch :69-108, gemm_blockscaled :134-216 on cuBLASLt).
//
// Format (OCP MX, the reference's MXFP8): e4m3 data, one power-of-two scale (UE8M0)
// per 32 consecutive K values of a row. gfx950's v_mfma_scale_f32_32x32x64_f8f6f4
// consumes exactly that: lane half h supplies the UE8M0 scale of K block h of each
// 64-value MFMA step (selected per operand by op_sel); see the operand layout note
// in mxfp8_gemm.
//
// Scale layout: the reference's 128 x 4 interleave (quantizer blockscale.cu:82,
// decoder tests/blockscale_test.cpp:15-17): scale (r, kb) at byte
// (r / 128) kbp 128 + (kb / 4) 512 + (r % 32) 16 + ((r % 128) / 32) 4 + kb % 4,
// kbp = K/32 rounded up to 4, rows padded to 128 (the reference's qscale_bytes size).
// The quantizer writes 127 (= 1.0) into every padding byte, so padded K blocks and
// rows contribute 0 (data 0 times a finite scale) instead of 0 x NaN (0xFF).
//
// GEMM (Y[M,N] bf16 = X[M,K] W[N,K]^T, both K-major): the largest tiles are 256 n x 256 m per
// 4-wave work-group, one wave per SIMD, each wave 128 n x 128 m = 4 x 4 MFMA blocks
// of 32 x 32 (C = W X^T: lane = one m column, 16 n rows; the 256 fp32 accumulators
// live in AGPRs). K advances in stages of 128 bytes DMA'd into LDS
// (buffer_load ... lds, 1 KB per op, rows past the matrix read as zeros), in a ring of
// slots; LDS rows are 128 B with their 16-byte chunks XOR'd by (row >> 1) & 7, so
// each 16-lane group of an operand read hits 16 distinct chunk slots. A stage's
// scales for a lane are one 16-byte load per operand (the interleave puts a 128-row
// band's four 32-row blocks side by side). The bf16 tile leaves through LDS as
// coalesced 16-byte row stores.
#include <type_traits>

#include "attn_common.hpp"

namespace mxa {

namespace {

constexpr int kMxBlock = 32;       // K values per UE8M0 scale
constexpr int kStage = 128;        // K bytes per LDS stage
constexpr int kGroupM = 4;         // tile rows per launch-order group

__host__ __device__ inline int64_t pad_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

// ---------------- quantizer ----------------
// One thread per 32-value block of a row: bmax = max |x|; e = the smallest power of
// two with bmax / 2^e <= 448 (frexp of bmax / 448: mantissa 0.5 -> e = ex - 1,
// else ex; clamped to [-127, 127]; bmax = 0 -> -127); q = e4m3(x * 2^-e), round to
// nearest even, saturate to +-448; scale byte e + 127 (reference :95-104).
__global__ void __launch_bounds__(256) mxfp8_quant(const uint16_t* __restrict__ x, int64_t ldx, int64_t rows,
                                                   int64_t K, uint8_t* __restrict__ q, uint8_t* __restrict__ sf,
                                                   int64_t kbp, int64_t rows_pad) {
  const int64_t nkb = K / kMxBlock;
  const int64_t id = int64_t(blockIdx.x) * 256 + threadIdx.x;  // over rows_pad * kbp
  if (id >= rows_pad * kbp) return;
  const int64_t r = id / kbp, kb = id % kbp;
  // the reference's 128 x 4 interleaved scale layout (blockscale.cu:82)
  const int64_t so = (r / 128) * kbp * 128 + (kb / 4) * 512 + (r % 32) * 16 + (r % 128) / 32 * 4 + kb % 4;
  if (r >= rows || kb >= nkb) {  // padding: scale 1.0
    sf[so] = 127;
    return;
  }
  const uint16_t* src = x + r * ldx + kb * kMxBlock;
  float v[32];
  float bmax = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u32x4 u = *reinterpret_cast<const u32x4*>(src + 8 * j);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      v[8 * j + t] = bf2f(uint16_t(u[t >> 1] >> ((t & 1) * 16)));
      bmax = fmaxf(bmax, fabsf(v[8 * j + t]));
    }
  }
  int e = -127;
  if (bmax > 0.f) {
    int ex;
    const float mant = frexpf(bmax / 448.f, &ex);
    e = mant == 0.5f ? ex - 1 : ex;
    e = e < -127 ? -127 : (e > 127 ? 127 : e);
  }
  const float inv = exp2f(float(-e));
  u32x4 w[2];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float a = __builtin_fminf(__builtin_fmaxf(v[4 * j] * inv, -448.f), 448.f);
    float b = __builtin_fminf(__builtin_fmaxf(v[4 * j + 1] * inv, -448.f), 448.f);
    float c = __builtin_fminf(__builtin_fmaxf(v[4 * j + 2] * inv, -448.f), 448.f);
    float d = __builtin_fminf(__builtin_fmaxf(v[4 * j + 3] * inv, -448.f), 448.f);
    const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    w[j >> 2][j & 3] = uint32_t(__builtin_amdgcn_cvt_pk_fp8_f32(c, d, lo, true));
  }
  u32x4* dst = reinterpret_cast<u32x4*>(q + r * K + kb * kMxBlock);
  dst[0] = w[0];
  dst[1] = w[1];
  sf[so] = uint8_t(e + 127);
}

// ---------------- GEMM ----------------
// One operand's DMA of stage k0: ops of 1 KB (8 rows x 128 B each); wave w of four
// issues ops j = 4 * jj + w. Lane i of op j fills physical chunk i % 8 of row
// 8 j + i / 8, i.e. logical chunk (i % 8) ^ ((row >> 1) & 7); ((row >> 1) & 7)
// depends on j only through its parity, which is the wave's. Both operands have
// row stride K, so one set of per-lane offsets serves both and the only
// scalar offset is k0.
template <int NV>
struct OpAddr {
  uint32_t vo[NV];  // row (8 j + lane / 8) * K + logical chunk * 16, j = 4 jj + wave
  uint32_t chunk;   // logical chunk * 16 (for the K-tail check)
};
template <int NV>
__device__ __forceinline__ OpAddr<NV> op_addr(int64_t K, int lane, int wave) {
  OpAddr<NV> a;
  const int rin = lane >> 3, p = lane & 7;
  const int row = 8 * (wave & 1) + rin;  // row modulo 16 is what the swizzle sees
  const int c = p ^ ((row >> 1) & 7);
  a.chunk = uint32_t(c * 16);
#pragma unroll
  for (int jj = 0; jj < NV; ++jj) a.vo[jj] = uint32_t(8 * (4 * jj + wave) + rin) * uint32_t(K) + a.chunk;
  return a;
}
// Lanes whose chunk lies past K read zeros (an offset past the buffer's range); for a
// stage wholly past K every lane does, and the DMA only clears LDS.
template <int NV>
__device__ __forceinline__ uint32_t past_k(const OpAddr<NV>& a, int64_t K, int k0) {
  return uint32_t(k0) + a.chunk >= uint32_t(K) ? 0x80000000u : 0u;
}
template <int NV>
__device__ __forceinline__ void dma_op(__amdgpu_buffer_rsrc_t rs, const OpAddr<NV>& a, int jj, uint32_t past, int k0,
                                       unsigned char* dst, int wave) {
  buf2lds16(rs, a.vo[jj] | past, uint32_t(k0), (MXA_LDS void*)(dst + (4 * jj + wave) * 1024));
}

// Epilogue through LDS: the TN x TM = 64 NI x 64 NJ bf16 Y tile (row m = 128 NI bytes of
// n) fills the stage buffers. Lane (m = lane % 32 of block j, h = lane / 32) holds n = 8g
// + 4h + (0..3) of block i; the 16-byte chunks of row m are XOR'd with m % 16
// so that 16 rows' same chunk covers every bank: the 8-byte writes and the 16-byte row
// reads are free of bank conflicts, and each row goes out as coalesced 16-byte stores.
// ALPHA: Y = alpha * C (+ Y).
template <int NI, int NJ, bool ALPHA>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[NI][NJ], unsigned char* lds, uint16_t* __restrict__ y,
                                           int64_t ldy, int M, int N, int m0, int n0, int wm, int wn, int lane,
                                           int beta, float alpha) {
  constexpr int CH = 8 * NI, RB = 16 * CH;  // chunks and bytes per row
  static_assert(NI == 2 || NI == 4, "rows of 256 or 512 bytes");
  const int n = lane & 31, h = lane >> 5;
  block_sync_lds();  // every wave is done with the operand buffers
  {
    const int xs = n & 15;  // m % 16: wm and 32 j are multiples of 16
    unsigned char* wp = lds + (wm + n) * RB + 8 * h + wn * 2;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        // chunk wn / 8 + 4 i + g of the row; NI = 4: wn / 8 is 0 or 16, outside the XOR
        const int q = 4 * i + g;
        unsigned char* wq = NI == 4 ? wp + ((q ^ xs) << 4) : lds + (wm + n) * RB + 8 * h + (((wn >> 3) + q) ^ xs) * 16;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const f32x16& c = acc[i][j];
          float v[4] = {c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
          if constexpr (ALPHA) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= alpha;
          }
          if (beta) {  // Y += C with one rounding: add the old values in fp32 here
            const int m = m0 + wm + 32 * j + n, nb = n0 + wn + 32 * i + 8 * g + 4 * h;
            if (m < M) {
              const uint16_t* p = y + int64_t(m) * ldy + nb;
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (nb + e < N) v[e] += bf2f(p[e]);
            }
          }
          *reinterpret_cast<u32x2*>(wq + j * 32 * RB) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
      }
  }
  block_sync_lds();  // the whole tile is written
  const bool vec = (reinterpret_cast<uintptr_t>(y) & 15) == 0 && ldy % 8 == 0;
#pragma unroll 4
  for (int it = 0; it < 2 * NJ * NI; ++it) {
    const int idx = it * 256 + int(threadIdx.x), r = idx / CH, c = idx % CH, m = m0 + r, nn = n0 + 8 * c;
    if (m >= M) break;
    const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * RB + ((c ^ (r & 15)) << 4));
    uint16_t* p = y + int64_t(m) * ldy + nn;
    if (vec && nn + 7 < N) {
      *reinterpret_cast<u32x4*>(p) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (nn + e < N) p[e] = uint16_t(v[e >> 1] >> ((e & 1) * 16));
    }
  }
}

// The scale words of NB consecutive 32-row blocks for the four K blocks of one stage, in
// the reference's 128 x 4 interleaved layout: byte (r / 128) kbp 128 + (kb / 4) 512 +
// (r % 32) 16 + ((r % 128) / 32) 4 + kb % 4. A 128-row band puts its four row blocks next
// to each other, so aligned runs of 4 or 2 blocks are one 16- or 8-byte load per lane.
__device__ __forceinline__ uint32_t scale_addr(int row0, int kbp, int n) {
  return uint32_t(row0 / 128) * uint32_t(kbp) * 128u + uint32_t(16 * n) + uint32_t((row0 % 128) / 32) * 4u;
}
template <int NB>
__device__ __forceinline__ void scale_load(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t soff, uint32_t (&w)[NB]) {
  static_assert(NB == 1 || NB == 2 || NB == 4, "an aligned run of row blocks");
  if constexpr (NB == 4) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, soff, 0));
    w[0] = v[0], w[1] = v[1], w[2] = v[2], w[3] = v[3];
  } else if constexpr (NB == 2) {
    const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, soff, 0));
    w[0] = v[0], w[1] = v[1];
  } else {
    w[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, soff, 0);
  }
}

// One LDS operand read of 16 bytes: chunk coff of row block blk (32 rows) of a stage.
__device__ __forceinline__ void op_read(const unsigned char* base, int blk, int coff, int hi, i32x8& d) {
  const i32x4 v = *reinterpret_cast<const i32x4*>(base + blk * 32 * kStage + coff);
  if (hi == 0) d = __builtin_shufflevector(v, v, 0, 1, 2, 3, -1, -1, -1, -1);
  else d = __builtin_shufflevector(d, __builtin_shufflevector(v, v, 0, 1, 2, 3, 0, 1, 2, 3), 0, 1, 2, 3, 8, 9, 10, 11);
}
#define MXA_SCHED __builtin_amdgcn_sched_barrier(0)

// MXFP8 GEMM on tiles of TN = 64 NI n x TM = 64 NJ m; wave (wn, wm) of 2 x 2 owns 32 NI x
// 32 NJ.
//
// What bounds it (8192 x 12288 x 4096, 256 x 256 tiles): a 64-wide K step is NI NJ MFMAs of
// 64 cycles, so a 128-byte stage cannot take less than 2048 cycles; its LDS-DMA (64 KB)
// takes 1300 cycles when every line hits L2 and ~2000 with this grid's misses, and four
// waves that issue more than one DMA op per ~80 cycles each fill the address queue, behind
// which the wave's next MFMA waits. So the order of a stage is written out instruction by
// instruction (MXA_SCHED keeps the compiler from regrouping it): one MFMA, then at most one
// LDS operand read of the next K step and at most one DMA op, DMA ops 1.25 MFMAs apart. The
// compiler's grouping (all 16 DMA ops within five MFMAs, and scale words unpacked after the
// first DMA ops, which waited for those to land) took 3150-3270 cycles a stage, this order
// 2340 (MFMAs and barriers alone: 2245); the chip then runs at its power limit (1.71
// instead of 2.05 GHz), so the GEMM gains less: 344 -> 310 us on operands resident in the
// caches; with the prefetch below, 377 -> 318 us on operands that come from HBM.
template <int NI, int NJ, int NBUF>
__global__ void __launch_bounds__(256, 1)
mxfp8_gemm(const uint8_t* __restrict__ wq, const uint8_t* __restrict__ wsf, const uint8_t* __restrict__ xq,
           const uint8_t* __restrict__ xsf, uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K, int beta,
           int ntn, int ntm) {
  constexpr int TN = 64 * NI, TM = 64 * NJ, SA = TN * kStage, SB = TM * kStage;
  constexpr int NV = 2 * (NI > NJ ? NI : NJ);
  constexpr bool TOUCH = NBUF == 2;  // L2 prefetch (below)
  // stage buffers: operand W at lds + (st % NBUF) * SA, operand X behind W's
  // (one LDS object: with a second one the compiler waits for every DMA before LDS reads)
  __shared__ __align__(16) unsigned char lds[NBUF * (SA + SB) + (TOUCH ? 4 * 256 : 0)];
  auto abuf = [&](int s) __attribute__((always_inline)) { return lds + s * SA; };
  auto bbuf = [&](int s) __attribute__((always_inline)) { return lds + NBUF * SA + s * SB; };
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  // grouped order: consecutive tiles walk kGroupM tile rows (m) before moving
  // along n, so the 32 concurrent tiles of one XCD (one L2) form a 4 x 8 block
  // and share 12 operand strips instead of 33
  const int gsz = kGroupM * ntn, grp = L / gsz, fm = grp * kGroupM;
  const int gm = min(ntm - fm, kGroupM), li = L - grp * gsz;
  const int tm = li % gm, tn = li / gm;
  const int n0 = tn * TN, m0 = (fm + tm) * TM;
  const int wn = (wave & 1) * (32 * NI), wm = (wave >> 1) * (32 * NJ);
  const int kbp = int(pad_up(K / kMxBlock, 4));
  const int nst = (K + kStage - 1) / kStage;

  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(wq + int64_t(n0) * K, uint32_t(int64_t(N - n0) * K));
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(xq + int64_t(m0) * K, uint32_t(int64_t(M - m0) * K));
  const OpAddr<NV> oa = op_addr<NV>(K, lane, wave_u);
  // scale words of a stage, loaded a stage ahead; blocks past the 128-padded matrix read as
  // zeros (their data is zero too)
  const int n = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rsw = buf_rsrc(wsf, uint32_t(pad_up(N, 128) * kbp));
  const __amdgpu_buffer_rsrc_t rsx = buf_rsrc(xsf, uint32_t(pad_up(M, 128) * kbp));
  const uint32_t sw = scale_addr(n0 + wn, kbp, n);
  const uint32_t sx = scale_addr(m0 + wm, kbp, n);

  // LDS operand reads: rows row0 + n of an operand tile for K step s. In the f8
  // operand of the 32x32x64 MFMA, bytes 0-15 of lane half h are K 16h .. 16h+15 and
  // bytes 16-31 are K 32 + 16h ..; the UE8M0 scale of lane half h applies to K block
  // h (K 32h .. 32h+31, i.e. bytes 0-15 of both halves for h = 0, bytes 16-31 for
  // h = 1). So lane half h takes logical chunks 4s + h (K block 2s) and 4s + 2 + h
  // (K block 2s + 1), and its scale is that of K block 2s + h. The per-lane part of
  // the address is one base plus the chunk offsets; the row block is a constant.
  const int x = (n >> 1) & 7;
  int coff[4];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    coff[2 * s] = ((4 * s + h) ^ x) << 4;
    coff[2 * s + 1] = ((4 * s + 2 + h) ^ x) << 4;
  }
  const int abase = (wn + n) * kStage, bbase = (wm + n) * kStage;

  f32x16 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      // opaque zeros: left as constants, the register allocator splits the
      // accumulators' live ranges at the loop header and spills them
      acc[i][j] = f32x16{};
      asm volatile("" : "+a"(acc[i][j]));
    }

  // MFMA slots of a stage: [0, SL) K step 0, [SL, 2 SL) K step 1, the stage barrier before
  // slot SL + PRE (PRE MFMAs keep the matrix core busy while a wave waits there). From there
  // on stage st's buffer is free and takes stage st + NBUF: its DMA op u goes into slot SL +
  // PRE + 5/8 * 2 SL * u / ND, the last ones into the first slots of stage st + 1.
  constexpr int SL = NI * NJ, PRE = SL >= 8 ? 2 : 1, ND = 2 * (NI + NJ), NP = 2 * (NI + NJ);
  auto dma_slot = [](int u) constexpr { return SL + PRE + u * 5 * SL / (4 * ND); };
  static_assert(dma_slot(ND - 1) < 3 * SL, "a stage's DMA ends before its wait");
  // DMA op u: operand u & 1 (X's ops run out first or last when NI != NJ), index u >> 1
  auto dma = [&](auto uc, int st, uint32_t past, unsigned char* da, unsigned char* db) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value, lo = 2 * (NI < NJ ? NI : NJ);
    constexpr bool isx = u < 2 * lo ? (u & 1) : NJ > NI;
    constexpr int jj = u < 2 * lo ? u >> 1 : u - lo;
    if constexpr (isx) dma_op(rx, oa, jj, past, st * kStage, db, wave_u);
    else dma_op(rw, oa, jj, past, st * kStage, da, wave_u);
  };
  // operand read piece u of K step S: blocks in the order a0, b0 .. b(NJ-1), a1 .., two halves each
  auto rd = [&](auto sc, auto uc, const unsigned char* ca, const unsigned char* cb, i32x8 (&av)[NI],
                i32x8 (&bv)[NJ]) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value, o = decltype(uc)::value >> 1, hi = decltype(uc)::value & 1;
    if constexpr (o == 0) op_read(ca + abase, 0, coff[2 * S + hi], hi, av[0]);
    else if constexpr (o <= NJ) op_read(cb + bbase, o - 1, coff[2 * S + hi], hi, bv[o - 1]);
    else op_read(ca + abase, o - NJ, coff[2 * S + hi], hi, av[o - NJ]);
  };
  // MFMA q of K step S: the UE8M0 byte of K block 2S + h is byte 2S of the scale word
  // shifted right by 8h
  auto mm = [&](auto sc, auto qc, const i32x8 (&av)[NI], const i32x8 (&bv)[NJ], const uint32_t (&ta)[NI],
                const uint32_t (&tb)[NJ]) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value, i = decltype(qc)::value / NJ, j = decltype(qc)::value % NJ;
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av[i], bv[j], acc[i][j], 0, 0, 2 * S, int(ta[i]),
                                                               2 * S, int(tb[j]));
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  constexpr int NR = NBUF == 2 ? 1 : NBUF;       // sets of raw scale words in flight
  uint32_t ra[NR][NI], rb[NR][NJ];               // by stage
  uint32_t ta[NBUF][NI], tb[NBUF][NJ];           // shifted words by stage
  i32x8 r0a[NI], r0b[NJ], r1a[NI], r1b[NJ];      // operands of K steps 0 and 1
  // (past the last stage: the last one's words again, never used; the stage is a scalar
  // offset, which the buffer's range check need not cover)
  auto scales = [&](int st, uint32_t (&a)[NI], uint32_t (&b)[NJ]) __attribute__((always_inline)) {
    const uint32_t so = uint32_t(min(st, nst - 1) * 512);
    scale_load<NI>(rsw, sw, so, a);
    scale_load<NJ>(rsx, sx, so, b);
  };
  // the words are consumed here, before the next loads into their registers are issued
  auto unpack = [&](const uint32_t (&a)[NI], const uint32_t (&b)[NJ], uint32_t (&u)[NI],
                    uint32_t (&v)[NJ]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      u[i] = a[i] >> (8 * h);
      asm volatile("" : "+v"(u[i]));
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      v[j] = b[j] >> (8 * h);
      asm volatile("" : "+v"(v[j]));
    }
  };
  // L2 prefetch: with two buffers a stage's DMA has one stage to land, less than a miss to
  // HBM takes, so four bytes of each line of stage st + kAhead are loaded (into LDS that
  // nothing reads) while stage st runs. The gm work-groups of one XCD that share a W strip
  // touch a gm-th of its lines each, the neighbours along n a quarter of the X strip. Waves
  // 0-1: W, 2-3: X. 8192 x 12288 x 4096 with operands that are not in any cache: 360 -> 318
  // us (resident operands: no change); touching half a strip each 328, two stages further
  // ahead 320.
  constexpr int kAhead = 4, kTouchSlot = SL / 2;
  const __amdgpu_buffer_rsrc_t rt = wave_u < 2 ? rw : rx;
  const int share = wave_u < 2 ? gm : min(ntn, 4), strip = wave_u < 2 ? TN : TM;
  const int per = (strip + share - 1) / share, slice = wave_u < 2 ? tm : tn % share;
  const uint32_t toff = uint32_t(slice * per + ((wave_u & 1) * 64 + lane) * per / 128) * uint32_t(K);
  auto touch = [&](int st) __attribute__((always_inline)) {
    if constexpr (TOUCH)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (MXA_LDS void*)(lds + NBUF * (SA + SB) + wave_u * 256), 4,
                                               st < nst ? toff : 0x80000000u, uint32_t(st < nst ? st * kStage : 0), 0, 0);
  };
  static_assert(!TOUCH || dma_slot(ND - 1) - 2 * SL < kTouchSlot, "the touch is the newest load at the stage's wait");
  for (int st = 1; st < kAhead; ++st) touch(st);
  constexpr int kEarly = [=] {  // DMA ops of a stage before the next one starts
    int n = 0;
    for (int u = 0; u < ND; ++u) n += dma_slot(u) < 2 * SL;
    return n;
  }();
  static_for<NBUF>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    const uint32_t past = past_k(oa, K, i * kStage);
    static_for<ND>([&](auto u) __attribute__((always_inline)) {  // the late ops of the last one are issued in stage 0
      if constexpr (i < NBUF - 1 || decltype(u)::value < kEarly) dma(u, i, past, abuf(i), bbuf(i));
    });
    if constexpr (NR > 1) scales(i, ra[i % NR], rb[i % NR]);
    else if constexpr (i == 0) scales(0, ra[0], rb[0]);
    MXA_SCHED;
    if constexpr (NBUF == 2 && i == 0) {
      wait_vm();
      unpack(ra[0], rb[0], ta[0], tb[0]);
      scales(1, ra[0], rb[0]);
    }
  });
  if constexpr (NBUF > 2) {
    wait_vm_n<(NBUF - 2) * ND + kEarly>();  // stage 0 landed (see the wait in `stage`)
    unpack(ra[0], rb[0], ta[0], tb[0]);
  }
  block_sync();
  static_for<NP>([&](auto u) __attribute__((always_inline)) { rd(S0{}, u, abuf(0), bbuf(0), r0a, r0b); });
  MXA_SCHED;

  // Stage st in buffer s (compile-time).
  auto stage = [&](int st, auto sc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value, sn = (s + 1) % NBUF, sp = (s + NBUF - 1) % NBUF;
    const uint32_t late = past_k(oa, K, (st + NBUF - 1) * kStage), past = past_k(oa, K, (st + NBUF) * kStage);
    static_for<SL>([&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
      mm(S0{}, qc, r0a, r0b, ta[s], tb[s]);
      static_for<NP>([&](auto u) __attribute__((always_inline)) {
        if constexpr (decltype(u)::value * SL / NP == q) rd(S1{}, u, abuf(s), bbuf(s), r1a, r1b);
      });
      static_for<ND>([&](auto u) __attribute__((always_inline)) {
        if constexpr (dma_slot(decltype(u)::value) - 2 * SL == q) dma(u, st + NBUF - 1, late, abuf(sp), bbuf(sp));
      });
      if constexpr (TOUCH && q == kTouchSlot) {
        MXA_SCHED;
        touch(st + kAhead);
      }
      MXA_SCHED;
    });
    static_for<PRE>([&](auto qc) __attribute__((always_inline)) {
      mm(S1{}, qc, r1a, r1b, ta[s], tb[s]);
      MXA_SCHED;
    });
    // this wave's DMA of stage st + 1 landed (newer: the stages up to st + NBUF - 1, a touch) ...
    // Only LDS-DMA ops are counted. The two scale loads of a stage lie between them, but in the
    // stages behind the loop over whole turns the compiler deletes those whose words nothing
    // uses: counted in, they let that many DMA ops of stage st + 1 stay in flight.
    wait_vm_n<(NBUF - 2) * ND + TOUCH>();
    // ... for every wave, and every wave has read stage st (the youngest operand reads were
    // issued only PRE MFMAs ago: they are waited for here, the next DMA op goes into their slot)
    block_sync_lds();
    MXA_SCHED;
    static_for<SL - PRE>([&](auto qc) __attribute__((always_inline)) {
      constexpr int q = decltype(qc)::value;
      mm(S1{}, std::integral_constant<int, PRE + q>{}, r1a, r1b, ta[s], tb[s]);
      static_for<ND>([&](auto u) __attribute__((always_inline)) {
        if constexpr (dma_slot(decltype(u)::value) - SL - PRE == q) dma(u, st + NBUF, past, abuf(s), bbuf(s));
      });
      static_for<NP>([&](auto u) __attribute__((always_inline)) {
        if constexpr (decltype(u)::value * (SL - PRE - (SL >= 8 ? 2 : 0)) / NP == q)
          rd(S0{}, u, abuf(sn), bbuf(sn), r0a, r0b);  // on the last stage: stale data, never used
      });
      if constexpr (q == 0) unpack(ra[sn % NR], rb[sn % NR], ta[sn], tb[sn]);
      if constexpr (q == (SL - PRE > 1 ? 1 : 0)) scales(st + NBUF, ra[s % NR], rb[s % NR]);
      MXA_SCHED;
    });
  };
  // whole turns of the ring, then the rest (a loop with an exit inside a group would make
  // the compiler wait for the youngest scale words on every turn)
  int st = 0;
  for (; st + NBUF <= nst; st += NBUF)
    static_for<NBUF>([&](auto s) __attribute__((always_inline)) { stage(st + decltype(s)::value, s); });
  static_for<NBUF - 1>([&](auto s) __attribute__((always_inline)) {
    if (st + decltype(s)::value < nst) stage(st + decltype(s)::value, s);
  });
  wait_vm();  // no LDS-DMA may land after the work-group ends

  store_tile<NI, NJ, false>(acc, lds, y, ldy, M, N, m0, n0, wm, wn, lane, beta, 1.f);
}


// ---------------- NVFP4 ----------------
// Format (the reference's NVFP4, blockscale.cu:36-93): e2m1 data, two per byte (the
// lower-index value in the low nibble), one e4m3 scale per 16 consecutive K values of
// a row (the same 128 x 4 interleave with K/16 blocks, padding bytes 0, as the
// reference's memset), and a per-tensor amax: g = amax / (6 * 448), block scale
// se = e4m3(bmax / (6 g)), codes e2m1(x / (se g)). The GEMM returns
// alpha * sum (e2m1 se)_X (e2m1 se)_W with alpha = gW gX.
constexpr int kFp4Block = 16;
constexpr float kFp4Range = 6.f * 448.f;

__global__ void nvfp4_amax_init(float* amax) {
  if (threadIdx.x == 0) *amax = 0.f;
}

__device__ __forceinline__ float max8(float m, u32x4 u) {  // max of m and 8 bf16 magnitudes
#pragma unroll
  for (int t = 0; t < 8; ++t) m = fmaxf(m, fabsf(bf2f(uint16_t(u[t >> 1] >> ((t & 1) * 16)))));
  return m;
}
__device__ __forceinline__ float block_max16(float m, float* wmax) {  // 16 waves; every thread gets the max
#pragma unroll
  for (int o = 32; o; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) m = fmaxf(m, wmax[w]);
  return m;
}

// max |x| of the tensor (reference amax_kernel :45-67): a 1024-thread work-group per
// range of rows, four 16-byte loads in flight per thread, a wave max, the work-group
// max through LDS, one atomic max per work-group on the value's bits (non-negative
// floats order as integers). At most 256 work-groups: atomics on one address
// serialise (one per wave cost ~40 us at 4096 x 4096).
__global__ void __launch_bounds__(1024) nvfp4_amax(const uint16_t* __restrict__ x, int64_t ldx, int64_t rows,
                                                   int64_t K, float* amax) {
  const int64_t nv = K / 8;
  const int64_t per = (rows + gridDim.x - 1) / gridDim.x;
  const int64_t r0 = int64_t(blockIdx.x) * per, r1 = r0 + per < rows ? r0 + per : rows;
  const int64_t n = r1 > r0 ? (r1 - r0) * nv : 0;
  float m = 0.f;
  for (int64_t i0 = threadIdx.x; i0 < n; i0 += 4 * 1024) {
    u32x4 u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t i = i0 + k * 1024;
      const int64_t r = r0 + i / nv, j = i - (i / nv) * nv;
      u[k] = i < n ? *reinterpret_cast<const u32x4*>(x + r * ldx + 8 * j) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) m = max8(m, u[k]);
  }
  __shared__ float wmax[16];
  m = block_max16(m, wmax);
  if (threadIdx.x == 0) atomicMax(reinterpret_cast<int*>(amax), __float_as_int(m));
}

// One thread per 16-value block of a row (reference quant_kernel NVFP4 branch :76-93);
// padding scale bytes get 0.
__device__ __forceinline__ void nvfp4_block(const uint16_t* __restrict__ x, int64_t ldx, int64_t rows, int64_t K,
                                            uint8_t* __restrict__ q, uint8_t* __restrict__ sf, float a, int64_t kbp,
                                            int64_t id) {
  const int64_t nkb = K / kFp4Block;
  const int64_t r = id / kbp, kb = id % kbp;
  const int64_t so = (r / 128) * kbp * 128 + (kb / 4) * 512 + (r % 32) * 16 + (r % 128) / 32 * 4 + kb % 4;
  if (r >= rows || kb >= nkb) {
    sf[so] = 0;
    return;
  }
  const uint16_t* src = x + r * ldx + kb * kFp4Block;
  float v[16];
  float bmax = 0.f;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const u32x4 u = *reinterpret_cast<const u32x4*>(src + 8 * j);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      v[8 * j + t] = bf2f(uint16_t(u[t >> 1] >> ((t & 1) * 16)));
      bmax = fmaxf(bmax, fabsf(v[8 * j + t]));
    }
  }
  const float g = a > 0.f ? a / kFp4Range : 1.f;
  const float inv6g = 1.f / (6.f * g);
  // e4m3 of bmax / (6 g), saturating: clamp to 448, then round to nearest even
  const float t = __builtin_fminf(bmax * inv6g, 448.f);
  const uint32_t se = uint32_t(__builtin_amdgcn_cvt_pk_fp8_f32(t, t, 0, false)) & 0xffu;
  const float sd = __builtin_amdgcn_cvt_f32_fp8(int(se), 0) * g;
  const float inv = sd > 0.f ? 1.f / sd : 0.f;
  // e2m1 codes: v_cvt_scalef32_pk_fp4_f32 (scale 1) rounds to the nearest magnitude of
  // {0, 0.5, 1, 1.5, 2, 3, 4, 6} with ties to the even code, saturates at 6 and sets the
  // sign bit for negative values: the reference's threshold sum (:38-42), checked on
  // the device against it over 2M value pairs (every midpoint +-1 ulp, -0, saturation);
  // two values per byte, the lower-index one in the low nibble
  u32x2 w = {0u, 0u};
  static_for<8>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    w[j >> 2] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w[j >> 2], v[2 * j] * inv, v[2 * j + 1] * inv, 1.f, j & 3);
  });
  *reinterpret_cast<u32x2*>(q + (r * K + kb * kFp4Block) / 2) = w;
  sf[so] = uint8_t(se);
}
__global__ void __launch_bounds__(256) nvfp4_quant(const uint16_t* __restrict__ x, int64_t ldx, int64_t rows,
                                                   int64_t K, uint8_t* __restrict__ q, uint8_t* __restrict__ sf,
                                                   const float* __restrict__ amax, int64_t kbp, int64_t rows_pad) {
  const int64_t id = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (id < rows_pad * kbp) nvfp4_block(x, ldx, rows, K, q, sf, *amax, kbp, id);
}

// The same in one launch for a tensor of few values: every work-group that holds values
// takes the maximum of the whole tensor itself (at most kFp4Small values, 128 KB that stay in
// L2), which is cheaper than two more launches: 1 x 3072 9.4 -> 4.2 us, 4 x 12288 9.6 -> 5.4,
// 16 x 4096 (the limit) 9.8 -> 5.8.
constexpr int kFp4Small = 65536;
__global__ void __launch_bounds__(1024) nvfp4_quant_small(const uint16_t* __restrict__ x, int64_t ldx, int rows, int K,
                                                          uint8_t* __restrict__ q, uint8_t* __restrict__ sf,
                                                          float* __restrict__ amax, int64_t kbp, int64_t rows_pad) {
  constexpr int NL = kFp4Small / 8 / 1024;  // 16-byte loads per thread
  __shared__ float wmax[16];
  const int64_t id = int64_t(blockIdx.x) * 1024 + threadIdx.x;
  float m = 0.f;
  if (int64_t(blockIdx.x) * 1024 < int64_t(rows) * kbp) {  // (else the work-group holds padding only)
    const int nv = K / 8, n = rows * nv;                   // n <= 1024 NL
    u32x4 u[NL];
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      const int i = int(threadIdx.x) + k * 1024, r = i / nv, j = i - r * nv;
      u[k] = i < n ? *reinterpret_cast<const u32x4*>(x + r * ldx + 8 * j) : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int k = 0; k < NL; ++k) m = max8(m, u[k]);
    m = block_max16(m, wmax);
    if (blockIdx.x == 0 && threadIdx.x == 0) *amax = m;
  }
  if (id < rows_pad * kbp) nvfp4_block(x, ldx, rows, K, q, sf, m, kbp, id);
}

// NVFP4 GEMM: the MXFP8 kernel's tiling (64 NI n x 64 NJ m per 4-wave work-group, fp32
// accumulators in AGPRs, K stages of 128 bytes = 256 values DMA'd into LDS
// with the same swizzle, XCD-grouped tile order, LDS epilogue), but the raw e2m1
// data is dequantized in registers and multiplied on the f16 MFMA (32x32x16). gfx950's
// scaled MFMA takes one power-of-two scale per 32 values, NVFP4 an e4m3 scale per 16;
// the product of an e2m1 value and an e4m3 scale has at most 6 significant bits, so
// e2m1 -> f16 (v_cvt_scalef32_pk_f16_fp4, scale 1) times the block scale in f16
// (v_pk_mul_f16) is exact, as are the MFMA's f16 products; accumulation is fp32, and
// alpha = gW gX scales the tile in the epilogue.
//
// Operand layout: the MFMA sums its 16 K values in any order, so the two lane halves
// take different 16-value blocks: lane half h of row r reads the 16 bytes of chunk 2c + h
// of a stage (blocks 4c + 2h + u, u = 0, 1) and feeds bytes 8u + 4w .. + 3 of them to MFMA
// step 4c + 2u + w; W and X use the same assignment, so every product pairs the same K.
//
// What bounds it: a step is NI NJ MFMAs of 32 cycles and 8 (NI + NJ) vector instructions of
// dequantization (4 x 4: 16 and 64), which fit beside the MFMAs only if they are spread
// between them. So the next step's operands are dequantized into a second register set while
// this step's MFMAs run, half a block after each MFMA, in a fixed order (MXA_SCHED); the
// compiler's own order put the dequantization of a step before its MFMAs, and 8-byte LDS
// reads of half a chunk waited for each other. M 4096 N 3072 K 12288: 327 -> 227 us (1.36
// PFLOP/s); M 8192 N 12288 K 4096: 660 -> 576 us (1.43 PFLOP/s, near the rate at which this
// chip's power limit holds bf16 library GEMMs: 1.4-1.6).
using f16x2 = __attribute__((ext_vector_type(2))) _Float16;
using f16x8 = __attribute__((ext_vector_type(8))) _Float16;

// Eight e2m1 values (a dword) times their block's scale in f16.
__device__ __forceinline__ f16x8 fp4x8_to_f16(uint32_t d, f16x2 s) {
  const f16x2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.f, 0) * s;
  const f16x2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.f, 1) * s;
  const f16x2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.f, 2) * s;
  const f16x2 e = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(d, 1.f, 3) * s;
  return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
}

// The block scales in the low two bytes of a word, as an f16 pair (exact).
__device__ __forceinline__ f16x2 fp4_scales(uint32_t word) {
  return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(word, 1.f, false);
}
__device__ __forceinline__ f16x2 splat16(f16x2 p, int u) { return u ? p.yy : p.xx; }
__device__ __forceinline__ float fp4_alpha(float aw, float ax) {
  return (aw > 0.f ? aw / kFp4Range : 1.f) * (ax > 0.f ? ax / kFp4Range : 1.f);
}

template <int NI, int NJ>
__global__ void __launch_bounds__(256, 1)
nvfp4_gemm(const uint8_t* __restrict__ wq, const uint8_t* __restrict__ wsf, const float* __restrict__ wamax,
           const uint8_t* __restrict__ xq, const uint8_t* __restrict__ xsf, const float* __restrict__ xamax,
           uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K, int beta, int ntn, int ntm) {
  constexpr int TN = 64 * NI, TM = 64 * NJ, SA = TN * kStage, SB = TM * kStage;
  constexpr int NV = 2 * (NI > NJ ? NI : NJ);
  // stage buffers: operand W at lds + (st & 1) * SA, operand X at lds + 2 SA + (st & 1) * SB
  __shared__ __align__(16) unsigned char lds[2 * (SA + SB)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int gsz = kGroupM * ntn, grp = L / gsz, fm = grp * kGroupM;
  const int gm = min(ntm - fm, kGroupM), li = L - grp * gsz;
  const int n0 = li / gm * TN, m0 = (fm + li % gm) * TM;
  const int wn = (wave & 1) * (32 * NI), wm = (wave >> 1) * (32 * NJ);
  const int RB = K / 2;                                  // bytes per row
  const int kbp = int(pad_up(K / kFp4Block, 4));
  const int nst = (RB + kStage - 1) / kStage;            // stages of 256 values

  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(wq + int64_t(n0) * RB, uint32_t(int64_t(N - n0) * RB));
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(xq + int64_t(m0) * RB, uint32_t(int64_t(M - m0) * RB));
  const OpAddr<NV> oa = op_addr<NV>(RB, lane, wave_u);
  const int n = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rsw = buf_rsrc(wsf, uint32_t(pad_up(N, 128) * kbp));
  const __amdgpu_buffer_rsrc_t rsx = buf_rsrc(xsf, uint32_t(pad_up(M, 128) * kbp));
  const uint32_t sw = scale_addr(n0 + wn, kbp, n);
  const uint32_t sx = scale_addr(m0 + wm, kbp, n);
  // LDS address of this half's chunk 2c + h of row (w* + 32 b + n): physical chunk
  // (2c + h) ^ ((row >> 1) & 7)
  const int x = (n >> 1) & 7;
  int co[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) co[c] = ((2 * c + h) ^ x) << 4;
  const int abase = (wn + n) * kStage, bbase = 2 * SA + (wm + n) * kStage;

  f32x16 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      acc[i][j] = f32x16{};
      asm volatile("" : "+a"(acc[i][j]));
    }

  constexpr int SL = NI * NJ, NB = NI + NJ, ND = 2 * NB;
  uint32_t wa[4][NI], wb[4][NJ];  // scale words of K blocks 4c .. 4c + 3 of a stage
  i32x4 raw[2][NB];               // e2m1 chunks of c (by parity): NI W blocks, then NJ X blocks
  f16x2 ps[2][NB];                // their two block scales
  f16x8 op[2][NB];                // dequantized operands of a step (by parity)
  auto words = [&](int st, auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value;
    const uint32_t so = uint32_t(min(4 * st + c, kbp / 4 - 1) * 512);  // (past the end: never used)
    scale_load<NI>(rsw, sw, so, wa[c]);
    scale_load<NJ>(rsx, sx, so, wb[c]);
  };
  auto read = [&](int buf, auto cc, auto bc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value, b = decltype(bc)::value;
    const unsigned char* p = b < NI ? lds + abase + buf * SA + b * 32 * kStage : lds + bbase + buf * SB + (b - NI) * 32 * kStage;
    raw[c & 1][b] = *reinterpret_cast<const i32x4*>(p + co[c]);
  };
  auto scale = [&](auto cc, auto bc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value, b = decltype(bc)::value;
    ps[c & 1][b] = fp4_scales((b < NI ? wa[c][b < NI ? b : 0] : wb[c][b < NI ? 0 : b - NI]) >> (16 * h));
  };
  // dequantization unit d (0 .. 2 NB - 1) of step k: half (4 values) of one block, in the
  // order the MFMAs need the blocks: W 0, X 0 .. NJ - 1, W 1 ..
  auto deq = [&](auto kc, auto dc) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value, c = k >> 2, u = (k >> 1) & 1, w = k & 1;
    constexpr int o = decltype(dc)::value >> 1, hi = decltype(dc)::value & 1;
    constexpr int b = o == 0 ? 0 : o <= NJ ? NI + o - 1 : o - NJ;
    const uint32_t v = uint32_t(raw[c & 1][b][2 * u + w]);
    const f16x2 s = splat16(ps[c & 1][b], u);
    const f16x2 e = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 1.f, 2 * hi) * s;
    const f16x2 f = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v, 1.f, 2 * hi + 1) * s;
    f16x8& d = op[k & 1][b];
    d[4 * hi] = e[0], d[4 * hi + 1] = e[1], d[4 * hi + 2] = f[0], d[4 * hi + 3] = f[1];
  };
  auto dma = [&](auto uc, int st, uint32_t past) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value, lo = 2 * (NI < NJ ? NI : NJ);
    constexpr bool isx = u < 2 * lo ? (u & 1) : NJ > NI;
    constexpr int jj = u < 2 * lo ? u >> 1 : u - lo;
    if constexpr (isx) dma_op(rx, oa, jj, past, st * kStage, lds + 2 * SA + (st & 1) * SB, wave_u);
    else dma_op(rw, oa, jj, past, st * kStage, lds + (st & 1) * SA, wave_u);
  };
  using C0 = std::integral_constant<int, 0>;
  // (the words first: the compiler waits for them by the number of younger loads)
  static_for<4>([&](auto c) __attribute__((always_inline)) { words(0, c); });
  static_for<ND>([&](auto u) __attribute__((always_inline)) { dma(u, 0, past_k(oa, RB, 0)); });
  wait_vm();
  block_sync();
  static_for<NB>([&](auto b) __attribute__((always_inline)) {
    read(0, C0{}, b);
    scale(C0{}, b);
  });
  MXA_SCHED;
  words(1, C0{});
  static_for<ND>([&](auto u) __attribute__((always_inline)) { dma(u, 1, past_k(oa, RB, kStage)); });
  static_for<2 * NB>([&](auto d) __attribute__((always_inline)) { deq(C0{}, d); });
  MXA_SCHED;

  // A stage is 16 steps of SL MFMA slots. Beside step k's MFMAs: step k + 1's dequantization;
  // in steps 4c + 1 and 4c + 2 the LDS reads and block scales of chunk c + 1; in step 13 the
  // stage barrier (stage st + 1 landed; every wave holds the last chunk of stage st in
  // registers), from then on the DMA of stage st + 2; a chunk's scale words of the next stage
  // as soon as this stage's are consumed.
  for (int st = 0; st < nst; ++st) {
    const int buf = st & 1;
    const uint32_t past = past_k(oa, RB, (st + 2) * kStage);
    static_for<16>([&](auto kc) __attribute__((always_inline)) {
      constexpr int k = decltype(kc)::value, c = k >> 2, r = k & 3, cn = (c + 1) & 3;
      if constexpr (k == 13) {
        wait_vm();
        block_sync();
        MXA_SCHED;
      }
      static_for<SL>([&](auto qc) __attribute__((always_inline)) {
        constexpr int q = decltype(qc)::value, i = q / NJ, j = q % NJ;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(op[k & 1][i], op[k & 1][NI + j], acc[i][j], 0, 0, 0);
        static_for<2 * NB>([&](auto d) __attribute__((always_inline)) {
          if constexpr (decltype(d)::value * SL / (2 * NB) == q) deq(std::integral_constant<int, (k + 1) & 15>{}, d);
        });
        static_for<NB>([&](auto b) __attribute__((always_inline)) {
          if constexpr (r == 1 && decltype(b)::value * SL / NB == q)
            read(c == 3 ? buf ^ 1 : buf, std::integral_constant<int, cn>{}, b);
          if constexpr (r == 2 && decltype(b)::value * SL / NB == q) scale(std::integral_constant<int, cn>{}, b);
        });
        if constexpr (r == 3 && q == 0) words(cn == 0 ? st + 2 : st + 1, std::integral_constant<int, cn>{});
        if constexpr (k >= 13)
          static_for<ND>([&](auto u) __attribute__((always_inline)) {
            if constexpr (decltype(u)::value * 3 * SL / ND == (k - 13) * SL + q) dma(u, st + 2, past);
          });
        MXA_SCHED;
      });
    });
  }
  wait_vm();  // no LDS-DMA may land after the work-group ends
  store_tile<NI, NJ, true>(acc, lds, y, ldy, M, N, m0, n0, wm, wn, lane, beta, fp4_alpha(*wamax, *xamax));
}

// ---------------- GEMM of few tiles: K split over the waves of a work-group ----------------
//
// A GEMM whose 64- or 128-row tiles leave CUs idle is bound by latency: one work-group
// walks K in series (M 256, N 3072, K 3072 on 12 tiles of 256 x 256: 24 stages, 34 us; 192
// tiles of 64 x 64 here: 9.2 us; M 1, N = K = 12288: 128 -> 35 us, 4.3 TB/s of W).
// Here a work-group of KS waves computes one small tile of TN = 32 NI x TM = 32 NJ and
// wave w takes the K stages w, w + KS, ..: every wave streams its own 128-byte K slices of
// the tile's rows into its own ring of NB stage buffers (LDS-DMA, no work-group barrier
// in the loop, only counted waits), so KS NB stages are in flight per work-group. The fp32
// partial tiles are added in wave order through LDS (no partial leaves the CU, the sum's
// order is fixed) and the sum is rounded once.
//
// F4: NVFP4. A lane half h reads the 16 bytes of chunk 2 c + h (32 values: two 16-value
// blocks, K blocks 4 c + 2 h + u) of its row, so the two halves of an f16 MFMA step hold
// different blocks; W and X use the same assignment and the MFMA sums its K values in any
// order. Otherwise MXFP8, with the operand layout of mxfp8_gemm.
template <bool F4, int NI, int NJ, int KS, int NB>
__global__ void __launch_bounds__(64 * KS, 1)
gemm_ksplit(const uint8_t* __restrict__ wq, const uint8_t* __restrict__ wsf, const float* __restrict__ wamax,
            const uint8_t* __restrict__ xq, const uint8_t* __restrict__ xsf, const float* __restrict__ xamax,
            uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K, int beta, int ntm) {
  constexpr int TN = 32 * NI, TM = 32 * NJ, SA = TN * kStage, ST = (TN + TM) * kStage;
  constexpr int NSC = F4 ? 4 : 1;                       // scale words per row block and stage
  constexpr int DMA = 4 * (NI + NJ);                    // LDS-DMA operations per stage
  constexpr int OPS = DMA + 2 * NSC;                    // with the scale loads
  constexpr int RED = NI * NJ * 4096;                   // bytes of one wave's partial tile
  static_assert((NB - 1) * OPS < 64, "the wait counter has 6 bits");
  __shared__ __align__(16) unsigned char lds[KS * NB * ST > KS * RED ? KS * NB * ST : KS * RED];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  // consecutive tiles share a W strip: the m tiles of one strip run on one XCD
  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int n0 = L / ntm * TN, m0 = L % ntm * TM;
  const int RB = F4 ? K / 2 : K;                        // bytes per row
  const int kbp = int(pad_up(K / (F4 ? kFp4Block : kMxBlock), 4));
  const int nst = (RB + kStage - 1) / kStage;
  const __amdgpu_buffer_rsrc_t rw = buf_rsrc(wq + int64_t(n0) * RB, uint32_t(int64_t(N - n0) * RB));
  const __amdgpu_buffer_rsrc_t rx = buf_rsrc(xq + int64_t(m0) * RB, uint32_t(int64_t(M - m0) * RB));
  const __amdgpu_buffer_rsrc_t rsw = buf_rsrc(wsf, uint32_t(pad_up(N, 128) * kbp));
  const __amdgpu_buffer_rsrc_t rsx = buf_rsrc(xsf, uint32_t(pad_up(M, 128) * kbp));
  const uint32_t sw = scale_addr(n0, kbp, n);
  const uint32_t sx = scale_addr(m0, kbp, n);
  // DMA op j (rows 8 j .. 8 j + 7): lane i fills physical chunk i % 8 of row 8 j + i / 8,
  // logical chunk (i % 8) ^ ((row >> 1) & 7), which depends on j through its parity
  constexpr int NV = 4 * (NI > NJ ? NI : NJ);
  const int c0 = (lane & 7) ^ (lane >> 4);
  uint32_t vo[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) vo[j] = uint32_t(8 * j + (lane >> 3)) * uint32_t(RB) + uint32_t((c0 ^ (4 * (j & 1))) * 16);
  unsigned char* const ring = lds + wave * NB * ST;
  uint32_t ra[NB][NSC][NI], rb[NB][NSC][NJ];
  // stage i of this wave (K stage wave + KS i; past the end: zeros, no traffic) into slot s
  auto issue = [&](int i, auto sc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    const int st = wave + KS * i, k0 = st * kStage;
    const uint32_t p0 = uint32_t(k0 + c0 * 16) >= uint32_t(RB) ? 0x80000000u : 0u;
    const uint32_t p1 = uint32_t(k0 + (c0 ^ 4) * 16) >= uint32_t(RB) ? 0x80000000u : 0u;
    unsigned char* d = ring + s * ST;
#pragma unroll
    for (int j = 0; j < 4 * NI; ++j) buf2lds16(rw, vo[j] | (j & 1 ? p1 : p0), uint32_t(k0), (MXA_LDS void*)(d + j * 1024));
#pragma unroll
    for (int j = 0; j < 4 * NJ; ++j)
      buf2lds16(rx, vo[j] | (j & 1 ? p1 : p0), uint32_t(k0), (MXA_LDS void*)(d + SA + j * 1024));
#pragma unroll
    for (int t = 0; t < NSC; ++t) {
      // (past the end: the last words again, their data is zero)
      const uint32_t so = uint32_t(min(st * NSC + t, kbp / 4 - 1) * 512);
      scale_load<NI>(rsw, sw, so, ra[s][t]);
      scale_load<NJ>(rsx, sx, so, rb[s][t]);
    }
    MXA_SCHED;
  };
  f32x16 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x16{};

  const int x = (n >> 1) & 7;
  const int cnt = (nst - wave + KS - 1) / KS;  // this wave's stages (wave < KS; may be 0)
  static_for<NB>([&](auto s) __attribute__((always_inline)) { issue(decltype(s)::value, s); });
  // (rest: the stages behind the whole turns, where the compiler deletes scale loads that nothing
  // uses: only the DMA ops of the younger stages are counted)
  auto body = [&](int i, auto sc, auto rest) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    wait_vm_n<(NB - 1) * (decltype(rest)::value ? DMA : OPS)>();
    const unsigned char* d = ring + s * ST + n * kStage;
    // this half's 16-byte chunks of a row: 2 r + h
    i32x4 av[NI][4], bv[NJ][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = ((2 * r + h) ^ x) << 4;
#pragma unroll
      for (int b = 0; b < NI; ++b) av[b][r] = *reinterpret_cast<const i32x4*>(d + b * 32 * kStage + co);
#pragma unroll
      for (int b = 0; b < NJ; ++b) bv[b][r] = *reinterpret_cast<const i32x4*>(d + SA + b * 32 * kStage + co);
    }
    uint32_t ta[NSC][NI], tb[NSC][NJ];
#pragma unroll
    for (int t = 0; t < NSC; ++t) {
#pragma unroll
      for (int b = 0; b < NI; ++b) ta[t][b] = ra[s][t][b] >> ((F4 ? 16 : 8) * h);
#pragma unroll
      for (int b = 0; b < NJ; ++b) tb[t][b] = rb[s][t][b] >> ((F4 ? 16 : 8) * h);
    }
    // every operand read has returned and the scale words are consumed before the slot is refilled
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int b = 0; b < NI; ++b) asm volatile("" : "+v"(av[b][r]));
#pragma unroll
      for (int b = 0; b < NJ; ++b) asm volatile("" : "+v"(bv[b][r]));
    }
#pragma unroll
    for (int t = 0; t < NSC; ++t) {
#pragma unroll
      for (int b = 0; b < NI; ++b) asm volatile("" : "+v"(ta[t][b]));
#pragma unroll
      for (int b = 0; b < NJ; ++b) asm volatile("" : "+v"(tb[t][b]));
    }
    issue(i + NB, sc);  // (ends with a scheduling barrier)
    if constexpr (!F4) {
      static_for<2>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
#pragma unroll
        for (int i2 = 0; i2 < NI; ++i2)
#pragma unroll
          for (int j2 = 0; j2 < NJ; ++j2)
            acc[i2][j2] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                __builtin_shufflevector(av[i2][2 * k], av[i2][2 * k + 1], 0, 1, 2, 3, 4, 5, 6, 7),
                __builtin_shufflevector(bv[j2][2 * k], bv[j2][2 * k + 1], 0, 1, 2, 3, 4, 5, 6, 7), acc[i2][j2], 0, 0,
                2 * k, int(ta[0][i2]), 2 * k, int(tb[0][j2]));
      });
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f16x2 pa[NI], pb[NJ];
#pragma unroll
          for (int b = 0; b < NI; ++b) pa[b] = splat16(fp4_scales(ta[r][b]), u);
#pragma unroll
          for (int b = 0; b < NJ; ++b) pb[b] = splat16(fp4_scales(tb[r][b]), u);
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            f16x8 fa[NI], fb[NJ];
#pragma unroll
            for (int b = 0; b < NI; ++b) fa[b] = fp4x8_to_f16(uint32_t(av[b][r][2 * u + w]), pa[b]);
#pragma unroll
            for (int b = 0; b < NJ; ++b) fb[b] = fp4x8_to_f16(uint32_t(bv[b][r][2 * u + w]), pb[b]);
#pragma unroll
            for (int i2 = 0; i2 < NI; ++i2)
#pragma unroll
              for (int j2 = 0; j2 < NJ; ++j2)
                acc[i2][j2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i2], fb[j2], acc[i2][j2], 0, 0, 0);
          }
        }
    }
    MXA_SCHED;
  };
  // whole turns of the ring, then the rest (see mxfp8_gemm)
  int i = 0;
  for (; i + NB <= cnt; i += NB)
    static_for<NB>([&](auto s) __attribute__((always_inline)) { body(i + decltype(s)::value, s, std::false_type{}); });
  static_for<NB - 1>([&](auto s) __attribute__((always_inline)) {
    if (i + decltype(s)::value < cnt) body(i + decltype(s)::value, s, std::true_type{});
  });
  wait_vm();        // no LDS-DMA may land in what the reduction writes
  __syncthreads();  // every wave is done with the rings

  // Reduction: [wave][block][g = 4 rows of n][2 halves][32 m] groups of four n in fp32, the m
  // slot XOR'd with the group's position along n so that reads along n are conflict-free.
  float alpha = 1.f;
  if constexpr (F4) alpha = fp4_alpha(*wamax, *xamax);
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int sl = n ^ (2 * g + h + 8 * (i & 1));
        *reinterpret_cast<f32x4*>(lds + wave * RED + (((i * NJ + j) * 4 + g) * 64 + h * 32 + sl) * 16) =
            f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
      }
  __syncthreads();
  const bool vec = (reinterpret_cast<uintptr_t>(y) & 7) == 0 && ldy % 4 == 0;
  constexpr int Q = TN / 4;  // groups of four n per row
  for (int t = threadIdx.x; t < Q * TM; t += 64 * KS) {
    const int q = t % Q, ml = t / Q, i = q >> 3, g = (q >> 1) & 3, hh = q & 1;
    const int sl = (ml & 31) ^ (2 * g + hh + 8 * (i & 1));
    const unsigned char* rp = lds + (((i * NJ + (ml >> 5)) * 4 + g) * 64 + hh * 32 + sl) * 16;
    f32x4 v = *reinterpret_cast<const f32x4*>(rp);
#pragma unroll
    for (int w = 1; w < KS; ++w) v += *reinterpret_cast<const f32x4*>(rp + w * RED);
    const int m = m0 + ml, nn = n0 + 4 * q;
    if (m >= M) continue;
    uint16_t* p = y + int64_t(m) * ldy + nn;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (F4) v[e] *= alpha;
      if (beta && nn + e < N) v[e] += bf2f(p[e]);
    }
    if (vec && nn + 3 < N) {
      *reinterpret_cast<u32x2*>(p) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (nn + e < N) p[e] = f2bf(v[e]);
    }
  }
}

}  // namespace

size_t mx_qscale_size(int64_t rows, int64_t K) { return size_t(pad_up(rows, 128) * pad_up(K / kMxBlock, 4)); }

hipError_t launch_mxfp8_quant(const uint16_t* x, int64_t ldx, int64_t rows, int64_t K, uint8_t* q, uint8_t* sf,
                              hipStream_t s) {
  const int64_t kbp = pad_up(K / kMxBlock, 4), rp = pad_up(rows, 128);
  const int64_t blocks = (rp * kbp + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(mxfp8_quant, dim3(unsigned(blocks)), dim3(256), 0, s, x, ldx, rows, K, q, sf, kbp, rp);
  return hipGetLastError();
}

namespace {

// The tile of a GEMM, by its estimated time in us: f0 + rounds (f + a nst), nst K stages of
// 128 bytes, rounds of C CUs x occ work-groups; `alone` replaces a where two work-groups
// fit a CU and no more than C run. The figures are fits to sweeps of M 1 .. 8192, N and K
// 1024 .. 12288 on an MI355X (C = 256), operands rotating through 3 buffers (us, best of the others):
//   M     N     K       256 x 256  256 x 128  128 x 128  64 x 64   64 x 64   64 x 32  32 x 32
//                                                        4 waves   2 waves
//   1     3072  3072    28.2       17.6       11.9       7.2       8.6       6.2      5.0
//   1     12288 12288   128        80         55         36        36        34       35
//   33    5120  5120    44         27         18         11.3      12.8      9.5      11.0
//   256   3072  3072    34         20.6       14.6       9.1       10.2      13.3     11.4
//   512   3072  3072    34         20.7       14.8       16.5      13.0      19.8     19.8
//   256   12288 3072    35         21.1       15.6       25.6      24.9      37       37
//   2048  3072  3072    33         23.1       30         64        44        80       90
//   3000  3072  3072    35         43         44         92        75        116      129
// The large tiles move fewer bytes per product and lose where they leave CUs idle; below
// them the time is the latency of K in series, which the K-split tiles divide by their waves.
enum GemmKind { kG256, kG256x128, kG128, kGk64, kGk64w2, kGk64x32, kGk32, kGKinds };
struct GemmTile {
  int tn, tm, occ, ks;  // ks: waves that K is split over
  double f0, f, a, alone;
};
constexpr GemmTile kMxTiles[kGKinds] = {
    {256, 256, 1, 1, 2.0, 8.0, 1.05, 0}, {256, 128, 1, 1, 0, 7.0, 0.58, 0},      {128, 128, 1, 1, 0, 5.5, 0.39, 0},
    {64, 64, 1, 4, 1.5, 3.4, 0.175, 0},  {64, 64, 2, 2, 1.1, 3.9, 0.325, 0.226}, {64, 32, 1, 4, 1.2, 3.0, 0.13, 0},
    {32, 32, 2, 4, 0.5, 2.8, 0.20, 0.095}};
GemmKind gemm_plan(const GemmTile (&tiles)[kGKinds], int M, int N, int nst, int C) {
  int best = 0;
  double bt = 0;
  for (int k = 0; k < kGKinds; ++k) {
    const GemmTile& t = tiles[k];
    const int64_t n = int64_t((N + t.tn - 1) / t.tn) * ((M + t.tm - 1) / t.tm);
    const double rounds = double((n + int64_t(C) * t.occ - 1) / (int64_t(C) * t.occ));
    const double us = t.f0 + rounds * (t.f + nst * (t.occ == 2 && n <= C ? t.alone : t.a));
    if (k == 0 || us < bt) best = k, bt = us;
  }
  return GemmKind(best);
}
GemmKind mxfp8_plan(int M, int N, int K, int C) { return gemm_plan(kMxTiles, M, N, (K + kStage - 1) / kStage, C); }

}  // namespace

// Preconditions (checked by the caller): K % 32 == 0, (N + 255) / 256 * 256 * K < 2^31,
// same for M; beta 0 or 1.
hipError_t launch_mxfp8_gemm(const uint8_t* wq, const uint8_t* wsf, const uint8_t* xq, const uint8_t* xsf,
                             uint16_t* y, int64_t ldy, int M, int N, int K, int beta, hipStream_t s) {
  const GemmKind kind = mxfp8_plan(M, N, K, current_cus());
  const int tn = kMxTiles[kind].tn, tm = kMxTiles[kind].tm, ntn = (N + tn - 1) / tn, ntm = (M + tm - 1) / tm;
  const int64_t blocks = int64_t(ntn) * ntm;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid{unsigned(blocks)};
  auto tiles = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, wq, wsf, xq, xsf, y, ldy, M, N, K, beta, ntn, ntm);
  };
  auto ksplit = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(64 * kMxTiles[kind].ks), 0, s, wq, wsf, (const float*)nullptr, xq, xsf,
                       (const float*)nullptr, y, ldy, M, N, K, beta, ntm);
  };
  switch (kind) {
    case kG256x128: tiles(mxfp8_gemm<4, 2, 3>); break;
    case kG128: tiles(mxfp8_gemm<2, 2, 4>); break;
    case kGk64: ksplit(gemm_ksplit<false, 2, 2, 4, 2>); break;
    case kGk64w2: ksplit(gemm_ksplit<false, 2, 2, 2, 2>); break;
    case kGk64x32: ksplit(gemm_ksplit<false, 2, 1, 4, 3>); break;
    case kGk32: ksplit(gemm_ksplit<false, 1, 1, 4, 2>); break;
    default: tiles(mxfp8_gemm<4, 4, 2>); break;
  }
  return hipGetLastError();
}

hipError_t launch_nvfp4_quant(const uint16_t* x, int64_t ldx, int64_t rows, int64_t K, uint8_t* q, uint8_t* sf,
                              float* amax, hipStream_t s) {
  const int64_t kbp = pad_up(K / kFp4Block, 4), rp = pad_up(rows, 128);
  const int64_t blocks = (rp * kbp + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  if (rows <= kFp4Small && K <= kFp4Small && rows * K <= kFp4Small) {
    hipLaunchKernelGGL(nvfp4_quant_small, dim3(unsigned((rp * kbp + 1023) / 1024)), dim3(1024), 0, s, x, ldx, int(rows),
                       int(K), q, sf, amax, kbp, rp);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(nvfp4_amax_init, dim3(1), dim3(64), 0, s, amax);
  hipLaunchKernelGGL(nvfp4_amax, dim3(unsigned(rows < 256 ? rows : 256)), dim3(1024), 0, s, x, ldx, rows, K, amax);
  hipLaunchKernelGGL(nvfp4_quant, dim3(unsigned(blocks)), dim3(256), 0, s, x, ldx, rows, K, q, sf,
                     (const float*)amax, kbp, rp);
  return hipGetLastError();
}

namespace {

// The same estimate for NVFP4 (stages of 256 values; the f16 MFMAs weigh more, so the
// large tiles hold on to smaller shapes). Measured us, as above:
//   M     N     K       256 x 256  256 x 128  128 x 128  64 x 64   64 x 64   64 x 32  32 x 32
//                                                        4 waves   2 waves
//   1     3072  3072    50         34         22         9.9       14.2      8.2      6.2
//   1     12288 12288   184        122        84         29        45        22       25
//   33    5120  5120    81         54         36         14.6      21.7      11.3     13.5
//   256   3072  3072    54         36         23         11.0      15.6      15.8     12.6
//   512   3072  3072    55         37         24         20.8      17.5      24       22
//   1024  3072  3072    55         37         25         31        32        47       40
//   2048  3072  3072    56         39         43         60        50        90       76
//   4096  3072  12288   227        283        262        350       337       461      547
constexpr GemmTile kF4Tiles[kGKinds] = {
    {256, 256, 1, 1, 0, 8.0, 3.9, 0},   {256, 128, 1, 1, 0, 7.7, 2.4, 0},    {128, 128, 2, 1, 0, 4.4, 3.2, 1.6},
    {64, 64, 1, 4, 1.0, 4.5, 0.45, 0},  {64, 64, 2, 2, 1.0, 4.2, 1.02, 0.87}, {64, 32, 1, 4, 0.9, 3.7, 0.32, 0},
    {32, 32, 2, 4, 0.5, 2.7, 0.53, 0.25}};
GemmKind nvfp4_plan(int M, int N, int K, int C) {
  return gemm_plan(kF4Tiles, M, N, (K / 2 + kStage - 1) / kStage, C);
}

}  // namespace

void gemm_blockscaled_tile(bool f4, int M, int N, int K, int cus, int* tile_n, int* tile_m, int* k_waves) {
  const GemmTile& t = f4 ? kF4Tiles[nvfp4_plan(M, N, K, cus)] : kMxTiles[mxfp8_plan(M, N, K, cus)];
  *tile_n = t.tn, *tile_m = t.tm, *k_waves = t.ks;
}

// Preconditions (checked by the caller): K % 32 == 0, (N + 255) / 256 * 256 * K / 2 < 2^31,
// same for M; beta 0 or 1; the amax pointers are device floats written by the quantizer.
hipError_t launch_nvfp4_gemm(const uint8_t* wq, const uint8_t* wsf, const float* wamax, const uint8_t* xq,
                             const uint8_t* xsf, const float* xamax, uint16_t* y, int64_t ldy, int M, int N, int K,
                             int beta, hipStream_t s) {
  const GemmKind kind = nvfp4_plan(M, N, K, current_cus());
  const int tn = kF4Tiles[kind].tn, tm = kF4Tiles[kind].tm, ntn = (N + tn - 1) / tn, ntm = (M + tm - 1) / tm;
  const int64_t blocks = int64_t(ntn) * ntm;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid{unsigned(blocks)};
  auto tiles = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, wq, wsf, wamax, xq, xsf, xamax, y, ldy, M, N, K, beta, ntn, ntm);
  };
  auto ksplit = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(64 * kF4Tiles[kind].ks), 0, s, wq, wsf, wamax, xq, xsf, xamax, y, ldy, M, N, K,
                       beta, ntm);
  };
  switch (kind) {
    case kG256x128: tiles(nvfp4_gemm<4, 2>); break;
    case kG128: tiles(nvfp4_gemm<2, 2>); break;
    case kGk64: ksplit(gemm_ksplit<true, 2, 2, 4, 2>); break;
    case kGk64w2: ksplit(gemm_ksplit<true, 2, 2, 2, 2>); break;
    case kGk64x32: ksplit(gemm_ksplit<true, 2, 1, 4, 3>); break;
    case kGk32: ksplit(gemm_ksplit<true, 1, 1, 4, 2>); break;
    default: tiles(nvfp4_gemm<4, 4>); break;
  }
  return hipGetLastError();
}

}  // namespace mxa
