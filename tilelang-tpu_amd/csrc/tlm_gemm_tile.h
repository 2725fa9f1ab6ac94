// Tiled GEMM for the sizes between one decode step and a whole prompt batch: C = A * B (row-major
// B) or A * B^T, where 256x256 tiles are too few to fill the 256 CUs. Shared by tlm_gemm.hip
// (fp16 / bf16) and tlm_gemm_fp8.hip (e4m3 / e5m2, B^T).
//
// What bounds it: with few rows, the stream of B (every weight is read once, from HBM); with more,
// the rate at which a CU takes operand tiles from L2 (about 50 B/clk), since a BM x BN tile reads
// (BM + BN) bytes per 2 BM BN flops. So the tile is as large as still gives every CU a workgroup,
// and where even 32- or 64-row tiles are fewer than the CUs, K is split over `ns` workgroups.
//
// Workgroup = 8 waves: BM/WTM x BN/WTN wave tiles times KG k-groups. The waves of a k-group take
// every KG-th 64-byte k-step of a tile, which keeps wave tiles large (LDS bytes per flop) with two
// waves on each SIMD; the k-groups' sums meet in LDS at the end. Tiles stream through an NST-stage LDS
// ring by LDS-DMA (NST - 1 tiles in flight, one barrier per tile); the operands of tile t are
// read from LDS while the MFMAs of tile t - 1 run.
// The MFMAs take B as the first operand, so a lane holds 4 consecutive columns of one row of C.
// Measured (us, the 256x256 kernel before -> here): bf16 500 x 4096 x 4096 79 -> 27, 64 x 2048 x 7168
// B^T 123 -> 11, 1024 x 4096 x 4096 80 -> 40, 2048 x 4096 x 4096 81 -> 66; e4m3 512 x 4096 x 4096
// 39 -> 22, 16 x 4096 x 4096 (one thread per output before) 1515 -> 9; M 16 B^T 14336 x 4096 (a
// 64-column strip kernel before) 31.9 -> 22.4, 5.2 TB/s.
//
// Split K: every workgroup stores its partial tile (fp32) with write-through stores and counts
// itself in on the tile's counter; the last to arrive adds the tiles in split order, writes C and
// resets the counter, so the result does not depend on the order of arrival.
#pragma once

#include "tlm_common.h"

#include <type_traits>

// Workspace of the split kernels for stream `s` on the current device (tlm_gemm.hip): tlm_split_bytes of
// partial tiles and TLM_SPLIT_TILES zeroed counters that a kernel leaves at zero. False when the
// stream owns none and none is free. 16-bit calls of one decode step (`decode`: 16 rows or fewer) have
// slots of their own: streams that run larger calls or fp8 do not take them, and a graph that keeps
// one can be replayed beside the larger calls of the stream it was captured on.
constexpr size_t tlm_split_bytes(bool decode) { return (size_t)(decode ? 8 : 16) << 20; }
constexpr int TLM_SPLIT_TILES = 512;
bool tlm_split_slot(bool decode, hipStream_t s, float** part, unsigned** arrivals);

namespace gt {

enum { EL_F16 = 0, EL_BF16 = 1, EL_E4M3 = 2, EL_E5M2 = 3 };

constexpr int THREADS = 512;
constexpr uint32_t OOB_OFF = 0xfffffff0u;  // past num_records: the load returns zeros
constexpr int RSRC3 = 0x00020000;

template <int EL_, bool TRANS_B_, int BM_, int BN_, int WTM_, int WTN_, int BKB_, int NST_,
          bool WIDE_ = false, bool DUAL_ = false>
struct Cfg {
  static constexpr int EL = EL_, BM = BM_, BN = BN_, WTM = WTM_, WTN = WTN_;
  static constexpr int BKB = BKB_;  // bytes of k per tile
  static constexpr int NST = NST_;
  static constexpr bool TRANS_B = TRANS_B_;
  static constexpr bool FP8 = EL >= EL_E4M3;
  static constexpr bool DUAL = DUAL_;  // two B^T matrices, SwiGLU of the two products
  static constexpr int BNC = DUAL ? BN / 2 : BN;  // columns of C
  static constexpr bool WIDE = WIDE_;  // fp8 operands multiplied as fp16
  static constexpr int ES = FP8 ? 1 : 2;
  static constexpr int BK = BKB / ES;
  static constexpr int WM = BM / WTM, WN = BN / WTN, KG = 8 / (WM * WN);
  static constexpr int STEPS = BKB / 64, SPG = STEPS / KG;  // 64-byte k-steps: per tile, per k-group
  static constexpr int SA = BM * BKB, SB = BN * BKB, ST = SA + SB;
  static constexpr int NA = SA / 8192, NB = SB / 8192;  // LDS-DMA instructions per wave and tile
  static constexpr int PER = NA + NB;
  static constexpr int TR = FP8 ? 32 : 16;                // rows / columns of an MFMA tile
  static constexpr int MT = WTM / TR, NT = WTN / TR;  // MFMA tiles of a wave
  static constexpr int Q = WTM * WTN / 256;               // f32x4 of accumulator per lane
  static constexpr int QO = Q / KG;                       // of which the wave finishes
  static_assert(WM * WN * KG == 8 && SPG * KG == STEPS && QO * KG == Q, "wave layout");
  static_assert(NA * 8192 == SA && NB * 8192 == SB, "whole LDS-DMA instructions per wave");
  static_assert(!FP8 || TRANS_B, "fp8 takes B^T");
  static_assert(!DUAL || (!FP8 && TRANS_B && NT % 2 == 0 && QO % 2 == 0), "pairs of column tiles");
  static constexpr int RED = KG > 1 ? 8 * Q * 1024 : 0;
  static constexpr int SMEM = NST * ST > RED ? NST * ST : RED;
  static_assert(SMEM <= 160 * 1024, "LDS");
};

using namespace ldsop;

TLM_DEV void lgkm_wait0() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
}
template <int N>
TLM_DEV void vm_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt(0x3f70 | (N & 15) | ((N >> 4) << 14));
}
TLM_DEV void tile_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// 16-byte chunk c of row r of an [rows][BKB bytes] tile sits at c ^ swz: 16 lanes that read one
// chunk column of 16 consecutive rows hit the 16 different 16-byte windows of all banks.
template <int BKB>
TLM_DEV int swz_row(int r) {
  return BKB == 128 ? (r >> 1) & 7 : r & 15;
}
// Row-major B tile [k][BN]: 32 lanes of a transposed read cover rows k0 .. k0 + 3 and k0 + 8 ..
// k0 + 11 of two neighbouring chunks; XOR with swz_k puts them in 16 different chunk positions of
// a 256-byte window (one row of 128 columns, two of 64).
template <int BN>
TLM_DEV int swz_k(int k) {
  return BN >= 128 ? 2 * ((k & 3) + 4 * ((k >> 3) & 1)) : 2 * (((k >> 1) & 1) + 2 * ((k >> 3) & 1));
}

template <int EL>
TLM_DEV f32x4 mma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (EL == EL_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
template <int EL>
TLM_DEV f32x16 mma8(u32x4 a0, u32x4 a1, u32x4 b0, u32x4 b1, f32x16 c) {
  constexpr int FMT = EL == EL_E5M2 ? 1 : 0;
  const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3],
                   (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
  const i32x8 b = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3],
                   (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, FMT, FMT, 0, 0, 0, 0);
}

// The same product on the fp16 matrix instruction (every e4m3 / e5m2 value is an fp16 value): the fp8
// one drops low bits of the sums (1.3e-5 of a K 4096 product against 3e-8 here).
template <int EL>
TLM_DEV f16x8 widen(uint32_t lo, uint32_t hi) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  f16x2 p[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int w = (int)(i ? hi : lo);
    if constexpr (EL == EL_E4M3) {
      p[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
      p[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
    } else {
      p[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, 1.0f, false);
      p[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(w, 1.0f, true);
    }
  }
  return f16x8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}
template <int EL>
TLM_DEV f32x16 mma8_wide(u32x4 a0, u32x4 a1, u32x4 b0, u32x4 b1, f32x16 c) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const u32x4 a = q < 2 ? a0 : a1, b = q < 2 ? b0 : b1;
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(widen<EL>(a[2 * (q & 1)], a[2 * (q & 1) + 1]),
                                               widen<EL>(b[2 * (q & 1)], b[2 * (q & 1) + 1]), c, 0, 0,
                                               0);
  }
  return c;
}

// Four consecutive output values (columns col .. col + 3 of one row).
template <int OUT>
TLM_DEV void store4(void* C, int64_t idx, f32x4 v, int valid, bool vec) {
  if constexpr (OUT == TLM_F32) {
    float* c = (float*)C + idx;
    if (vec) {
      *(f32x4*)c = v;
      return;
    }
    for (int i = 0; i < valid; ++i) c[i] = v[i];
  } else if constexpr (OUT == TLM_F16 || OUT == TLM_BF16) {
    using H = h16<OUT == TLM_BF16>;
    const u32x2 p = {H::pack(v[0], v[1]), H::pack(v[2], v[3])};
    uint16_t* c = (uint16_t*)C + idx;
    if (vec) {
      *(u32x2*)c = p;
      return;
    }
    if (valid > 0) c[0] = (uint16_t)p[0];
    if (valid > 1) c[1] = (uint16_t)(p[0] >> 16);
    if (valid > 2) c[2] = (uint16_t)p[1];
    if (valid > 3) c[3] = (uint16_t)(p[1] >> 16);
  } else {  // fp8: round to nearest even, no saturation (torch's cast)
    uint32_t p;
    if constexpr (OUT == TLM_F8E4M3) {
      p = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
      p = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], (int)p, true);
    } else {
      p = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(v[0], v[1], 0, false);
      p = (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(v[2], v[3], (int)p, true);
    }
    uint8_t* c = (uint8_t*)C + idx;
    if (vec) {
      *(uint32_t*)c = p;
      return;
    }
    for (int i = 0; i < valid; ++i) c[i] = (uint8_t)(p >> (8 * i));
  }
}
template <int OUT>
constexpr int out_size() {
  return OUT == TLM_F32 ? 4 : (OUT == TLM_F16 || OUT == TLM_BF16) ? 2 : 1;
}

// Requires: A, B 16-byte aligned, rows of A (and B^T) and row-major B's rows whole 16-byte chunks,
// BM K and BN K (B^T) or BK N (row-major) bytes below 2^31 - 16; ns > 1: part and
// arrivals of tlm_split_slot with grid tiles <= TLM_SPLIT_TILES and grid * BM * BN * 4 <=
// tlm_split_bytes. Grid: ns * ceil(M / BM) * ceil(N / BN) workgroups of THREADS.
template <typename CF, int OUT>
__global__ __launch_bounds__(THREADS, 1) void gemm_tile(const uint8_t* __restrict__ A,
                                                       const uint8_t* __restrict__ B,
                                                       void* __restrict__ C, int M, int N, int K,
                                                       int ns, float* __restrict__ part,
                                                       unsigned* __restrict__ arrivals,
                                                       const uint8_t* __restrict__ B2) {
  constexpr int BM = CF::BM, BN = CF::BN, BKB = CF::BKB, ES = CF::ES, KG = CF::KG;
  constexpr bool FP8 = CF::FP8, TRANS_B = CF::TRANS_B;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[CF::SMEM];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sp = wave / KG, kg = wave % KG;  // the waves of one SIMD (w, w + 4) take the same kg
  const int wm = sp / CF::WN, wn = sp % CF::WN;

  // Workgroup ids go round-robin over the 8 XCDs: XCD x takes a contiguous range of (split, column
  // tile, row tile), row tiles fastest, so that the row tiles that share a strip of B, and the
  // strips that share a k range of A, meet in one L2.
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + CF::BNC - 1) / CF::BNC;
  const int total = tiles_m * tiles_n * ns;
  const int xcd = blockIdx.x & 7, xi = blockIdx.x >> 3;
  const int lin = xcd * (total >> 3) + min(xcd, total & 7) + xi;
  const int tile = lin % (tiles_m * tiles_n), split = lin / (tiles_m * tiles_n);
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * CF::BNC;
  const int KT = (int)(((int64_t)K * ES + BKB - 1) / BKB);
  const int kt_lo = (int)((int64_t)split * KT / ns);
  const int n = (int)((int64_t)(split + 1) * KT / ns) - kt_lo;

  // ---- LDS-DMA: instruction j of a wave fills 1 KB of A (j < NA) or B; the lane's byte offset from
  // the k-tile's base does not change from tile to tile. Lanes outside the matrix read zeros.
  uint32_t off[CF::PER];
  int kch[CF::PER];  // first k of the lane's chunk within the tile (row of row-major B)
#pragma unroll
  for (int j = 0; j < CF::PER; ++j) {
    const int ins = 8 * (j < CF::NA ? j : j - CF::NA) + wave;
    if (j < CF::NA || TRANS_B) {
      constexpr int CPR = BKB / 16;
      const int r = ins * (64 / CPR) + lane / CPR;
      const int c = (lane % CPR) ^ swz_row<BKB>(r);
      // DUAL: 16-row blocks of the tile alternate between the two matrices
      const int rr = CF::DUAL && j >= CF::NA ? (r >> 5) * 16 + (r & 15) : r;
      const bool ok = j < CF::NA ? m0 + rr < M : n0 + rr < N;
      off[j] = ok ? (uint32_t)(rr * K * ES + 16 * c) : OOB_OFF;
      kch[j] = c * (16 / ES);
    } else {
      constexpr int CPR = BN * 2 / 16;
      const int k = ins * (64 / CPR) + lane / CPR;
      const int c = (lane % CPR) ^ swz_k<BN>(k);
      off[j] = n0 + 8 * c < N ? (uint32_t)(k * N * 2 + 16 * c) : OOB_OFF;
      kch[j] = k;
    }
  }
  const uint8_t* const a_base = A + (int64_t)m0 * K * ES;
  // (a wave's instructions fill blocks of one of them: 8 instructions are whole pairs of blocks)
  const bool second = CF::DUAL && (wave * (1024 / BKB) >> 4 & 1);
  const uint8_t* const b_base =
      TRANS_B ? (second ? B2 : B) + (int64_t)n0 * K * ES : B + (int64_t)n0 * 2;
  struct Fill {  // a tile's operand bases and LDS stage
    const uint8_t* a;
    const uint8_t* b;
    uint8_t* st;
    int kmax;
  };
  auto fill_of = [&](int t, int stage) __attribute__((always_inline)) {
    const int k0 = (kt_lo + t) * CF::BK;
    return Fill{a_base + (int64_t)k0 * ES,
                TRANS_B ? b_base + (int64_t)k0 * ES : b_base + (int64_t)k0 * N * 2,
                smem + stage * CF::ST + wave * 1024, K - k0};
  };
  auto fill1 = [&](const Fill& f, auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    constexpr bool isa = j < CF::NA;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(isa ? f.a : f.b), (short)0, 0x7ffffff0, RSRC3);
    const uint32_t o = kch[j] < f.kmax ? off[j] : OOB_OFF;
    uint8_t* const dst = f.st + (isa ? j * 8192 : CF::SA + (j - CF::NA) * 8192);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void*)dst, 16, o, 0, 0, 0);
  };
  auto issue = [&](int t, int stage) __attribute__((always_inline)) {
    const Fill f = fill_of(t, stage);
    unroll<0, CF::PER>([&](auto jc) __attribute__((always_inline)) { fill1(f, jc); });
  };

  // ---- operand reads (byte addresses within stage 0)
  const uint32_t s0 = lds_u32(smem);
  const int lr = lane & (CF::TR - 1);          // row of A / column of B within an MFMA tile
  const int lq = lane / CF::TR;                // 16-byte chunk within the k-step
  uint32_t a_addr[CF::SPG][FP8 ? 2 : 1];       // + mt * TR rows
  uint32_t b_addr[CF::SPG][FP8 ? 2 : 1];       // B^T: + nt * TR rows
  uint32_t bt_addr[CF::NT];                    // row-major: + 32 k-rows per step
#pragma unroll
  for (int s = 0; s < CF::SPG; ++s)
#pragma unroll
    for (int p = 0; p < (FP8 ? 2 : 1); ++p) {
      const int c = 4 * (kg * CF::SPG + s) + lq + 2 * p;
      const int x = 16 * (c ^ swz_row<BKB>(lr));
      a_addr[s][p] = s0 + (uint32_t)((wm * CF::WTM + lr) * BKB + x);
      b_addr[s][p] = s0 + (uint32_t)(CF::SA + (wn * CF::WTN + lr) * BKB + x);
    }
  if constexpr (!TRANS_B) {
    // 16-lane group h, lane j: 8 bytes at columns 4 (j % 4) of k-row 8 h + j / 4 (+ 4 for the
    // second read); the lane receives column j of the four rows
    const int h = lane >> 4, j = lane & 15;
    const int k = 8 * h + (j >> 2);
#pragma unroll
    for (int nt = 0; nt < CF::NT; ++nt) {
      const int c = (wn * CF::WTN + 16 * nt) / 8 + ((j & 3) >> 1);
      bt_addr[nt] = s0 + (uint32_t)(CF::SA + (32 * kg * CF::SPG + k) * (BN * 2) +
                                    16 * (c ^ swz_k<BN>(k)) + 8 * (j & 1));
    }
  }
  struct Ops {
    u32x4 a[CF::SPG][CF::MT][FP8 ? 2 : 1];
    u32x4 b[CF::SPG][CF::NT][FP8 ? 2 : 1];  // B^T
    u32x2 bt[CF::SPG][CF::NT][2];            // row-major
  };
  // read i of a tile's operands: per k-step the MT A operands, then the NT B operands
  constexpr int P = FP8 ? 2 : 1, PB = TRANS_B ? P : 2;
  constexpr int RPS = CF::MT * P + CF::NT * PB, NR = CF::SPG * RPS;
  auto read1 = [&](Ops& o, uint32_t so, auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value, s = i / RPS, r = i % RPS;
    if constexpr (r < CF::MT * P) {
      ds_b128<r / P * CF::TR * BKB>(o.a[s][r / P][r % P], a_addr[s][r % P] + so);
    } else {
      constexpr int nt = (r - CF::MT * P) / PB, p = (r - CF::MT * P) % PB;
      if constexpr (TRANS_B)
        ds_b128<nt * CF::TR * BKB>(o.b[s][nt][p], b_addr[s][p] + so);
      else
        ds_tr16<(32 * s + 4 * p) * BN * 2>(o.bt[s][nt][p], bt_addr[nt] + so);
    }
  };
  auto read_ops = [&](Ops& o, int stage) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)(stage * CF::ST);
    unroll<0, NR>([&](auto ic) __attribute__((always_inline)) { read1(o, so, ic); });
  };
  auto ops_landed = [&](Ops& o) __attribute__((always_inline)) {
    lgkm_wait0();
#pragma unroll
    for (int s = 0; s < CF::SPG; ++s) {
#pragma unroll
      for (int mt = 0; mt < CF::MT; ++mt)
#pragma unroll
        for (int p = 0; p < (FP8 ? 2 : 1); ++p) landed(o.a[s][mt][p]);
#pragma unroll
      for (int nt = 0; nt < CF::NT; ++nt) {
        if constexpr (TRANS_B) {
#pragma unroll
          for (int p = 0; p < (FP8 ? 2 : 1); ++p) landed(o.b[s][nt][p]);
        } else {
          landed(o.bt[s][nt][0]);
          landed(o.bt[s][nt][1]);
        }
      }
    }
  };
  using Acc = std::conditional_t<FP8, f32x16, f32x4>;
  Acc acc[CF::MT][CF::NT];
#pragma unroll
  for (int mt = 0; mt < CF::MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < CF::NT; ++nt) acc[mt][nt] = Acc{};
  constexpr int NM = CF::SPG * CF::NT * CF::MT;  // MFMAs of a tile
  auto mul1 = [&](const Ops& o, auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value, mt = i % CF::MT, nt = i / CF::MT % CF::NT,
                  s = i / (CF::MT * CF::NT);
    if constexpr (CF::WIDE) {
      acc[mt][nt] = mma8_wide<CF::EL>(o.b[s][nt][0], o.b[s][nt][1], o.a[s][mt][0], o.a[s][mt][1],
                                      acc[mt][nt]);
    } else if constexpr (FP8) {
      acc[mt][nt] = mma8<CF::EL>(o.b[s][nt][0], o.b[s][nt][1], o.a[s][mt][0], o.a[s][mt][1],
                                 acc[mt][nt]);
    } else if constexpr (TRANS_B) {
      acc[mt][nt] = mma16<CF::EL>(o.b[s][nt][0], o.a[s][mt][0], acc[mt][nt]);
    } else {
      const u32x4 b = {o.bt[s][nt][0][0], o.bt[s][nt][0][1], o.bt[s][nt][1][0], o.bt[s][nt][1][1]};
      acc[mt][nt] = mma16<CF::EL>(b, o.a[s][mt][0], acc[mt][nt]);
    }
  };
  auto multiply = [&](const Ops& o) __attribute__((always_inline)) {
    unroll<0, NM>([&](auto ic) __attribute__((always_inline)) { mul1(o, ic); });
  };

  // ---- main loop: tile t lives in stage t % NST. At step t a wave waits for its own share of tile t, and
  // after the barrier every wave has: tile t is whole, and tile t - 1's stage, read by
  // every wave before the barrier, takes tile t + NST - 1.
  constexpr int AHEAD = CF::NST - 1;
#pragma unroll
  for (int t = 0; t < AHEAD; ++t)
    if (t < n) issue(t, t);
  int stage = 0;
  auto enter = [&](int t) __attribute__((always_inline)) {
    const int left = min(AHEAD - 1, n - 1 - t);  // tiles after t whose loads may stay in flight
    __builtin_amdgcn_sched_barrier(0);
    unroll<0, AHEAD>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      if (left == i) vm_wait<i * CF::PER>();
    });
    tile_barrier();
  };
  auto refill_stage = [&]() __attribute__((always_inline)) {
    return stage == 0 ? AHEAD : stage - 1;
  };
  auto next = [&]() __attribute__((always_inline)) { stage = stage == AHEAD ? 0 : stage + 1; };
  // The reads of tile t and the refill are spread over the MFMAs of tile t - 1: issued in a burst,
  // they hold the wave until the LDS has taken them and its MFMAs start late.
  auto step = [&](int t, Ops& cur, const Ops& prev) __attribute__((always_inline)) {
    enter(t);
    const uint32_t so = (uint32_t)(stage * CF::ST);
    const bool more = t + AHEAD < n;
    const Fill f = fill_of(more ? t + AHEAD : t, refill_stage());
    unroll<0, NM>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      constexpr int RS = NM * 3 / 4 > 0 ? NM * 3 / 4 : 1;  // the reads go out in the first 3/4
      unroll<(i < RS ? i * NR / RS : NR), (i + 1 < RS ? (i + 1) * NR / RS : NR)>(
          [&](auto rc) __attribute__((always_inline)) { read1(cur, so, rc); });
      if constexpr ((i + 1) * CF::PER / NM > i * CF::PER / NM)
        if (more)
          unroll<i * CF::PER / NM, (i + 1) * CF::PER / NM>(
              [&](auto jc) __attribute__((always_inline)) { fill1(f, jc); });
      mul1(prev, ic);
      __builtin_amdgcn_sched_barrier(0);
    });
    ops_landed(cur);
    next();
  };
  if (n > 0) {
    Ops x, y;
    enter(0);
    read_ops(x, 0);
    if (AHEAD < n) issue(AHEAD, refill_stage());
    ops_landed(x);
    next();
    int t = 1;
    for (; t + 1 < n; t += 2) {
      step(t, y, x);
      step(t + 1, x, y);
    }
    if (t < n) {
      step(t, y, x);
      multiply(y);
    } else {
      multiply(x);
    }
  }

  // ---- the k-groups' sums: quad u (f32x4) of a wave tile is finished by k-group u / QO
  auto quad = [&](auto uc) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    if constexpr (FP8) {
      const f32x16& v = acc[u / 4 / CF::NT][u / 4 % CF::NT];
      constexpr int q = 4 * (u % 4);
      return f32x4{v[q], v[q + 1], v[q + 2], v[q + 3]};
    } else {
      return acc[u / CF::NT][u % CF::NT];
    }
  };
  f32x4 fin[CF::QO];
  if constexpr (KG > 1) {
    f32x4* const red = (f32x4*)smem;
    __syncthreads();  // every operand read is done
    unroll<0, CF::Q>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      if (kg != u / CF::QO) red[(wave * CF::Q + u) * 64 + lane] = quad(uc);
    });
    __syncthreads();
    unroll<0, CF::Q>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      if (kg == u / CF::QO) {
        f32x4 s = {};
#pragma unroll
        for (int g = 0; g < KG; ++g)
          s += g == u / CF::QO ? quad(uc) : red[((sp * KG + g) * CF::Q + u) * 64 + lane];
        fin[u % CF::QO] = s;
      }
    });
  } else {
    unroll<0, CF::Q>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value;
      fin[u] = quad(uc);
    });
  }

  // ---- split K: as in gemm_skinny_split, the tiles meet in memory through write-through stores and
  // loads that miss every cache
  if (ns > 1) {
    unsigned* const last = (unsigned*)smem;  // the k-groups' sums have been read by the barrier below
    const int lo = ((wave * CF::QO) * 64 + lane) * 16;
    float* const mine = part + ((int64_t)split * tiles_m * tiles_n + tile) * (BM * BN);
#pragma unroll
    for (int v = 0; v < CF::QO; ++v)
      st_cp<CP_SC01>(mine, lo + v * 1024, __builtin_bit_cast(u32x4, fin[v]));
    __builtin_amdgcn_s_waitcnt(0x3f70);  // vmcnt(0): the tile has been written
    __syncthreads();
    if (tid == 0) *last = atomicAdd(&arrivals[tile], 1u) == (unsigned)(ns - 1);
    __syncthreads();
    if (!*last) return;
    constexpr int BATCH = 16 / CF::QO > 8 ? 8 : 16 / CF::QO < 1 ? 1 : 16 / CF::QO;
    f32x4 sum[CF::QO];
#pragma unroll
    for (int v = 0; v < CF::QO; ++v) sum[v] = f32x4{};
    for (int s0_ = 0; s0_ < ns; s0_ += BATCH) {  // uniform; BATCH splits' tiles requested together
      f32x4 t[BATCH][CF::QO];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const int s = s0_ + i;
        const float* const src = part + ((int64_t)s * tiles_m * tiles_n + tile) * (BM * BN);
#pragma unroll
        for (int v = 0; v < CF::QO; ++v) {
          t[i][v] = fin[v];
          if (s < ns && s != split)
            t[i][v] = __builtin_bit_cast(f32x4, ld_cp<CP_SC01>(src, lo + v * 1024));
        }
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (s0_ + i < ns)
#pragma unroll
          for (int v = 0; v < CF::QO; ++v) sum[v] += t[i][v];
    }
#pragma unroll
    for (int v = 0; v < CF::QO; ++v) fin[v] = sum[v];
    if (tid == 0) atomicExch(&arrivals[tile], 0u);
  }

  // ---- C: the lane's quads are 4 consecutive columns of row m
  const bool vec_c = N % 4 == 0 && ((uintptr_t)C % (4 * out_size<OUT>())) == 0;
  if constexpr (CF::DUAL) {
    // column tiles nt, nt + 1 hold the same columns of the two products, rounded to the storage type as
    // if stored, then up * gate / (1 + exp(-gate)) as tlm_swiglu
    using H = h16<OUT == TLM_BF16>;
    unroll<0, CF::Q / 2>([&](auto pc) __attribute__((always_inline)) {
      constexpr int u = 2 * decltype(pc)::value, v = u % CF::QO;
      if (kg == u / CF::QO) {
        constexpr int mt = u / CF::NT, nt = u % CF::NT;
        const int m = m0 + wm * CF::WTM + mt * CF::TR + lr;
        const int c = n0 + (wn * CF::WTN + nt * CF::TR) / 2 + 4 * lq;
        f32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = H::to_f32(H::from_f32(fin[v][i]));
          const float up = H::to_f32(H::from_f32(fin[v + 1][i]));
          o[i] = up * (g * __builtin_amdgcn_rcpf(fast_exp(-g) + 1.0f));
        }
        if (m < M && c < N) store4<OUT>(C, (int64_t)m * N + c, o, min(4, N - c), vec_c);
      }
    });
    return;
  }
  unroll<0, CF::Q>([&](auto uc) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    if (kg == u / CF::QO) {
      constexpr int tu = FP8 ? u / 4 : u;
      constexpr int mt = tu / CF::NT, nt = tu % CF::NT;
      const int m = m0 + wm * CF::WTM + mt * CF::TR + lr;
      const int c = n0 + wn * CF::WTN + nt * CF::TR + (FP8 ? 8 * (u % 4) : 0) + 4 * lq;
      if (m < M && c < N)
        store4<OUT>(C, (int64_t)m * N + c, fin[u % CF::QO], min(4, N - c), vec_c);
    }
  });
}

// ---- choice of tile and split on the host
enum { T32 = 0, T32W, T64N, T64, T128, T256, T_COUNT };  // the tiles below; -1: the 256 x 256 kernel
struct Shape {
  int bm, bn, bkb;
};
constexpr Shape SHAPES[T_COUNT] = {{32, 64, 256},  {32, 128, 256},  {64, 64, 256},
                                   {64, 64, 256},  {128, 128, 128}, {256, 128, 128}};
// T32, T32W and T64N hold all rows (B is read once), the others share B in L2 between row tiles. T64N and T64 are
// one kernel with two cost lines: one row tile, or several. The ring holds at most 64 KB in flight
// per CU: more stages made the LDS-DMA instructions wait at issue (T128 at 1024 x 4096 x 4096: 39 us with
// 3 stages, 44 with 4).
template <int EL, bool TB>
using C32 = Cfg<EL, TB, 32, 64, 32, 32, 256, 4>;
template <int EL, bool TB>
using C32W = Cfg<EL, TB, 32, 128, 32, 32, 256, 3>;
template <int EL, bool TB>
using C64 = Cfg<EL, TB, 64, 64, 32, 32, 256, 3>;
template <int EL, bool TB>
using C128 = Cfg<EL, TB, 128, 128, 64, 64, 128, 3>;
template <int EL, bool TB>
using C256 = Cfg<EL, TB, 256, 128, 64, 64, 128, 3>;

struct Plan {
  int tile, ns;
};
// The cheapest (tile, split) by a model of the time in us: a launch, its rounds of 256 workgroups
// times their k-tiles (dearer the more CUs share L2 and memory), and for a split the exchange. The
// coefficients are a fit to measured times of the tiles and splits at M 1-4096, N and K 512-57344.
// max_ns 1: no split.
// dual: both matrices of run_swiglu, N columns in all; only_tiles: not the 256 x 256 kernel.
inline Plan choose(bool fp8, bool trans_b, int64_t M, int64_t N, int64_t K, int max_ns,
                   bool dual = false, bool only_tiles = false) {
  struct Cost {
    double a, b0, b1;  // launch; per k-tile alone; more per k-tile with every CU at work
  };
  static constexpr Cost C16[T_COUNT + 1] = {{4.35, 0.25, 0.27}, {4.34, 0.365, 0.385}, {4.8, 0.555, 0.065},
                                            {4.7, 0.23, 0.32},  {6.0, 0.37, 0.16},    {6.3, 0.54, 0.355},
                                            {7.6, 1.05, 0.27}};
  static constexpr Cost C8[T_COUNT + 1] = {{0.9, 0.305, 0.02}, {0, 1e9, 0},       {6.0, 0.265, 0.01},
                                           {3.7, 0.2, 0.445},  {6.5, 0.3, 0.25},  {7.0, 0.86, 0.025},
                                           {16.0, 0.21, 1.04}};
  const int64_t kb = K * (fp8 ? 1 : 2);
  auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  auto run = [](const Cost& c, int64_t wg, int64_t kt) {
    const double rounds = (double)((wg + 255) / 256);
    return c.a + rounds * (double)kt * (c.b0 + c.b1 * (double)wg / rounds / 256.0);
  };
  const Cost* const cost = fp8 ? C8 : C16;
  const bool only32 = fp8 && M <= 16;  // the one tile with an fp16 product
  const size_t part_bytes = tlm_split_bytes(!fp8 && !dual && M <= 16);
  Plan best{-1, 1};
  double t_best = only32 || only_tiles ? 1e300 : run(cost[T_COUNT], tiles(256, 256), (kb + 127) / 128);
  if (dual) t_best += 10.0 + (double)M * (double)N * 3e-6 / 6.0;  // two more launches, SwiGLU's bytes
  for (int t = 0; t < T_COUNT; ++t) {
    if (only32 && t != T32) continue;
    if ((t == T32 || t == T32W) && M > 32) continue;
    // wider rows for row-major B; the pairs of column tiles of a dual product
    if ((t == T32W && trans_b && !dual) || (t == T32 && dual)) continue;
    if ((t == T64N) != (M <= 64) && (t == T64N || t == T64)) continue;
    const Shape s = SHAPES[t];
    const int64_t tl = tiles(s.bm, s.bn), kt = (kb + s.bkb - 1) / s.bkb;
    for (int ns = 1; ns <= max_ns; ++ns) {
      const int64_t wg = tl * ns;
      if (wg * THREADS > UINT32_MAX) break;  // a launch counts its threads in 32 bits
      if (ns > 1 && (wg > TLM_SPLIT_TILES || kt < 2 * ns ||
                     (size_t)wg * s.bm * s.bn * 4 > part_bytes))
        break;
      double t_us = run(cost[t], wg, (kt + ns - 1) / ns);
      if (ns > 1)
        t_us += 0.6 + 0.1 * ns + 0.5 * s.bm * s.bn / 4096.0 * (wg < 256 ? (double)wg / 256.0 : 1.0);
      if (t_us < t_best) {
        t_best = t_us;
        best = Plan{t, ns};
      }
    }
  }
  return best;
}

template <typename CF, int OUT>
void launch_tile(const void* A, const void* B, void* C, int M, int N, int K, int ns, float* part,
                 unsigned* arrivals, hipStream_t s, const uint8_t* B2 = nullptr) {
  const int64_t wg = (int64_t)((M + CF::BM - 1) / CF::BM) * ((N + CF::BNC - 1) / CF::BNC) * ns;
  gemm_tile<CF, OUT><<<(unsigned)wg, THREADS, 0, s>>>((const uint8_t*)A, (const uint8_t*)B, C, M, N,
                                                      K, ns, part, arrivals, B2);
}

// Whether a call on stream `s` may split K. hipStreamPerThread is one handle for a stream of every thread, so
// it can own no workspace. Inside a capture only calls that may keep the captured stream's workspace
// (`graph_ok`) split, so that other graphs captured on one stream may be replayed side by side.
inline bool may_split(hipStream_t s, bool captured, bool graph_ok) {
  return s != hipStreamPerThread && (graph_ok || !captured);
}
inline bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}
inline bool split_workspace(bool decode, hipStream_t s, bool graph_ok, float** part,
                            unsigned** arrivals) {
  return may_split(s, s != hipStreamPerThread && !graph_ok && capturing(s), graph_ok) &&
         tlm_split_slot(decode, s, part, arrivals);
}

// The tile and split of a call on 16-byte aligned operands; tile -1: the 256 x 256 kernel (also where the shape
// does not fit the tiles' 32-bit offsets).
inline Plan plan_tiles(bool fp8, bool trans_b, int64_t M, int64_t N, int64_t K, bool split) {
  constexpr int64_t LIM = 0x7ffffff0;
  if (256 * K * (fp8 ? 1 : 2) >= LIM || (!trans_b && 128 * N * 2 >= LIM) || K <= 0) return Plan{-1, 1};
  return choose(fp8, trans_b, M, N, K, split ? 16 : 1);
}

// Runs the plan's tile; false for tile -1.
template <int EL, bool TB, int OUT>
bool run_tiles(Plan p, const void* A, const void* B, void* C, int M, int N, int K, float* part,
               unsigned* arrivals, hipStream_t s) {
  constexpr bool FP8 = EL >= EL_E4M3;
  switch (p.tile) {
    case T32:
      // 16 rows or fewer of fp8 are multiplied as fp16, which costs nothing beside B's stream and
      // keeps the accuracy of the per-output kernel that took them before
      if constexpr (FP8) {
        if (M <= 16) {
          launch_tile<Cfg<EL, TB, 32, 64, 32, 32, 256, 4, true>, OUT>(A, B, C, M, N, K, p.ns, part,
                                                                           arrivals, s);
          return true;
        }
      }
      launch_tile<C32<EL, TB>, OUT>(A, B, C, M, N, K, p.ns, part, arrivals, s);
      return true;
    case T32W:
      if constexpr (!TB) launch_tile<C32W<EL, TB>, OUT>(A, B, C, M, N, K, p.ns, part, arrivals, s);
      return !TB;
    case T64N:
    case T64: launch_tile<C64<EL, TB>, OUT>(A, B, C, M, N, K, p.ns, part, arrivals, s); return true;
    case T128: launch_tile<C128<EL, TB>, OUT>(A, B, C, M, N, K, p.ns, part, arrivals, s); return true;
    case T256: launch_tile<C256<EL, TB>, OUT>(A, B, C, M, N, K, p.ns, part, arrivals, s); return true;
    default: return false;
  }
}

// ---- up * silu(gate) of two products with one A: gate = A B^T, up = A B2^T, both [M, N]. The MLP of
// 64 tokens (7168 x 2048) spent its time in launches and their gaps: two products, SwiGLU (4.6 us for
// 0.8 MB) and the down product took 46.5 us; with the first three in one kernel 27.3.
// Without a split a call that may not split still takes a tile, so that tlm_gemm_swiglu_tmp_bytes holds for
// every stream.
inline Plan dual_plan(int64_t M, int64_t N, int64_t K, bool split) {
  if (256 * K * 2 >= 0x7ffffff0 || K <= 0 || K % 8) return Plan{-1, 1};
  const Plan p = choose(false, true, M, 2 * N, K, 16, true);
  return p.tile < 0 || p.ns == 1 || split ? p : choose(false, true, M, 2 * N, K, 1, true, true);
}
template <int EL, int OUT>
void run_swiglu(Plan p, const void* A, const void* B, const void* B2, void* C, int M, int N, int K,
                hipStream_t s) {
  float* part = nullptr;
  unsigned* arrivals = nullptr;
  if (p.ns > 1 && !split_workspace(false, s, false, &part, &arrivals)) p = dual_plan(M, N, K, false);
  const uint8_t* const b2 = (const uint8_t*)B2;
  switch (p.tile) {
    case T32W:
      launch_tile<Cfg<EL, true, 32, 128, 32, 64, 256, 3, false, true>, OUT>(
          A, B, C, M, N, K, p.ns, part, arrivals, s, b2);
      break;
    case T64N:
    case T64:
      launch_tile<Cfg<EL, true, 64, 64, 32, 32, 256, 3, false, true>, OUT>(
          A, B, C, M, N, K, p.ns, part, arrivals, s, b2);
      break;
    case T128:
      launch_tile<Cfg<EL, true, 128, 128, 64, 64, 128, 3, false, true>, OUT>(
          A, B, C, M, N, K, p.ns, part, arrivals, s, b2);
      break;
    default:
      launch_tile<Cfg<EL, true, 256, 128, 64, 64, 128, 3, false, true>, OUT>(
          A, B, C, M, N, K, p.ns, part, arrivals, s, b2);
  }
}

}  // namespace gt
