// MLA paged decode over a 16-bit (fp16 / bf16) latent cache on the matrix cores, balanced over the batch.
//
// Reference: examples/deepseek_mla/example_mla_decode_paged.py:100-221 (see tlm_mla.hip); the result
// of its split kernel and combine without the program's own split partition. dv 512, dpe 64, query
// heads a multiple of 64.
//
// What bounds it: fixed costs at small batches, the tile's own chain at large ones. 8 sequences of
// 500 .. 4,000 tokens, 128 heads (bf16): 26.0 us and 8.2 us for the combine, where the split kernel that
// it replaced took 67.2 and 14.7; 20.7 MB of cache rows would take 3.1 us. Inside a workgroup 1.6 us go to the
// scan, 5 to the block table and Q, 2.6 to the first tile and 2 to 4 to the partial rows (33 MB of fp32 for
// 128 ranges, written and read again); the rest is the launch. 16 x 4,000 .. 8,000 tokens: 65 to 67 us, of which
// a 32-token tile takes 1.9 with the next ones already there. It has 1,100 cycles of MFMA issue per SIMD
// and 1,450 of LDS reads per CU (K and V^T operands, 140 KB); leaving out the loads or the MFMAs, or
// taking the rows from L2, changes the kernel's time by less than 5 %: the chain read, multiply, exchange,
// softmax, barrier is what remains, with two waves per SIMD to overlap it.
//
//   * Partition: sequence b costs its 32-token tiles plus MH_PIECE for fetching Q and writing rows; the cost
//     line of the batch is cut into G equal ranges, one per workgroup and 64 heads. A sequence
//     inside one range is written to the output directly; the pieces of others go to slots (fp32
//     normalised O and log2 sum-exp) that mla_h16_combine merges. Every workgroup finds its own range
//     from the lengths (a block scan), so there is no preparing launch.
//   * Wave (hg, th, dh): 32 heads (hg). For S^T, 16 of the tile's tokens (th) over one half of the 576 dims
//     (Q in 72 registers; all of Q would take 144 and spill). The four waves of a head group then exchange their
//     partial sums (12 KB of LDS traffic a tile) so that each finishes 32 tokens x 8 heads, whose maximum it
//     has in its own lanes. P^T goes through LDS, and the wave multiplies V^T rows 128 (2 th + dh) .. + 127 of
//     all 32 tokens. The earlier kernel split the 576 dims four ways, exchanged 160 KB of partial scores per 32
//     tokens and repeated the softmax in four waves.
//   * Softmax against the running maximum of each head, so that the largest weight is exactly 1 in 16 bits
//     and a piece may start with tiles that score -inf. O is rescaled beside the MFMAs. Against a reference that
//     only the first tile set (kept until some P left the 16-bit range, error 2.0e-3 of fp64 instead of 1.9e-3
//     in bf16): 16 x 4,000 .. 8,000 tokens 66.4 -> 69.6 us, 8 x 500 .. 4,000 31.4 -> 31.8. Finishing 16 tokens x
//     16 heads per wave, the halves' maxima meeting in LDS behind a fourth barrier: 72.2 and 32.3.
//   * Tiles stream through a four-stage LDS ring by LDS-DMA (latent rows one 1 KB instruction per token, rope
//     rows 8 tokens per instruction). The cache rows of 512 tokens at a time are looked up half a block
//     ahead into an LDS table. 16-byte chunk c of token r sits at c ^ f(r), f(r) = 2 (r % 8) + r / 8 % 2:
//     16 tokens' reads of one chunk column (S^T) and the transposed reads of 8 tokens x 2 chunks (V^T)
//     both fall on all banks.
#include "tlm_common.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace {

constexpr int MH_DV = 512, MH_DPE = 64;
constexpr int MH_HEADS = 64;                    // heads per workgroup
constexpr int MH_BN = 32;                       // tokens per tile
constexpr int MH_PIECE = 6;                     // cost of a piece beside its tiles, in tiles
constexpr int MH_LAT = MH_BN * MH_DV * 2;       // bytes of a tile's latent rows
constexpr int MH_STAGE = MH_LAT + MH_BN * MH_DPE * 2;
constexpr int MH_NST = 4;
// Per wave 1.5 KB: the half scores of its 8 heads that the three other waves of its 32 heads bring (3 x 512
// bytes) and, once it has read them, its P^T block (512 bytes) and 8 factors, row sums and maxima.
constexpr int MH_P = MH_NST * MH_STAGE, MH_BOX = 1536, MH_BOX_X = 512;
constexpr int MH_TBL = 512;                     // tokens of a look-up block; two blocks
constexpr int MH_TBL_TILES = MH_TBL / MH_BN;
constexpr uint32_t MH_NO_ROW = 0xffffffffu;  // (rows are 1 KB or more: memory ends before the 2^32nd)
constexpr int MH_ROWS = MH_P + 8 * MH_BOX;
constexpr int MH_SMEM = MH_ROWS + 2 * MH_TBL * 4;
static_assert(MH_SMEM <= 160 * 1024, "LDS");

struct MhArgs {
  const uint16_t* q;
  const uint16_t* q_pe;
  int64_t qs, qpes;
  const uint8_t* kv;
  const uint8_t* k_pe;
  int64_t kvs_b, kpes_b, kv_rows;
  const int32_t* bt;
  const int32_t* sl;
  uint16_t* out;
  float* ws_o;    // [slots][Hq][512]
  float* ws_lse;  // [slots][Hq]
  int B, Hq, page, max_pages, G;
  float c;  // sm_scale log2(e)
};

template <bool BF16>
TLM_DEV f32x4 mh_mma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

using namespace ldsop;
template <int OFF>
TLM_DEV void ds_b64(u32x2& r, uint32_t a) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset is 16 bits");
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(a), "i"(OFF) : "memory");
}
// An accumulator: the compiler does not see an asm operand's hazard with the MFMA that has just been
// issued for it, and 16 wait states cover a 16x16x32 MFMA's result.
TLM_DEV void ds_put_acc(uint32_t a, f32x4 v) {
  asm volatile("s_nop 15\n\tds_write_b128 %0, %1" ::"v"(a), "v"(v) : "memory");
}
TLM_DEV void ds_put64(uint32_t a, u32x2 v) {
  asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(v) : "memory");
}
TLM_DEV void ds_put32(uint32_t a, uint32_t v) {
  asm volatile("ds_write_b32 %0, %1" ::"v"(a), "v"(v) : "memory");
}
TLM_DEV uint32_t ds_get32(uint32_t a) {  // waits for the value
  uint32_t r;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(r) : "v"(a) : "memory");
  return r;
}
template <int N>
TLM_DEV void lgkm_wait() {
  static_assert(N >= 0 && N < 16, "lgkmcnt is 4 bits");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f | (N << 8));
  __builtin_amdgcn_sched_barrier(0);
}
template <int N>
TLM_DEV void vm_wait() {  // all but the last N vector loads and LDS-DMA instructions of this wave have landed
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x3f70 | (N & 15) | ((N >> 4) << 14));
  __builtin_amdgcn_sched_barrier(0);
}
// Workgroup barrier: this wave's LDS accesses are done; LDS-DMA loads stay in flight.
TLM_DEV void mh_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
TLM_DEV float mh_ror8(float x) {  // of lane l ^ 8
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x128, 0xf, 0xf, false));
}
TLM_DEV int mh_tiles(const MhArgs& a, int b) {
  const int L = max(0, min(a.sl[b], a.max_pages * a.page));
  return (L + MH_BN - 1) / MH_BN;
}
TLM_DEV int mh_cost(int tiles) { return tiles > 0 ? tiles + MH_PIECE : 0; }

// Slots. The G - 1 cuts between ranges give at most one piece per range r >= 1 that starts inside a
// sequence (slot r - 1), and the piece at the start of a cut sequence: one per sequence or one per range
// but the last, whichever are fewer.
TLM_DEV int mh_tail_slot(int r) { return r - 1; }
TLM_DEV int mh_head_slot(const MhArgs& a, int r, int b) { return a.G - 1 + (a.B < a.G ? b : r); }

// Ranges of the cost line: range r of g starts at floor(r total / g) (g <= 256: 32-bit products).
TLM_DEV int mh_range(int total, int g, int r) {
  const uint32_t q = (uint32_t)total / (uint32_t)g, rem = (uint32_t)total % (uint32_t)g;
  return (int)(q * (uint32_t)r + rem * (uint32_t)r / (uint32_t)g);
}
TLM_DEV int mh_range_of(int total, int g, int x) {  // the range that holds position x
  int r = min(g - 1, (int)((float)x * (float)g / (float)total));
  while (mh_range(total, g, r) > x) --r;
  while (r + 1 < g && mh_range(total, g, r + 1) <= x) ++r;
  return r;
}

// Cost line of the batch, by a block of NT threads: each takes a contiguous chunk of sequences (one in
// batches of up to NT, whose length it then loads once). The chunk that holds the wanted point, a position
// (FIND_SEQ = false) or a sequence, reports the sequence and the cost before it. `sh`: NT / 64 + 2 ints.
struct MhPoint {
  int total, seq, before;
};
template <int NT, bool FIND_SEQ, typename F>
TLM_DEV MhPoint mh_scan(const MhArgs& a, int* sh, F&& want) {
  const int tid = threadIdx.x;
  const int per = (a.B + NT - 1) / NT;
  const int b0 = min(a.B, tid * per), b1 = min(a.B, b0 + per);
  int mine = 0;
  for (int b = b0; b < b1; ++b) mine += mh_cost(mh_tiles(a, b));
  // inclusive scan over the wave, then over the waves
  int x = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if ((tid & 63) >= o) x += y;
  }
  if ((tid & 63) == 63) sh[tid >> 6] = x;
  __syncthreads();
  MhPoint pt{0, 0, 0};
  int pre = x - mine;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    const int v = sh[i];
    if (i < tid >> 6) pre += v;
    pt.total += v;
  }
  const int at = want(pt.total);
  if (FIND_SEQ ? at >= b0 && at < b1 : at >= pre && at < pre + mine) {
    int p = pre, b = b0;
    for (; b < b1 - 1; ++b) {
      if (FIND_SEQ && b == at) break;
      const int cst = mh_cost(mh_tiles(a, b));
      if (!FIND_SEQ && at < p + cst) break;
      p += cst;
    }
    sh[NT / 64] = b;
    sh[NT / 64 + 1] = p;
  }
  __syncthreads();
  pt.seq = sh[NT / 64];
  pt.before = sh[NT / 64 + 1];
  return pt;
}

__device__ const u32x4 mh_zero_row[MH_DPE * 2 / 16] = {};  // rope row of a token without one

template <bool BF16, bool O_BF16>
__global__ __launch_bounds__(512, 1) void mla_h16_decode(const MhArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // device builtins inside generic lambdas: no host instantiation
  using HH = h16<BF16>;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[MH_SMEM];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hg = wave >> 2, w = wave & 3;
  const int th = w >> 1, dh = w & 1;  // S^T: token half, dim half
  const int g = lane >> 4, jl = lane & 15;
  const int hblocks = a.Hq / MH_HEADS;
  // the head blocks of a range share its tiles: on one XCD (id % 8) where the ranges divide evenly
  int hb, r;
  if (a.G % 8 == 0) {
    hb = (blockIdx.x >> 3) % hblocks;
    r = (blockIdx.x >> 3) / hblocks * 8 + (blockIdx.x & 7);
  } else {
    hb = blockIdx.x % hblocks;
    r = blockIdx.x / hblocks;
  }

  // fewer cost units than ranges: one each for the first
  int lo = 0, hi = 0;
  const MhPoint start = mh_scan<512, false>(a, (int*)(smem + MH_P), [&](int total) {
    const int ng = min(a.G, total);
    if (r < ng) {
      lo = mh_range(total, ng, r);
      hi = mh_range(total, ng, r + 1);
    }
    return r < ng ? lo : -1;
  });
  if (lo >= hi) return;  // whole workgroup
  int seq_before = start.before;

  const uint32_t s0 = lds_u32(smem);  // 1 KB aligned: the XORs below stay within a row
  auto f_swz = [](int t) { return ((t & 7) << 1) | ((t >> 3) & 1); };
  // S^T: A operand = K row 16 th + jl, chunk 4 ks + g (rope: chunk g of the rope row): k_a ^ 64 (ks % 4), ks / 4
  // as an immediate
  const uint32_t k_a = s0 + (uint32_t)((16 * th + jl) * (MH_DV * 2) + 16 * (g ^ f_swz(jl)));
  const uint32_t r_a = s0 + (uint32_t)(MH_LAT + (16 * th + jl) * (MH_DPE * 2) +
                                       16 * (g ^ ((jl >> 1) & 7)));  // ^ 64 for the upper half
  // V^T: 16-lane group g, lane jl reads 4 dims 16 dt + 4 (jl % 4) of token 4 g + jl / 4 (+ 16 for the second
  // read) and receives dim 16 dt + jl of the four tokens. The chunk of d-tile dt is 16 w + 2 dt +
  // (jl % 4) / 2, stored at ^ f(token): v_a ^ 32 dt; tokens 16 apart share f.
  const int vt = 4 * g + (jl >> 2);
  const uint32_t v_a = s0 + (uint32_t)(vt * (MH_DV * 2) + 256 * w +
                                       16 * (((jl & 3) >> 1) ^ f_swz(vt)) + 8 * (jl & 1));
  // Exchange (the boxes of the four waves of a head group). Wave w finishes heads 8 w .. + 7 of the group's 32:
  // lane (g, jl) head 8 w + jl % 8 and, where jl / 8 == dh, the wave's own 16 tokens 4 g + i, else the other
  // half's. Block 0 of its box comes from the wave of the other dims (the own quarter stays in
  // registers), blocks 1 and 2 from the waves of the other tokens; the ^ 8 and ^ 2 keep the two
  // halves jl / 8 of an access on different banks.
  const int oct = jl >> 3, pos = g * 8 + (jl & 7);
  const bool own = oct == dh;
  const int t_fin = own ? th : 1 - th;  // token half that the lane finishes
  const uint32_t box_hg = s0 + MH_P + (uint32_t)(4 * hg) * MH_BOX, box = box_hg + (uint32_t)w * MH_BOX;
  const uint32_t put_dims = box_hg + (uint32_t)((w ^ 1) * MH_BOX + (pos ^ 8 * (dh ^ 1)) * 16);
  const uint32_t put_toks = box_hg + (uint32_t)((2 * (1 - th) + oct) * MH_BOX + (1 + dh) * 512 +
                                                (pos ^ 8 * (oct ^ dh ^ 1)) * 16);
  const uint32_t get_1 = box + (uint32_t)((own ? 0 : 512) + (pos ^ 8 * (own ? dh : dh ^ 1)) * 16);
  const uint32_t get_2 = box + (uint32_t)(1024 + (pos ^ 8 * dh) * 16);
  // P^T: token half t2, lane group, head, 4 tokens; the reader takes head jl of the group's tiles hh (+ 2 hh boxes)
  const uint32_t put_p = box + (uint32_t)(t_fin * 256 + (g ^ 2 * (t_fin ^ dh)) * 64 + (jl & 7) * 8);
  const uint32_t get_p0 = box_hg + (uint32_t)(oct * MH_BOX + (g ^ 2 * oct) * 64 + (jl & 7) * 8);
  const uint32_t get_p1 = box_hg + (uint32_t)(oct * MH_BOX + 256 + (g ^ 2 * (oct ^ 1)) * 64 + (jl & 7) * 8);
  // one value per head (every lane of a head writes the same)
  const uint32_t put_x = box + (uint32_t)(MH_BOX_X + (jl & 7) * 4);
  const uint32_t get_x = box_hg + (uint32_t)(oct * MH_BOX + MH_BOX_X + (jl & 7) * 4);
  const uint32_t row_tbl = s0 + MH_ROWS;
  const bool rope_wave = wave < 4;

  for (int b = start.seq; b < a.B && seq_before < hi; ++b) {
    const int L = max(0, min(a.sl[b], a.max_pages * a.page));
    const int tiles = (L + MH_BN - 1) / MH_BN;
    const int cst = mh_cost(tiles);
    const int first = seq_before + MH_PIECE;  // cost position of tile 0
    const int t0 = max(0, min(tiles, lo - first));
    const int t1 = max(0, min(tiles, hi - first));
    seq_before += cst;
    if (t0 >= t1) continue;
    const int n = t1 - t0;

    // ---- cache rows of look-up block k (512 tokens from tile t0 + 16 k): one token per thread
    const int32_t* const bt = a.bt + (int64_t)b * a.max_pages;
    auto token = [&](int k) { return t0 * MH_BN + k * MH_TBL + tid; };
    auto entry = [&](int k) { return token(k) < L ? bt[token(k) / a.page] : -1; };
    auto put_row = [&](int k, int e) {
      const int64_t row = (int64_t)e * a.page + token(k) % a.page;
      const bool ok = token(k) < L && e >= 0 && row < a.kv_rows && row < MH_NO_ROW;
      ds_put32(row_tbl + (uint32_t)(((k & 1) * MH_TBL + tid) * 4), ok ? (uint32_t)row : MH_NO_ROW);
    };
    // ---- loads of tile i of the piece: the wave's four latent rows, and eight rope rows (waves 0 .. 3)
    auto issue = [&](int i) __attribute__((always_inline)) {
      // lane l < 32: row of token l of the tile
      const uint32_t rv = ds_get32(row_tbl + (uint32_t)((i & (2 * MH_TBL_TILES - 1)) * MH_BN * 4 + (lane & 31) * 4));
      const int stage = i & (MH_NST - 1);
      uint8_t* const dst = smem + stage * MH_STAGE;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t ri = __builtin_amdgcn_readlane(rv, 4 * wave + k);
        const bool ok = ri != MH_NO_ROW;  // uniform; rows outside the pool and past the length read as zeros
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(a.kv + (int64_t)(ok ? ri : 0) * a.kvs_b), (short)0, ok ? MH_DV * 2 : 0, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rs, (__attribute__((address_space(3))) void*)(dst + (4 * wave + k) * (MH_DV * 2)), 16,
            16 * (lane ^ f_swz(4 * wave + k)), 0, 0, 0);
      }
      if (rope_wave) {
        const int t = 8 * wave + (lane >> 3);
        const uint32_t ri = (uint32_t)__shfl((int)rv, t, 64);
        const uint8_t* const src =
            ri != MH_NO_ROW ? a.k_pe + (int64_t)ri * a.kpes_b : (const uint8_t*)mh_zero_row;
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(src + 16 * ((lane & 7) ^ ((t >> 1) & 7))),
            (__attribute__((address_space(3))) void*)(dst + MH_LAT + 1024 * wave), 16, 0, 0);
      }
    };

    const int ent0 = entry(0);
    // ---- Q^T operand: heads 16 hh + jl of the wave's 32, dims 32 ks + 8 g .. of k-steps ks = 9 dh + i
    u32x4 qreg[2][9];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int64_t row = (int64_t)b * a.Hq + hb * MH_HEADS + 32 * hg + 16 * hh + jl;
      const uint16_t* const qr = a.q + row * a.qs + 288 * dh + 8 * g;
      const uint16_t* const pr = a.q_pe + row * a.qpes + 8 * g;
#pragma unroll
      for (int i = 0; i < 9; ++i)
        qreg[hh][i] = *(const u32x4*)(dh && i >= 7 ? pr + 32 * (i - 7) : qr + 32 * i);
    }
    mh_barrier();  // the previous piece's (or the scan's) last LDS accesses
    put_row(0, ent0);
    mh_barrier();  // the table's first block
    issue(0);
    // waited for here, behind the first tile's loads only: inside the loop the compiler would wait for every
    // load
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int i = 0; i < 9; ++i) landed(qreg[hh][i]);
#pragma unroll
    for (int i = 1; i < MH_NST - 1; ++i)
      if (i < n) issue(i);
    int ent = -1;
    f32x4 oacc[8][2];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) oacc[dt][0] = oacc[dt][1] = f32x4{};
    float m = -INFINITY, l = 0.f;  // of the head that the lane finishes (l: of its tokens)

    for (int t = 0; t < n; ++t) {
      const int left = min(MH_NST - 2, n - 1 - t);  // later tiles whose loads may stay in flight
      if (left == 2) {
        if (rope_wave) vm_wait<10>(); else vm_wait<8>();
      } else if (left == 1) {
        if (rope_wave) vm_wait<5>(); else vm_wait<4>();
      } else {
        vm_wait<0>();
      }
      mh_barrier();  // tile t is whole; tile t - 1's stage is free
      if ((t & (MH_TBL_TILES - 1)) == 0) {
        if (t + MH_TBL_TILES < n) ent = entry(t / MH_TBL_TILES + 1);
      } else if ((t & (MH_TBL_TILES - 1)) == MH_TBL_TILES / 2) {
        if (t + MH_TBL_TILES / 2 < n) put_row(t / MH_TBL_TILES + 1, ent);
      }
      if (t + MH_NST - 1 < n) issue(t + MH_NST - 1);
      const uint32_t so = (uint32_t)((t & (MH_NST - 1)) * MH_STAGE);

      // ---- S^T = K Q^T: half the dims of 16 tokens x 32 heads, then the sums of 32 tokens x 8 heads
      f32x4 h[2] = {f32x4{}, f32x4{}};
      auto scores = [&](auto dc) __attribute__((always_inline)) {
        constexpr int DH = decltype(dc)::value, DEPTH = 6;
        u32x4 op[DEPTH];
        const uint32_t ka = k_a + so, ra = r_a + so;
        auto read = [&](auto ic) __attribute__((always_inline)) {
          constexpr int n_ = decltype(ic)::value, ks = 9 * DH + n_;
          if constexpr (n_ < 9) {
            if constexpr (ks < 16)
              ds_b128<(ks >> 2) * 256>(op[n_ % DEPTH], ka ^ (64 * (ks & 3)));
            else
              ds_b128<0>(op[n_ % DEPTH], ra ^ (64 * (ks - 16)));
          }
        };
        unroll<0, DEPTH - 1>(read);
        unroll<0, 9>([&](auto ic) __attribute__((always_inline)) {
          constexpr int n_ = decltype(ic)::value;
          read(std::integral_constant<int, n_ + DEPTH - 1>{});
          constexpr int ahead = 8 - n_ < DEPTH - 1 ? 8 - n_ : DEPTH - 1;
          lgkm_wait<ahead>();
          landed(op[n_ % DEPTH]);
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) h[hh] = mh_mma<BF16>(op[n_ % DEPTH], qreg[hh][n_], h[hh]);
        });
      };
      if (dh == 0)
        scores(std::integral_constant<int, 0>{});
      else
        scores(std::integral_constant<int, 1>{});
      const f32x4 h_own = th ? h[1] : h[0], h_oth = th ? h[0] : h[1];
      if (!own) ds_put_acc(put_dims, h_own);
      ds_put_acc(put_toks, h_oth);
      mh_barrier();
      f32x4 s;
      {
        u32x4 in1, in2;
        ds_b128<0>(in1, get_1);
        ds_b128<0>(in2, get_2);
        lgkm_wait<0>();
        landed(in1);
        landed(in2);
        s = __builtin_bit_cast(f32x4, in1) + (own ? h_own : __builtin_bit_cast(f32x4, in2));
      }
      // the first V^T operands: they arrive while the weights are made
      constexpr int VDEPTH = 5;
      u32x2 vl[VDEPTH], vh[VDEPTH];
      const uint32_t va = v_a + so;
      auto read_v = [&](auto ic) __attribute__((always_inline)) {
        constexpr int dt = decltype(ic)::value;
        if constexpr (dt < 8) {
          ds_tr16<0>(vl[dt % VDEPTH], va ^ (32 * dt));
          ds_tr16<16 * MH_DV * 2>(vh[dt % VDEPTH], va ^ (32 * dt));
        }
      };
      unroll<0, VDEPTH - 1>(read_v);
      // ---- weights against the running maximum of the lane's head
      const int tok = (t0 + t) * MH_BN + 16 * t_fin + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = tok + i < L ? s[i] * a.c : -INFINITY;
      {
        float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        mx = fmaxf(mx, mh_ror8(mx));
        mx = fmaxf(m, xhalf_max(xrow_max(mx)));
        const float al = mx == -INFINITY ? 1.f : fast_exp2(m - mx);
        const float mm = mx == -INFINITY ? 0.f : mx;
        m = mx;
        f32x4 p;
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = fast_exp2(s[i] - mm);
        l = l * al + ((p[0] + p[1]) + (p[2] + p[3]));
        ds_put64(put_p, u32x2{HH::pack(p[0], p[1]), HH::pack(p[2], p[3])});
        ds_put32(put_x, __float_as_uint(al));
      }
      mh_barrier();  // every wave's P^T and factors are in LDS, and this wave's V^T operands have landed
#pragma unroll
      for (int i = 0; i < VDEPTH - 1; ++i) {
        landed(vl[i]);
        landed(vh[i]);
      }

      // ---- O^T += V^T P^T: dims 128 w .. of the wave's 32 heads over the tile's 32 tokens
      u32x2 pb[2][2], al;  // [head tile][token half]; the factors of the two head tiles
      asm volatile("ds_read2st64_b32 %0, %1 offset1:%2" : "=v"(al) : "v"(get_x), "i"(2 * MH_BOX / 256) : "memory");
      unroll<0, 2>([&](auto ic) __attribute__((always_inline)) {
        constexpr int hh = decltype(ic)::value;
        ds_b64<2 * hh * MH_BOX>(pb[hh][0], get_p0);
        ds_b64<2 * hh * MH_BOX>(pb[hh][1], get_p1);
      });
      lgkm_wait<0>();
      landed(al);
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        landed(pb[hh][0]);
        landed(pb[hh][1]);
      }
      // O's rescale of d-tile dt + 1 runs beside the MFMAs of d-tile dt
      auto rescale = [&](auto ic) __attribute__((always_inline)) {
        constexpr int dt = decltype(ic)::value;
        if constexpr (dt < 8) {
          oacc[dt][0] *= __uint_as_float(al[0]);
          oacc[dt][1] *= __uint_as_float(al[1]);
        }
      };
      rescale(std::integral_constant<int, 0>{});
      unroll<0, 8>([&](auto ic) __attribute__((always_inline)) {
        constexpr int dt = decltype(ic)::value;
        read_v(std::integral_constant<int, dt + VDEPTH - 1>{});
        if constexpr (dt >= VDEPTH - 1) {
          constexpr int ahead = 2 * (7 - dt < VDEPTH - 1 ? 7 - dt : VDEPTH - 1);
          lgkm_wait<ahead>();
          landed(vl[dt % VDEPTH]);
          landed(vh[dt % VDEPTH]);
        }
        const u32x4 v = {vl[dt % VDEPTH][0], vl[dt % VDEPTH][1], vh[dt % VDEPTH][0], vh[dt % VDEPTH][1]};
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const u32x4 p = {pb[hh][0][0], pb[hh][0][1], pb[hh][1][0], pb[hh][1][1]};
          oacc[dt][hh] = mh_mma<BF16>(v, p, oacc[dt][hh]);
        }
        rescale(std::integral_constant<int, dt + 1>{});
      });
    }

    // ---- end of the piece: row sums over the lanes of a head
    mh_barrier();  // the exchange area's last readers are done
    {
      float x = l + mh_ror8(l);
      x += __shfl_xor(x, 16, 64);
      x += __shfl_xor(x, 32, 64);
      ds_put32(put_x, __float_as_uint(x));
      ds_put32(put_x + 32, __float_as_uint(m));
    }
    mh_barrier();
    const bool whole = t0 == 0 && t1 == tiles;
    const int64_t slot = t0 == 0 ? mh_head_slot(a, r, b) : mh_tail_slot(r);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const float lt = __uint_as_float(ds_get32(get_x + 2 * hh * MH_BOX));
      const float inv = lt > 0.f ? 1.0f / lt : 0.f;
      const int head = hb * MH_HEADS + 32 * hg + 16 * hh + jl;
      if (whole) {
        using HO = h16<O_BF16>;
        uint16_t* const o = a.out + ((int64_t)b * a.Hq + head) * MH_DV + 128 * w + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          const f32x4 v = oacc[dt][hh] * inv;
          *(u32x2*)(o + 16 * dt) = u32x2{HO::pack(v[0], v[1]), HO::pack(v[2], v[3])};
        }
      } else {
        float* const o = a.ws_o + (slot * a.Hq + head) * MH_DV + 128 * w + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) *(f32x4*)(o + 16 * dt) = oacc[dt][hh] * inv;
        const float mt = __uint_as_float(ds_get32(get_x + 32 + 2 * hh * MH_BOX));
        if (w == 0 && g == 0) a.ws_lse[slot * a.Hq + head] = lt > 0.f ? mt + __log2f(lt) : -INFINITY;
      }
    }
  }
#endif
}

// Merge of the pieces of every sequence that no range holds whole, and zero rows for empty sequences. A wave
// per head and step, 8 dims per lane; MH_BATCH pieces' rows requested together. Bound by the partial rows
// (4 to 5 TB/s of 33 MB) after two dependent loads. Every workgroup scans the lengths, so a large batch has
// few per sequence: with one for every 4 heads, 4,096 sequences of 16 tokens took 1,307 us in all (now
// 413; the split kernel 1,102). Two waves a workgroup instead of four: 8.2 -> 8.0 us at 8 x 500 .. 4,000
// tokens, 11.0 -> 9.1 at 1 x 2,000.
constexpr int MH_CW = 2;  // waves per workgroup
constexpr int MH_CWGS = 4096;  // workgroups wanted
constexpr int MH_BATCH = 8;
template <bool O_BF16>
__global__ __launch_bounds__(64 * MH_CW) void mla_h16_combine(const MhArgs a) {
  __shared__ int sh[MH_CW + 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per_seq = gridDim.x / a.B, b = blockIdx.x / per_seq;
  const int head0 = blockIdx.x % per_seq * MH_CW + wave, step = per_seq * MH_CW;
  const int tiles = mh_tiles(a, b);
  using HO = h16<O_BF16>;
  uint16_t* const out_b = a.out + (int64_t)b * a.Hq * MH_DV + 8 * lane;
  if (tiles == 0) {
    for (int head = head0; head < a.Hq; head += step) {
      uint16_t* const out = out_b + (int64_t)head * MH_DV;
      *(u32x2*)out = u32x2{0, 0};
      *(u32x2*)(out + 4) = u32x2{0, 0};
    }
    return;
  }
  const MhPoint pt = mh_scan<64 * MH_CW, true>(a, sh, [&](int) { return b; });
  const int ng = min(a.G, pt.total), x0 = pt.before + MH_PIECE;
  const int r0 = mh_range_of(pt.total, ng, x0), r1 = mh_range_of(pt.total, ng, x0 + tiles - 1);
  if (r0 == r1) return;  // written whole
  const int np = r1 - r0 + 1;
  for (int head = head0; head < a.Hq; head += step) {
    uint16_t* const out = out_b + (int64_t)head * MH_DV;
    float mx = -INFINITY, sum = 0.f;
    f32x4 acc[2] = {f32x4{}, f32x4{}};
    for (int p0 = 0; p0 < np; p0 += MH_BATCH) {
      f32x4 v[MH_BATCH][2];
      float ls[MH_BATCH], top = mx;
#pragma unroll
      for (int i = 0; i < MH_BATCH; ++i) {
        ls[i] = -INFINITY;
        v[i][0] = v[i][1] = f32x4{};
        if (p0 + i < np) {
          const int p = p0 + i;
          const int64_t s = (int64_t)(p == 0 ? mh_head_slot(a, r0, b) : mh_tail_slot(r0 + p)) * a.Hq + head;
          ls[i] = a.ws_lse[s];
          const float* const o = a.ws_o + s * MH_DV + 8 * lane;
          v[i][0] = *(const f32x4*)o;
          v[i][1] = *(const f32x4*)(o + 4);
        }
      }
#pragma unroll
      for (int i = 0; i < MH_BATCH; ++i) top = fmaxf(top, ls[i]);
      const float al = mx == -INFINITY ? 0.f : fast_exp2(mx - top);
      mx = top;
      sum *= al;
      acc[0] *= al;
      acc[1] *= al;
#pragma unroll
      for (int i = 0; i < MH_BATCH; ++i) {
        const float wt = ls[i] == -INFINITY ? 0.f : fast_exp2(ls[i] - mx);
        sum += wt;
        acc[0] += v[i][0] * wt;
        acc[1] += v[i][1] * wt;
      }
    }
    const float inv = sum > 0.f ? 1.0f / sum : 0.f;
    acc[0] *= inv;
    acc[1] *= inv;
    *(u32x2*)out = u32x2{HO::pack(acc[0][0], acc[0][1]), HO::pack(acc[0][2], acc[0][3])};
    *(u32x2*)(out + 4) = u32x2{HO::pack(acc[1][0], acc[1][1]), HO::pack(acc[1][2], acc[1][3])};
  }
}

template <bool BF16, bool O_BF16>
int mh_launch(const MhArgs& a, hipStream_t st) {
  mla_h16_decode<BF16, O_BF16><<<(unsigned)(a.G * (a.Hq / MH_HEADS)), 512, 0, st>>>(a);
  TLM_LAUNCH_CHECK("tlm_mla_decode (16-bit)");
  const int per_seq = std::max(1, std::min(MH_CWGS / a.B, a.Hq / MH_CW));
  mla_h16_combine<O_BF16><<<(unsigned)(a.B * per_seq), 64 * MH_CW, 0, st>>>(a);
  TLM_LAUNCH_CHECK("tlm_mla_decode (16-bit combine)");
  return TLM_OK;
}

}  // namespace

// Ranges of a decode: one workgroup per CU at most, each holds a CU's whole LDS (one more starts when the first
// ends and takes as long: 16 x 8,000 tokens of 192 heads 199 us with 258 workgroups, 116 with 255), and
// as many as the slots (of Hq rows of 513 floats) take: G ranges use at most G - 1 + min(B, G - 1).
extern "C" int64_t tlm_mla_h16_ranges(int64_t B, int64_t Hq, size_t ws_bytes) {
  if (B <= 0 || Hq < MH_HEADS) return 0;
  const int64_t slots = (int64_t)(ws_bytes / ((size_t)Hq * (MH_DV + 1) * sizeof(float)));
  return std::max<int64_t>(
      1, std::min(256 / (Hq / MH_HEADS), std::max(slots - B, slots / 2) + 1));
}

// Balanced decode over a 16-bit cache on validated arguments of the matrix-core shape (tlm_mla.hip: dv 512,
// dpe 64, Hq a multiple of 64, 16-byte aligned rows). TLM_EUNSUPPORTED where every workgroup's own scan of the
// lengths would cost more than it saves.
int tlm_mla_h16_launch(const void* q, const void* q_pe, int64_t q_stride, int64_t q_pe_stride,
                       const void* kv, const void* k_pe, int64_t kv_stride, int64_t kpe_stride,
                       int64_t kv_rows, const int32_t* block_table, const int32_t* seqlens, void* o,
                       void* ws, size_t ws_bytes, int64_t B, int64_t Hq, int64_t page,
                       int64_t max_pages, float score_scale, bool bf16, bool o_bf16, void* stream) {
  // token and cost positions are 32-bit
  if (B > 4096 || max_pages * page > INT32_MAX / 2 ||
      B * (max_pages * page / MH_BN + 1 + MH_PIECE) > INT32_MAX / 2)
    return TLM_EUNSUPPORTED;
  const int64_t G = tlm_mla_h16_ranges(B, Hq, ws_bytes);
  MhArgs a;
  a.q = (const uint16_t*)q;
  a.q_pe = (const uint16_t*)q_pe;
  a.qs = q_stride;
  a.qpes = q_pe_stride;
  a.kv = (const uint8_t*)kv;
  a.k_pe = (const uint8_t*)k_pe;
  a.kvs_b = 2 * kv_stride;
  a.kpes_b = 2 * kpe_stride;
  a.kv_rows = kv_rows;
  a.bt = block_table;
  a.sl = seqlens;
  a.out = (uint16_t*)o;
  a.ws_o = (float*)ws;
  a.ws_lse = a.ws_o + (G - 1 + std::min(B, G - 1)) * Hq * MH_DV;
  a.B = (int)B;
  a.Hq = (int)Hq;
  a.page = (int)page;
  a.max_pages = (int)max_pages;
  a.G = (int)G;
  a.c = score_scale;
  hipStream_t st = (hipStream_t)stream;
  return bf16 ? (o_bf16 ? mh_launch<true, true>(a, st) : mh_launch<true, false>(a, st))
              : (o_bf16 ? mh_launch<false, true>(a, st) : mh_launch<false, false>(a, st));
}
