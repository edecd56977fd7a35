// expert_gemm.hip -- grouped int4 (Q4_0) expert SwiGLU FFN for gfx950 on the
// matrix cores: calls of about a dozen positions per expert or more, with enough
// work for the chip, run as GEMMs (gemm_regime).
//
// Reference operator: kernels/sparse_moe/sparse_matmul.cu:120-215 and its
// dense branch (:322-365, cuBLAS GEMMs for gate/up and down, SwiGLU between),
// with the expert weights of python/phantom/loader/gguf_loader.py:362-381.
//
// Operands are exact, as in the decode regime, and fp16 for
// v_mfma_f32_16x16x32_f16, so the products are exact and only the fp32
// accumulation rounds:
//   A  gate/up: x as fp16, each token scaled by the power of two that puts its
//      largest element in [2^14, 2^15) (the router's prep; undone in the
//      epilogue), so bf16 values down to 2^-31 of the largest are exact and
//      smaller ones within 2^-39 of it; down: h as the fp16 pair hi + lo
//      written by the gate/up epilogue (|h - hi - lo| <= 2^-22 |h| down to
//      2^-14, and 2^-25 below).
//   B  the integers q = n - 8 as fp16: the nibble becomes the fp16 value
//      1024 + n (or 1024 + 16 n) by one v_and_or_b32 per pair, and one packed
//      fp16 add (or fma) gives q.
// Per 32-group g, an MFMA gives the exact group sums P = A . q (fp32), and
// acc += d[n][g] * P scales them in fp32 (four FMAs per MFMA output tile).
// (Weights rounded to fp16 as q * d, one MFMA and no scaling, cost 9e-3 of
// max-abs error on outputs of magnitude 40 per rounded stage; the layer
// tolerance is 1e-2.)
//
// What bounds it.  The scaling is the kernel's floor beside the weights'
// bytes: a wave issues one vector or matrix instruction per four cycles, an
// MFMA keeps its unit busy for sixteen, so MFMA + four FMAs is twenty cycles
// per 16 x 16 x 32 product.  With operands in registers that pattern reaches
// 1.2 PFLOP/s (gate/up) and 0.75 PFLOP/s (down, two MFMAs a product) here;
// plain MFMAs reach 1.5.
//
// Two (gate/up) or three (down) workgroups of four waves per CU.  A workgroup
// owns BM consecutive positions of one expert segment and 4 x 2 row tiles of
// weights, so a CU holds items that share no barrier: one's prologue (item
// lookup, first copies), epilogue (SwiGLU, stores) and barrier waits run under
// another's MFMAs.  (One eight-wave workgroup per CU spent 28% of gate/up and
// 36% of down outside the K loop at 4096 tokens: all eight waves were in the
// prologue or the epilogue at the same time.)  Down's blocks of 64 positions
// need half the accumulators, so three of its workgroups fit: 1417 -> 1226 us
// at DeepSeek-V3 2048 tokens, 257 -> 241 at Qwen3 4096, against two with a
// deeper ring (ahead only where the launch has one workgroup per CU: Mixtral
// at 64 tokens 99 against 115).
//
// Operand ring.  Both operands come by direct-to-LDS loads, issued from inline
// assembly (dma_b128_unseen) so that the compiler adds no waits of its own;
// each wave copies its own weight tiles and a share of the A rows, waits for
// its copies of the step about to be read, and one workgroup barrier per step
// publishes them (and says that every wave has left the slot about to be
// refilled).  A workgroup has 75 KB (gate/up) or 50 KB (down) of a CU's 160 KB
// for its ring (RingCfg).  Gate/up up to 64 positions: a step is a whole K quad
// of both operands and the ring is three to five steps deep, which is what
// streams weights from HBM.  Above, and in down: a step is half a quad of A
// (three slots, or two) and the weights keep a ring of quads (three, or two).
// A rows are stored with 16-byte unit s of row r at s ^ a_swizzle(r): no
// ds_read_b128 of A has a bank conflict.
//
// Tiling.  Every wave multiplies all BM positions with two weight row tiles of
// its own, so each B operand feeds one MFMA (down: two) per 16-position tile
// that holds a segment position.
//   gate/up (BM 128): wave w takes the gate and the up operand of one 16-row
//            tile of I, so its epilogue has both factors of every output; the
//            workgroup's 4 tiles are half a quad of I, written as down
//            operand units via LDS.
//   down (BM 64, A rows of hi and lo): wave w takes two 16-row tiles of H.
//
// Schedule.  The A reads of group g + 1 are issued while the MFMAs of group g
// run, and the fp32 scaling of a tile's sums runs while the next tile's MFMAs
// execute, so no instruction waits on the one just issued.  (Left to itself
// the compiler issued each A read right before its two MFMAs, with a wait for
// it: one LDS round trip per two MFMAs.)
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "expert_common.h"
#include "moe_common.h"
#include "moe_launch.h"

namespace pmoe {

struct GemmK {
  SegSrc seg;
  int32_t* items;         // [8] counters of the item queue, items_stride words apart, cleared by the router
  int items_stride;
  const uint16_t* a_src;  // fp16 rows [rows][Kq][half quad][part][group][AW x 8] in MFMA operand order
  int64_t a_rows;         // rows of a_src
  const float* a_unscale; // gate/up: per token, the power of two that undoes its scaling
  int64_t Kq;             // quads of K
  int64_t Kg;             // real 32-groups of K (padded groups of a_src are not multiplied)
  int64_t N;              // rows of the weight matrices (I for gate/up, H for down)
  // weights: [E][N/16][Kq][1 KiB] nibbles, [E][N/16][Kq][64] fp16 scales;
  // w1 = gate (or down), w2 = up (gate/up only); sh_* the shared expert's
  const uint8_t* nib1;
  const uint16_t* sc1;
  const uint8_t* nib2;
  const uint16_t* sc2;
  const uint8_t* sh_nib1;
  const uint16_t* sh_sc1;
  const uint8_t* sh_nib2;
  const uint16_t* sh_sc2;
  // gate/up output: h as fp16 hi + lo [rows][KqI][half quad][part][group][hi 8, lo 8],
  // the down GEMM's A operand
  uint16_t* hq16;
  int64_t KqI;
  // down output: fp32 [rows][H]
  float* outbuf;
};

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

// B operand of one 32-group: the lane's four nibble bytes w (bytes 4p..4p+3 of
// the group's qs for its row) -> the eight fp16 integers n - 8 in kmap order.
// mask holds 0x000F000F; the nibbles at bits 4..7 need no shift of their own:
// in place they make 1024 + 16 n, and (1024 + 16 n) / 16 - 72 is n - 8, exactly.
__device__ inline u32x4 dequant_int_f16(uint32_t w, uint32_t mask) {
  const h2_t off = {(_Float16)1032.0f, (_Float16)1032.0f};
  const h2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const h2_t off16 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const uint32_t w8 = w >> 8, mask16 = mask << 4;
  auto h2 = [](uint32_t v) { return __builtin_bit_cast(h2_t, v); };
  auto bits = [](h2_t v) { return __builtin_bit_cast(uint32_t, v); };
  u32x4 out;
  out.x = bits(h2(and_or(w, mask, 0x64006400u)) - off);
  out.y = bits(__builtin_elementwise_fma(h2(and_or(w, mask16, 0x64006400u)), sixteenth, off16));
  out.z = bits(h2(and_or(w8, mask, 0x64006400u)) - off);
  out.w = bits(__builtin_elementwise_fma(h2(and_or(w8, mask16, 0x64006400u)), sixteenth, off16));
  return out;
}

// SwiGLU of one output, silu(g) * u, from the hardware exp2 and reciprocal
// (v_exp_f32, v_rcp_f32; about 1 ulp each, against some 35 instructions for
// expf and an IEEE division).  g log2(e) is rounded before the exp2, so for
// negative g the relative error grows as |g| 2^-24 (1.2e-6 at -20), as the
// rounding of g itself does.  A layer's error against 64 bits at mean g -2.7, -8
// and -16 is 8.1e-8, 1.8e-7 and 5.1e-6; of the decode kernels, with expf, 3.7e-6,
// 4.1e-6 and 6.5e-6 (H 1024, I 1024).
__device__ inline float swiglu_fast(float g, float u) {
  const float e = __builtin_amdgcn_exp2f(-g * 1.44269504088896341f);
  return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
}

// s_waitcnt vmcnt(N) lgkmcnt(0), gfx9 encoding.
template <int N>
__device__ inline void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

// Item space: for each active segment u (active slots come first),
// ceil(len_u / BM) position blocks times n_nb row blocks.  s_mb[u] = first
// position block of segment u (an exclusive prefix over segments, by wave 0).
// All descriptor loads are issued before the scan: a loop over 64 slots at a
// time paid a memory round trip each, twice (7 us of a launch at 257 slots).
struct BlockPlan {
  int n_act, n_mb;
};
template <int BM>
__device__ inline BlockPlan plan_blocks(const SegSrc& seg, int* s_mb, BlockPlan* s_plan) {
  constexpr int kChunks = (kMaxExperts + 1 + kWave - 1) / kWave;
  if (threadIdx.x < kWave) {
    const int lane = threadIdx.x;
    int4 d[kChunks];
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      const int u = i * kWave + lane;
      d[i] = seg.desc[u < seg.max_slots ? u : seg.max_slots - 1];
    }
    int carry = 0, n_act = 0;
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
      if (i * kWave >= seg.max_slots) break;
      const int u = i * kWave + lane;
      const bool act = u < seg.max_slots && d[i].x >= 0;
      const int v = act ? (d[i].z - d[i].y + BM - 1) / BM : 0;
      int inc = v;
#pragma unroll
      for (int off = 1; off < kWave; off <<= 1) {
        const int t = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += t;
      }
      if (act) s_mb[u] = carry + inc - v;
      carry += __shfl(inc, kWave - 1, kWave);
      n_act += __popcll(__ballot(act));
    }
    // (loads past the last slot are never used: wait for them here, or the
    // compiler waits for them, vmcnt(0), in every loop that reuses their
    // registers)
    wait_vm_lgkm0<0>();
    if (lane == 0) {
      s_mb[n_act] = carry;
      *s_plan = BlockPlan{n_act, carry};
    }
  }
  lds_barrier();
  return BlockPlan{__builtin_amdgcn_readfirstlane(s_plan->n_act), __builtin_amdgcn_readfirstlane(s_plan->n_mb)};
}

// Segment holding position block mb: the last u with s_mb[u] <= mb (binary
// search; every lane computes the same answer).
__device__ inline int segment_of_block(const int* s_mb, int n_act, int mb) {
  int lo = 0, hi = n_act - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (s_mb[mid] <= mb) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// XCD-aware item order.  Workgroups are dispatched to the 8 XCDs round-robin
// (workgroup b on XCD b % 8), each XCD with its own L2.  The position blocks,
// in segment order, are cut into 8 contiguous ranges, one per XCD, and an
// XCD's items run block by block with the row blocks innermost.  The
// workgroups of an XCD that run at one time then share the A rows of each
// block (its row blocks run side by side) and the weights of each segment
// (its position blocks are neighbours in the range), so both come from HBM
// about once.  (Blocks dealt round-robin over the XCDs put the 2-3 blocks of
// a segment on different XCDs, each streaming the segment's weights.)  Fewer
// blocks than XCDs are cut between their row blocks instead, or some XCDs would
// have no items (one block of 64 positions at H 2048, I 1024 134 -> 53 us a
// layer, four experts at 96 tokens of H 2048, I 2048 106 -> 68), and so are 9 to
// 15 blocks, of which some XCDs would have two and some one (nine experts and
// the shared one at 33 tokens of H 5120, I 8192 339 -> 238; at 150 tokens of H
// 2048, I 2048 92 -> 68).  In down only where no segment has two blocks: cut
// apart, their XCDs would both stream its weights (Mixtral at 256 tokens 399
// -> 433 us).
//
// Items are drawn, not dealt: a workgroup starts with item l of its XCD's
// range and then draws from the range's counter, and from the other ranges'
// once its own is empty.  Drawing keeps an XCD's workgroups on neighbouring
// items, so they go on sharing A rows and weights in L2, and evens out items
// of different cost (a segment's last block may hold one position).  Dealt in
// rounds against drawn (us, gate/up + down): Qwen3 4096 tokens 316 + 270
// against 284 + 267, DeepSeek-V3 2048 tokens 2084 + 1643 against 1660 + 1409.
// With fewer than kDrawRounds rounds of items all are dealt: a drawn item waits
// for an atomic, which at 64 to 1024 tokens of Qwen3 (three rounds) cost 5 to
// 8 us a kernel.  The router clears the counters.
constexpr int kDrawRounds = 4;
struct ItemQueue {
  int32_t* next;  // items drawn of each range, `stride` words apart
  int stride;
  const int* first;  // LDS: [9] the ranges' first items
  int nx, x0;        // ranges, this workgroup's own
  bool drawing;
  int item, step, end;  // the next item dealt to this workgroup, and the end of those
  __device__ int workgroups(int x) const { return ((int)gridDim.x - x + nx - 1) / nx; }
  __device__ int drawn(int x, int t) const {  // the t-th item drawn of range x, or -1 past its end
    const int i = first[x] + workgroups(x) + t;
    return i < first[x + 1] ? i : -1;
  }
  __device__ int take(int x) const {
    return __hip_atomic_fetch_add(next + x * stride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // A drawn item, or -1 when every range is empty (one thread).  Other ranges
  // are looked at before they are drawn from: 512 workgroups drawing from
  // eight empty ranges cost 40 us at about 10 ns an atomic.
  __device__ int draw() const {
    if (!drawing) return -1;
    const int own = drawn(x0, take(x0));
    if (own >= 0) return own;
    int t[8];
#pragma unroll
    for (int v = 1; v < 8; ++v)
      t[v] = v < nx ? __hip_atomic_load(next + (x0 + v) % nx * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    wait_vm_lgkm0<0>();  // as in plan_blocks: some of these are never used
#pragma unroll
    for (int v = 1; v < 8; ++v) {
      const int x = (x0 + v) % nx;
      if (v >= nx || drawn(x, t[v]) < 0) continue;
      const int i = drawn(x, take(x));
      if (i >= 0) return i;
    }
    return -1;
  }
  // This workgroup's next item (every thread calls it) into *s_item, by
  // thread 0: the caller reads it after a barrier.
  __device__ void next_item(int* s_item) {
    if (threadIdx.x == 0) *s_item = item < end ? item : draw();
    item = item < end ? item + step : end;
  }
};

// s_first: [9] ints of LDS.  Item counts stay far below 2^31: an item writes
// 32 KB of workspace.
// by_segment: two blocks of a segment should share an XCD.
__device__ inline ItemQueue item_queue(int32_t* next, int stride, BlockPlan plan, bool by_segment, int n_nb,
                                       int* s_first) {
  ItemQueue q;
  q.next = next;
  q.stride = stride;
  q.first = s_first;
  q.nx = gridDim.x < 8 ? (int)gridDim.x : 8;
  q.x0 = (int)(blockIdx.x % q.nx);
  const int n_mb = plan.n_mb, xr = (int)threadIdx.x;
  const bool uneven = n_mb < q.nx || (n_mb < 2 * q.nx && n_mb != q.nx && !(by_segment && n_mb > plan.n_act));
  if (xr <= q.nx) s_first[xr] = uneven ? n_mb * n_nb * xr / q.nx : n_mb * xr / q.nx * n_nb;
  lds_barrier();
  const int f0 = __builtin_amdgcn_readfirstlane(s_first[q.x0]);
  q.item = f0 + (int)blockIdx.x / q.nx;
  q.step = q.workgroups(q.x0);
  const int f1 = __builtin_amdgcn_readfirstlane(s_first[q.x0 + 1]);
  q.drawing = n_mb * n_nb >= kDrawRounds * (int)gridDim.x;
  q.end = q.drawing && f0 + q.step < f1 ? f0 + q.step : f1;  // drawing: one dealt item each
  return q;
}

struct TileCoord {
  int e;
  int64_t m0, end;
  int64_t nb;
};

__device__ inline int4 sload_int4(const int4* p) {
  typedef int v4 __attribute__((ext_vector_type(4)));
  const v4 v = *(const __attribute__((address_space(4))) v4*)(uintptr_t)uniform_ptr(p);
  return make_int4(v.x, v.y, v.z, v.w);
}

// Segment, positions and row block of an item.
template <int BM>
__device__ inline TileCoord tile_coord(const GemmK& a, const int* s_mb, int n_act, int item, int n_nb) {
  TileCoord c;
  const int mb = item / n_nb;
  c.nb = item - mb * n_nb;
  const int u = __builtin_amdgcn_readfirstlane(segment_of_block(s_mb, n_act, mb));
  // a scalar load (the descriptors were written by an earlier launch): a vector
  // load's wait would also wait for the copies and stores in flight
  const int4 d = sload_int4(a.seg.desc + u);
  c.e = d.x;
  c.m0 = (int64_t)d.y + (int64_t)(mb - __builtin_amdgcn_readfirstlane(s_mb[u])) * BM;
  c.end = d.z;
  return c;
}

// ------------------------------------------------------------ the kernels
constexpr int kGateUpBM = 128;  // segment positions per gate/up item
constexpr int kDownBM = 64;      // and per down item
constexpr int kG2Waves = 4;
constexpr int kG2NB = 2;  // weight row tiles per wave in both kernels
constexpr int kG2BNib = kG2Waves * kG2NB * kWave;          // nibbles: one 1 KiB unit row per operand
constexpr int kG2BUnits = kG2BNib + kG2Waves * kG2NB * 8;  // and 128 B of scales per operand
constexpr int kG2BLoads = 2 * kG2NB;                       // weight copies per wave per quad
// Ring of a workgroup: 75 KB for gate/up (two workgroups and their tables in a
// CU's 160 KB), 50 KB for down (three; its blocks need fewer registers).
template <int AW>
constexpr int kG2RingUnits = AW == 1 ? 4800 : 3200;
template <int AW>
constexpr int kG2PerCu = AW == 1 ? 2 : 3;

// The ring of a block whose leading VT 16-position tiles are multiplied
// (16-byte units).
template <int AW, int VT>
struct RingCfg {
  static constexpr int kRing = kG2RingUnits<AW>;
  // a step is a quad of both operands (gate/up, few positions), else half a quad of A
  static constexpr bool kHalf = AW == 2 || VT > 4;
  static constexpr int kUpr = (kHalf ? 8 : 16) * AW;  // units per A row per step
  static constexpr int kRpd = kWave / kUpr;           // A rows per copy
  // A copies per wave per step: only those that reach a multiplied tile
  static constexpr int kALoads = (16 * VT + kG2Waves * kRpd - 1) / (kG2Waves * kRpd);
  static constexpr int kAUnits = kALoads * kG2Waves * kWave;
  // whole quads: slots of the ring
  static constexpr int kSlot = kAUnits + kG2BUnits;
  static constexpr int kSlots = kRing / kSlot > 5 ? 5 : kRing / kSlot;
  // half quads: A slots (halves) and B slots (quads)
  static constexpr int kSlotsA = 3 * kAUnits + 2 * kG2BUnits <= kRing ? 3 : 2;
  static constexpr int kSlotsB = kSlotsA == 3 && 3 * kSlot <= kRing ? 3 : 2;
  static_assert(kHalf ? kSlotsA * kAUnits + kSlotsB * kG2BUnits <= kRing : kSlots >= 3, "the ring fits");
};

// Column swizzle of the A rows in LDS.  gfx950 serves a wave's ds_read_b128
// in four cycles of 16 lanes, lane l in cycle group (b0 ^ b1 ^ b2, b3) of its
// quad q = l / 4 (measured: two lanes conflict exactly when they share a
// group, a 16-byte column of a 256-byte LDS row, and not the row).  Lane
// (n, p) of an A read takes row n + 16 tt and logical unit AW (2p + gi % 2)
// (+ 8 AW for the quad's second half, + 1 for lo), so in one cycle group p's
// low bit is n2 ^ n3 (or its complement): unit s of row r at s ^ a_swizzle(r)
// puts the group's 16 lanes in distinct columns.  UPR 8 (two rows per 256
// bytes), 16 with AW 1, and 16 or 32 with AW 2 need a map each.
template <int AW, int UPR>
__device__ inline uint32_t a_swizzle(uint32_t row) {
  const uint32_t n = row & 15u;
  if constexpr (UPR == 8) return ((n >> 2) & 1u) | (n & 2u) | ((n >> 1) & 4u);
  else if constexpr (AW == 1) return n;
  else return ((n & 3u) << 2) | (n >> 2);
}

// The multiply-accumulate of NG consecutive groups (one ring step) into acc,
// shared by both kernels.  sa: the step's A rows; sb: this wave's nibble units
// of the quad, ss its scales; g0: the step's first group within the quad (0 or
// 2).  VT: the leading 16-position tiles of the block that are multiplied (the
// number that hold a segment position); the rest lie past the segment end, so
// their MFMAs, A reads and scaling are skipped and their accumulators never
// stored.  A compile-time count keeps the loop branch-free: a run-time test
// per tile broke the software pipelining and cost 30%.  RAGGED: only the first
// n_valid (uniform) groups are multiplied.
template <int AW, int VT, int BMT, bool RAGGED>
__device__ __attribute__((always_inline)) inline void step_math(const u32x4* sa, const u32x4* sb, const uint2* ss,
                                                                int g0, int n_valid, uint32_t a_lane, uint32_t mask,
                                                                f32x4 (&acc)[kG2NB][BMT]) {
  typedef RingCfg<AW, VT> C;
  constexpr int NB = kG2NB;
  constexpr int NG = C::kHalf ? 2 : 4;
  const int lane = threadIdx.x % kWave;
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  // One group: MFMAs of every tile (hi then lo), the scaling of tile tt - 1
  // after the MFMAs of tile tt.
  auto group_math = [&](const u32x4 (&ah)[VT], const u32x4 (&al)[VT], const u32x4 (&bq)[NB], const float (&d)[NB]) {
    f32x4 pv[2][NB];
#pragma unroll
    for (int tt = 0; tt < VT; ++tt) {
#pragma unroll
      for (int b = 0; b < NB; ++b) pv[tt & 1][b] = mfma_f16_16x16x32(ah[tt], bq[b], z);
      if constexpr (AW == 2) {
#pragma unroll
        for (int b = 0; b < NB; ++b) pv[tt & 1][b] = mfma_f16_16x16x32(al[tt], bq[b], pv[tt & 1][b]);
      }
      if (tt > 0) {
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[b][tt - 1] += d[b] * pv[(tt - 1) & 1][b];
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][VT - 1] += d[b] * pv[(VT - 1) & 1][b];
  };
  // logical unit AW (8 (gi / 2) + gi % 2) (+ 1) on top of the lane's own
  // a_lane = n UPR + (2 AW p ^ a_swizzle(n)): the parts occupy different bits
  auto read_a = [&](int gi, u32x4 (&ah)[VT], u32x4 (&al)[VT]) {
    const uint32_t u = a_lane ^ (uint32_t)(AW * (8 * (gi >> 1) + (gi & 1)));
#pragma unroll
    for (int tt = 0; tt < VT; ++tt) {
      ah[tt] = sa[u + tt * 16 * C::kUpr];
      if constexpr (AW == 2) al[tt] = sa[(u ^ 1u) + tt * 16 * C::kUpr];
      else al[tt] = ah[tt];
    }
  };
  uint32_t bw[NB][NG];
  uint32_t bs[NB][NG / 2];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if constexpr (C::kHalf) {
      const uint2 v = reinterpret_cast<const uint2*>(sb + b * kWave + lane)[g0 >> 1];
      bw[b][0] = v.x;
      bw[b][1] = v.y;
      bs[b][0] = reinterpret_cast<const uint32_t*>(ss + b * 16 + lane % 16)[g0 >> 1];
    } else {
      const u32x4 v = sb[b * kWave + lane];
#pragma unroll
      for (int gi = 0; gi < NG; ++gi) bw[b][gi] = v[gi];
      const uint2 s2 = ss[b * 16 + lane % 16];
      bs[b][0] = s2.x;
      bs[b][1] = s2.y;
    }
  }
  auto operands = [&](int gi, u32x4 (&bq)[NB], float (&d)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t s2 = bs[b][gi >> 1];
      d[b] = half_bits_to_float((uint16_t)((gi % 2) ? (s2 >> 16) : (s2 & 0xffffu)));
      // the scale as fp32 in a register: the scaling is then v_fmac_f32,
      // not the slower mixed-precision v_fma_mix_f32 the compiler would
      // fold the conversion into
      asm volatile("" : "+v"(d[b]));
      bq[b] = dequant_int_f16(bw[b][gi], mask);
    }
  };
  if constexpr (!RAGGED) {
    u32x4 ah[2][VT], al[2][VT];
    read_a(0, ah[0], al[0]);
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
      if (gi + 1 < NG) read_a(gi + 1, ah[(gi + 1) & 1], al[(gi + 1) & 1]);
      u32x4 bq[NB];
      float d[NB];
      operands(gi, bq, d);
      group_math(ah[gi & 1], al[gi & 1], bq, d);
    }
  } else {
#pragma unroll
    for (int gi = 0; gi < NG; ++gi) {
      if (gi >= n_valid) break;
      u32x4 ah[VT], al[VT];
      read_a(gi, ah, al);
      u32x4 bq[NB];
      float d[NB];
      operands(gi, bq, d);
      group_math(ah, al, bq, d);
    }
  }
  // The sums stay in this step: otherwise the compiler sinks an even step's
  // scaling below the next barrier, which keeps 128 registers of group sums
  // alive and leaves its MFMAs nothing to overlap with.
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int tt = 0; tt < VT; ++tt) asm volatile("" : "+v"(acc[b][tt]));
}

// One item's K loop through the LDS ring.  s_row: A row of each position;
// rt: this wave's row tiles; nr / sr: the resources of their weights.
template <int AW, int VT, int BMT>
__device__ __attribute__((always_inline)) inline void gemm_tile(const GemmK& a, const uint32_t* s_row, u32x4* lds,
                                                                const i32x4& ar, const i32x4 (&nr)[kG2NB],
                                                                const i32x4 (&sr)[kG2NB], const int64_t (&rt)[kG2NB],
                                                                f32x4 (&acc)[kG2NB][BMT]) {
  typedef RingCfg<AW, VT> C;
  constexpr int NB = kG2NB;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t mask = vgpr_const(0x000F000Fu);
  const uint32_t row_bytes = (uint32_t)(a.Kq * 256 * AW);
  const uint32_t Kq = (uint32_t)a.Kq, Kg = (uint32_t)a.Kg;
  // A copy i of this wave fills rows [j Rpd, (j + 1) Rpd), j = w + 4 i: lane l
  // the unit l % Upr of row j Rpd + l / Upr, from logical unit (l % Upr) ^ a_swizzle
  uint32_t voff[C::kALoads];
#pragma unroll
  for (int i = 0; i < C::kALoads; ++i) {
    const uint32_t row = (uint32_t)((w + kG2Waves * i) * C::kRpd + lane / C::kUpr);
    const uint32_t unit = (uint32_t)(lane % C::kUpr) ^ a_swizzle<AW, C::kUpr>(row);
    voff[i] = s_row[row] * row_bytes + unit * 16u;
  }
  const uint32_t a_lane = (uint32_t)(lane % 16) * C::kUpr +
                          ((uint32_t)(lane / 16) * 2u * AW ^ a_swizzle<AW, C::kUpr>((uint32_t)(lane % 16)));
  const uint32_t lds0 = lds_addr(lds);
  auto uni = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  auto copy_a = [&](uint32_t step, uint32_t unit0) {
    const uint32_t aoff = uni(step * (uint32_t)(C::kUpr * 16));
#pragma unroll
    for (int i = 0; i < C::kALoads; ++i)
      dma_b128_unseen(ar, uni(lds0 + (unit0 + (uint32_t)(w + kG2Waves * i) * kWave) * 16u), voff[i], aoff);
  };
  auto copy_b = [&](uint32_t q, uint32_t unit0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint32_t tq = uni((uint32_t)rt[b] * Kq + q);
      dma_b128_unseen(nr[b], uni(lds0 + (unit0 + (uint32_t)(w * NB + b) * kWave) * 16u), (uint32_t)lane * 16u,
                      tq * kQuadNibBytes);
      // the 128 scale bytes: eight lanes
      if (lane < 8)
        dma_b128_unseen(sr[b], uni(lds0 + (unit0 + (uint32_t)kG2BNib + (uint32_t)(w * NB + b) * 8u) * 16u),
                        (uint32_t)lane * 16u, tq * (kQuadScales * 2));
    }
  };
  auto nib_of = [&](uint32_t unit0) { return lds + unit0 + w * NB * kWave; };
  auto scale_of = [&](uint32_t unit0) {
    return reinterpret_cast<const uint2*>(lds + unit0 + kG2BNib + w * NB * 8);
  };
  if constexpr (!C::kHalf) {
    // S slots of one quad each; quads q + 1 .. q + S - 1 in flight behind q
    constexpr uint32_t S = C::kSlots;
    constexpr int kLoads = C::kALoads + kG2BLoads;
    auto copy = [&](uint32_t q, uint32_t slot) {
      copy_a(q, slot * C::kSlot);
      copy_b(q, slot * C::kSlot + C::kAUnits);
    };
#pragma unroll
    for (uint32_t i = 0; i + 1 < S; ++i)
      if (i < Kq) copy(i, i);
    uint32_t slot = 0;
    auto top = [&](uint32_t q) {
      asm volatile("" ::: "memory");
      const uint32_t left = Kq - 1 - q;  // quads behind q still to come
      if (left >= S - 2) wait_vm_lgkm0<(int)(S - 2) * kLoads>();
      else if (S > 4 && left == 2) wait_vm_lgkm0<2 * kLoads>();
      else if (S > 3 && left == 1) wait_vm_lgkm0<kLoads>();
      else wait_vm_lgkm0<0>();
      __builtin_amdgcn_s_barrier();  // every copy of quad q is in; quad q - 1's slot is free
      asm volatile("" ::: "memory");
      if (q + S - 1 < Kq) copy(q + S - 1, slot == 0 ? S - 1 : slot - 1);
      const uint32_t u0 = slot * C::kSlot;
      slot = slot == S - 1 ? 0u : slot + 1u;
      return u0;
    };
    const uint32_t full = Kg / 4;
    for (uint32_t q = 0; q < full; ++q) {
      const uint32_t u0 = top(q);
      step_math<AW, VT, BMT, false>(lds + u0, nib_of(u0 + C::kAUnits), scale_of(u0 + C::kAUnits), 0, 4, a_lane, mask,
                                    acc);
    }
    if (full < Kq) {
      const uint32_t u0 = top(full);
      step_math<AW, VT, BMT, true>(lds + u0, nib_of(u0 + C::kAUnits), scale_of(u0 + C::kAUnits), 0, (int)(Kg % 4),
                                   a_lane, mask, acc);
    }
  } else {
    // A in NA slots of half a quad, B in NQ slots of a quad, each refilled as
    // far ahead as its slots allow, B on even steps
    constexpr uint32_t NA = C::kSlotsA, NQ = C::kSlotsB;
    constexpr uint32_t kB0 = NA * C::kAUnits;
    const uint32_t n_steps = (Kg + 1) / 2;
    copy_b(0, kB0);
    if (NQ == 3 && Kq > 1) copy_b(1, kB0 + kG2BUnits);
    copy_a(0, 0);
    if (NA == 3 && n_steps > 1) copy_a(1, C::kAUnits);
    uint32_t sa = 0, sb = 0;
    auto top = [&](uint32_t s, bool odd) {
      asm volatile("" ::: "memory");
      if constexpr (NA == 3) {
        // newer than this step's A: the next step's, and the weights copied before it
        if (s + 1 >= n_steps) wait_vm_lgkm0<0>();
        else if (odd && (s >> 1) + NQ - 1 < Kq) wait_vm_lgkm0<C::kALoads + kG2BLoads>();
        else wait_vm_lgkm0<C::kALoads>();
      } else {
        // this step's A was copied a step ago, the weights after it
        if (odd && (s >> 1) + NQ - 1 < Kq) wait_vm_lgkm0<kG2BLoads>();
        else wait_vm_lgkm0<0>();
      }
      __builtin_amdgcn_s_barrier();  // every copy of step s is in; step s - 1's slots are free
      asm volatile("" ::: "memory");
      auto refill_b = [&] {
        if (!odd && (s >> 1) + NQ - 1 < Kq)
          copy_b((s >> 1) + NQ - 1, kB0 + (sb == 0 ? NQ - 1 : sb - 1u) * kG2BUnits);
      };
      if constexpr (NA == 3) refill_b();
      if (s + NA - 1 < n_steps) copy_a(s + NA - 1, (sa == 0 ? NA - 1 : sa - 1u) * C::kAUnits);
      if constexpr (NA == 2) refill_b();
    };
    auto math = [&](auto ragged, bool odd) {
      const uint32_t ub = kB0 + sb * kG2BUnits;
      step_math<AW, VT, BMT, decltype(ragged)::value>(lds + sa * C::kAUnits, nib_of(ub), scale_of(ub), odd ? 2 : 0, 1,
                                                      a_lane, mask, acc);
      sa = sa == NA - 1 ? 0u : sa + 1u;
    };
    const uint32_t full = Kg / 2;  // steps with both groups
    uint32_t s = 0;
    for (; s + 1 < full; s += 2) {
      top(s, false);
      math(std::false_type(), false);
      top(s + 1, true);
      math(std::false_type(), true);
      sb = sb == NQ - 1 ? 0u : sb + 1u;
    }
    if (s < full) {
      top(s, false);
      math(std::false_type(), false);
      ++s;
    }
    if (s < n_steps) {
      const bool odd = (s & 1) != 0;
      top(s, odd);
      math(std::true_type(), odd);
    }
  }
  lds_barrier();  // every wave has left the ring before it is reused
}

// Multiplies an item with exactly the tiles that hold a position (a block of
// 65 positions takes 5 tiles, not 8: at about 64 positions an expert,
// DeepSeek-V3's prefill multiplied half again its positions with rounding to
// 2, 4 or 8).
template <int AW, int TT, int VT = 1, typename... Args>
__device__ __attribute__((always_inline)) inline void gemm_tiles(int vt, Args&&... args) {
  if constexpr (VT == TT) {
    gemm_tile<AW, VT, TT>(args...);
  } else {
    if (vt == VT) gemm_tile<AW, VT, TT>(args...);
    else gemm_tiles<AW, TT, VT + 1>(vt, args...);
  }
}

__global__ __launch_bounds__(kG2Waves * kWave, kG2PerCu<1>) void gemm_gate_up_kernel(GemmK a) {
  constexpr int BM = kGateUpBM;
  constexpr int TT = BM / 16;
  constexpr int kTiles = kG2Waves;  // row tiles of I per workgroup: half a quad of h,
  constexpr int kUr = 16;           // 16 units of 16 bytes per position
  __shared__ u32x4 lds_a[kG2RingUnits<1>];
  __shared__ int s_mb[kMaxExperts + 2];
  __shared__ uint32_t s_row[BM];
  __shared__ __align__(16) float s_un[BM];  // read as float4
  __shared__ BlockPlan s_plan;
  __shared__ int s_first[9], s_item;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n = lane % 16;
  const int p = lane / 16;
  const i32x4 ar = buf_rsrc_words(a.a_src, (uint32_t)(a.a_rows * a.Kq * 256));
  const BlockPlan plan = plan_blocks<BM>(a.seg, s_mb, &s_plan);
  const int64_t n_tiles = a.N / kRowTile;
  const int n_nb = (int)ceil_div(n_tiles, kTiles);
  ItemQueue queue = item_queue(a.items, a.items_stride, plan, false, n_nb, s_first);
  const uint32_t nib_bytes = (uint32_t)(a.N * a.Kq * 64), sc_bytes = (uint32_t)(a.N * a.Kq * 8);
  // positions past the segment repeat its last row (computed, not stored)
  auto token_of = [&](const TileCoord& t) {
    const int64_t pos = t.m0 + threadIdx.x;
    return threadIdx.x < BM ? a.seg.seg_tok[pos < t.end ? pos : t.end - 1] : 0;
  };
  queue.next_item(&s_item);
  lds_barrier();
  int item = __builtin_amdgcn_readfirstlane(s_item);
  if (item < 0) return;
  TileCoord c = tile_coord<BM>(a, s_mb, plan.n_act, item, n_nb);
  int tok = token_of(c);
  while (true) {
    if (threadIdx.x < BM) {
      s_row[threadIdx.x] = (uint32_t)tok;
      s_un[threadIdx.x] = a.a_unscale[tok];
    }
    lds_barrier();
    const bool routed = c.e < a.seg.E;
    const i32x4 ng = buf_rsrc_words(routed ? a.nib1 + (int64_t)c.e * nib_bytes : a.sh_nib1, nib_bytes);
    const i32x4 nu = buf_rsrc_words(routed ? a.nib2 + (int64_t)c.e * nib_bytes : a.sh_nib2, nib_bytes);
    const i32x4 sg = buf_rsrc_words(routed ? reinterpret_cast<const uint8_t*>(a.sc1) + (int64_t)c.e * sc_bytes
                                           : reinterpret_cast<const uint8_t*>(a.sh_sc1), sc_bytes);
    const i32x4 su = buf_rsrc_words(routed ? reinterpret_cast<const uint8_t*>(a.sc2) + (int64_t)c.e * sc_bytes
                                           : reinterpret_cast<const uint8_t*>(a.sh_sc2), sc_bytes);
    const i32x4 nr[2] = {ng, nu}, sr[2] = {sg, su};
    const int64_t t = c.nb * kTiles + w;
    const int64_t tc = t < n_tiles ? t : n_tiles - 1;  // a tile past I computes, unstored
    const int64_t rt[2] = {tc, tc};
    f32x4 acc[2][TT];
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[b][tt] = z;
    const int64_t left = c.end - c.m0;
    const int len = (int)(left < BM ? left : BM);  // positions of the block
    const int vt = __builtin_amdgcn_readfirstlane((len + 15) / 16);
    gemm_tiles<1, TT>(vt, a, s_row, lds_a, ar, nr, sr, rt, acc);
    queue.next_item(&s_item);

    // SwiGLU, then h as the fp16 pair hi + lo into LDS as the workgroup's half
    // quad of each position's down operand row: 256 bytes, 16-byte unit
    // 4 p' + 2 gl + (0 hi, 1 lo) for part p' and group gl.  Element
    // half * 16 + n of a group sits at j' = kmap^-1(p', .) of part p' = n / 4.
    // Unit u of position m is stored at u ^ (m / 4 % 4), so the four rows that
    // a wave's write touches lie in different banks.
    uint16_t* hs = reinterpret_cast<uint16_t*>(lds_a);
    const int gl = w / 2;  // group of the half quad this wave's tile belongs to
    const int rr = n % 4;
    const int jj = ((rr & 1) ? 4 : 0) + (rr >> 1) + 2 * (w % 2);
    const int u0 = 4 * (n / 4) + 2 * gl;
    const int uh = (u0 ^ p) * 8 + jj, ul = ((u0 + 1) ^ p) * 8 + jj;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      if (tt >= vt) break;  // tiles past the segment hold no position that is stored
      const float4 un = reinterpret_cast<const float4*>(s_un)[tt * 4 + p];
      const float uns[4] = {un.x, un.y, un.z, un.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float hv = swiglu_fast(acc[0][tt][j] * uns[j], acc[1][tt][j] * uns[j]);
        const uint32_t hb = float_to_half_bits(hv);
        const uint32_t lb = float_to_half_bits(hv - half_bits_to_float32(hb));
        uint16_t* row = hs + (tt * 16 + 4 * p + j) * (kUr * 8);
        row[uh] = (uint16_t)hb;
        row[ul] = (uint16_t)lb;
      }
    }
    lds_barrier();
    // the next item's tokens are on their way while this one's h is stored
    item = __builtin_amdgcn_readfirstlane(s_item);
    const TileCoord cn = item < 0 ? c : tile_coord<BM>(a, s_mb, plan.n_act, item, n_nb);
    tok = token_of(cn);
    // 16 lanes store a position's 256 bytes (group 1 of a half quad past I is skipped)
    const bool two = 2 * (c.nb * 2 + 1) + 1 < n_tiles;
    for (int cidx = threadIdx.x; cidx < len * kUr; cidx += kG2Waves * kWave) {
      const int m = cidx / kUr, u = cidx % kUr;
      if (two || (u & 2) == 0) {
        const u32x4 v = lds_a[m * kUr + (u ^ ((m >> 2) & 3))];
        *reinterpret_cast<u32x4*>(a.hq16 + ((c.m0 + m) * a.KqI * 32 + c.nb * kUr + u) * 8) = v;
      }
    }
    if (item < 0) return;
    lds_barrier();
    c = cn;
  }
}

__global__ __launch_bounds__(kG2Waves * kWave, kG2PerCu<2>) void gemm_down_kernel(GemmK a) {
  constexpr int BM = kDownBM;
  constexpr int TT = BM / 16;
  constexpr int NB = kG2NB;
  constexpr int kRows = kG2Waves * 16 * NB;  // rows of H per workgroup
  static_assert(BM * kRows / 4 <= kG2RingUnits<2>, "the epilogue's rows fit the ring");
  __shared__ u32x4 lds_a[kG2RingUnits<2>];
  __shared__ int s_mb[kMaxExperts + 2];
  __shared__ uint32_t s_row[BM];
  __shared__ BlockPlan s_plan;
  __shared__ int s_first[9], s_item;
  const int lane = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n = lane % 16;
  const int p = lane / 16;
  const BlockPlan plan = plan_blocks<BM>(a.seg, s_mb, &s_plan);
  const int n_nb = (int)ceil_div(a.N, kRows);
  const int64_t n_tiles = a.N / kRowTile;
  ItemQueue queue = item_queue(a.items, a.items_stride, plan, true, n_nb, s_first);
  const uint32_t nib_bytes = (uint32_t)(a.N * a.Kq * 64), sc_bytes = (uint32_t)(a.N * a.Kq * 8);
  queue.next_item(&s_item);
  lds_barrier();
  int item = __builtin_amdgcn_readfirstlane(s_item);
  while (item >= 0) {
    const TileCoord c = tile_coord<BM>(a, s_mb, plan.n_act, item, n_nb);
    const int64_t left = c.end - c.m0;
    const int len = (int)(left < BM ? left : BM);  // positions of the block
    // the block's rows are consecutive; those past the segment repeat its last
    // (computed, not stored)
    if (threadIdx.x < BM) s_row[threadIdx.x] = (uint32_t)((int)threadIdx.x < len ? (int)threadIdx.x : len - 1);
    lds_barrier();
    const i32x4 ar = buf_rsrc_words(reinterpret_cast<const uint8_t*>(a.a_src) + c.m0 * a.Kq * 512,
                                    (uint32_t)((int64_t)len * a.Kq * 512));
    const bool routed = c.e < a.seg.E;
    const i32x4 nw = buf_rsrc_words(routed ? a.nib1 + (int64_t)c.e * nib_bytes : a.sh_nib1, nib_bytes);
    const i32x4 sw = buf_rsrc_words(routed ? reinterpret_cast<const uint8_t*>(a.sc1) + (int64_t)c.e * sc_bytes
                                           : reinterpret_cast<const uint8_t*>(a.sh_sc1), sc_bytes);
    const i32x4 nr[NB] = {nw, nw};
    const i32x4 sr[NB] = {sw, sw};
    int64_t rt[NB];
    f32x4 acc[NB][TT];
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int64_t t = (c.nb * kG2Waves + w) * NB + b;
      rt[b] = t < n_tiles ? t : n_tiles - 1;  // a tile past H computes, unstored
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) acc[b][tt] = z;
    }
    const int vt = __builtin_amdgcn_readfirstlane((len + 15) / 16);
    gemm_tiles<2, TT>(vt, a, s_row, lds_a, ar, nr, sr, rt, acc);
    queue.next_item(&s_item);
    // The block's outputs through LDS, so that a position's 512 bytes are
    // stored by 32 consecutive lanes (straight from the accumulators a store
    // instruction wrote four 64-byte pieces).  64-byte unit u of position m is
    // stored at u ^ (m / 4 % 4): the four positions of a wave's write lie in
    // different banks.
    float* os = reinterpret_cast<float*>(lds_a);
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      if (tt >= vt) break;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float* row = os + (tt * 16 + 4 * p) * kRows + ((w * NB + b) ^ p) * 16 + n;
#pragma unroll
        for (int j = 0; j < 4; ++j) row[j * kRows] = acc[b][tt][j];
      }
    }
    lds_barrier();
    item = __builtin_amdgcn_readfirstlane(s_item);
    const int cols = (int)(a.N - c.nb * kRows < kRows ? a.N - c.nb * kRows : kRows);  // a multiple of 32
    float* out = a.outbuf + c.m0 * a.N + c.nb * kRows;
    for (int i = threadIdx.x; i < len * (kRows / 4); i += kG2Waves * kWave) {
      const int m = i / (kRows / 4), u = i % (kRows / 4);  // 16-byte unit u of position m
      if (4 * u < cols)
        *reinterpret_cast<u32x4*>(out + (int64_t)m * a.N + 4 * u) = lds_a[m * (kRows / 4) + (u ^ (((m >> 2) & 3) << 2))];
    }
    lds_barrier();
  }
}

bool dense_segments(int64_t T, int k, int E) {
  const int64_t slots = T * k;
  return slots >= kDenseSlotsPerExpert * (slots < E ? slots : E);
}

// Where the lines lie below 64 slots per expert: drawn so that a call is not
// slower than on the decode kernels, over 1648 timed calls of 428 shapes (H 256
// to 7168, I 128 to 14336, 4 to 256 experts, 1 to 1024 tokens); three are, by 6
// to 8%, and none of 419 others by more than 3%.  (With a line at 12 slots per
// expert alone, 149 of the first 1265 were, by up to 63%.)  Us a layer, decode
// kernels / GEMMs:
//   token-tile shapes, positions.  Those kernels read an expert's weights once
//     per 16-position tile, so they are ahead as long as few experts have more
//     than 16 positions: Qwen3 at 8, 12, 16, 32 slots per expert 152 / 129,
//     157 / 135, 162 / 143, 296 / 168; Mixtral at 8, 12, 14, 16, 32 171 / 208,
//     203 / 215, 281 / 248, 310 / 247, 512 / 319.  The second tile comes from
//     cache where weights are few: E 141, H 3200, I 416 210 / 237 at 13, E 16,
//     H 256, I 2048 41 / 47 at 12.
//   token-tile shapes, positions x I.  A GEMM item is one workgroup's chain
//     through K, so a launch needs items for the chip: E 10, H 2048, I 1024
//     57 / 66 at 40 slots per expert (0.4 M), E 16, H 2048, I 1024 55 / 51 at 24
//     (0.4 M) and 79 / 70 at 32 (0.5 M).  Where the K-split kernel would run
//     down (short H), it takes longer for many positions, and the GEMMs are
//     ahead sooner: E 20, H 512, I 768 60 / 51 at 32 slots per expert (0.5 M),
//     most of all for a shared expert, one segment of all tokens: E 25, H 320,
//     I 192 at 342 tokens 99 / 47 (0.19 M), E 26, H 352, I 448 at 201 78 / 50
//     (0.26 M).
//   shapes of the K-split kernels (rows of H too long for a token tile's
//     operand in LDS): DeepSeek-V3 at 1, 2, 4, 8 slots per expert 833 / 765,
//     1189 / 1078, 1452 / 1298, 1904 / 1397.  Few tokens or short I again: H
//     5120, E 160, I 448 173 / 183 at 64 tokens (0.23 M), H 7168, E 128, I 768
//     181 / 214 at 32 tokens (0.10 M); H 5376, E 128, I 1024 and a shared expert
//     305 / 238 at 48 (0.25 M).
bool gemm_regime(int64_t T, int64_t H, int64_t I, int k, int E, int has_shared) {
  if (dense_segments(T, k, E)) return true;
  if (lib_config().force_ksplit) return false;
  const int64_t slots = T * k, experts = slots < E ? slots : E;
  const int64_t work = (slots + (has_shared ? T : 0)) * I / 1024;
  const int64_t Kq = ceil_div(H, kQuad), KqI = ceil_div(I, kQuad);
  const int64_t lim = (int64_t)1 << 31;
  if (T * Kq * 256 >= lim || I * Kq * 64 >= lim || H * KqI * 64 >= lim) return false;  // 32-bit offsets
  if (gate_up_tile_regime(T, H, I, E, k, has_shared)) {
    const bool down_tile = down_tile_regime(T, H, I, E, k, has_shared);
    const bool long_down = !down_tile && has_shared && T >= 64;
    const int line = experts >= 16 && I >= 512 && work >= 512 ? 12 : (I >= 512 || long_down ? 14 : 16);
    return slots >= line * experts && work >= (down_tile ? 512 : (long_down ? 160 : 320));
  }
  return slots >= E && slots + (has_shared ? T : 0) >= 64 && work >= 225 &&
         experts * ceil_div(I, kG2Waves * 16) >= 4 * (int64_t)device_cus();
}

// One launch: position blocks of BM times row blocks of `rows`, on the
// workgroups resident at once.
template <typename Kernel>
static hipError_t launch_tiles(Kernel kernel, const ExpertArgs& x, const GemmK& g, int BM, int rows,
                               hipStream_t stream) {
  const int64_t positions = x.T * x.k + (x.has_shared ? x.T : 0);
  const int64_t max_items = (ceil_div(positions, BM) + max_active_experts(x)) * ceil_div(g.N, rows);
  hipLaunchKernelGGL(kernel, dim3(resident_grid(kernel, kG2Waves * kWave, max_items)), dim3(kG2Waves * kWave), 0,
                     stream, g);
  return hipGetLastError();
}

hipError_t launch_gemm_gate_up(const ExpertArgs& x, const Workspace& ws, hipStream_t stream) {
  GemmK g = {};
  g.seg = segments_of(x, ws);
  const GemmItems items = gemm_items(ws, x.T, x.H);
  g.items = items.counters;
  g.items_stride = items.stride;
  g.a_src = ws.xq;
  g.a_rows = x.T;
  g.a_unscale = ws.xs;
  g.Kq = ceil_div(x.H, kQuad);
  g.Kg = x.H / kGroup;
  g.N = x.I;
  g.nib1 = x.gate_nib;
  g.sc1 = x.gate_scale;
  g.nib2 = x.up_nib;
  g.sc2 = x.up_scale;
  g.sh_nib1 = x.sh_gate_nib;
  g.sh_sc1 = x.sh_gate_scale;
  g.sh_nib2 = x.sh_up_nib;
  g.sh_sc2 = x.sh_up_scale;
  g.hq16 = ws.hq;
  g.KqI = ceil_div(x.I, kQuad);
  return launch_tiles(gemm_gate_up_kernel, x, g, kGateUpBM, kG2Waves * 16, stream);
}

hipError_t launch_gemm_down(const ExpertArgs& x, const Workspace& ws, hipStream_t stream) {
  GemmK g = {};
  g.seg = segments_of(x, ws);
  const GemmItems items = gemm_items(ws, x.T, x.H);
  g.items = items.counters + 8 * items.stride;
  g.items_stride = items.stride;
  g.a_src = ws.hq;
  g.a_rows = x.T * x.k + (x.has_shared ? x.T : 0);
  g.Kq = ceil_div(x.I, kQuad);
  g.Kg = x.I / kGroup;
  g.N = x.H;
  g.nib1 = x.down_nib;
  g.sc1 = x.down_scale;
  g.sh_nib1 = x.sh_down_nib;
  g.sh_sc1 = x.sh_down_scale;
  g.outbuf = ws.outbuf;
  return launch_tiles(gemm_down_kernel, x, g, kDownBM, kG2Waves * 16 * kG2NB, stream);
}

}  // namespace pmoe
