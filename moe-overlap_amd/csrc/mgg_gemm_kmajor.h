// The 256x256 tile of the grouped GEMM for K-major 16-bit B ([E, N, K], a
// linear layer's weights) and even N, where K is long or tiles are many
// (four_waves in mgg_gemm.hip).  (N-major B, the other tiles, odd N, fp8 and
// short K run mgg_gemm_kernel.h, whose queue, tickets and static rounds this
// kernel shares.)
//
// What bounds it: the matrix cores, at the clock that power leaves them, and
// the L2-to-LDS path behind them.  Four waves, one per SIMD, each 128 x 128 of
// the tile as 8 x 8 blocks of v_mfma_f32_16x16x32: 256 accumulators per lane
// (AGPRs) and a third fewer LDS reads per MFMA than eight waves of 128 x 64.
// K advances in 64-deep stages (128-byte rows of both operands), two in LDS.
// A lane holds the fragments of two K steps of 32, so a stage's slot is free
// as soon as its second step's fragments are read, halfway into its first:
//   step 0: 64 MFMAs on fragment set 0; set 1 (the stage's second step) is
//           read; barrier after MFMA kFreeAt: every wave has read this stage,
//           and the DMAs of the stage after the next start into its slot, one
//           per kDmaGap MFMAs;
//   wait for the next stage's DMAs, barrier;
//   step 1: 64 MFMAs on set 1; the rest of the DMAs; set 0 of the next stage.
// (One DMA per MFMA holds up the only wave of its SIMD: 1323 TFLOP/s from
// MFMA 47 on, 1475 from 35 on at a gap of 4, on a dense 16384 x 4096 x 8192
// problem; a gap of 3 from 33 on is level there and 1-6% behind on the shapes
// below.)  The stage
// stream does not stop at a tile's end: its last two bodies issue the next
// tile's stages 0 and 1, so they load behind the finished tile's epilogue, and
// its stores drain behind the next tile's MFMAs.
//
// Measured against the eight-wave kernel (ring of two 64-deep stages,
// v_mfma_f32_32x32x16), one process, inputs in rotation, atomic: E = 16, 1024
// rows routed, K = 2048, N = 4096 297.7 -> 247.2 us; E = 8 x 2048 rows, N = 8192
// 496.3 -> 429.5; E = 32, 300 rows, K = 1024, N = 2048 70.4 -> 60.2; one m-tile
// per expert in halves of K (16 x 256 rows, K = 7168, N = 2048) 146.1 -> 125.1;
// the dense problem 890.9 -> 745.3.  The same kernel with N-major B
// (transposing reads) ran behind the eight-wave A-block kernel and is not built.
#pragma once

#include "mgg_gemm_kernel.h"

namespace mgg {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(Bf16, u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(F16, u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

constexpr int kFreeAt = 35, kDmaGap = 4;
constexpr int kKmThreads = 256;
constexpr int kKmStage = 64;                 // K per stage
constexpr int kKmSlot = 65536;               // LDS bytes of a stage: A, then B
constexpr int kKmRow = 4096;                 // epilogue staging bytes per wave

// The kernel's arguments through an opaque pointer: each use loads what it
// needs.  Hoisted to the kernel's start, the fields that tiles are decoded and
// stored with fill the scalar registers and spill into the vector registers
// that the fragments need.
typedef const __attribute__((address_space(4))) GemmParams* KernelArgs;
__device__ __forceinline__ KernelArgs kernel_args() {
  auto a = (KernelArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}

// A pointer that is the same in every lane, in scalar registers (a buffer
// descriptor made of one the compiler takes to vary costs a loop per access).
template <class P>
__device__ __forceinline__ P* uniform_ptr(P* ptr) {
  const uint64_t a = reinterpret_cast<uint64_t>(ptr);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return reinterpret_cast<P*>(((uint64_t)hi << 32) | lo);
}

// dma16 with no scalar offset: the lane offset and the record count alone decide
// what is read (whether the range check sees a scalar offset is not relied on).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16_at(i32x4 rsrc, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop
// The descriptor `bytes` further on: its base moved, its records as many fewer
// (none below none).
__device__ __forceinline__ void advance_rsrc(i32x4& r, int bytes) {
  const uint64_t base = (((uint64_t)(uint32_t)r[1] << 32) | (uint32_t)r[0]) + (uint64_t)bytes;
  r[0] = (int32_t)(uint32_t)base;
  r[1] = (int32_t)(uint32_t)(base >> 32);
  r[2] = r[2] > bytes ? r[2] - bytes : 0;
}

template <class T, int EPI>
__device__ __forceinline__ void run_kmajor(const GemmParams& p0, int32_t W_tiles, int32_t w_report,
                                           int32_t first, int n_tiles, const int32_t* s_prefix,
                                           int32_t* s_item, uint8_t* lds, uint8_t* s_rows) {
  constexpr int kEpi = EPI;
  static_assert(T::kBKMajor, "B's rows run along K");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1;
  const int wn = wave >> 1;
  const int G = gridDim.x;
  const int K = (int)p0.k;
  const bool atomic = p0.atomic != 0;
  const bool derived = p0.num_work < 0;
  auto opaque_lane = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };

  // ---- work items: run_worker's split last round and static rounds --------
  constexpr int kGran = kKmStage;
  const int n_gran = (K + kGran - 1) / kGran;
  constexpr int kMinPartGran = MGG_SPLIT_MIN_K / kGran;
  constexpr int kStagger = MGG_SPLIT_STAGGER_K / kGran;
  int32_t w_base = W_tiles;
  int32_t W = W_tiles;
  int split_s = 1;
  if (atomic && derived && p0.split_flags != nullptr) {
    const int32_t rem = W_tiles > G ? W_tiles % G : W_tiles;
    for (int sp = MGG_SPLIT_MAX; sp >= 2 && split_s == 1; --sp)
      if (rem > 0 && (int64_t)rem * sp <= G && (int64_t)rem * sp <= p0.split_slots && n_gran >= kMinPartGran * sp)
        split_s = sp;
    if (split_s > 1) {
      w_base = W_tiles - rem;
      W = w_base + rem * split_s;
    }
  }
  auto dyn_base = [&]() -> int32_t {
    return atomic && derived && W_tiles >= 2 * G ? W_tiles / G * G : G;
  };
  auto by_ticket_after = [&](int32_t item) -> bool { return atomic && item + G >= dyn_base(); };
  auto resolve = [&](unsigned long long raw) -> int32_t {
    const KernelArgs p = kernel_args();
    const int32_t t = ticket_from(raw, p->counter, p->epoch);
    if (t == (W > G ? W - dyn_base() + G - 1 : W - 1)) {
      __hip_atomic_store(p->counter, (unsigned long long)p->next_epoch << 32, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      if (p->report != nullptr) atomicExch(p->report, w_report + G);
    }
    return dyn_base() + t;
  };

  struct Coords {
    int32_t e;
    int32_t rows_valid;
    int64_t row_base;
    int64_t n0;
    int32_t slot;  // -1: the whole tile; s*t + q: part q of K of split tile t
  };
  // The expert of a device-derived item: the last e with s_prefix[e] <= item,
  // found 64 entries at a time by the whole wave (a binary search's chain of
  // LDS reads would stall the only wave of the SIMD).
  auto expert_of = [&](int32_t item) -> int {
    const KernelArgs p = kernel_args();
    const int l = opaque_lane();
    int lo = 0, n = p->num_experts;
    if (n > 64) {
      const int step = (n + 63) / 64;  // at most 32
      const int at = l * step;
      const uint64_t m = __ballot(at < n && s_prefix[at < n ? at : 0] <= item);
      lo = (63 - __builtin_clzll(m | 1ull)) * step;
      n = n - lo < step ? n - lo : step;
    }
    const int at = lo + (l < n ? l : 0);
    const uint64_t m = __ballot(l < n && s_prefix[at] <= item);
    return lo + 63 - __builtin_clzll(m | 1ull);
  };
  auto decode = [&](int32_t item, Coords& c) -> bool {
    const KernelArgs p = kernel_args();
    c.slot = -1;
    if (item >= w_base) {
      c.slot = item - w_base;
      item = w_base + c.slot / split_s;
    }
    int e, tm, tn;
    int32_t off_lo, off_hi;
    if (p->num_work >= 0) {
      e = __builtin_amdgcn_readfirstlane(p->q_expert[item]);
      tm = __builtin_amdgcn_readfirstlane(p->q_tile_m[item]);
      tn = __builtin_amdgcn_readfirstlane(p->q_tile_n[item]);
      if ((uint32_t)e >= (uint32_t)p->num_experts || tm < 0 || (uint32_t)tn >= (uint32_t)n_tiles)
        return false;
      off_lo = __builtin_amdgcn_readfirstlane(p->offsets[e]);
      off_hi = __builtin_amdgcn_readfirstlane(p->offsets[e + 1]);
    } else {
      e = __builtin_amdgcn_readfirstlane(expert_of(item));
      off_lo = __builtin_amdgcn_readfirstlane(p->offsets[e]);
      off_hi = __builtin_amdgcn_readfirstlane(p->offsets[e + 1]);
      const int32_t local = item - __builtin_amdgcn_readfirstlane(s_prefix[e]);
      const int32_t mt_e = (int32_t)(((int64_t)off_hi - off_lo + 255) / 256);
      const int32_t span = MGG_GROUP_M * n_tiles;
      const int32_t g = local / span;
      const int32_t gm = min(MGG_GROUP_M, mt_e - g * MGG_GROUP_M);
      const int32_t sub = local - g * span;
      tn = sub / gm;
      tm = g * MGG_GROUP_M + (sub - tn * gm);
    }
    const int64_t m0 = (int64_t)tm * 256;
    const int64_t left = (int64_t)off_hi - off_lo - m0;
    if (left <= 0) return false;
    c.e = e;
    c.row_base = off_lo + m0;
    c.rows_valid = left < 256 ? (int)left : 256;
    c.n0 = (int64_t)tn * 256;
    return true;
  };

  // ---- the stage stream's source: the tile whose stages are being issued --
  // Chunk (row, K position) a lane moves in its wave's t-th A or B DMA of a
  // stage: 8 rows of 128 bytes each; chunk c of row r lies at
  // c ^ ((r >> 1) & 7).
  i32x4 a_rsrc, b_rsrc;  // from the next stage to issue on
  int iss_k0 = 0;    // K position of that stage
  int iss_klen = 0;  // K extent of the source tile (a part's, for a split tile)
  auto row_of = [&](int l, int t) { return 8 * (8 * wave + t) + (l >> 3); };
  auto kpos_of = [&](int l, int t) { return 8 * ((l & 7) ^ ((l >> 4) | (4 * (t & 1)))); };
  auto set_source = [&](const Coords& c) {
    const KernelArgs p = kernel_args();
    int kb = 0, klen = K;
    if (c.slot >= 0) {
      const int q = c.slot % split_s;
      auto pc_sum = [](int pb) {
        int t = 0;
        for (int j = 1; j < pb; ++j) t += __builtin_popcount(j);
        return t;
      };
      auto bound = [&](int pb) {
        return pb * (n_gran + kStagger * pc_sum(split_s)) / split_s - kStagger * pc_sum(pb);
      };
      kb = q == 0 ? 0 : bound(q) * kGran;
      klen = (q == split_s - 1 ? K : bound(q + 1) * kGran) - kb;
    }
    iss_k0 = 0;
    iss_klen = klen;
    const uint8_t* a_bytes = reinterpret_cast<const uint8_t*>(p->a);
    const uint8_t* b_bytes = reinterpret_cast<const uint8_t*>(p->b);
    const int64_t r0 = c.row_base < 0 ? 0 : (c.row_base > p->m ? p->m : c.row_base);
    const int64_t r_end = c.row_base + c.rows_valid < p->m ? c.row_base + c.rows_valid : p->m;
    a_rsrc = make_rsrc4(a_bytes + (r0 * p->lda + kb) * 2,
                        r0 < r_end ? ((r_end - 1 - r0) * p->lda + klen) * 2 : 0);
    b_rsrc = make_rsrc4(b_bytes + ((int64_t)c.e * p->ldb_e + c.n0 * p->ldb_k + kb) * 2,
                        c.n0 < p->n ? ((p->n - 1 - c.n0) * p->ldb_k + klen) * 2 : 0);
  };
  // The lane offsets of the source's DMAs.  Computed afresh for every run of
  // stages, like the fragment addresses below: kept live across the epilogue
  // they spill, and the K loop would reload them.  A stage that ends past K
  // (`left` < 64 of K): chunks at and past K get offsets past the
  // descriptors, so they write zeros.
  uint32_t a_voff[8], b_voff[8];
  auto set_offsets = [&](int left) {
    const KernelArgs p = kernel_args();
    const int l = opaque_lane();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int kp = kpos_of(l, t);
      a_voff[t] = kp < left ? (uint32_t)((row_of(l, t) * p->lda + kp) * 2) : kOutOfRange;
      b_voff[t] = kp < left ? (uint32_t)((row_of(l, t) * p->ldb_k + kp) * 2) : kOutOfRange;
    }
  };
  const uint32_t lds0 = lds_addr(lds);
  const uint32_t dst0 = lds0 + wave * 8192;
  // DMA d (0-7 B, 8-15 A) of the next stage into the slot at byte `slot`.
  auto issue = [&](uint32_t slot, int d) {
    dma16_at(d < 8 ? b_rsrc : a_rsrc, d < 8 ? b_voff[d] : a_voff[d - 8],
             dst0 + slot + (d < 8 ? 32768 : 0) + d % 8 * 1024);
  };
  auto next_stage = [&]() {
    iss_k0 += kKmStage;
    advance_rsrc(a_rsrc, kKmStage * 2);
    advance_rsrc(b_rsrc, kKmStage * 2);
  };
  auto no_source = [&]() {  // nothing left to load: every DMA writes zeros
    a_rsrc[2] = 0;
    b_rsrc[2] = 0;
    iss_k0 = 0;
    iss_klen = 2 * kKmStage;
  };

  // ---- fragments ----------------------------------------------------------
  // Lane l of a 16x16x32 operand holds row l%16, K 8*(l/16) .. +7: one 16-byte
  // read, conflict-free under the swizzle above.
  uint32_t row_off[2];
  auto set_frag_offsets = [&]() {
    const int l = opaque_lane();
    const int frow = l & 15, fq = l >> 4;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      row_off[kk] = (uint32_t)(frow * 128 + (((kk * 4 + fq) ^ ((frow >> 1) & 7)) * 16));
  };
  u32x4 fa[2][8], fb[2][8];
  auto read_a = [&](int f, uint32_t slot, int j) {
    fa[f][j] = lds_load(lds, (int)(slot + wm * 16384 + j * 2048 + row_off[f]));
  };
  auto read_b = [&](int f, uint32_t slot, int i) {
    fb[f][i] = lds_load(lds, (int)(slot + 32768 + wn * 16384 + i * 2048 + row_off[f]));
  };

  // acc[i][j]: columns 16i .. +15, rows 16j .. +15 of the wave's quarter; lane
  // l holds row l%16, columns 4*(l/16) .. +3 (the product is C^T = B^T A^T).
  f32x4 acc[8][8];

  // ---- split tiles ----------------------------------------------------------
  // The s parts of a split tile meet on one flag word (word (s - 1) * t of the
  // launch's flags).  A worker that finds s - 1 parts done is the last; any
  // other writes its sums to its slot s*t + q, waits until they are complete
  // and takes a ticket on the flag, and is the last if it draws s - 1.  The
  // last worker adds the other slots' sums to its own on their way out, as
  // (p0 + p1) + (p2 + p3) whichever part is its own, so the tile is the same
  // whoever comes last; the others are done.  No worker waits for another.
  // The accumulators are read by stores alone (memory here, LDS below), which
  // take them from the AGPRs: arithmetic on them would need each of the 256
  // in a vector register at the K loop's end, and spills.
  static_assert(MGG_SPLIT_MAX <= 4, "the parts' sums are added as (p0 + p1) + (p2 + p3)");
  constexpr int kPartWords = 65536;
  auto split_flag = [&](KernelArgs p, const Coords& c) {
    return p->split_flags + (int64_t)(split_s - 1) * (c.slot / split_s);
  };
  auto broadcast = [&]() -> bool {  // s_item[1], written by thread 0
    __syncthreads();
    const bool v = __builtin_amdgcn_readfirstlane(s_item[1]) != 0;
    __syncthreads();
    return v;
  };
  auto others_done = [&](const Coords& c) -> bool {
    const KernelArgs p = kernel_args();
    if (tid == 0) {
      const unsigned long long f =
          __hip_atomic_load(split_flag(p, c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_item[1] = ((uint32_t)(f >> 32) == p->epoch && (uint32_t)f == (uint32_t)(split_s - 1)) ? 1 : 0;
    }
    return broadcast();
  };
  auto last_to_write = [&](const Coords& c) -> bool {
    const KernelArgs p = kernel_args();
    wait_dma<0>();  // this wave's partial stores are complete (vmcnt counts stores too)
    __syncthreads();
    if (tid == 0) s_item[1] = first_ticket(split_flag(p, c), p->epoch) == split_s - 1 ? 1 : 0;
    return broadcast();
  };

  // ---- epilogue -------------------------------------------------------------
  // 16 rows x 64 columns of fp32 sums at a time through the wave's LDS (256
  // bytes a row, 16-byte chunk ch of row r at ch ^ r, conflict-free both
  // ways); each lane takes 8 consecutive columns back, applies the epilogue
  // and stores 16 bytes, 128 consecutive bytes of a row per 8 lanes (64 per 4
  // with SwiGLU, whose 64 columns are 32 gates and their 32 ups).  Where C's
  // rows are whole 16-byte chunks they go as buffer stores, rows and columns
  // that do not exist masked by offset, so that every such tile issues kStores
  // of them and the next tile's first wait counts past them.
  constexpr int kStores = kEpi == kEpiSwiglu ? 16 : 32;
  uint8_t* const rows_lds = s_rows + wave * kKmRow;
  auto counted = [&]() {
    const KernelArgs p = kernel_args();
    const int64_t c_cols = kEpi == kEpiSwiglu ? p->n / 2 : p->n;
    return ((c_cols | p->ldc) & 7) == 0 && p->ldc < (1 << 21);
  };
  // kMode kOutBuffered: as above; kOutPlain: any other C; kOutPartial: a
  // part's sums to its slot, as they come back from LDS (quad n of a lane at
  // n * 4096 + wave * 1024 + 16 * lane).  kOthers: how many other parts' sums
  // are added (3 also for two, the missing one reading as zeros).  They lie in
  // uncached memory, microseconds away, so they are read kAhead of the 16
  // steps ahead, as many as the registers hold without a spill (the plain
  // stores' addresses leave room for none).  Read in their own step, the
  // halves of 8 experts x 256 rows, K = 2048, N = 4096 took 65.2 us, now 50.5
  // (whole tiles 62.1).
  constexpr int kOutBuffered = 0, kOutPlain = 1, kOutPartial = 2;
  auto epilogue = [&](auto Mode, auto Others, const Coords& c) {
    constexpr int kMode = decltype(Mode)::value;
    constexpr int kOthers = decltype(Others)::value;
    constexpr bool kBuf = kMode == kOutBuffered;
    constexpr bool kParts = kOthers > 0;
    constexpr int kAhead = !kBuf ? 0 : kOthers == 1 ? 4 : 1;
    constexpr int kLanes = kEpi == kEpiSwiglu ? 4 : 8;  // lanes to a row
    const KernelArgs p = kernel_args();
    const int64_t c_cols = kEpi == kEpiSwiglu ? p->n / 2 : p->n;
    const int l = opaque_lane();
    const int r16 = l & 15, q4 = l >> 4;
    const int ch = l % kLanes;
    const int64_t col0 = (kEpi == kEpiSwiglu ? c.n0 / 2 + wn * 64 : c.n0 + wn * 128) + 8 * ch;
    const auto c_rsrc = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(p->c + c.row_base * p->ldc),
                                                          (short)0, 0x7FFFFFF0, 0x00020000);
    // The other parts' slots: the one its own is paired with, then the other
    // pair's (a part that does not exist reads as zeros).
    const int own = kParts ? c.slot % split_s : 0;
    auto part_rsrc = [&](int k) {
      const bool there = kParts && k < split_s;
      return __builtin_amdgcn_make_buffer_rsrc(
          uniform_ptr(p->split_partials + (int64_t)(there ? c.slot - own + k : 0) * kPartWords), (short)0,
          __builtin_amdgcn_readfirstlane(there ? kPartWords * 4 : 0), 0x00020000);
    };
    const auto r_pair = part_rsrc(own ^ 1), r_far0 = part_rsrc((own & 2) ^ 2),
               r_far1 = part_rsrc((own & 2) ^ 3);
    const int part_off = wave * 1024 + 16 * l;
    auto quad_at = [](int n, int g, int hh) { return ((n * 2 + g) * 2 + hh) * 4096; };
    auto read_back = [&](int u, int up, int hh) -> f32x4 {
      const int rr = 64 / kLanes * u + l / kLanes;
      const int cc = 8 * up + 2 * ch + hh;
      return *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(
          lds_ptr(rows_lds) + rr * 256 + ((cc ^ rr) * 16));
    };
    constexpr int kRing = kAhead > 0 ? kAhead : 1;
    f32x4 others[kRing][kParts ? kOthers : 1][2][2];  // step n's at n % kRing
    auto read_part = [&](auto r, int at) -> f32x4 {
      return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, part_off, at, 17));
    };
    auto read_others = [&](int n) {
      if constexpr (kParts) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const int at = quad_at(n, g, hh);
            others[n % kRing][0][g][hh] = read_part(r_pair, at);
            if constexpr (kOthers == 3) {
              others[n % kRing][1][g][hh] = read_part(r_far0, at);
              others[n % kRing][2][g][hh] = read_part(r_far1, at);
            }
          }
      }
    };
    auto summed = [&](f32x4 v, int n, int g, int hh) -> f32x4 {
      if constexpr (kParts) v += others[n % kRing][0][g][hh];
      if constexpr (kOthers == 3) v += others[n % kRing][1][g][hh] + others[n % kRing][2][g][hh];
      return v;
    };
    const auto r_own = __builtin_amdgcn_make_buffer_rsrc(
        uniform_ptr(p->split_partials + (int64_t)(kMode == kOutPartial ? c.slot : 0) * kPartWords), (short)0,
        kPartWords * 4, 0x00020000);
    auto store_quad = [&](const f32x4& v, int at) {
      const u32x4 u = {__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
      __builtin_amdgcn_raw_buffer_store_b128(u, r_own, part_off, at, 17);
    };
    // Rows of the tile that exist: [row_lo, row_hi).
    const int row_lo = c.row_base < 0 ? (int)(-c.row_base < 256 ? -c.row_base : 256) : 0;
    const int row_hi = (int)(c.row_base + c.rows_valid <= p->m ? c.rows_valid
                             : p->m > c.row_base              ? p->m - c.row_base
                                                              : 0);
    // Sums of step n = 2j + h (row block j, half h): [pass u or up][hh].  A
    // step's are read back while the step before it is stored (LDS operations
    // of a wave run in order, so its writes need no wait for those reads).
    f32x4 back[2][2][2];
    if constexpr (kParts) {
#pragma unroll
      for (int n = 0; n < kAhead; ++n) read_others(n);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int n = 0; n <= 16; ++n) {
      if (n < 16) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(
              lds_ptr(rows_lds) + r16 * 256 + (((4 * i + q4) ^ r16) * 16)) = acc[4 * (n & 1) + i][n / 2];
        // Lanes read what other lanes of the wave wrote.
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
            back[n & 1][g][hh] = kEpi == kEpiSwiglu ? read_back(0, g, hh) : read_back(g, 0, hh);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (n == 0) continue;
      const int j = (n - 1) / 2, h = (n - 1) & 1;
      if constexpr (kMode == kOutPartial) {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) store_quad(back[(n - 1) & 1][g][hh], quad_at(n - 1, g, hh));
      } else {
        if (kParts && kAhead == 0) read_others(n - 1);
        f32x4 v[2][2];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) v[g][hh] = summed(back[(n - 1) & 1][g][hh], n - 1, g, hh);
        if (kAhead > 0 && n - 1 + kAhead < 16) read_others(n - 1 + kAhead);
#pragma unroll
        for (int u = 0; u < kLanes / 4; ++u) {
          float y[8];
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            const float f = v[u][x / 4][x % 4];
            y[x] = kEpi == kEpiSwiglu ? silu_mul(f, v[1][x / 4][x % 4]) : kEpi == kEpiGelu ? gelu_erf(f) : f;
          }
          const u32x4 w = {T::pack(y[0], y[1]), T::pack(y[2], y[3]), T::pack(y[4], y[5]),
                           T::pack(y[6], y[7])};
          const int mr = wm * 128 + 16 * j + 64 / kLanes * u + l / kLanes;
          const int64_t col = col0 + h * (kEpi == kEpiSwiglu ? 32 : 64);
          const bool ok = mr >= row_lo && mr < row_hi && col < c_cols;
          if constexpr (kBuf) {
            const uint32_t off = (uint32_t)((mr * (int32_t)p->ldc + (int32_t)col) * 2);
            __builtin_amdgcn_raw_buffer_store_b128(w, c_rsrc, ok ? (int)off : (int)kOutOfRange, 0, 2);
          } else if (ok) {
            uint16_t* crow = p->c + (c.row_base + mr) * p->ldc;
            if (col + 8 <= c_cols) {
              __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(crow + col));
            } else {
#pragma unroll
              for (int d = 0; d < 4; ++d)
                if (col + 2 * d < c_cols)
                  __builtin_nontemporal_store(w[d], reinterpret_cast<uint32_t*>(crow + col) + d);
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- the persistent loop ---------------------------------------------------
  auto take_ticket_now = [&]() -> int32_t {
    const KernelArgs p = kernel_args();
    if (tid == 0) *s_item = resolve(atomicAdd(p->counter, 1ull));
    __syncthreads();
    const int32_t t = __builtin_amdgcn_readfirstlane(*s_item);
    __syncthreads();
    return t;
  };
  auto find_valid = [&](int32_t item, Coords& c) -> int32_t {
    while ((uint32_t)item < (uint32_t)W && !decode(item, c))
      item = by_ticket_after(item) ? take_ticket_now() : item + G;
    return item;
  };
  auto stages_of = [&](int klen) {
    const int n = (klen + kKmStage - 1) / kKmStage;
    return n < 2 ? 2 : n;  // the stream runs two stages ahead
  };

  Coords cur, nxt;
  int32_t w = find_valid(first, cur);
  if ((uint32_t)w >= (uint32_t)W) return;
  set_source(cur);
  int ns = stages_of(iss_klen);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    set_offsets(iss_klen - iss_k0);
#pragma unroll
    for (int d = 0; d < 16; ++d) issue(s * kKmSlot, d);
    next_stage();
  }
  wait_dma<16>();
  __syncthreads();
  uint32_t slot = 0;           // LDS byte offset of the stage being multiplied
  int stores_behind = 0;       // 1: kStores stores were issued after stage 1's DMAs
  int s = 0;
  bool ticketed = false, more = false;
  unsigned long long ticket = 0;
  int32_t next = 0;
  int ns_next = 2;
  // (The last body of a tile has read set 0 of the next tile's stage 0 too:
  // kept across the epilogue its 64 registers spill, and a reload there waits
  // for the stores before it.)
  auto start_tile = [&]() {
    set_frag_offsets();
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      read_a(0, slot, x);
      read_b(0, slot, x);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    ticketed = by_ticket_after(w);
    next = w + G;
    if (ticketed && tid == 0) ticket = atomicAdd(kernel_args()->counter, 1ull);
    s = 0;
  };
  start_tile();
  for (;;) {
    // Between runs of stages: two stages before the tile's end the stream
    // turns to the next tile, and a stage that ends past K is masked.
    if (s == ns - 2) {
      if (ticketed) {
        if (tid == 0) *s_item = resolve(ticket);
        __syncthreads();
        next = __builtin_amdgcn_readfirstlane(*s_item);
        __syncthreads();
      }
      next = find_valid(next, nxt);
      more = (uint32_t)next < (uint32_t)W;
      if (more) {
        set_source(nxt);
      } else {
        no_source();
      }
      ns_next = stages_of(iss_klen);
    }
    const int whole = (iss_klen - iss_k0) / kKmStage;  // stages the source has before a partial one
    int run = (s < ns - 2 ? ns - 2 : ns) - s;
    run = min(run, whole < 1 ? 1 : whole);
    // All that the loops carry is the same in every lane; the compiler, which
    // takes the one-lane atomics' and the meetings' results to vary, is told so
    // here, where the K loop's scalar registers come from.
    auto same = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    run = same(run);
    s = same(s) + run;
    ns = same(ns);
    slot = same(slot);
    iss_k0 = same(iss_k0);
    iss_klen = same(iss_klen);
    stores_behind = same(stores_behind);
    more = same(more ? 1 : 0) != 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      a_rsrc[x] = same(a_rsrc[x]);
      b_rsrc[x] = same(b_rsrc[x]);
    }
    set_offsets(iss_klen - iss_k0);
    set_frag_offsets();
#pragma clang loop unroll(disable)
    for (; run > 0; --run) {
#pragma unroll
      for (int x = 0; x < 64; ++x) {
        const int i = x / 8, j = x % 8;
        acc[i][j] = mfma16(T{}, fb[0][i], fa[0][j], acc[i][j]);
        if (x % 2 == 0 && x < 32) {
          if (x % 4 == 0) read_a(1, slot, x / 4);
          else read_b(1, slot, x / 4);
        }
        if (x == kFreeAt) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
        }
        if (x > kFreeAt && (x - kFreeAt) % kDmaGap == 0) issue(slot, (x - kFreeAt) / kDmaGap - 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      constexpr int kOut = (63 - kFreeAt) / kDmaGap;  // DMAs of this body so far
      static_assert(kOut + (62 / kDmaGap + 1) >= 16, "a body issues a stage's sixteen DMAs");
      if (stores_behind != 0) {
        wait_dma<kStores + kOut>();
        stores_behind = 0;
      } else {
        wait_dma<kOut>();
      }
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t other = kKmSlot - slot;
#pragma unroll
      for (int x = 0; x < 64; ++x) {
        const int i = x / 8, j = x % 8;
        acc[i][j] = mfma16(T{}, fb[1][i], fa[1][j], acc[i][j]);
        if (x % 2 == 0 && x < 32) {
          if (x % 4 == 0) read_a(0, other, x / 4);
          else read_b(0, other, x / 4);
        }
        if (x % kDmaGap == 1 && kOut + x / kDmaGap < 16) issue(slot, kOut + x / kDmaGap);
        __builtin_amdgcn_sched_barrier(0);
      }
      next_stage();
      slot = other;
    }
    if (s < ns) continue;
    if (cur.slot >= 0) {
      int last = same(others_done(cur) ? 1 : 0);
      if (last == 0) {
        epilogue(IntConst<kOutPartial>{}, IntConst<0>{}, cur);
        last = same(last_to_write(cur) ? 1 : 0);
      }
      if (last != 0) {
        if (tid == 0)
          __hip_atomic_store(split_flag(kernel_args(), cur), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!counted())
          epilogue(IntConst<kOutPlain>{}, IntConst<3>{}, cur);
        else if (split_s == 2)
          epilogue(IntConst<kOutBuffered>{}, IntConst<1>{}, cur);
        else
          epilogue(IntConst<kOutBuffered>{}, IntConst<3>{}, cur);
      }
    } else if (counted()) {
      epilogue(IntConst<kOutBuffered>{}, IntConst<0>{}, cur);
      stores_behind = 1;
    } else {
      epilogue(IntConst<kOutPlain>{}, IntConst<0>{}, cur);
    }
    if (!more) break;
    cur = nxt;
    w = next;
    ns = ns_next;
    start_tile();
  }
  wait_dma<0>();
}

template <class T, int EPI>
__global__ __attribute__((amdgpu_flat_work_group_size(kKmThreads, kKmThreads),
                          amdgpu_waves_per_eu(1, 1))) void
grouped_gemm_kmajor_kernel(GemmParams p) {
  constexpr int NT = kKmThreads;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * kKmSlot];
  __shared__ __attribute__((aligned(1024))) uint8_t s_rows[NT / 64 * kKmRow];
  __shared__ int32_t s_prefix[kMaxLdsExpertsGemm + 1];
  __shared__ int32_t s_scan[NT];
  __shared__ int32_t s_item[2];  // [0] ticket broadcast, [1] split-tile meeting

  const int G = gridDim.x;
  const int n_tiles = (int)((p.n + 255) / 256);
  const bool probe = p.clock_probe != nullptr && blockIdx.x < 8 && threadIdx.x < 64;
  unsigned long long clk0 = 0;
  if (probe) clk0 = __builtin_amdgcn_s_memtime();
  const bool rep_other =
      p.atomic && p.report != nullptr && (p.report_bm != 256 || p.report_bn != 256);
  const int rep_tiles = rep_other ? (int)((p.n + p.report_bn - 1) / p.report_bn) : 0;
  int32_t w_report = 0;
  int32_t W;
  if (p.num_work >= 0) {
    W = p.num_work;
    w_report = rep_other ? queue_length<NT>(p, p.report_bm, rep_tiles, s_scan) : W;
  } else {
    W = derive_prefix<256, NT>(p, n_tiles, s_prefix, nullptr, s_scan, rep_tiles, &w_report);
  }
  if (W == 0) {
    if (p.atomic && blockIdx.x == 0 && threadIdx.x == 0)
      __hip_atomic_store(p.counter, (unsigned long long)p.next_epoch << 32, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    zero_fill<false>(p, EPI == kEpiSwiglu ? p.n / 2 : p.n);
    return;
  }
  // XCD-aware worker numbering, as in grouped_gemm_kernel.
  int v = blockIdx.x;
  if (p.remap_xcd && (G & 7) == 0) v = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  // (What LDS or memory holds for the whole workgroup is made uniform for the
  // compiler where it is read.)
  run_kmajor<T, EPI>(p, __builtin_amdgcn_readfirstlane(W), __builtin_amdgcn_readfirstlane(w_report), v, n_tiles, s_prefix, s_item, lds, s_rows);
  if (probe) {
    const unsigned long long clk1 = __builtin_amdgcn_s_memtime();
    if (threadIdx.x == 0) {
      atomicAdd(p.clock_probe, clk1 - clk0);
      atomicAdd(p.clock_probe + 1, 1ull);
    }
  }
}

}  // namespace
}  // namespace mgg
