// Shared parts of the grouped GEMM kernels: the device-side tile scheduler,
// MFMA operand tiles and fragment readers, and the launch arguments.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace nt {

enum GemmMode { kFwd = 0, kDx = 1, kDw = 2 };

struct GemmArgs {
  const void* a;  // fwd: X     dX: dOut   dW: X
  const void* b;  // fwd: W     dX: W      dW: dOut
  const int32_t* offsets;
  int32_t E;
  int64_t A, K, N;
  void* out;
  int32_t ntn;      // output tiles along the n dimension
  int32_t ntm;      // dW only: output tiles along K
  int64_t mtiles;   // m-tile slots enumerated by the grid (upper bound for fwd / dX)
  void* out2;       // fused GELU forward: gelu'(h), same layout as out
  const void* aux;  // fused GELU backward: gelu'(h), same layout as out
  int32_t chunk;    // dW: rows per reduction chunk (0: one chunk per expert)
  float* partial;   // dW: fp32 partial slabs [split chunks][K][N] when chunk > 0
  // SwiGLU forward: b2 = W_val (b = W_gate), out = hidden, out2 = gate,
  // out3 = value. SwiGLU backward: aux = gate, aux2 = value, out = dgate,
  // out2 = dvalue. Two-part dX: a2 / b2 = dOut / W of the second product.
  const void* a2;
  const void* b2;
  void* out3;
  const void* aux2;
  int32_t split_thr;  // dW: experts with more rows than this are split (when chunk > 0)
  int32_t slab_cap;   // dW: partial slabs the workspace holds (when chunk > 0)
  int32_t stagger;    // start delay of half the workgroups, 100 MHz ticks (0: none)
  // Paired dW with split experts: arrival counters, one per (split expert,
  // 256x256 output tile), tagged with done_epoch; the last chunk of a tile
  // to arrive sums its slabs (fold_split_tile). Null: a reduce pass does.
  unsigned long long* done;
  unsigned long long done_epoch;
  // Tail split (tail_pieces): fp32 partials, one 128x128 slot per workgroup
  // that can be resident (tail_slots of them, a multiple of 8; 0: no split),
  // and one arrival counter per slot, tagged with tail_epoch.
  int32_t tail_slots;
  float* tail_partial;
  unsigned long long* tail_ctr;
  unsigned long long tail_epoch;
};

// Epilogues: plain store; forward GELU (out = gelu(h), out2 = gelu'(h), h
// itself is not stored); backward GELU (out = C * aux, aux = gelu'(h));
// SwiGLU forward (gate and value tiles of one output tile computed side by
// side: out = silu(gate) * value, out2 = gate, out3 = value); SwiGLU
// backward (C = dhidden: out = dgate, out2 = dvalue from aux = gate, aux2 =
// value); two-part dX (plain store, C = dOut @ W^T + dOut2 @ W2^T over one
// concatenated reduction).
enum GemmEpilogue {
  kEpiPlain = 0,
  kEpiGelu = 1,
  kEpiGeluGrad = 2,
  kEpiSwiGLU = 3,
  kEpiSwiGLUGrad = 4,
  kEpiDualK = 5
};

namespace {

// ------------------------------------------------------------ scheduling

// Row range of expert e, clamped to [0, A] and made non-decreasing, so a
// malformed offsets array can never move an access outside the buffers.
__device__ __forceinline__ void expert_rows(const int32_t* __restrict__ offsets, int e, int64_t A,
                                            int64_t& r0, int64_t& r1) {
  int64_t a = offsets[e], b = offsets[e + 1];
  a = a < 0 ? 0 : (a > A ? A : a);
  b = b < a ? a : (b > A ? A : b);
  r0 = a;
  r1 = b;
}

// s_pref[e] = number of BM-row tiles of experts < e (s_pref[E] = total),
// built by the first wave; ends with a workgroup barrier.
__device__ void build_m_prefix(const int32_t* __restrict__ offsets, int E, int64_t A, int BM,
                               int32_t* s_pref) {
  if (threadIdx.x < kWave) {
    const int lane = lane_id();
    int carry = 0;
    for (int s = 0; s < E; s += kWave) {
      const int e = s + lane;
      int v = 0;
      if (e < E) {
        int64_t a, b;
        expert_rows(offsets, e, A, a, b);
        v = (int)ceil_div(b - a, BM);
      }
      const int incl = wave_incl_scan(v);
      if (e < E) s_pref[e + 1] = carry + incl;
      carry += __shfl(incl, kWave - 1, kWave);
    }
    if (lane == 0) s_pref[0] = 0;
  }
  __syncthreads();
}

// dW reduction chunks. An expert with more than `thr` rows is cut into
// nch(e) = ceil(M_e / R) chunks of R rows (R <= thr); every other expert is
// one chunk (an empty expert keeps one empty chunk, so its dW is still
// written, as zeros). s_pref[e] = chunks of experts < e; s_split[e] = chunks
// of experts < e that have at least two (those write fp32 partials, one slab
// per chunk, and a reduce pass sums them in chunk order). R = 0 means one
// chunk per expert.
//
// The workspace holds `cap` slabs, enough whenever the experts' row ranges
// are disjoint (non-decreasing offsets). expert_rows clamps each expert on
// its own, so a non-monotone offsets array can give ranges that overlap and
// more split chunks than that; then every expert is one chunk (no partial
// slab is written, and split_total() tells the reduce pass to do nothing).
// Ends with a workgroup barrier.
__device__ __forceinline__ int dw_chunks(int64_t rows, int32_t R, int32_t thr) {
  if (R <= 0 || rows <= thr) return 1;
  return (int)ceil_div(rows, R);
}
// Wave-wide: chunks of the split experts (those with two or more) over all
// E experts, the same on every lane.
__device__ int split_total(const int32_t* __restrict__ offsets, int E, int64_t A, int32_t R,
                           int32_t thr) {
  int tot = 0;
  for (int s = 0; s < E; s += kWave) {
    const int e = s + lane_id();
    int v = 0;
    if (e < E) {
      int64_t a, b;
      expert_rows(offsets, e, A, a, b);
      v = dw_chunks(b - a, R, thr);
      v = v >= 2 ? v : 0;
    }
    tot += wave_sum_int(v);
  }
  return tot;
}
__device__ void build_chunk_prefix(const int32_t* __restrict__ offsets, int E, int64_t A,
                                   int32_t R, int32_t thr, int32_t cap, int32_t* s_pref,
                                   int32_t* s_split) {
  if (threadIdx.x < kWave) {
    const int lane = lane_id();
    if (R > 0 && split_total(offsets, E, A, R, thr) > cap) R = 0;
    int carry = 0, carry_s = 0;
    for (int s = 0; s < E; s += kWave) {
      const int e = s + lane;
      int v = 0, vs = 0;
      if (e < E) {
        int64_t a, b;
        expert_rows(offsets, e, A, a, b);
        v = dw_chunks(b - a, R, thr);
        vs = v >= 2 ? v : 0;
      }
      const int incl = wave_incl_scan(v);
      const int incl_s = wave_incl_scan(vs);
      if (e < E) {
        s_pref[e + 1] = carry + incl;
        s_split[e + 1] = carry_s + incl_s;
      }
      carry += __shfl(incl, kWave - 1, kWave);
      carry_s += __shfl(incl_s, kWave - 1, kWave);
    }
    if (lane == 0) {
      s_pref[0] = 0;
      s_split[0] = 0;
    }
  }
  __syncthreads();
}

// Expert owning m-tile `mt_global` (expert-major order) and the tile's row
// range; false when mt_global is past the last tile.
__device__ bool find_m_tile(const int32_t* __restrict__ offsets, int E, int64_t A,
                            const int32_t* s_pref, int64_t mt_global, int& e_out, int64_t& r0,
                            int64_t& r1, int64_t& mt_local) {
  if (mt_global >= s_pref[E]) return false;
  int lo = 0, hi = E - 1;  // largest e with s_pref[e] <= mt_global
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_pref[mid] <= mt_global) lo = mid;
    else hi = mid - 1;
  }
  e_out = lo;
  expert_rows(offsets, lo, A, r0, r1);
  mt_local = mt_global - s_pref[lo];
  return true;
}

__device__ bool map_m_tile(const int32_t* __restrict__ offsets, int E, int64_t A, int BM,
                           int64_t mt_global, int32_t* s_pref, int& e_out, int64_t& r0,
                           int64_t& r1, int64_t& mt_local) {
  build_m_prefix(offsets, E, A, BM, s_pref);
  return find_m_tile(offsets, E, A, s_pref, mt_global, e_out, r0, r1, mt_local);
}

// ------------------------------------------------------- MFMA operand tiles

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));

// The 16-bit GEMMs run on v_mfma_f32_16x16x32: the same operand registers
// (8 elements per lane) and flops per register as 32x32x16, at lower power
// per flop. The GPU holds its power limit by lowering the clock, so this
// raises the sustained rate (measured on MI355X, MFMA chains from registers:
// 1,916-1,922 TF/s at 1.92 GHz against 1,660-1,681 at 1.64-1.67 GHz; this
// kernel's k-step with operands from LDS: 1,422-1,441 against 1,342-1,360;
// the GEMMs, outputs bit-identical: C4 forward 1,171 -> 1,245 TF/s, dX
// 1,120 -> 1,198, dW 1,090 -> 1,140, C2 layer step 1.028 -> 0.964 ms).
template <typename T>
struct mfma_op;
template <>
struct mfma_op<bf16> {
  typedef bf16x8_t vec;
  __device__ static f32x4_t run(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct mfma_op<f16> {
  typedef f16x8_t vec;
  __device__ static f32x4_t run(vec a, vec b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Accumulators of one wave: acc[i][j][g] holds 16x16 block g of the 32x32
// sub-tile (i, j) of the wave's output block, with the B fragment issued as
// the MFMA's first operand, so that lane l, element q holds
//   C[32 i + acc_row(g, l)][32 j + acc_col(g, l) + q]:
// 4 consecutive output columns of one row per block.
template <int TM, int TN>
using AccTile = f32x4_t[TM][TN][4];
__device__ __forceinline__ int acc_row(int g, int lane) { return 16 * (g >> 1) + (lane & 15); }
__device__ __forceinline__ int acc_col(int g, int lane) { return 16 * (g & 1) + 4 * (lane >> 4); }

// Two fp32 values rounded to nearest-even and packed into 32 bits (first
// value in the low half). bf16 uses the hardware pair conversion
// (v_cvt_pk_bf16_f32, RNE); fp16 converts each value (v_cvt_f16_f32, RNE).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b);
template <>
__device__ __forceinline__ uint32_t pack2<bf16>(float a, float b) {
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
template <>
__device__ __forceinline__ uint32_t pack2<f16>(float a, float b) {
  return (uint32_t)f32_to_f16(a) | ((uint32_t)f32_to_f16(b) << 16);
}

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int kMfmaThreads = 512;  // 8 waves, two per SIMD
constexpr int kMfmaWaves = kMfmaThreads / kWave;

// Operand tiles are fetched with raw buffer loads that write straight into
// LDS (buffer_load_dwordx4 ... lds): lane i of one instruction lands at
// 16*i bytes past the instruction's LDS base (M0), so one instruction fills
// 1 KiB of LDS and the lane -> global-address map chooses the LDS layout.
// The descriptor's range check turns any offset past the range into a zero
// fill; lanes whose chunk lies past the reduction end get kOob.
//
// The loads are issued from inline assembly: the compiler then does not
// treat them as LDS writes that every later LDS read must wait for (it
// would wait for the next stage's loads before reading the current stage).
// Completion is explicit instead: s_waitcnt vmcnt(0) and a workgroup
// barrier before a stage is read.
constexpr uint32_t kBufConfig = 0x00020000u;  // gfx9 buffer descriptor word 3
constexpr uint32_t kOob = 0x80000000u;
constexpr int kCpolNT = 2;  // buffer instruction cache policy: non-temporal

__device__ __forceinline__ i32x4_t make_rsrc(const void* base, int64_t bytes) {
  const int32_t n = (int32_t)(bytes <= 0 ? 0 : (bytes > 0x7ffffff0 ? 0x7ffffff0 : bytes));
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu));  // stride 0
  r[2] = __builtin_amdgcn_readfirstlane(n);
  r[3] = (int)kBufConfig;
  return r;
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void*)p);
}

__device__ __forceinline__ void load16_to_lds(i32x4_t rsrc, uint32_t voff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, 0 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(lds)
      : "memory", "m0");
}

// a + b (b wave-uniform) as an instruction the compiler cannot move or fold.
__device__ __forceinline__ uint32_t add_opaque(uint32_t a, uint32_t b) {
  uint32_t r;
  asm volatile("v_add_u32 %0, %1, %2" : "=v"(r) : "s"(b), "v"(a));
  return r;
}

// Wait until at most N of this wave's vector-memory operations are in
// flight. The counter retires loads and stores in issue order, so every
// older operation is complete.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Buffer descriptor for the epilogue's stores to one output tile. Lanes
// outside the tile store at offset kOob, which the range check drops, so
// every wave issues the same number of store instructions per tile (the
// next tile's first wait counts them).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t out_rsrc(const void* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
                     ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32))
                      << 32);
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(u), 0, 0x7ffffff0,
                                           (int)kBufConfig);
}

__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  const u32x4_t d = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
  return make_uint4(d[0], d[1], d[2], d[3]);
}

__device__ __forceinline__ void store16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint4 v) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  const u32x4_t d = {v.x, v.y, v.z, v.w};
  // Non-temporal (cache policy NT): output tiles are written once and read
  // by a later kernel, so they should not displace the operand panels the
  // XCD's L2 shares between concurrent tiles (measured: -5 to -19 us per
  // C2-sized GEMM).
  __builtin_amdgcn_raw_buffer_store_b128(d, r, (int)off, 0, kCpolNT);
}

// One operand tile in LDS, ROWS (m or n) x BK (reduction, 64 or 32) 16-bit
// elements.
//
// K-major (the reduction index is contiguous in HBM): row r of the tile is
// BK elements = CPR chunks of 16 B; RPW = 16 / CPR rows share one 256-byte
// sweep of the 64 banks. Chunk c of row r is stored at c ^ ((r / RPW) % CPR).
// An MFMA fragment read (ds_read_b128, 16 lanes per LDS cycle: rows
// r..r+15, one chunk) then touches all 64 banks once.
//
// MN-major (m / n contiguous in HBM): row k of the tile holds ROWS elements
// (ROWS/8 chunks), chunk c stored at c ^ mn_swizzle(k). Fragments come from
// ds_read_b64_tr_b16, which transposes 4x4 blocks of 16-bit elements across
// each 16-lane group: source lane 4j+q reads the 4 elements at (k0 + j,
// mn0 + 4q .. 4q+3); destination lane 4q+e receives (k0 + 0..3, mn0 + 4q + e).
// Two such reads (k0 and k0 + 4) give a lane the 8 consecutive reduction
// elements of one m / n index that v_mfma_f32_16x16x32 takes; lane group g
// reads rows 8g .. 8g+7 of the substep. 32 lanes per LDS cycle (groups 0
// and 1, or 2 and 3) read rows k0 + 0..3 and k0 + 8..11, two chunks each;
// the XOR (bits 0, 1 and 3 of k) places those 16 chunks on all 64 banks.
//
// Wave w issues instructions w, w+NW, ...; where the rows of successive
// instructions differ by a whole number of XOR periods (16 rows), one
// per-lane offset plus a uniform stride per instruction covers them, else
// two offsets (even and odd instructions).
__device__ __forceinline__ int mn_swizzle(int k) { return 4 * (k & 3) + 2 * ((k >> 3) & 1); }
template <int ROWS, bool KMAJ, int BK, int NW>
struct OperandTile {
  static_assert(BK == 32 || BK == 64, "k-step of 32 or 64 elements");
  static constexpr int kBytes = ROWS * BK * 2;
  static constexpr int kInsts = kBytes / 1024;   // 1 KiB per load instruction
  static constexpr int kPer = kInsts / NW;
  static_assert(kPer >= 1 && kInsts % NW == 0, "tile too small for the wave count");
  static_assert(KMAJ || ROWS >= 128, "MN-major tiles need at least 16 chunks per row");
  static constexpr int kRowBytes = KMAJ ? BK * 2 : ROWS * 2;
  static constexpr int kRowsPerInst = 1024 / kRowBytes;
  static constexpr int kCpr = KMAJ ? BK / 8 : ROWS / 8;  // chunks per row
  static constexpr int kRpw = 16 / (BK / 8);             // K-major rows per bank sweep
  static constexpr int kStepRows = NW * kRowsPerInst;    // rows between a wave's instructions
  static constexpr bool kTwo = !KMAJ && kStepRows % 16 != 0;
  static_assert(KMAJ || kStepRows % 8 == 0, "MN-major swizzle: 8-row steps");
  static_assert(!kTwo || kPer % 2 == 0, "MN-major swizzle: even instruction count");

  uint32_t off;     // byte offset of this lane's chunk (instruction `wave`) from the tile origin
  uint32_t off2;    // kTwo: the same for instruction `wave` + NW
  uint32_t kchunk;  // K-major: first reduction index of the lane's chunk
  uint32_t ustep;   // byte stride between this wave's successive instructions (kTwo: of
                    // every second one)

  __device__ void init(int64_t ld, int wave, int lane) {
    const int r = kRowsPerInst * wave + lane / kCpr;
    const int c = KMAJ ? (lane % kCpr) ^ ((r / kRpw) % kCpr) : (lane % kCpr) ^ mn_swizzle(r);
    off = (uint32_t)((int64_t)r * ld + c * 8) * 2u;
    kchunk = (uint32_t)(c * 8);
    if (kTwo) {
      const int r2 = r + kStepRows;
      off2 = (uint32_t)((int64_t)r2 * ld + ((lane % kCpr) ^ mn_swizzle(r2)) * 8) * 2u;
    }
    ustep = (uint32_t)__builtin_amdgcn_readfirstlane((int)((kTwo ? 2 : 1) * kStepRows * ld * 2));
  }

  // Issue this wave's share of the tile's loads. `base` is the tile origin
  // for this k-step; `range` bytes from it are readable; `kv` reduction
  // elements are valid (K-major chunks past kv are zero-filled; MN-major
  // rows past kv fall outside `range`).
  __device__ void issue(const void* base, int64_t range, char* lds, int64_t kv, int wave) const {
    const i32x4_t rs = make_rsrc(base, range);
    const uint32_t l0 = lds_addr(lds) + (uint32_t)wave * 1024u;
    uint32_t v = off;
    if (KMAJ && kv < BK && (int64_t)kchunk >= kv) v = kOob;
    // Instruction u reads u * ustep bytes further on. The offset advances
    // through an opaque add, so the compiler keeps one offset register
    // instead of hoisting kPer of them out of the k-loop.
    if constexpr (kTwo) {
      uint32_t v2 = off2;
#pragma unroll
      for (int u = 0; u < kPer; u += 2) {
        load16_to_lds(rs, v, __builtin_amdgcn_readfirstlane(l0 + (uint32_t)(u * NW * 1024)));
        load16_to_lds(rs, v2, __builtin_amdgcn_readfirstlane(l0 + (uint32_t)((u + 1) * NW * 1024)));
        if (u + 2 < kPer) {
          v = add_opaque(v, ustep);
          v2 = add_opaque(v2, ustep);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        load16_to_lds(rs, v, __builtin_amdgcn_readfirstlane(l0 + (uint32_t)(u * NW * 1024)));
        if (u + 1 < kPer) v = add_opaque(v, ustep);
      }
    }
  }
};

// Per-lane LDS byte offsets of the fragment reads of one operand: TS 16-row
// blocks starting at row `row0` of the tile, for each of the BK/32
// k-substeps of 32 elements. Lane l supplies index l % 16 of a block and
// reduction elements 8 (l / 16) .. +7 of the substep.
template <int ROWS, bool KMAJ, int TS, int BK>
struct FragReader {
  static constexpr int kRowBytes = KMAJ ? BK * 2 : ROWS * 2;
  static constexpr int kCpr = BK / 8;
  static constexpr int kRpw = 16 / kCpr;
  uint32_t base[KMAJ ? BK / 32 : TS];
  __device__ void init(int row0, int lane) {
    if (KMAJ) {
      // the K-major XOR repeats every 16 rows, so blocks differ by a stride
      const int r = row0 + (lane & 15);
#pragma unroll
      for (int ks = 0; ks < BK / 32; ++ks) {
        const int c = (4 * ks + (lane >> 4)) ^ ((r / kRpw) % kCpr);
        base[ks] = (uint32_t)(r * kRowBytes + c * 16);
      }
    } else {
      // mn_swizzle repeats every 16 rows and ignores bit 2, so the substep
      // (32 rows on) and the second read (4 rows on) are strides
      const int g = lane >> 4, s = lane & 15, j = s >> 2, q = s & 3;
      const int k = 8 * g + j;
#pragma unroll
      for (int t = 0; t < TS; ++t) {
        const int mn = row0 + 16 * t + 4 * q;
        const int c = (mn >> 3) ^ mn_swizzle(k);
        base[t] = (uint32_t)(k * kRowBytes + c * 16 + (mn & 7) * 2);
      }
    }
  }
  template <typename V>
  __device__ V read(const char* lds, int t, int ks) const {
    if (KMAJ) {
      return *reinterpret_cast<const V*>(lds + base[ks] + t * 16 * kRowBytes);
    } else {
      const char* p = lds + base[t] + 32 * ks * kRowBytes;
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * kRowBytes));
      const s16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(V, v);
    }
  }
};

// Logical tile -> (m-tile, n-tile): groups of kGroupM m-tiles, m fastest
// inside a group, so neighbouring logical tiles reuse both A and B panels.
constexpr int kGroupM = 8;
__device__ __forceinline__ void tile_coords(int64_t logical, int64_t mtiles, int ntn, int64_t& mt,
                                            int& nt) {
  const int64_t per_group = (int64_t)kGroupM * ntn;
  const int64_t grp = logical / per_group;
  const int64_t rem = logical - grp * per_group;
  const int64_t gm0 = grp * kGroupM;
  const int64_t gsz = (mtiles - gm0) < kGroupM ? (mtiles - gm0) : kGroupM;
  mt = gm0 + rem % gsz;
  nt = (int)(rem / gsz);
}

// Row-tiled modes (forward, dX): logical tile -> (expert, m-tile within the
// expert, n-tile). Expert e's tiles are the block [P_e * ntn, P_{e+1} * ntn)
// of the logical order (P = s_pref, its m-tile prefix), so that tiles
// which run at the same time share the expert's weight panels. Inside the
// block the expert's m-tiles form ceil(mt_e / kGroupM) groups of balanced
// sizes (never crossing into the next expert, and with no stub group for
// an expert one m-tile past a multiple of kGroupM), each walked m fastest.
__device__ __forceinline__ void expert_tile_coords(int64_t logical, const int32_t* s_pref, int E,
                                                   int ntn, int& e_out, int64_t& mtl, int& nt) {
  const int64_t mt_global = logical / ntn;
  int lo = 0, hi = E - 1;  // largest e with s_pref[e] <= mt_global
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_pref[mid] <= mt_global) lo = mid;
    else hi = mid - 1;
  }
  const int64_t mt_e = s_pref[lo + 1] - s_pref[lo];
  const int64_t l = logical - (int64_t)s_pref[lo] * ntn;
  const int64_t ng = ceil_div(mt_e, (int64_t)kGroupM);
  const int64_t base = mt_e / ng, rem = mt_e % ng;  // rem groups of base + 1, then base
  const int64_t big = rem * (base + 1) * ntn;       // tiles in the larger groups
  int64_t gi, gsz, gm0;
  if (l < big) {
    gi = l / ((base + 1) * ntn);
    gsz = base + 1;
    gm0 = gi * (base + 1);
  } else {
    gi = (l - big) / (base * ntn);
    gsz = base;
    gm0 = rem * (base + 1) + gi * base;
    gi += rem;
  }
  const int64_t r = l - gm0 * ntn;
  e_out = lo;
  mtl = gm0 + r % gsz;
  nt = (int)(r / gsz);
}

// Start of the logical-tile range of the workgroups before `before` (of G):
// the proportional share, moved to the nearest expert boundary when that
// is within 1/16 of one XCD's share (so an XCD's range holds whole experts
// where the routing allows it, without unbalancing the XCDs).
__device__ __forceinline__ int64_t xcd_range_start(int64_t total, int64_t before, int64_t G,
                                                   const int32_t* s_pref, int E, int ntn) {
  const int64_t b = total * before / G;
  if (b <= 0 || b >= total) return b;
  const int64_t mt = b / ntn;
  int lo = 0, hi = E - 1;  // largest e with s_pref[e] <= mt
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (s_pref[mid] <= mt) lo = mid;
    else hi = mid - 1;
  }
  const int64_t e0 = (int64_t)s_pref[lo] * ntn, e1 = (int64_t)s_pref[lo + 1] * ntn;
  const int64_t near = (b - e0 <= e1 - b) ? e0 : e1;
  const int64_t tol = total / 8 / 16;
  const int64_t dist = near > b ? near - b : b - near;
  return dist <= tol ? near : b;
}

// fp32 rounded to T (RNE) and back.
template <typename T>
__device__ __forceinline__ float round_to(float x) {
  return elem<T>::load(elem<T>::store(x));
}
// Accumulator type of the generic and register-staged paths.
template <typename T>
struct acc_type {
  typedef float type;
};
template <>
struct acc_type<double> {
  typedef double type;
};

template <typename T>
__device__ __forceinline__ typename acc_type<T>::type to_acc(typename elem<T>::storage v) {
  return elem<T>::load(v);
}
template <>
__device__ __forceinline__ double to_acc<double>(double v) {
  return v;
}
template <typename T>
__device__ __forceinline__ typename elem<T>::storage from_acc(typename acc_type<T>::type v) {
  return elem<T>::store(v);
}
template <>
__device__ __forceinline__ double from_acc<double>(double v) {
  return v;
}

// Activations of the generic and register-staged paths, in AT (float, or
// double for fp64), on values already rounded to T.
template <typename AT>
__device__ __forceinline__ void gelu_both(AT x, AT& y, AT& dy) {
  const AT cdf = AT(0.5) * (AT(1) + erf(x * AT(0.70710678118654752440)));
  const AT pdf = exp(AT(-0.5) * x * x) * AT(0.39894228040143267794);
  y = x * cdf;
  dy = cdf + x * pdf;
}
template <typename T, typename AT>
__device__ __forceinline__ AT swiglu_fwd(AT g, AT v) {
  const AT sg = AT(1) / (AT(1) + exp(-g));
  const AT silu = to_acc<T>(from_acc<T>(g * sg));
  return silu * v;
}
template <typename T, typename AT>
__device__ __forceinline__ void swiglu_bwd(AT dh, AT g, AT v, AT& dg, AT& dv) {
  const AT sg = AT(1) / (AT(1) + exp(-g));
  const AT silu = to_acc<T>(from_acc<T>(g * sg));
  const AT ds = to_acc<T>(from_acc<T>(dh * v));
  dg = (ds * sg) * (AT(1) + g * (AT(1) - sg));
  dv = dh * silu;
}

// The next of `limit` items from a counter tagged with the launch's epoch:
// high 40 bits the epoch, low 24 the number of claims so far. A claim is one
// atomic add. An add that finds a word from before this launch (another
// epoch: an earlier launch's count, or any other leftover data) installs
// this launch's epoch with one claim taken, by compare-and-swap; if another
// workgroup installed it first, the claim is counted again by an add. So the
// counters need no clearing before a launch, and only the first claims of a
// launch can take more than one atomic.
constexpr int kClaimBits = 24;
__device__ int64_t claim_tagged(unsigned long long* ctr, unsigned long long epoch,
                                int64_t limit) {
  constexpr unsigned long long kCount = (1ull << kClaimBits) - 1;
  unsigned long long v = atomicAdd(ctr, 1ull);
  while ((v >> kClaimBits) != epoch) {
    const unsigned long long cur =
        __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((cur >> kClaimBits) == epoch) {
      v = atomicAdd(ctr, 1ull);
    } else if (atomicCAS(ctr, cur, (epoch << kClaimBits) | 1ull) == cur) {
      return limit > 0 ? 0 : -1;
    }
  }
  const int64_t cnt = (int64_t)(v & kCount);
  return cnt < limit ? cnt : -1;
}

// Tail split of forward / dX launches. The R tiles of an XCD's last round on
// `cus` compute units are cut along their nk k-steps into S pieces of at
// least four, one workgroup each; the last piece of a tile to finish sums the
// fp32 partials of all, in piece order, and runs the epilogue. S is the one
// with the shortest round: R S pieces of nk / S k-steps on `cus` units (up to
// `slots` of them resident), plus base + per S k-steps for the sum.
__device__ __forceinline__ int tail_pieces(int64_t R, int64_t cus, int64_t slots, int64_t nk,
                                           int base, int per) {
  if (R <= 0) return 1;
  int best = 1;
  int64_t cost = 840 * nk;  // in 1 / 840 of a k-step; 840 = lcm(1..8)
  for (int S = 2; S <= 8 && R * S <= slots && 4 * S <= nk; ++S) {
    const int64_t c = ceil_div(R * S, cus) * nk * (840 / S) + 840 * (base + per * S);
    if (c < cost) {
      cost = c;
      best = S;
    }
  }
  return best;
}

// One piece's 128x128 tile (4 waves of 64x64) to its slot, then: true in the
// workgroup that finished the tile last, with every piece's partials summed
// into acc in piece order. `slot0` is the tile's first slot, `ctr` its
// counter, s_flag an LDS word. Rows past `rows` are neither stored nor read.
//
// The slots are written and read with agent-scope accesses (through the L2s,
// whichever XCD a workgroup runs on), and a wave's writes are complete once
// its vmcnt is zero; the counter is touched only after that, behind the
// workgroup's barrier. Agent-scope fences instead write back and invalidate
// the whole L2 for every piece: they made the GEMMs around them 1.5 to 3
// times slower than no split.
__device__ __forceinline__ bool tail_fold(f32x4_t (&acc)[2][2][4], float* slot0, int piece, int S,
                                          unsigned long long* ctr, unsigned long long epoch,
                                          int m0, int rows, int32_t* s_flag) {
  typedef unsigned long long u64;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  auto at = [&](int p, int i, int j, int q) {
    return reinterpret_cast<u64*>(slot0 + (int64_t)p * (128 * 128)) +
           ((((wave * 2 + i) * 2 + j) * 4 + q) * 2 * kWave + lane);
  };
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (m0 + 32 * i + 16 * (q >> 1) >= rows) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u64 v[2];
        __builtin_memcpy(v, &acc[i][j][q], sizeof(v));
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(at(piece, i, j, q) + h * kWave, v[h], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  wait_vmcnt<0>();
  __syncthreads();
  if (threadIdx.x == 0) *s_flag = claim_tagged(ctr, epoch, S) == S - 1 ? 1 : 0;
  __syncthreads();
  if (*s_flag == 0) return false;
  // Sixteen loads in flight per lane and piece (block by block, each waited
  // for, the sum took longer than a piece's k-steps). Rows past `rows` in a
  // block read what their slots hold; those outputs are not stored.
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (m0 + 32 * i >= rows) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[i][j][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int p = 0; p < S; ++p) {
      u64 v[2][4][2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            v[j][q][h] = __hip_atomic_load(at(p, i, j, q) + h * kWave, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4_t x;
          __builtin_memcpy(&x, v[j][q], sizeof(x));
          acc[i][j][q] += x;
        }
    }
  }
  return true;
}

// Tile bookkeeping shared by the launchers: n-tiles, m-tile slots and the
// grid size (one workgroup per tile).
template <int MODE>
int64_t plan_tiles(GemmArgs& g, int64_t out_cols, int BM, int BN) {
  g.ntn = (int32_t)ceil_div(out_cols, BN);
  if (MODE == kDw) {
    g.ntm = (int32_t)ceil_div(g.K, BM);
    // Chunks: at most one per expert plus A / chunk (upper bound).
    const int64_t chunks = g.chunk > 0 ? g.E + g.A / g.chunk : g.E;
    g.mtiles = chunks * g.ntm;
  } else {
    g.ntm = 0;
    g.mtiles = ceil_div(g.A, BM) + g.E;  // upper bound: each expert's last tile may be partial
  }
  return g.mtiles * g.ntn;
}

}  // namespace

// grouped_gemm.hip. CUs of the device that `s` launches on.
int device_cus(hipStream_t s);

// staged_gemm.hip: whether the register-staged kernel takes this GEMM, and
// its launch (epilogue fused).
bool staged_ok(int mode, int dtype, const GemmArgs& g);
int launch_staged_gemm(int mode, int epi, int dtype, const GemmArgs& g, int64_t out_cols,
                       hipStream_t s);

}  // namespace nt
