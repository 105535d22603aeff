// Grouped GEMM forward, dX and dW for operands that the direct-to-LDS kernel
// does not take: fp32, and bf16 / fp16 off 16-byte chunks.
#include <algorithm>

#include "gemm_common.hpp"

namespace nt {
namespace {

// ------------------------------------------- register-staged MFMA kernel
// fp32 operands of any shape, and bf16 / fp16 operands whose rows are not
// whole aligned 16-byte chunks (K or N not a multiple of 8, or pointers off
// 16 bytes; a SwiGLU width of 8 d / 3 is both). The direct-to-LDS loads of
// gg_mfma_kernel need aligned chunks; here each thread loads its chunks (8
// elements along the contiguous dimension, at the element's alignment) into
// registers while the MFMAs of the k-step before run, and writes them to
// LDS in the layouts of OperandTile, so FragReader and the transposing
// reads serve both kernels. A 16-byte load at an odd multiple of 2 bytes
// runs at two thirds of the aligned rate (measured on MI355X, 32 MB from
// cache: 6.4 against 9.6 TB/s; from HBM 4.9 against 6.3), far above what a
// tile needs.
//
// fp32 runs on the bf16 MFMA: each value is the sum of three bf16 terms
// (x = h + m + l, each the round-to-nearest of what is left: 24 bits), and
// a product is the six term products down to 2^-18 (h l, m m, l h, then
// h m, m h, h h) in fp32 accumulators; the dropped ones (m l, l m: each up
// to 2^-25; l l) are below 2^-24 of the product, one fp32 rounding. Six
// products on a matrix core that runs bf16 at 16 times the fp32 rate. Two
// kinds of tile are reduced again with v_mfma_f32_16x16x4 on the unsplit
// values: one with a non-finite result (an infinite operand has no finite
// remainder to split, so only that keeps inf and NaN as fp32 arithmetic
// gives them), and one with an operand that the three terms do not hold: below
// 2^-110 its last bits lie under bf16's smallest subnormal, 2^-133 (the bf16
// MFMA keeps subnormal operands). Measured on MI355X, 132-term sums, largest
// error over sum |a||b|: 9.5e-8 down to 2^-110; split below it 2.2e-6 at 2^-118
// and 5.7e-4 at 2^-126, unsplit 1.3e-7 throughout.
//
// 128x128 outputs, 4 waves of 64x64, one LDS stage of 32 KiB (16-bit, 64
// deep) or 48 KiB (fp32, 32 deep): two (fp32) or three (16-bit) workgroups
// share a CU, so one's conversions, barriers and stores run under the
// others' MFMAs.
//
// Measured on MI355X, layer forward + backward, against the kernels before
// (fp32 on v_mfma_f32_32x32x2 with separate GELU passes; 16-bit on the VALU
// kernel): fp32, 4,096 tokens, 8 experts 512 -> 2048 -> 512, top-2, 1,295 ->
// 863 us (the GEMMs 80 -> 110 TFLOP/s), distance from float64 9.4e-7 ->
// 8.0e-7; bf16 SwiGLU, 5,003 tokens, 8 experts 512 -> 1365 -> 512, 3,470 ->
// 407 us (36 -> 320 TFLOP/s).
template <typename T>
struct staged_traits {
  typedef T mma;  // MFMA operand type
  static constexpr int kPlanes = 1, kBK = 64, kOcc = 3;
};
template <>
struct staged_traits<float> {
  typedef bf16 mma;
  static constexpr int kPlanes = 3, kBK = 32, kOcc = 2;
};
constexpr int kStagedThreads = 256;
constexpr int kStagedTile = 128;
// The largest row pitch whose 32-bit byte offsets within a tile cannot wrap.
constexpr int64_t kStagedMaxDim = int64_t(1) << 21;

// 16 bytes at any element boundary.
struct __attribute__((packed, aligned(2))) unaligned16 {
  uint32_t w[4];
};
struct __attribute__((packed, aligned(2))) unaligned8 {
  uint32_t w[2];
};
struct __attribute__((packed, aligned(4))) aligned4x4 {
  float f[4];
};

// Staging of one operand tile (128 rows x BK, K-major or MN-major like
// OperandTile): thread t holds chunks t, t + 256, ... of the tile.
template <typename S, bool KMAJ, int BK>
struct StagedTile {
  static constexpr int kRows = kStagedTile;
  static constexpr int kPer = kRows * BK / 8 / kStagedThreads;  // chunks per thread
  static constexpr int kCpr = KMAJ ? BK / 8 : kRows / 8;        // chunks per tile row
  static constexpr int kRowStep = kStagedThreads / kCpr;        // tile rows between chunks
  static constexpr int kRpw = 16 / (BK / 8);                    // K-major rows per bank sweep
  static constexpr int kRowBytes = (KMAJ ? BK : kRows) * 2;     // LDS bytes per tile row
  static constexpr int kWords = (int)sizeof(S) * 8 / 16;        // 16-byte words per chunk
  static constexpr int kChunkBytes = (int)sizeof(S) * 8;
  static constexpr int kBytes = kRows * BK * 2;                 // LDS bytes per plane
  static_assert(kRowStep % 16 == 0, "the LDS swizzles repeat every 16 rows");
  uint32_t off[kPer];  // byte offset of each chunk from the k-step's origin
  int32_t kq;          // reduction index (within the k-step) of chunk 0
  uint32_t lds;        // LDS byte offset of chunk 0 within a plane
  int64_t span;        // bytes past the origin that no chunk of a k-step exceeds
  // `valid` rows (K-major) or columns (MN-major) exist; chunks past them
  // read the last row / first columns instead (their products land in
  // outputs that are not stored). `halves`: columns 64.. are those of a
  // second operand at the same offsets (SwiGLU forward).
  __device__ void init(int64_t ld, int64_t valid, int tid, bool halves) {
    const int r = tid / kCpr, c = tid % kCpr;
    const int v = (int)(valid < kRows ? valid : kRows);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int ru = r + u * kRowStep;
      if (KMAJ) {
        const int rr = ru < v ? ru : v - 1;
        off[u] = (uint32_t)((rr * ld + c * 8) * (int64_t)sizeof(S));
      } else {
        const int cl = halves ? c & (kCpr / 2 - 1) : c;
        off[u] = (uint32_t)((ru * ld + (cl * 8 < v ? cl * 8 : 0)) * (int64_t)sizeof(S));
      }
    }
    kq = KMAJ ? c * 8 : r;
    lds = (uint32_t)(r * kRowBytes +
                     ((KMAJ ? c ^ ((r / kRpw) % kCpr) : c ^ mn_swizzle(r)) * 16));
    span = KMAJ ? ((int64_t)(v - 1) * ld + BK) * (int64_t)sizeof(S)
                : ((int64_t)(BK - 1) * ld + round_up(v, 8)) * (int64_t)sizeof(S);
  }
  __device__ int k_of(int u) const { return KMAJ ? kq : kq + u * kRowStep; }
  // Valid reduction elements (0..8) of chunk u when `kleft` are left.
  __device__ int n_valid(int u, int64_t kleft) const {
    const int64_t n = kleft - k_of(u);
    if (KMAJ) return n < 0 ? 0 : (n > 8 ? 8 : (int)n);
    return n > 0 ? 8 : 0;
  }
  // Load the chunks of the k-step at `base`. `end` is the end of the
  // operand's memory: no byte at or past it is read.
  __device__ void fetch(const char* base, const char* end, int64_t kleft,
                        uint4 (&reg)[kPer][kWords]) const {
    const bool inside = end - base >= span;  // every chunk lies inside
    if (inside && kleft >= BK) {
#pragma unroll
      for (int u = 0; u < kPer; ++u)
#pragma unroll
        for (int w = 0; w < kWords; ++w) reg[u][w] = word(base + off[u] + 16 * w);
      return;
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      // Chunks wholly past the reduction read the origin (mask zeroes them).
      // A chunk that would cross the end is loaded from the last chunk of
      // the memory and shifted down by the elements that lie before it.
      const char* p = base + (k_of(u) < kleft ? off[u] : 0u);
      const char* last = end - kChunkBytes;
      const uint32_t sh = p > last ? (uint32_t)(p - last) / (uint32_t)sizeof(S) : 0u;
      p = p > last ? last : p;
      uint32_t x[4 * kWords];
#pragma unroll
      for (int w = 0; w < kWords; ++w) {
        const uint4 v = word(p + 16 * w);
        x[4 * w] = v.x; x[4 * w + 1] = v.y; x[4 * w + 2] = v.z; x[4 * w + 3] = v.w;
      }
      uint32_t ws = sh;  // words to shift by
      if (sizeof(S) == 2) {
        if (sh & 1) {
#pragma unroll
          for (int i = 0; i < 4 * kWords; ++i)
            x[i] = (x[i] >> 16) | (i + 1 < 4 * kWords ? x[i + 1] << 16 : 0u);
        }
        ws = sh >> 1;
      }
#pragma unroll
      for (int b = 1; b < 4 * kWords; b *= 2) {
#pragma unroll
        for (int i = 0; i < 4 * kWords; ++i)
          x[i] = (ws & b) ? (i + b < 4 * kWords ? x[i + b] : 0u) : x[i];
      }
#pragma unroll
      for (int w = 0; w < kWords; ++w)
        reg[u][w] = make_uint4(x[4 * w], x[4 * w + 1], x[4 * w + 2], x[4 * w + 3]);
    }
  }
  __device__ static uint4 word(const char* p) {
    const unaligned16 v = *reinterpret_cast<const unaligned16*>(p);
    return make_uint4(v.w[0], v.w[1], v.w[2], v.w[3]);
  }
  // Zero the elements past the reduction (last k-step only).
  __device__ void mask(int64_t kleft, uint4 (&reg)[kPer][kWords]) const {
    constexpr int kEpw = 4 / (int)sizeof(S);  // elements per 32-bit word
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int n = n_valid(u, kleft);
      uint32_t x[4 * kWords];
      __builtin_memcpy(x, &reg[u][0], sizeof(x));
#pragma unroll
      for (int i = 0; i < 4 * kWords; ++i) {
        if (kEpw == 1) x[i] = i < n ? x[i] : 0u;
        else x[i] = 2 * i + 1 < n ? x[i] : (2 * i < n ? x[i] & 0xffffu : 0u);
      }
      __builtin_memcpy(&reg[u][0], x, sizeof(x));
    }
  }
  // Write the chunks to LDS: as they are (16-bit), or as three bf16 planes.
  // The third term is exact if what the first two leave is a bf16 value, the
  // upper half of an fp32 one: `lost` collects the bits of the lower halves.
  __device__ void store(char* smem, const uint4 (&reg)[kPer][kWords], uint32_t& lost) const {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      char* p = smem + lds + u * kRowStep * kRowBytes;
      if constexpr (kWords == 1) {
        *reinterpret_cast<uint4*>(p) = reg[u][0];
      } else {
        float x[8];
        __builtin_memcpy(x, &reg[u][0], sizeof(x));
        uint32_t t[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
          for (int pl = 0; pl < 3; ++pl) {
            if (pl == 2) lost |= __float_as_uint(a) | __float_as_uint(b);
            t[pl][i] = pack2<bf16>(a, b);
            a -= __uint_as_float(t[pl][i] << 16);
            b -= __uint_as_float(t[pl][i] & 0xffff0000u);
          }
        }
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          *reinterpret_cast<uint4*>(p + pl * kBytes) =
              make_uint4(t[pl][0], t[pl][1], t[pl][2], t[pl][3]);
      }
    }
  }
  // fp32 fallback: the chunks unsplit, element (row, k) at row * kPitch + k.
  static constexpr int kPitch = 33;
  __device__ void store_f32(float* s, const uint4 (&reg)[kPer][kWords], int tid) const {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      float x[4 * kWords];
      __builtin_memcpy(x, &reg[u][0], sizeof(x));
      const int r = tid / kCpr + u * kRowStep, c = (tid % kCpr) * 8;
#pragma unroll
      for (int i = 0; i < 4 * kWords; ++i)
        s[KMAJ ? r * kPitch + c + i : (c + i) * kPitch + r] = x[i];
    }
  }
};

// n (1..4) consecutive outputs / inputs at an element boundary.
template <typename T>
__device__ __forceinline__ void staged_store4(typename elem<T>::storage* p, const float (&v)[4],
                                              int n) {
  if (n >= 4) {
    if constexpr (sizeof(*p) == 4) {
      *reinterpret_cast<aligned4x4*>(p) = aligned4x4{{v[0], v[1], v[2], v[3]}};
    } else {
      *reinterpret_cast<unaligned8*>(p) = unaligned8{{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])}};
    }
  } else {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q < n) p[q] = elem<T>::store(v[q]);
  }
}
template <typename T>
__device__ __forceinline__ void staged_load4(const typename elem<T>::storage* p, float (&v)[4],
                                             int n) {
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = 0.f;
  if (n >= 4) {
    if constexpr (sizeof(*p) == 4) {
      const aligned4x4 x = *reinterpret_cast<const aligned4x4*>(p);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = x.f[q];
    } else {
      const unaligned8 x = *reinterpret_cast<const unaligned8*>(p);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = elem<T>::load((uint16_t)(x.w[q / 2] >> (16 * (q & 1))));
    }
  } else {
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (q < n) v[q] = elem<T>::load(p[q]);
  }
}

template <typename T, int MODE, int EPI>
__global__ void __launch_bounds__(kStagedThreads, staged_traits<T>::kOcc)
gg_staged_kernel(GemmArgs g) {
  typedef typename elem<T>::storage S;
  typedef typename staged_traits<T>::mma M;
  constexpr int NP = staged_traits<T>::kPlanes, BK = staged_traits<T>::kBK;
  constexpr int BT = kStagedTile;
  constexpr bool kAK = MODE != kDw, kBKm = MODE == kDx;
  constexpr bool kHalves = EPI == kEpiSwiGLU;  // B tile: 64 gate | 64 value columns
  typedef StagedTile<S, kAK, BK> TA;
  typedef StagedTile<S, kBKm, BK> TB;
  constexpr int kSmem = NP * (TA::kBytes + TB::kBytes);
  static_assert(NP == 1 || 2 * BT * TA::kPitch * 4 <= kSmem, "fallback stage fits");
  __shared__ __attribute__((aligned(1024))) char smem[kSmem];
  __shared__ int32_t s_pref[MODE == kDw ? 1 : NT_MAX_EXPERTS + 1];

  // XCD x (workgroup b runs on XCD b % 8) walks a contiguous eighth of the
  // tiles, so tiles that share operand panels share an L2. The grid is a
  // multiple of 8 with at least one workgroup per tile.
  int64_t total;
  if (MODE != kDw) {
    build_m_prefix(g.offsets, g.E, g.A, BT, s_pref);
    total = (int64_t)s_pref[g.E] * g.ntn;
  } else {
    total = g.mtiles * g.ntn;
  }
  const int xcd = blockIdx.x % 8;
  const int64_t t0 = total * xcd / 8, t1 = total * (xcd + 1) / 8;
  int64_t logical = t0 + blockIdx.x / 8;
  // Tail split: the XCD's last R tiles are np workgroups each.
  int np = 1, piece = 0;
  int64_t slot0 = 0;  // the tile's first partial slot
  if (MODE != kDw && g.tail_slots > 0) {
    // One workgroup per CU counts as a full round: alone on its CU it runs at
    // 85-90% of the rate of two or three together.
    const int64_t red = MODE == kFwd ? g.K : g.N, slots = g.tail_slots / 8, cus = slots / 2;
    const int64_t R = (t1 - t0) % cus, full = t1 - t0 - R;
    np = tail_pieces(R, cus, slots, ceil_div(red, BK) * (EPI == kEpiDualK ? 2 : 1), 4, 1);
    const int64_t r = blockIdx.x / 8 - full;
    if (np >= 2 && r >= 0) {
      if (r >= R * np) return;
      logical = t0 + full + r / np;
      piece = (int)(r % np);
      slot0 = xcd * slots + r - piece;
    } else {
      np = 1;
    }
  }
  if (logical >= t1) return;

  const S *pa, *pb, *pa2 = nullptr, *pb2 = nullptr;
  int64_t lda, ldb, rv, cv, klen, klen2 = 0, ldo, oofs;
  if (MODE == kDw) {
    const int64_t mt = logical / g.ntn;
    const int nt = (int)(logical % g.ntn);
    const int e = (int)(mt / g.ntm);
    const int64_t m0 = (mt % g.ntm) * BT, n0 = (int64_t)nt * BT;
    int64_t r0, r1;
    expert_rows(g.offsets, e, g.A, r0, r1);
    pa = static_cast<const S*>(g.a) + r0 * g.K + m0;
    pb = static_cast<const S*>(g.b) + r0 * g.N + n0;
    lda = g.K;
    ldb = g.N;
    rv = g.K - m0;
    cv = g.N - n0;
    klen = r1 - r0;
    ldo = g.N;
    oofs = (int64_t)e * g.K * g.N + m0 * g.N + n0;
  } else {
    int e, nt;
    int64_t mtl, r0, r1;
    expert_tile_coords(logical, s_pref, g.E, g.ntn, e, mtl, nt);
    expert_rows(g.offsets, e, g.A, r0, r1);
    const int64_t row0 = r0 + mtl * BT;
    const int64_t n0 = (int64_t)nt * (kHalves ? BT / 2 : BT);
    const int64_t wofs = (int64_t)e * g.K * g.N + (MODE == kFwd ? n0 : n0 * g.N);
    lda = MODE == kFwd ? g.K : g.N;
    ldb = g.N;
    pa = static_cast<const S*>(g.a) + row0 * lda;
    pb = static_cast<const S*>(g.b) + wofs;
    if (EPI == kEpiDualK) {
      pa2 = static_cast<const S*>(g.a2) + row0 * lda;
      klen2 = g.N;
    }
    if (EPI == kEpiDualK || kHalves) pb2 = static_cast<const S*>(g.b2) + wofs;
    rv = r1 - row0;
    ldo = MODE == kFwd ? g.N : g.K;
    cv = ldo - n0;
    klen = lda;
    oofs = row0 * ldo + n0;
  }
  // Ends of the operands' memory.
  const int64_t na = g.A * lda, nb = MODE == kDw ? g.A * g.N : (int64_t)g.E * g.K * g.N;
  const char* ea = reinterpret_cast<const char*>(static_cast<const S*>(g.a) + na);
  const char* eb = reinterpret_cast<const char*>(static_cast<const S*>(g.b) + nb);
  const char* ea2 = EPI == kEpiDualK
                        ? reinterpret_cast<const char*>(static_cast<const S*>(g.a2) + na) : nullptr;
  const char* eb2 = EPI == kEpiDualK || kHalves
                        ? reinterpret_cast<const char*>(static_cast<const S*>(g.b2) + nb) : nullptr;

  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 2, wn = wave % 2;
  TA ta;
  TB tb;
  ta.init(lda, rv, tid, false);
  tb.init(ldb, cv, tid, kHalves);
  const bool second = kHalves && tid % TB::kCpr >= TB::kCpr / 2;  // this thread's half of B
  uint4 ra[TA::kPer][TA::kWords], rb[TB::kPer][TB::kWords];
  // k-step kt: the first nk1 of (pa, pb), then (two-part dX) of (pa2, pb2).
  const int64_t nk1 = ceil_div(klen, BK);
  const int64_t nk = nk1 + (EPI == kEpiDualK ? ceil_div(klen2, BK) : 0);
  const int64_t kb = nk * piece / np, ke = nk * (piece + 1) / np;  // this workgroup's k-steps
  auto left_of = [&](int64_t kt) -> int64_t {
    return EPI == kEpiDualK && kt >= nk1 ? klen2 - (kt - nk1) * BK : klen - kt * BK;
  };
  auto fetch = [&](int64_t kt) {
    const bool p2 = EPI == kEpiDualK && kt >= nk1;
    const int64_t kl = (p2 ? kt - nk1 : kt) * BK;
    const int64_t left = left_of(kt);
    const S* a = (p2 ? pa2 : pa) + (kAK ? kl : kl * lda);
    const S* b = (p2 || second ? pb2 : pb) + (kBKm ? kl : kl * ldb);
    ta.fetch(reinterpret_cast<const char*>(a), p2 ? ea2 : ea, left, ra);
    tb.fetch(reinterpret_cast<const char*>(b), p2 || second ? eb2 : eb, left, rb);
  };

  AccTile<2, 2> acc;
  auto zero = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[i][j][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  zero();
  char* sa = smem;
  char* sb = smem + NP * TA::kBytes;
  // Wave columns: two 32-column sub-tiles; with halves, one gate and one
  // value sub-tile of the same outputs.
  FragReader<BT, kAK, 4, BK> fa;
  FragReader<BT, kBKm, 2, BK> fb[2];
  fa.init(wm * 64, lane);
  fb[0].init(kHalves ? wn * 32 : wn * 64, lane);
  fb[1].init(kHalves ? 64 + wn * 32 : wn * 64 + 32, lane);
  typedef typename mfma_op<M>::vec vec;

  uint32_t lost = 0;
  if (kb < ke) fetch(kb);
  for (int64_t kt = kb; kt < ke; ++kt) {
    __syncthreads();  // the stage's readers are done
    const int64_t left = left_of(kt);
    if (left < BK) {
      ta.mask(left, ra);
      tb.mask(left, rb);
    }
    ta.store(sa, ra, lost);
    tb.store(sb, rb, lost);
    __syncthreads();
    if (kt + 1 < ke) fetch(kt + 1);
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      vec bv[NP][4];
#pragma unroll
      for (int pl = 0; pl < NP; ++pl)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          bv[pl][j] = fb[j >> 1].template read<vec>(sb + pl * TB::kBytes, j & 1, ks);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        vec av[NP];
#pragma unroll
        for (int pl = 0; pl < NP; ++pl)
          av[pl] = fa.template read<vec>(sa + pl * TA::kBytes, i, ks);
        auto mma = [&](int x, int y) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            f32x4_t& c = acc[i >> 1][j >> 1][2 * (i & 1) + (j & 1)];
            c = mfma_op<M>::run(bv[y][j], av[x], c);
          }
        };
        if constexpr (NP == 3) {
          mma(2, 0);
          mma(0, 2);
          mma(1, 1);
          mma(1, 0);
          mma(0, 1);
        }
        mma(0, 0);
      }
    }
  }

  const int rvi = (int)(rv < BT ? rv : BT);
  const int cvi = (int)(cv < (kHalves ? BT / 2 : BT) ? cv : (kHalves ? BT / 2 : BT));
  auto row_of = [&](int i, int q) { return wm * 64 + i * 32 + acc_row(q, lane); };
  auto col_of = [&](int j, int q) {
    return kHalves ? wn * 32 + acc_col(q, lane) : wn * 64 + j * 32 + acc_col(q, lane);
  };
  if constexpr (NP == 3) {
    bool bad = (lost & 0xffffu) != 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            bad |= !(fabsf(acc[i][j][q][v]) <= 3.402823466e38f) && row_of(i, q) < rvi &&
                   col_of(j, q) + v < cvi;
    if (__syncthreads_or(bad)) {
      // Again on the fp32 matrix instruction, with the operands unsplit.
      zero();
      float* fsa = reinterpret_cast<float*>(smem);
      float* fsb = fsa + BT * TA::kPitch;
      for (int64_t kt = kb; kt < ke; ++kt) {
        fetch(kt);
        const int64_t left = left_of(kt);
        if (left < BK) {
          ta.mask(left, ra);
          tb.mask(left, rb);
        }
        __syncthreads();
        ta.store_f32(fsa, ra, tid);
        tb.store_f32(fsb, rb, tid);
        __syncthreads();
        const int kl = lane >> 4, rl = lane & 15;
        for (int k4 = 0; k4 < BK; k4 += 4) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float a = fsa[(wm * 64 + 16 * i + rl) * TA::kPitch + k4 + kl];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int n = kHalves ? (j >> 1) * 64 + wn * 32 + 16 * (j & 1) : wn * 64 + 16 * j;
              const float b = fsb[(n + rl) * TB::kPitch + k4 + kl];
              f32x4_t& c = acc[i >> 1][j >> 1][2 * (i & 1) + (j & 1)];
              c = __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, c, 0, 0, 0);
            }
          }
        }
      }
    }
  }

  if (MODE != kDw && np > 1) {
    __shared__ int32_t s_last;
    if (!tail_fold(acc, g.tail_partial + slot0 * (BT * BT), piece, np, g.tail_ctr + slot0,
                   g.tail_epoch, wm * 64, rvi, &s_last))
      return;
  }

  S* po = static_cast<S*>(g.out) + oofs;
  S* po2 = static_cast<S*>(g.out2);
  S* po3 = static_cast<S*>(g.out3);
  const S* px = static_cast<const S*>(g.aux);
  const S* px2 = static_cast<const S*>(g.aux2);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = row_of(i, q);
      if (m >= rvi) continue;
#pragma unroll
      for (int j = 0; j < (kHalves ? 1 : 2); ++j) {
        const int n = col_of(j, q);
        const int nv = cvi - n;
        if (nv <= 0) continue;
        const int64_t o = (int64_t)m * ldo + n;
        float c[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) c[v] = round_to<T>(acc[i][j][q][v]);
        if constexpr (EPI == kEpiGelu) {
          float d[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float x = c[v];
            gelu_both<float>(x, c[v], d[v]);
          }
          staged_store4<T>(po2 + oofs + o, d, nv);
        } else if constexpr (EPI == kEpiGeluGrad) {
          float d[4];
          staged_load4<T>(px + oofs + o, d, nv);
#pragma unroll
          for (int v = 0; v < 4; ++v) c[v] *= d[v];
        } else if constexpr (EPI == kEpiSwiGLU) {
          float val[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) val[v] = round_to<T>(acc[i][1][q][v]);
          staged_store4<T>(po2 + oofs + o, c, nv);
          staged_store4<T>(po3 + oofs + o, val, nv);
#pragma unroll
          for (int v = 0; v < 4; ++v) c[v] = swiglu_fwd<T, float>(c[v], val[v]);
        } else if constexpr (EPI == kEpiSwiGLUGrad) {
          float gt[4], vl[4], dv[4];
          staged_load4<T>(px + oofs + o, gt, nv);
          staged_load4<T>(px2 + oofs + o, vl, nv);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float dh = c[v];
            swiglu_bwd<T, float>(dh, gt[v], vl[v], c[v], dv[v]);
          }
          staged_store4<T>(po2 + oofs + o, dv, nv);
        }
        staged_store4<T>(po + o, c, nv);
      }
    }
}

template <int MODE, int EPI>
int launch_staged(int dtype, GemmArgs g, int64_t out_cols, hipStream_t s) {
  constexpr int BT = kStagedTile;
  g.chunk = 0;
  int64_t tiles = plan_tiles<MODE>(g, out_cols, BT, EPI == kEpiSwiGLU ? BT / 2 : BT);
  if (tiles == 0) return NT_OK;
  if (MODE == kDw) g.tail_slots = 0;
  if (g.tail_slots > 0) {
    g.tail_slots = std::min<int32_t>(g.tail_slots / 16, device_cus(s) / 8) * 16;  // two per CU
    tiles += g.tail_slots;
  }
  tiles = round_up(tiles, 8);
  if (tiles > INT32_MAX) return NT_ERR_TOO_LARGE;
  const dim3 grid((unsigned)tiles), block(kStagedThreads);
  switch (dtype) {
    case NT_F32: hipLaunchKernelGGL((gg_staged_kernel<float, MODE, EPI>), grid, block, 0, s, g); break;
    case NT_F16: hipLaunchKernelGGL((gg_staged_kernel<f16, MODE, EPI>), grid, block, 0, s, g); break;
    case NT_BF16: hipLaunchKernelGGL((gg_staged_kernel<bf16, MODE, EPI>), grid, block, 0, s, g); break;
    default: return NT_ERR_DTYPE;
  }
  return launch_status();
}

}  // namespace

// Shapes the register-staged kernel takes: any in fp32, bf16 and fp16 whose
// row pitches keep its 32-bit offsets, with operands of at least one chunk
// (8 elements) in memory.
bool staged_ok(int mode, int dtype, const GemmArgs& g) {
  const int64_t na = g.A * (mode == kDx ? g.N : g.K);
  const int64_t nb = mode == kDw ? g.A * g.N : g.E * g.K * g.N;
  return dtype != NT_F64 && g.K <= kStagedMaxDim && g.N <= kStagedMaxDim && na >= 8 && nb >= 8;
}

// (mode, epilogue) pairs: the forward takes plain, GELU and SwiGLU, dX plain,
// GELU / SwiGLU backward and two-part, dW plain.
int launch_staged_gemm(int mode, int epi, int dtype, const GemmArgs& g, int64_t out_cols,
                       hipStream_t s) {
  switch (mode * 8 + epi) {
    case kFwd * 8 + kEpiPlain: return launch_staged<kFwd, kEpiPlain>(dtype, g, out_cols, s);
    case kFwd * 8 + kEpiGelu: return launch_staged<kFwd, kEpiGelu>(dtype, g, out_cols, s);
    case kFwd * 8 + kEpiSwiGLU: return launch_staged<kFwd, kEpiSwiGLU>(dtype, g, out_cols, s);
    case kDx * 8 + kEpiPlain: return launch_staged<kDx, kEpiPlain>(dtype, g, out_cols, s);
    case kDx * 8 + kEpiGeluGrad: return launch_staged<kDx, kEpiGeluGrad>(dtype, g, out_cols, s);
    case kDx * 8 + kEpiSwiGLUGrad: return launch_staged<kDx, kEpiSwiGLUGrad>(dtype, g, out_cols, s);
    case kDx * 8 + kEpiDualK: return launch_staged<kDx, kEpiDualK>(dtype, g, out_cols, s);
    case kDw * 8 + kEpiPlain: return launch_staged<kDw, kEpiPlain>(dtype, g, out_cols, s);
  }
  return NT_ERR_INVALID_ARG;
}

}  // namespace nt
