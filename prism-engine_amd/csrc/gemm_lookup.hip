// gemm_lookup.hip -- the palettized GEMM: the weights looked up straight into
// MFMA operands (k_gemm_lookup, k_gemm_lookup_x), and X packed into operand
// order (k_pack_x).
//
// Y[M x N] = X[M x K] . W^T, fp32 accumulation and fp16 (RNE) output: M
// independent lut_gemv_cpu rows (compute-core/src/lut/evaluator.rs:21-44).
//
// v_mfma_f32_32x32x16_f16 takes 32 weight rows as its A operand (lane (r, h)
// = (l % 32, l / 32): row r, eight consecutive k) and 32 tokens as its B
// operand.  The A operand comes out of lookup tables in LDS: at 4 bits a
// row's 256-entry pair table (entry b = LUT[b & 15] | LUT[b >> 4] << 16 at
// dword 64 b + row), so an index dword is four v_perm addresses and four
// ds_read_b32, with no packing; at 8 bits the LUT itself at dword 64 b +
// row, eight lookups and four packing v_perms.  A decode in registers takes
// 29 VALU operations for the same eight elements (lut_perm.hpp).  In step s
// lane (r, h) takes index chunk 2 s + h of its row (16 bytes); MFMA j of the
// step takes elements 8 j .. 8 j + 7 of that chunk, and x is read with the
// same permutation of k.
//
// RAGGED (K is not a multiple of what one iteration takes): both operands
// are zero at k >= K, whatever bytes follow the row.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_lookup.hpp"
#include "gemv_kernels.hpp"
#include "gemv_lpr_args.hpp"

namespace prism {

namespace {

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8v __attribute__((ext_vector_type(8)));

constexpr uint32_t kOut = 0x80000000u;  // a buffer offset past every range: the load returns zeros

template <int BITS>
struct LkShape {
  static constexpr int EPC = 128 / BITS;      // elements per 16-byte index chunk
  static constexpr int SK = 2 * EPC;          // k of a step
  static constexpr int NJ = SK / 16;          // MFMAs of a step per row and token tile
  static constexpr int PIECES = SK / 8;       // 16-byte pieces of a token's x per step
};

// Block b runs on XCD b % 8: each XCD takes a contiguous range of the tiles,
// whose token blocks share their weight rows in its L2.
__device__ __forceinline__ uint32_t lk_tile() {
  const uint32_t t = blockIdx.x, per = gridDim.x / 8, rem = gridDim.x % 8, xcd = t % 8;
  return xcd * per + (xcd < rem ? xcd : rem) + t / 8;
}

// The weights' buffer descriptors and per-lane offsets.  Rows past N read the
// last row (their results are not stored).
template <int BITS>
struct LkWeights {
  __amdgpu_buffer_rsrc_t rl, ri;
  uint32_t N, K, G, cstride;
  __device__ explicit LkWeights(const LkArgs& a) : N(a.N), K(a.K), G(a.G) {
    const uint32_t bytes = G ? (uint32_t)gi_bytes(G, N, K, BITS) : N * (K * BITS / 8);
    rl = __builtin_amdgcn_make_buffer_rsrc((void*)a.lut, (short)0, (int)(G ? bytes : N * (2u << BITS)), kBufferWord3);
    ri = __builtin_amdgcn_make_buffer_rsrc((void*)a.idx, (short)0, (int)bytes, kBufferWord3);
    cstride = G ? G * kGiChunk : kGiChunk;  // bytes from a row's chunk to its next
  }
  __device__ uint32_t lut_at(uint32_t row) const {
    const uint32_t r = row < N ? row : N - 1;
    return G ? (uint32_t)gi_lut_offset(G, r, K, BITS) : r * (2u << BITS);
  }
  __device__ uint32_t chunk_at(uint32_t row) const {
    const uint32_t r = row < N ? row : N - 1;
    return G ? (uint32_t)gi_chunk_offset(G, r, 0, K, BITS) : r * (K * BITS / 8);
  }
};

// Lookup tables of 64 or 128 rows from row n0 on.  Every wave builds 1/8 of
// every row's entries: at 4 bits from the row's whole LUT, at 8 bits from
// its own 64 bytes of it.  4 bits: rows 64.. follow at dword 256 * 64; 8
// bits: they take the high halves.
template <int BITS, int R>
struct LkTables {
  static constexpr int Q = R / 64, NL = BITS == 4 ? 2 : 4;
  static constexpr int kDwords = (BITS == 4 ? Q : 1) * kLprTableDw;
  u32x4v L[Q][NL];
  __device__ void load(const LkWeights<BITS>& wt, uint32_t n0, uint32_t lane, uint32_t w) {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const uint32_t lo = wt.lut_at(n0 + 64 * q + lane) + (BITS == 8 ? 64u * w : 0u);
#pragma unroll
      for (int i = 0; i < NL; i++) L[q][i] = __builtin_amdgcn_raw_buffer_load_b128(wt.rl, lo + 16u * i, 0u, 0);
    }
  }
  __device__ void build(uint32_t* lds, uint32_t lane, uint32_t w) const {
    if constexpr (BITS == 4) {
#pragma unroll
      for (int q = 0; q < Q; q++) {
        uint32_t d[8], lo[2];
#pragma unroll
        for (int i = 0; i < 8; i++) d[i] = L[q][i >> 2][i & 3];
        // entries w + 8 i: low nibble w + 8 (i % 2), high nibble i / 2
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const uint32_t e = w + 8u * j;
          uint32_t v = d[0];
#pragma unroll
          for (int k = 1; k < 8; k++) v = (e >> 1) == (uint32_t)k ? d[k] : v;
          lo[j] = (e & 1) ? (v >> 16) : (v & 0xFFFFu);
        }
#pragma unroll
        for (int i = 0; i < 32; i++)
          lds[q * kLprTableDw + (w + 8 * i) * 64 + lane] =
              __builtin_amdgcn_perm(d[i / 4], lo[i % 2], (i / 2 & 1) ? 0x07060100u : 0x05040100u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const uint32_t e = w * 32 + 8 * i + 2 * c, lo = L[0][i][c], hi = Q > 1 ? L[Q - 1][i][c] : 0u;
          lds[e * 64 + lane] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
          lds[(e + 1) * 64 + lane] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        }
    }
  }
};

// The A operand of MFMA j of a step for row 32 q + r32: its raw lookups, and
// the operand made of them.
template <int BITS>
struct LkOperand {
  static constexpr int V = BITS == 4 ? 4 : 8;
  uint32_t v[V];
  __device__ __forceinline__ void look(const uint32_t* lds, u32x4v chunk, int j, int q, uint32_t r32) {
    const bool far = BITS == 4 && q >= 2;  // 4-bit rows 64..: the second 64 KB
    const uint32_t row = r32 * 4u + (q & 1) * 128u + (far ? 0x10000u : 0u);
#pragma unroll
    for (int e = 0; e < V; e++) {
      const uint32_t wd = chunk[BITS == 4 ? j : 2 * j + (e >> 2)];
      const uint32_t ad = __builtin_amdgcn_perm(wd, row, (far ? 0x0C020000u : 0x0C0C0000u) | ((4u + (e & 3)) << 8));
      v[e] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(lds) + ad);
    }
  }
  __device__ __forceinline__ u32x4v get(int q) const {
    if constexpr (BITS == 4) {
      return u32x4v{v[0], v[1], v[2], v[3]};
    } else {
      const uint32_t sel = q >= 2 ? 0x07060302u : 0x05040100u;
      return u32x4v{__builtin_amdgcn_perm(v[1], v[0], sel), __builtin_amdgcn_perm(v[3], v[2], sel),
                    __builtin_amdgcn_perm(v[V - 3], v[V - 4], sel), __builtin_amdgcn_perm(v[V - 1], v[V - 2], sel)};
    }
  }
};

__device__ __forceinline__ f32x16v lk_mfma(u32x4v A, u32x4v B, f32x16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8v, A), __builtin_bit_cast(f16x8v, B), c, 0, 0, 0);
}

// Orders a wave's own LDS accesses for the compiler (the LDS executes one
// wave's accesses in order, so no wait is needed).
__device__ __forceinline__ void lk_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); }

// Rows r .. r + 3 (r % 4 == 0) of token m: fp32 to this split's partials, or
// fp16 to Y.
__device__ __forceinline__ bool lk_quads(const LkArgs& a) {  // all four below N, and one store's alignment
  return a.N % 4 == 0 && (a.P || (a.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(a.Y) % 8 == 0));
}
__device__ __forceinline__ void lk_store(const LkArgs& a, bool quads, uint32_t m, uint32_t r, f32x4v v) {
  if (r >= a.N) return;
  if (a.P) {
    float* const p = a.P + ((size_t)blockIdx.y * a.M + m) * a.N + r;
    if (quads) {
      *reinterpret_cast<f32x4v*>(p) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (r + e < a.N) p[e] = v[e];
    }
    return;
  }
  uint16_t* const p = a.Y + (size_t)m * a.ldy + r;
  const uint16_t y[4] = {f2h(v.x), f2h(v.y), f2h(v.z), f2h(v.w)};
  if (quads) {
    *reinterpret_cast<uint64_t*>(p) =
        (uint64_t)y[0] | (uint64_t)y[1] << 16 | (uint64_t)y[2] << 32 | (uint64_t)y[3] << 48;
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (r + e < a.N) p[e] = y[e];
  }
}

}  // namespace

// X [M][K] -> Xp [token tile of 32][step][j][lane][8 halves]: the B operands
// of k_gemm_lookup, zero past M and K, so that each of its x loads reads one
// contiguous KB.  A thread moves 16 bytes; a wave's threads cover the
// pieces of one step of consecutive tokens, so both sides move whole lines.
template <int BITS>
__global__ __launch_bounds__(256) void k_pack_x(const uint16_t* __restrict__ X, uint16_t* __restrict__ Xp, uint32_t M,
                                                uint32_t K, uint32_t steps, uint32_t tiles) {
  using S = LkShape<BITS>;
  constexpr uint32_t PC = S::PIECES;
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const uint32_t o = i % PC, n = i / PC % 32, ts = i / (32 * PC);
  const uint32_t s = ts % steps, u = ts / steps;
  if (u >= tiles) return;
  const uint32_t m = u * 32 + n, k = s * S::SK + 8 * o;
  u32x4v v = {0u, 0u, 0u, 0u};
  if (m < M && k < K) v = *reinterpret_cast<const u32x4v*>(X + (size_t)m * K + k);
  const uint32_t h = o / (PC / 2), j = o % (PC / 2);
  *reinterpret_cast<u32x4v*>(Xp + (((size_t)ts * S::NJ + j) * 64 + 32 * h + n) * 8) = v;
}

// The GEMM of more than a few tokens, over packed X.
//  * A workgroup of 8 waves holds the tables of R = 32 RT rows (64 or 128);
//    wave w takes 32 TT tokens of its token group w / KS and slice w % KS of
//    the K range.  No wave waits for another between the table barrier and
//    the reduction.
//  * Per MFMA step a wave makes RT operands by lookup and reads TT operands
//    of x from L2: 128 x 64 (4 bits) or 64 x 128 (8 bits, whose lookups cost
//    twice) keeps lookups, x loads and MFMAs near balance.
//    14336 x 4096 x 2048 on MI355X: 4 bits 128 x 64 218 us, 64 x 128 234, 64
//    x 64 284; 8 bits 64 x 128 273, 128 x 64 302, 64 x 64 350.
//  * Software pipeline, pinned by the scheduling barriers: item i = (MFMA
//    step j, row tile q) issues its TT MFMAs while the lookups of item i + 3
//    are issued; a step's x registers are refilled as soon as its MFMAs of
//    step j are issued (one step ahead; two where registers allow) and its
//    index chunks once their last lookup is issued (two steps ahead).  Left
//    to the compiler the loads sank to their uses or the loop spilled.
//  * KS > 1: the slices' tiles are added pairwise in a fixed tree, each wave
//    handing its partner half of what it holds.
// Bounded by no single unit: at 14336 x 4096 x 2048 the matrix cores are busy for 63 %
// (4 bits) and 50 % (8 bits) of the cycles, the lookups' LDS for 33 and 27 (no bank
// conflicts), the VALU for 30, and a wave waits for 36..40 % of its time; the clock falls
// to 1.7 GHz.
template <int BITS, int RT, int TT, bool RAGGED>
__global__ __launch_bounds__(512) void k_gemm_lookup(LkArgs a) {
  using S = LkShape<BITS>;
  constexpr int R = 32 * RT, TM = 32 * TT;
  constexpr int BD = BITS == 4 && RT * TT > 4 ? 1 : 2;  // steps of x in flight
  constexpr int NI = S::NJ * RT;                        // items of a step
  constexpr int LA = 3, RING = 4;                       // items of lookups in flight
  constexpr int UN = RT * TT * 4;                       // quads of accumulators
  constexpr int TP = R / 2 + 4;                         // dwords of a token's output in LDS
  constexpr int HALF = 8 * 64 * UN * 2, OUT = 8 * 32 * TP;
  constexpr int TAB = LkTables<BITS, R>::kDwords, RED = HALF > OUT ? HALF : OUT;
  __shared__ __attribute__((aligned(16))) uint32_t lds[TAB > RED ? TAB : RED];

  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t r32 = lane & 31, h = lane >> 5;
  const uint32_t KS = a.KS, TG = kLkWaves / KS, ks = w % KS, tg = w / KS;
  const uint32_t nmb = (a.M + TM * TG - 1) / (TM * TG);
  const uint32_t t = lk_tile();
  const uint32_t n0 = (t / nmb) * R, m0 = (t % nmb) * (TM * TG) + tg * TM;
  // the wave's steps, always in pairs
  const uint32_t pairs = (a.K + 2 * S::SK - 1) / (2 * S::SK), steps = 2 * pairs;
  const uint32_t pb = blockIdx.y * a.per_split;
  const uint32_t np = pairs - pb < a.per_split ? pairs - pb : a.per_split;
  const uint32_t s0 = 2 * (pb + ks * np / KS), s1 = m0 < a.M ? 2 * (pb + (ks + 1) * np / KS) : s0;

  const LkWeights<BITS> wt(a);
  const uint32_t tiles = (a.M + 31) / 32, u0 = m0 / 32;
  const uint32_t tbytes = steps * (S::NJ * 1024u);  // a token tile's operands
  const uint32_t lt = u0 < tiles ? (tiles - u0 < (uint32_t)TT ? tiles - u0 : (uint32_t)TT) : 0u;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.X + (size_t)(lt ? u0 : 0u) * (tbytes / 2)), (short)0, (int)(lt * tbytes), kBufferWord3);

  LkTables<BITS, R> tab;
  tab.load(wt, n0, lane, w);
  uint32_t ibase[RT];
#pragma unroll
  for (int q = 0; q < RT; q++) ibase[q] = wt.chunk_at(n0 + 32 * q + r32) + h * wt.cstride;
  u32x4v ir[2][RT], xr[BD][S::NJ][TT];
  // steps past the wave's range get offsets past the buffers: zeros, and no
  // memory access.  The whole index offset is in the checked part: a ragged
  // row's last chunks may lie past the end of the buffer.
  auto load_i = [&](uint32_t s, int slot) {
    const uint32_t out = s < s1 ? 0u : kOut;
#pragma unroll
    for (int q = 0; q < RT; q++)
      ir[slot][q] = __builtin_amdgcn_raw_buffer_load_b128(wt.ri, (ibase[q] + s * 2u * wt.cstride) | out, 0u, 0);
  };
  auto load_x = [&](uint32_t s, int slot, int j) {
    const uint32_t out = s < s1 ? 0u : kOut;
#pragma unroll
    for (int u = 0; u < TT; u++)
      xr[slot][j][u] =
          __builtin_amdgcn_raw_buffer_load_b128(rx, (u * tbytes + lane * 16u) | out, (s * S::NJ + j) * 1024u, 0);
  };
  load_i(s0, 0);
  load_i(s0 + 1, 1);
#pragma unroll
  for (int u = 0; u < BD; u++)
#pragma unroll
    for (int j = 0; j < S::NJ; j++) load_x(s0 + u, u, j);
  tab.build(lds, lane, w);
  __syncthreads();

  f32x16v acc[RT][TT];
#pragma unroll
  for (int q = 0; q < RT; q++)
#pragma unroll
    for (int u = 0; u < TT; u++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[q][u][e] = 0.0f;
  LkOperand<BITS> op[RING];
  auto look = [&](int slot, int i) { op[i % RING].look(lds, ir[slot][i % RT], i / RT, i % RT, r32); };
  auto step = [&](uint32_t s, int slot, int xslot) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int j = i / RT, q = i % RT;
      u32x4v A = op[i % RING].get(q);
      if constexpr (RAGGED) {
        const bool in = s * S::SK + h * S::EPC + 8u * j < a.K;
#pragma unroll
        for (int e = 0; e < 4; e++) A[e] = in ? A[e] : 0u;
      }
#pragma unroll
      for (int u = 0; u < TT; u++) acc[q][u] = lk_mfma(A, xr[xslot][j][u], acc[q][u]);
      // (past the wave's last step: lookups of zeros, not used)
      if (i + LA < NI)
        look(slot, i + LA);
      else
        look(slot ^ 1, i + LA - NI);
#pragma unroll
      for (int u = 0; u < TT; u++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                           // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, LkOperand<BITS>::V / TT, 0);     // VALU
        __builtin_amdgcn_sched_group_barrier(0x100, LkOperand<BITS>::V / TT, 0);     // DS read
      }
      if (q == RT - 1) load_x(s + BD, xslot, j);
      if (i + LA == NI - 1) load_i(s + 2, slot);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int i = 0; i < LA; i++) look(0, i);
  for (uint32_t s = s0; s < s1; s += 2) {
    step(s, 0, 0);
    step(s + 1, 1, BD - 1);
  }

  // ---- the K slices: at each level a wave hands its partner half of the
  // quads it holds and adds the partner's half of those it keeps.  All waves
  // end with UN / KS finished quads, fl[0 ..], the tile's quads base ..
  f32x4v fl[UN];
#pragma unroll
  for (int q = 0; q < RT; q++)
#pragma unroll
    for (int u = 0; u < TT; u++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        fl[(q * TT + u) * 4 + g] =
            f32x4v{acc[q][u][4 * g], acc[q][u][4 * g + 1], acc[q][u][4 * g + 2], acc[q][u][4 * g + 3]};
  f32x4v* const red = reinterpret_cast<f32x4v*>(lds);
  uint32_t base = 0, cnt = UN;
  auto level = [&](auto n_tag, uint32_t dist) {
    constexpr int H = decltype(n_tag)::value / 2;  // quads kept
    const bool upper = ks & dist;
    f32x4v* const mine = red + w * (H * 64) + lane;
    const f32x4v* const theirs = red + (w ^ dist) * (H * 64) + lane;
    __syncthreads();
    if (upper) {
#pragma unroll
      for (int i = 0; i < H; i++) mine[i * 64] = fl[i];
    } else {
#pragma unroll
      for (int i = 0; i < H; i++) mine[i * 64] = fl[H + i];
    }
    __syncthreads();
    if (upper) {
#pragma unroll
      for (int i = 0; i < H; i++) {
        fl[i] = theirs[i * 64] + fl[H + i];
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (all loads at once would spill)
      }
    } else {
#pragma unroll
      for (int i = 0; i < H; i++) {
        fl[i] += theirs[i * 64];
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    cnt = H;
    base += upper ? H : 0;
  };
  if (KS >= 2) level(std::integral_constant<int, UN>{}, KS / 2);
  if (KS >= 4) level(std::integral_constant<int, UN / 2>{}, KS / 4);
  if (KS >= 8) level(std::integral_constant<int, UN / 4>{}, KS / 8);

  // ---- D: lane (n, h) holds token n, rows 8 g + 4 h .. + 3 of a row tile
  if (KS == 1 && !a.P && a.N % 8 == 0 && a.ldy % 8 == 0 && reinterpret_cast<uintptr_t>(a.Y) % 16 == 0) {
    // whole tiles go through the wave's own part of the LDS, so that a store
    // instruction writes R consecutive rows of each token
    constexpr int PER = R / 8;  // 16-byte pieces of a token
    uint32_t* const ts = lds + w * (32 * TP);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TT; u++) {
      lk_order();
#pragma unroll
      for (int q = 0; q < RT; q++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const f32x4v v = fl[(q * TT + u) * 4 + g];
          uint32_t* const z = ts + r32 * TP + 16 * q + 4 * g + 2 * h;
          z[0] = (uint32_t)f2h(v.x) | (uint32_t)f2h(v.y) << 16;
          z[1] = (uint32_t)f2h(v.z) | (uint32_t)f2h(v.w) << 16;
        }
      lk_order();
#pragma unroll
      for (int i = 0; i < 32 * PER / 64; i++) {
        const uint32_t pc = lane + 64 * i, n = pc / PER, r = n0 + 8 * (pc % PER), m = m0 + 32 * u + n;
        const u32x4v v = *reinterpret_cast<const u32x4v*>(ts + n * TP + 4 * (pc % PER));
        if (m < a.M && r < a.N) *reinterpret_cast<u32x4v*>(a.Y + (size_t)m * a.ldy + r) = v;
      }
    }
    return;
  }
  const bool quads = lk_quads(a);
#pragma unroll
  for (int i = 0; i < UN; i++) {
    const uint32_t un = base + i;
    const uint32_t m = m0 + 32 * (un / 4 % TT) + r32, r = n0 + 32 * (un / (4 * TT)) + 8 * (un % 4) + 4 * h;
    if ((uint32_t)i < cnt && m < a.M) lk_store(a, quads, m, r, fl[i]);
  }
}

// The GEMM of a few tokens: X as it is, through LDS, and no launch before it.
//  * A workgroup of 8 waves takes 64 rows x 32 TT tokens; wave w takes slice w
//    of the K range.  Each wave copies its own slice of x, a step at a time,
//    from registers (two steps in flight) to its own part of the LDS, tokens
//    PIECES pieces and one of padding apart, and reads it back as B operands:
//    the lanes of an operand are 32 tokens, which as direct global reads cost
//    the texture path a line per lane.  No wave waits for another until the
//    partial tiles are added in wave order.
// Bounded by the chain of a workgroup's phases (14336 x 4096, 4 bits, 32
// tokens, MI355X: LUT load and tables 2.5 us, the wave's 8 steps 5..7, the
// sum 1.5): 12 us against 25.1 for two passes of k_gemv_mfma, 16 tokens 11.0
// against 12.6; 8 bits 16 tokens 15.4 against 20.9.
template <int BITS, int TT, bool RAGGED>
__global__ __launch_bounds__(512) void k_gemm_lookup_x(LkArgs a) {
  using S = LkShape<BITS>;
  constexpr int R = 64, MT = 32 * TT;
  constexpr int XP = S::SK / 2 + 4;            // LDS dwords from one token's x to the next
  constexpr int TPI = 64 / S::PIECES;          // tokens of an x load
  constexpr int D = 2;                         // steps in flight
  constexpr int XL = MT / TPI;                 // x loads per lane and step
  constexpr int RP = R + 4;                    // floats from one token's partial sums to the next
  constexpr int TAB = LkTables<BITS, R>::kDwords;
  constexpr int STAGE = TAB + kLkWaves * MT * XP, RED = kLkWaves * MT * RP;
  __shared__ __attribute__((aligned(16))) uint32_t lds[STAGE > RED ? STAGE : RED];

  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t r32 = lane & 31, h = lane >> 5;
  const uint32_t K = a.K, nmb = (a.M + MT - 1) / MT, t = lk_tile();
  const uint32_t n0 = (t / nmb) * R, m0 = (t % nmb) * MT;
  const uint32_t steps = (K + S::SK - 1) / S::SK;
  const uint32_t sb = blockIdx.y * a.per_split;
  const uint32_t ns = steps - sb < a.per_split ? steps - sb : a.per_split;
  const uint32_t s0 = sb + w * ns / kLkWaves, s1 = sb + (w + 1) * ns / kLkWaves;
  const uint32_t live = a.M - m0 < (uint32_t)MT ? a.M - m0 : (uint32_t)MT;

  const LkWeights<BITS> wt(a);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc((void*)(a.X + (size_t)m0 * K), (short)0, (int)(live * K * 2u), kBufferWord3);
  LkTables<BITS, R> tab;
  tab.load(wt, n0, lane, w);
  uint32_t ibase[2];
#pragma unroll
  for (int q = 0; q < 2; q++) ibase[q] = wt.chunk_at(n0 + 32 * q + r32) + h * wt.cstride;
  const uint32_t xk = 8u * (lane % S::PIECES);
  const uint32_t xbase = (lane / S::PIECES) * K * 2u + xk * 2u;
  u32x4v ir[D][2], xr[D][XL];
  auto load = [&](uint32_t s, int slot) {
#pragma unroll
    for (int q = 0; q < 2; q++)
      ir[slot][q] = __builtin_amdgcn_raw_buffer_load_b128(wt.ri, ibase[q] + s * 2u * wt.cstride, 0u, 0);
    const bool in = !RAGGED || s * S::SK + xk < K;
#pragma unroll
    for (int i = 0; i < XL; i++)
      xr[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(
          rx, in ? xbase + s * (S::SK * 2u) + i * TPI * K * 2u : kOut, 0u, 0);
  };
#pragma unroll
  for (int u = 0; u < D; u++)
    if (s0 + u < s1) load(s0 + u, u);
  tab.build(lds, lane, w);
  __syncthreads();

  uint32_t* const xs = lds + TAB + w * MT * XP;
  uint32_t* const xw = xs + (lane / S::PIECES) * XP + 4 * (lane % S::PIECES);
  const uint32_t* const xp = xs + r32 * XP + h * (S::EPC / 2);
  f32x16v acc[2][TT];
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int u = 0; u < TT; u++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[q][u][e] = 0.0f;
  auto step = [&](uint32_t s, int slot) {
    lk_order();
#pragma unroll
    for (int i = 0; i < XL; i++) *reinterpret_cast<u32x4v*>(xw + i * TPI * XP) = xr[slot][i];
    lk_order();
#pragma unroll
    for (int j = 0; j < S::NJ; j++) {
      u32x4v A[2], B[TT];
#pragma unroll
      for (int u = 0; u < TT; u++) B[u] = *reinterpret_cast<const u32x4v*>(xp + 32 * u * XP + 4 * j);
#pragma unroll
      for (int q = 0; q < 2; q++) {
        LkOperand<BITS> op;
        op.look(lds, ir[slot][q], j, q, r32);
        A[q] = op.get(q);
        if constexpr (RAGGED) {
          const bool in = s * S::SK + h * S::EPC + 8u * j < K;
#pragma unroll
          for (int e = 0; e < 4; e++) A[q][e] = in ? A[q][e] : 0u;
        }
      }
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int u = 0; u < TT; u++) acc[q][u] = lk_mfma(A[q], B[u], acc[q][u]);
    }
  };
  // whole rounds of D steps with the next round in flight, then what is left
  uint32_t s = s0;
  for (; s + 2 * D <= s1; s += D) {
#pragma unroll
    for (int u = 0; u < D; u++) {
      step(s + u, u);
      load(s + u + D, u);
    }
  }
#pragma unroll
  for (int u = 0; u < D; u++)
    if (s + u < s1) {
      step(s + u, u);
      if (s + u + D < s1) load(s + u + D, u);
    }
#pragma unroll
  for (int u = 0; u < D; u++)
    if (s + u + D < s1) step(s + u + D, u);

  // ---- the waves' partial tiles [wave][token][row], added in wave order
  float* const red = reinterpret_cast<float*>(lds);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int u = 0; u < TT; u++)
#pragma unroll
      for (int g = 0; g < 4; g++)
        *reinterpret_cast<f32x4v*>(red + (w * MT + 32 * u + r32) * RP + 32 * q + 8 * g + 4 * h) =
            f32x4v{acc[q][u][4 * g], acc[q][u][4 * g + 1], acc[q][u][4 * g + 2], acc[q][u][4 * g + 3]};
  __syncthreads();
  const bool quads = lk_quads(a);
#pragma unroll
  for (int i = 0; i < MT * 16 / 512; i++) {
    const uint32_t p = tid + 512u * i, m = p / 16, r = 4 * (p % 16);
    f32x4v v = *reinterpret_cast<const f32x4v*>(red + m * RP + r);
#pragma unroll
    for (int k = 1; k < (int)kLkWaves; k++) v += *reinterpret_cast<const f32x4v*>(red + (k * MT + m) * RP + r);
    if (m < live) lk_store(a, quads, m0 + m, n0 + r, v);
  }
}

const void* lk_kernel(uint32_t bits, int rt, int tt, bool ragged) {
#define PRISM_LK(B_, R_, T_)                                                        \
  if (bits == B_ && rt == R_ && tt == T_)                                           \
    return ragged ? reinterpret_cast<const void*>(&k_gemm_lookup<B_, R_, T_, true>) \
                  : reinterpret_cast<const void*>(&k_gemm_lookup<B_, R_, T_, false>);
  PRISM_LK(4, 2, 2)
  PRISM_LK(4, 4, 2)
  PRISM_LK(8, 2, 2)
  PRISM_LK(8, 2, 4)
#undef PRISM_LK
  return nullptr;
}

const void* lkx_kernel(uint32_t bits, int tt, bool ragged) {
#define PRISM_LKX(B_, T_)                                                          \
  if (bits == B_ && tt == T_)                                                      \
    return ragged ? reinterpret_cast<const void*>(&k_gemm_lookup_x<B_, T_, true>)  \
                  : reinterpret_cast<const void*>(&k_gemm_lookup_x<B_, T_, false>);
  PRISM_LKX(4, 1)
  PRISM_LKX(4, 2)
  PRISM_LKX(8, 1)
  PRISM_LKX(8, 2)
#undef PRISM_LKX
  return nullptr;
}

const void* lk_pack_kernel(uint32_t bits) {
  return bits == 4 ? reinterpret_cast<const void*>(&k_pack_x<4>) : reinterpret_cast<const void*>(&k_pack_x<8>);
}

}  // namespace prism
