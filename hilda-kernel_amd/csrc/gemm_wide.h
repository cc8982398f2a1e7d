// The 16-bit GEMM of the fused-linear ops on gfx950 MFMA: C[M,N] = sum_k
// A(m,k) B(n,k), bf16 or fp16 inputs, fp32 accumulation, epilogues as gemm_nt.h
// declares them. Each operand is K-contiguous (K a multiple of 64) or
// MN-contiguous (any K: k-rows past its stored extent read zero).
//
// Bound by the matrix pipes and, in long runs, by the part's power limit. One
// 256x256 tile a workgroup of 4 waves, one wave a SIMD, each wave 128x128
// (8x8 16x16x32 MFMAs, 256 accumulators in AGPRs): a wave tile of 128x64 on 8
// waves, which this replaces, reads half as many LDS bytes again per FLOP. K advances
// 64 a stage through two 64 KiB LDS stages filled by buffer-to-LDS DMA.
//
// With one wave a SIMD nothing hides a stall but the order of the instructions,
// so the K loop is written in issue order and kept there: the MFMAs are
// volatile asm with the accumulator as one in-out AGPR operand (the builtin
// form let the register allocator copy accumulators between tuples, 500 moves a
// stage), and the LDS reads and the DMA sit at fixed slots between them. Per
// stage, in slots of one MFMA (16 cycles, four issue slots):
//   first half:  64 MFMAs on k 0..31 of the stage, the reads of its k 32..63 at
//                every 2nd, the next DMA buffers' scalar set-up;
//   wait for the own DMA of the next stage and the own reads, one barrier;
//   second half: 64 MFMAs on k 32..63, the DMA of the stage after next into the
//                buffer just read at every 4th (16 at once, or at every 2nd or
//                3rd, were 2-7% slower: they crowd the LDS reads out), the next
//                stage's k 0..31 reads at every 3rd.
// MN-contiguous operands go through ds_read_b64_tr_b16. The compiler holds that
// read back until every DMA into LDS has landed unless alias scopes tell the
// stages apart: hence core() and its restrict pointers, one per operand and
// stage. (Without them every stage waited for the next one's loads.)
//
// Persistent: a workgroup walks its tiles (blockIdx.x, + gridDim.x, ..) and fetches the next tile's first two stages
// during this one's last two, so the accumulators go out (WideOut below) while those land and no tile starts on an
// empty pipeline.
//
// Measured, TFLOP/s, kernel alone, 8 waves and one tile a workgroup -> this; M x N x K:
//   both K-contiguous                  8192x32768x4096 1280 -> 1454-1484
//   both MN-contiguous                 8192x32768x4096 1060 -> 1373-1382   8192x4096x4096 1170 -> 1493-1524
//   B MN-contiguous, read-modify-write 8192x4096x4096  1070 -> 1393-1458
// A tile's time beyond its K loop (the intercept over K at 8192x32768): 13 us one tile a workgroup -> 7 us, with a
// read-modify-write epilogue 51 -> 21 us. torch.matmul's best layout at 8192x32000x4096: 1494. In long runs the
// matrix pipes are 72-80% busy at 1.6-1.8 GHz: the power limit (logits, dX and dW of 16384 rows, H 4096, V 128256: 6.2,
// 6.2 and 12.1 ms).
#pragma once

#include "hk_common.h"

#include <type_traits>

namespace hk {
namespace gemm {

// A lambda inlined with the function it stands in (before that function is inlined elsewhere, where its alias
// scopes are attached).
#define HK_INLINE __attribute__((always_inline))

struct Wide {
  static constexpr int BM = 256, BN = 256, BK = 64, NT = 256;
  static constexpr int GROUP_M = 4;  // tiles an XCD runs at once: 4 A panels x 8 B panels (2, 8 and 16: 0-6% slower)
  static constexpr int kOpBytes = 256 * BK * 2;    // one operand's stage
  static constexpr int kLdsBytes = 4 * kOpBytes;   // [A0][A1][B0][B1]; the epilogue stages half a tile in it
  // slots of the K loop (see above)
  static constexpr int kRead1 = 2, kRead0 = 3, kDma = 4, kSetupA = 36, kSetupB = 48;
};

// Two 16-byte chunks of k per row: swizzles of the stage tiles.
// K-contiguous [256][64]: chunk ^ (row / 2) % 8, so the 16 rows a fragment read
// serves together cover the 64 banks. MN-contiguous [64][256]: chunk ^ 4 (k % 4)
// ^ 2 (k / 8 % 2), so the 4 k-rows of a 16-lane transposed read, and the two
// groups of a half-wave (8 k-rows apart), do.
__device__ __forceinline__ int wide_swz_k(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int wide_swz_mn(int k) { return (4 * (k & 3)) ^ (2 * ((k >> 3) & 1)); }

// A tile's operand panels: the element offset of their first row (column) and first k, their rows inside the matrix,
// the stored k past that start (MN-contiguous operands), and the tile's stages.
struct WideTile {
  int64_t at_a, at_b;
  int rows_a, rows_b, KT, ka, kb;
};

// Every tile of this workgroup: next(tile) gives the first and each following one (false: none left), done(acc) takes
// a finished one's accumulators, early() runs a stage before that. a0 a1 b0 b1: the LDS stages.
template <typename T, bool AMN, bool BMN, class Next, class Early, class Done>
__device__ __forceinline__ void wide_core(unsigned char* __restrict__ a0, unsigned char* __restrict__ a1,
                                          unsigned char* __restrict__ b0, unsigned char* __restrict__ b1,
                                          const T* __restrict__ A, const T* __restrict__ B, int64_t lda, int64_t ldb,
                                          int wave, int lane, Next&& next, Early&& early, Done&& done) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(sizeof(T) == 2, "bf16 or fp16 inputs");
  const int wm = wave >> 1, wn = wave & 1, fr = lane & 15, fk = lane >> 4;
  f32x4_t acc[8][8];
  auto clear = [&]() HK_INLINE {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };

  // LDS read bases. K-contiguous fragment t of half h: lane l holds row 16 t + l % 16, k = 32 h + 8 (l / 16)
  // .. + 7, one ds_read_b128 (one base per half, t in the immediate). MN-contiguous: two transposed reads (k
  // + 0..3, + 4..7); within each 16-lane group, lane i points at k-row i / 4 and row 4 (i % 4) and receives
  // row i's four k (one base per fragment, the half in the immediate).
  auto read_base = [&](bool mn, int R, int t) HK_INLINE -> uint32_t {
    if (mn) {
      const int kq = fr >> 2, r = R + 16 * t + 4 * (fr & 3), k = 8 * fk + kq;
      return (uint32_t)((k * 256 + ((r >> 3) ^ wide_swz_mn(k)) * 8 + (r & 7)) * 2);
    }
    return (uint32_t)((R + fr) * 128 + (((4 * t + fk) ^ wide_swz_k(fr)) << 4));
  };
  uint32_t abase[AMN ? 8 : 2], bbase[BMN ? 8 : 2];
#pragma unroll
  for (int t = 0; t < (AMN ? 8 : 2); ++t) {
    abase[t] = read_base(AMN, wm * 128, t);
    asm volatile("" : "+v"(abase[t]));  // kept in registers, not recomputed per read
  }
#pragma unroll
  for (int t = 0; t < (BMN ? 8 : 2); ++t) {
    bbase[t] = read_base(BMN, wn * 128, t);
    asm volatile("" : "+v"(bbase[t]));
  }

  // DMA: a 1 KiB load lands 16 bytes a lane, in lane order, so each lane fetches the chunk its LDS place
  // holds. K-contiguous: the panel's rows, the stage's k in the scalar offset; rows past the matrix are past
  // the buffer's end. MN-contiguous: the buffer starts at the stage's first k-row and ends with the stored
  // k-rows; chunks past the matrix's rows are redirected out of it.
  uint32_t va[8], vb[8];
  auto dma_offset = [&](bool mn, int q, int64_t ld, int rows) HK_INLINE -> uint32_t {
    if (mn) {
      const int k = q / 32, r = ((q % 32) ^ wide_swz_mn(k)) * 8;
      return r < rows ? (uint32_t)(k * ld + r) * 2u : kOobOffset;
    }
    const int r = q / 8;
    return (uint32_t)(r * ld + ((q % 8) ^ wide_swz_k(r)) * 8) * 2u;
  };
  // one operand's next stage: its buffer and scalar offset, advanced a stage per call. Scalar values only
  // (readfirstlane): a buffer in vector registers would turn every load into a loop over its lanes.
  // (the pointer is the kernel's argument plus a scalar offset: its alias scope has to be seen, too.)
  struct Feed {
    int64_t at;  // bytes
    int left, off, bytes;
  };
  auto scalar = [](int64_t v) HK_INLINE {
    return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
                     ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)((uint64_t)v >> 32)) << 32));
  };
  Feed na{}, nb{};
  // the feeds at a tile's start; without one (`any` false) they end at once and their loads return zeros
  auto feed = [&](const WideTile& t, bool any) HK_INLINE {
    // (an MN-contiguous operand of an odd stage count ends at KT stages: the trailing one reads zeros)
    na = Feed{scalar(t.at_a * 2),
              __builtin_amdgcn_readfirstlane(any ? (AMN ? min(t.ka, t.KT * 64) : t.KT * 64) : 0), -128,
              AMN ? (int)lda * 2 : __builtin_amdgcn_readfirstlane((int)(t.rows_a * lda * 2))};
    nb = Feed{scalar(t.at_b * 2),
              __builtin_amdgcn_readfirstlane(any ? (BMN ? min(t.kb, t.KT * 64) : t.KT * 64) : 0), -128,
              BMN ? (int)ldb * 2 : __builtin_amdgcn_readfirstlane((int)(t.rows_b * ldb * 2))};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      va[i] = dma_offset(AMN, (wave * 8 + i) * 64 + lane, lda, t.rows_a);
      vb[i] = dma_offset(BMN, (wave * 8 + i) * 64 + lane, ldb, t.rows_b);
    }
  };
  __amdgpu_buffer_rsrc_t rsa, rsb;
  auto setup = [&](bool mn, Feed& n, const T* p, int64_t ld, __amdgpu_buffer_rsrc_t& rs) HK_INLINE {
    char* const base = const_cast<char*>(reinterpret_cast<const char*>(p)) + scalar(n.at);
    if (mn) {  // n.bytes: a k-row's
      const int bytes = __builtin_amdgcn_readfirstlane(max(0, min(64, n.left)) * n.bytes);
      rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, kRsrcWord3);
      n.at += 128 * ld;
      n.off = 0;
    } else {  // n.bytes: the panel's; past the last stage a zero-length buffer, the loads return zeros
      rs = __builtin_amdgcn_make_buffer_rsrc(base, 0, __builtin_amdgcn_readfirstlane(n.left > 0 ? n.bytes : 0),
                                             kRsrcWord3);
      n.off = n.left > 0 ? n.off + 128 : 0;
    }
    n.left -= 64;
  };
  auto dma = [&](auto stage, int t) HK_INLINE {  // load t (A 0..7, B 8..15) of the stage set up last
    constexpr int st = decltype(stage)::value;
    if (t < 8)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (st ? a1 : a0) + (wave * 8 + t) * 1024, 16, va[t], na.off, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (st ? b1 : b0) + (wave * 8 + t - 8) * 1024, 16, vb[t - 8],
                                               nb.off, 0, 0);
  };

  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  auto frag = [&](bool mn, unsigned char* p, uint32_t base_t, uint32_t base_h, int h, int t) HK_INLINE -> u32x4 {
    if (mn) {
      v4i16 v[2];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        v[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + base_t + (32 * h + 4 * q) * 512));
      const u32x2 lo = __builtin_bit_cast(u32x2, v[0]), hi = __builtin_bit_cast(u32x2, v[1]);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
    return *reinterpret_cast<const u32x4*>(p + base_h + t * 2048);
  };
  u32x4 fa[2][8], fb[2][8];
  // read s (0..15) of half h, in the order the MFMAs need them: b0 a0 b1 .. b7 a1 .. a7
  auto read = [&](auto stage, int h, int s) HK_INLINE {
    constexpr int st = decltype(stage)::value;
    const bool is_b = s == 0 || (s >= 2 && s <= 8);
    const int t = s <= 1 ? 0 : s <= 8 ? s - 1 : s - 8;
    if (is_b) fb[h][t] = frag(BMN, st ? b1 : b0, bbase[BMN ? t : 0], bbase[BMN ? 0 : h], h, t);
    else fa[h][t] = frag(AMN, st ? a1 : a0, abase[AMN ? t : 0], abase[AMN ? 0 : h], h, t);
  };
  // MFMA m of half h: fed B then A, so a lane holds C row 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3
  auto mma = [&](int h, int m) HK_INLINE {
    const int i = m >> 3, j = m & 7;
    if constexpr (std::is_same<T, __bf16>::value)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[h][j]), "v"(fa[h][i]));
    else
      asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[h][j]), "v"(fa[h][i]));
  };
  // The compiler does not know the asm above as MFMAs: before their first use and after their last, every
  // accumulator waits out the longest MFMA hazard.
  auto settle = [&]() HK_INLINE {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      asm volatile("s_nop 15"
                   : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]),
                     "+a"(acc[i][5]), "+a"(acc[i][6]), "+a"(acc[i][7]));
  };
  // s_waitcnt as an instruction the compiler counts (asm text it would not)
  auto wait = [](auto cnt) HK_INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(decltype(cnt)::value);
    asm volatile("" ::: "memory");
  };
  using Lgkm0 = std::integral_constant<int, 0xc07f>;
  using Vm0Lgkm0 = std::integral_constant<int, 0x0070>;
  using Vm16 = std::integral_constant<int, 0x4f70>;
  auto barrier = []() HK_INLINE {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  auto body = [&](auto cur) HK_INLINE {
    using Nx = std::integral_constant<int, decltype(cur)::value ^ 1>;
    wait(Lgkm0{});
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      mma(0, m);
      if (m % Wide::kRead1 == 0 && m / Wide::kRead1 < 16) read(cur, 1, m / Wide::kRead1);
      if (m == Wide::kSetupA) setup(AMN, na, A, lda, rsa);
      if (m == Wide::kSetupB) setup(BMN, nb, B, ldb, rsb);
    }
    wait(Vm0Lgkm0{});  // this wave's DMA of the next stage, and its reads of this one
    barrier();         // every wave's
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      mma(1, m);
      if (m % Wide::kDma == 0) dma(cur, m / Wide::kDma);
      if (m % Wide::kRead0 == 1 && m / Wide::kRead0 < 16) read(Nx{}, 0, m / Wide::kRead0);
    }
  };

  WideTile cur;
  if (!next(cur)) return;
  feed(cur, true);
  setup(AMN, na, A, lda, rsa);
  setup(BMN, nb, B, ldb, rsb);
#pragma unroll
  for (int t = 0; t < 16; ++t) dma(S0{}, t);
  setup(AMN, na, A, lda, rsa);
  setup(BMN, nb, B, ldb, rsb);
#pragma unroll
  for (int t = 0; t < 16; ++t) dma(S1{}, t);
  wait(Vm16{});  // stage 0
  barrier();
#pragma unroll
  for (int s = 0; s < 16; ++s) read(S0{}, 0, s);
  for (bool more = true; more;) {
    clear();
    settle();
    // an odd stage count gets a trailing stage of zeros
    for (int kt = (__builtin_amdgcn_readfirstlane(cur.KT) + 1) / 2; kt > 1; --kt) {
      body(S0{});
      body(S1{});
    }
    // the tile's last two stages, fetching the next tile's first two; the accumulators go out while those land
    more = next(cur);
    feed(cur, more);
    early();
    body(S0{});
    body(S1{});
    settle();
    done(acc);
  }
  wait(Vm0Lgkm0{});  // the zero-length loads past the end target LDS: landed before the workgroup ends
#endif
}

// A finished 128x128 wave tile goes out from the accumulators, with no LDS (the next tile's stages land there) and no
// barrier: a lane holds 4 consecutive columns of a row, two half- and quarter-wave swaps make that 8. An epilogue
// functor takes them in
//   static constexpr bool kReads; using Prior8 = what load8 returns;
//   int64_t out_row(int row) const;                                              // where a row goes
//   Prior8 load8(int64_t out, int col, int n) const;                             // (kReads)
//   void store8(int64_t out, int col, const float* v, int n, const Prior8&) const;
// with n of the 8 columns from col inside the matrix. An epilogue that reads gets the loads of kBatch chunks in
// flight, the first batch issued a stage before the tile ends. (Staged through LDS, half a tile at a time, the
// read-modify-write of a tile took 51 us: four round trips of 8-byte loads with the matrix pipes idle.) One code
// path for whole and edge tiles: with two, the compiler read all 256 accumulators before their branch and spilled them.
// Accumulation in a 16-bit output (EpiDw<T, 1>) still spills 24 bytes a lane with B MN-contiguous and 48 with both,
// beside the transposed reads' bases; the other forms have no scratch. Its GEMM (8192x4096x4096, B MN-contiguous) takes
// 459 us against 389 without the accumulation, a quarter of the waves' time in waits.
template <class Epi>
struct WideOut {
  static constexpr int kBatch = Epi::kReads ? 32 / (int)(sizeof(typename Epi::Prior8) / 4) : 1;  // 32 registers
  Epi e;
  int m = 0, n = 0, row0 = 0, col0 = 0;  // the matrix; this lane's first row and column
  typename Epi::Prior8 prior[kBatch];

  __device__ __forceinline__ void load(int b) {
    if constexpr (Epi::kReads) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int c = b * kBatch + u, row = row0 + 16 * (c / 4), col = col0 + 32 * (c % 4);
        if (row < m && col < n) prior[u] = e.load8(e.out_row(row), col, min(8, n - col));
      }
    }
  }
  __device__ __forceinline__ void store(const f32x4_t (&acc)[8][8]) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = row0 + 16 * i;
      const int64_t out = row < m ? e.out_row(row) : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = 4 * i + j, col = col0 + 32 * j;
        float v[8];
        // (whole vectors are cast: __builtin_bit_cast of one vector element reads element 0 with this compiler)
        const u32x4 lo = __builtin_bit_cast(u32x4, acc[i][2 * j]), hi = __builtin_bit_cast(u32x4, acc[i][2 * j + 1]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const auto x = __builtin_amdgcn_permlane32_swap(lo[q], hi[q], false, false);
          const auto y = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
          v[q] = __builtin_bit_cast(float, (uint32_t)y[0]);
          v[4 + q] = __builtin_bit_cast(float, (uint32_t)y[1]);
        }
        if (row < m && col < n) e.store8(out, col, v, min(8, n - col), prior[c % kBatch]);
        if (Epi::kReads && c % kBatch == kBatch - 1 && c < 31) load(c / kBatch + 1);
      }
    }
#endif
  }
};

template <typename T, class Epi, bool AMN, bool BMN>
__global__ __launch_bounds__(Wide::NT, 1) void gemm_wide_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                                Shape g, Epi epi) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[Wide::kLdsBytes];
  apply_bound(g, Wide::BK);
  const int nbm = (g.M + Wide::BM - 1) / Wide::BM, nbn = (g.N + Wide::BN - 1) / Wide::BN;
  const int tiles = nbm * nbn;
  const int KTall = (g.K + Wide::BK - 1) / Wide::BK;  // >= 1 (checked by the launcher)
  const int nsplit = auto_splits(tiles, KTall, g.ksplit), total = tiles * nsplit;
  const int per = (KTall + nsplit - 1) / nsplit;  // stages a split (auto_splits keeps every split non-empty)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this workgroup's tiles: blockIdx.x, + gridDim.x, ... (a multiple of 8 workgroups keeps each XCD's band)
  int unit = (int)blockIdx.x;
  WideOut<Epi> out{epi}, pend{epi};  // the tile in flight, the one being fetched
  auto next = [&](WideTile& t) -> bool {
    if (unit >= total) return false;  // uniform: past the last tile, or a device-side bound
    const int split = unit / tiles;
    int tm, tn;
    tile_of_block<Wide::GROUP_M>(unit - split * tiles, nbm, nbn, &tm, &tn);
    unit += (int)gridDim.x;
    const int m0 = tm * Wide::BM, n0 = tn * Wide::BN, kt0 = split * per;
    const int64_t k0 = (int64_t)kt0 * Wide::BK;
    t.at_a = AMN ? k0 * g.lda + m0 : m0 * g.lda + k0;
    t.at_b = BMN ? k0 * g.ldb + n0 : n0 * g.ldb + k0;
    t.rows_a = min(Wide::BM, g.M - m0);
    t.rows_b = min(Wide::BN, g.N - n0);
    t.KT = min(per, KTall - kt0);
    t.ka = g.ka - (int)k0;
    t.kb = g.kb - (int)k0;
    apply_split(pend.e, split, nsplit, g.M, 0);
    pend.m = g.M;
    pend.n = g.N;
    pend.row0 = m0 + (wave >> 1) * 128 + (lane & 15);
    pend.col0 = n0 + (wave & 1) * 128 + 8 * (lane >> 4);
    return true;
  };
  constexpr int S = Wide::kOpBytes;
  wide_core<T, AMN, BMN>(
      lds_raw, lds_raw + S, lds_raw + 2 * S, lds_raw + 3 * S, A, B, g.lda, g.ldb, wave, lane,
      [&](WideTile& t) {
        out = pend;
        return next(t);
      },
      [&]() { out.load(0); }, [&](f32x4_t(&acc)[8][8]) { out.store(acc); });
}

}  // namespace gemm
}  // namespace hk
