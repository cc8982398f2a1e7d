// The 16-bit GEMM of the fused-linear ops on gfx950 MFMA: C[M,N] = sum_k
// A(m,k) B(n,k), bf16 or fp16 inputs, fp32 accumulation, epilogues as gemm_nt.h
// declares them. Each operand is K-contiguous (K a multiple of 64) or
// MN-contiguous (any K: k-rows past its stored extent read zero).
//
// Bound by the matrix pipes and, in long runs, by the part's power limit. One
// 256x256 tile a workgroup of 4 waves, one wave a SIMD, each wave 128x128
// (8x8 16x16x32 MFMAs, 256 accumulators in AGPRs): a wave tile of 128x64 on 8
// waves, which this replaces, reads a third more LDS bytes per FLOP. K advances
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
// Measured, TFLOP/s, kernel alone, before (8 waves) -> after; M x N x K:
//   both K-contiguous   8192x32000x4096 1280 -> 1426   8192x4096x32000 1285 -> 1422
//   B MN-contiguous     8192x32000x4096 1115 -> 1419   8192x4096x32000 1107 -> 1443
//   both MN-contiguous  8192x32000x4096 1057 -> 1431   8192x4096x32000 1075 -> 1474
// torch.matmul on the first shape, its own layout: 1494. The matrix pipes are
// 73% busy at 1.9 GHz in all three.
#pragma once

#include "hk_common.h"

#include <type_traits>

namespace hk {
namespace gemm {

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

// The K loop: acc += the tile's products over KT stages of 64 k.
// a0 a1 b0 b1: the LDS stages. pa, pb: the operand panels at this workgroup's
// first row (column) and first k. ra, rb: their rows inside the matrix. ka, kb:
// stored k past that start (MN-contiguous operands).
template <typename T, bool AMN, bool BMN>
__device__ __forceinline__ void wide_core(f32x4_t (&acc)[8][8], unsigned char* __restrict__ a0,
                                          unsigned char* __restrict__ a1, unsigned char* __restrict__ b0,
                                          unsigned char* __restrict__ b1, const T* __restrict__ pa,
                                          const T* __restrict__ pb, int64_t lda, int64_t ldb, int rows_a, int rows_b,
                                          int KT, int ka, int kb, int wave, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(sizeof(T) == 2, "bf16 or fp16 inputs");
  const int wm = wave >> 1, wn = wave & 1, fr = lane & 15, fk = lane >> 4;
  KT = __builtin_amdgcn_readfirstlane(KT);

  // LDS read bases. K-contiguous fragment t of half h: lane l holds row 16 t + l % 16, k = 32 h + 8 (l / 16)
  // .. + 7, one ds_read_b128 (one base per half, t in the immediate). MN-contiguous: two transposed reads (k
  // + 0..3, + 4..7); within each 16-lane group, lane i points at k-row i / 4 and row 4 (i % 4) and receives
  // row i's four k (one base per fragment, the half in the immediate).
  auto read_base = [&](bool mn, int R, int t) -> uint32_t {
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
  auto dma_offset = [&](bool mn, int q, int64_t ld, int rows) -> uint32_t {
    if (mn) {
      const int k = q / 32, r = ((q % 32) ^ wide_swz_mn(k)) * 8;
      return r < rows ? (uint32_t)(k * ld + r) * 2u : kOobOffset;
    }
    const int r = q / 8;
    return (uint32_t)(r * ld + ((q % 8) ^ wide_swz_k(r)) * 8) * 2u;
  };
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    va[i] = dma_offset(AMN, (wave * 8 + i) * 64 + lane, lda, rows_a);
    vb[i] = dma_offset(BMN, (wave * 8 + i) * 64 + lane, ldb, rows_b);
  }
  // one operand's next stage: its buffer and scalar offset, advanced a stage per call. Scalar values only
  // (readfirstlane): a buffer in vector registers would turn every load into a loop over its lanes.
  struct Next {
    const char* p;
    int64_t step;
    int ld2, left, off;
  };
  auto scalar = [](const char* p) {
    const uint64_t v = (uint64_t)p;
    return const_cast<char*>(reinterpret_cast<const char*>(
        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32)));
  };
  const int bytes_a = AMN ? 0 : (int)(rows_a * lda * 2), bytes_b = BMN ? 0 : (int)(rows_b * ldb * 2);
  // (an MN-contiguous operand of an odd stage count ends at KT stages: the trailing one reads zeros)
  Next na{(const char*)pa, 64 * lda * 2, (int)lda * 2, __builtin_amdgcn_readfirstlane(AMN ? min(ka, KT * 64) : KT * 64),
          -128};
  Next nb{(const char*)pb, 64 * ldb * 2, (int)ldb * 2, __builtin_amdgcn_readfirstlane(BMN ? min(kb, KT * 64) : KT * 64),
          -128};
  __amdgpu_buffer_rsrc_t rsa, rsb;
  auto setup = [&](bool mn, Next& n, int panel_bytes, __amdgpu_buffer_rsrc_t& rs) {
    if (mn) {
      const int bytes = __builtin_amdgcn_readfirstlane(max(0, min(64, n.left)) * n.ld2);
      rs = __builtin_amdgcn_make_buffer_rsrc(scalar(n.p), 0, bytes, kRsrcWord3);
      n.p += n.step;
      n.off = 0;
    } else {  // past the last stage: a zero-length buffer, the loads return zeros
      rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(n.p), 0, n.left > 0 ? panel_bytes : 0, kRsrcWord3);
      n.off = n.left > 0 ? n.off + 128 : 0;
    }
    n.left -= 64;
  };
  auto dma = [&](auto stage, int t) {  // load t (A 0..7, B 8..15) of the stage set up last
    constexpr int st = decltype(stage)::value;
    if (t < 8)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (st ? a1 : a0) + (wave * 8 + t) * 1024, 16, va[t], na.off, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (st ? b1 : b0) + (wave * 8 + t - 8) * 1024, 16, vb[t - 8],
                                               nb.off, 0, 0);
  };

  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  auto frag = [&](bool mn, unsigned char* p, uint32_t base_t, uint32_t base_h, int h, int t) -> u32x4 {
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
  auto read = [&](auto stage, int h, int s) {
    constexpr int st = decltype(stage)::value;
    const bool is_b = s == 0 || (s >= 2 && s <= 8);
    const int t = s <= 1 ? 0 : s <= 8 ? s - 1 : s - 8;
    if (is_b) fb[h][t] = frag(BMN, st ? b1 : b0, bbase[BMN ? t : 0], bbase[BMN ? 0 : h], h, t);
    else fa[h][t] = frag(AMN, st ? a1 : a0, abase[AMN ? t : 0], abase[AMN ? 0 : h], h, t);
  };
  // MFMA m of half h: fed B then A, so a lane holds C row 16 i + l % 16, columns 16 j + 4 (l / 16) .. + 3
  auto mma = [&](int h, int m) {
    const int i = m >> 3, j = m & 7;
    if constexpr (std::is_same<T, __bf16>::value)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[h][j]), "v"(fa[h][i]));
    else
      asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[h][j]), "v"(fa[h][i]));
  };
  // The compiler does not know the asm above as MFMAs: before their first use and after their last, every
  // accumulator waits out the longest MFMA hazard.
  auto settle = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      asm volatile("s_nop 15"
                   : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]),
                     "+a"(acc[i][5]), "+a"(acc[i][6]), "+a"(acc[i][7]));
  };
  // s_waitcnt as an instruction the compiler counts (asm text it would not)
  auto wait = [](auto cnt) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(decltype(cnt)::value);
    asm volatile("" ::: "memory");
  };
  using Lgkm0 = std::integral_constant<int, 0xc07f>;
  using Vm0Lgkm0 = std::integral_constant<int, 0x0070>;
  using Vm16 = std::integral_constant<int, 0x4f70>;
  auto barrier = []() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;

  auto body = [&](auto cur) {
    using Nx = std::integral_constant<int, decltype(cur)::value ^ 1>;
    wait(Lgkm0{});
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      mma(0, m);
      if (m % Wide::kRead1 == 0 && m / Wide::kRead1 < 16) read(cur, 1, m / Wide::kRead1);
      if (m == Wide::kSetupA) setup(AMN, na, bytes_a, rsa);
      if (m == Wide::kSetupB) setup(BMN, nb, bytes_b, rsb);
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

  settle();
  setup(AMN, na, bytes_a, rsa);
  setup(BMN, nb, bytes_b, rsb);
#pragma unroll
  for (int t = 0; t < 16; ++t) dma(S0{}, t);
  setup(AMN, na, bytes_a, rsa);
  setup(BMN, nb, bytes_b, rsb);
#pragma unroll
  for (int t = 0; t < 16; ++t) dma(S1{}, t);
  wait(Vm16{});  // stage 0
  barrier();
#pragma unroll
  for (int s = 0; s < 16; ++s) read(S0{}, 0, s);
  const int KT2 = KT + (KT & 1);  // an odd count gets a trailing stage of zeros
  for (int kt = 0; kt + 2 < KT2; kt += 2) {
    body(S0{});
    body(S1{});
  }
  body(S0{});
  wait(Lgkm0{});
#pragma unroll
  for (int m = 0; m < 64; ++m) {
    mma(0, m);
    if (m < 16) read(S1{}, 1, m);
  }
#pragma unroll
  for (int m = 0; m < 64; ++m) mma(1, m);
  settle();
  wait(Vm0Lgkm0{});  // the zero-length loads past the end target LDS too: drained before it is reused
  barrier();
#endif
}

// The epilogue contract of gemm_nt.h, from this kernel's accumulators: half a
// tile (the 128 rows of two waves) is staged in LDS at a time, its 16-byte
// chunks XOR-swizzled by the row, and read back as row chunks.
template <class Epi>
__device__ __forceinline__ void wide_epilogue(const f32x4_t (&acc)[8][8], unsigned char* lds_raw, int m0, int n0,
                                              const Shape& g, const Epi& epi) {
  using S = typename Epi::Stage;
  constexpr int EPC = 16 / (int)sizeof(S);           // elements per chunk
  constexpr int CPR = 256 / EPC;                     // chunks per staged row
  constexpr int SH = sizeof(S) == 4 ? 2 : 1;         // the swizzle spreads 16 rows of 4 (2) chunks over the banks
  constexpr int PER_T = 128 * CPR / Wide::NT, BATCH = 16;
  static_assert(128 * 256 * sizeof(S) <= Wide::kLdsBytes && PER_T % BATCH == 0, "epilogue split");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, fr = lane & 15, fk = lane >> 4;
  auto barrier = []() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  S* const st = reinterpret_cast<S*>(lds_raw);
  auto at = [&](int row, int chunk) { return st + row * 256 + (chunk ^ ((row & 15) << SH)) * EPC; };
#pragma unroll 1
  for (int p = 0; p < 2; ++p) {
    if (wm == p) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int c = wn * 128 + j * 16 + fk * 4;
          S* const d = at(i * 16 + fr, c / EPC) + c % EPC;
          if constexpr (sizeof(S) == 4) {
            *reinterpret_cast<f32x4_t*>(d) = acc[i][j];
          } else {
            *reinterpret_cast<u32x2*>(d) =
                u32x2{pack2<S>(acc[i][j][0], acc[i][j][1]), pack2<S>(acc[i][j][2], acc[i][j][3])};
          }
        }
    }
    barrier();
    const int rbase = m0 + p * 128;
#pragma unroll
    for (int b0 = 0; b0 < PER_T; b0 += BATCH) {
      typename Epi::Prior prior[BATCH];
      if constexpr (Epi::kReads) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
          const int c = (b0 + u) * Wide::NT + tid, r = c / CPR, col = n0 + (c % CPR) * EPC;
          if (rbase + r < g.M && col < g.N) prior[u] = epi.load(rbase + r, col, min(EPC, g.N - col));
        }
      }
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        const int c = (b0 + u) * Wide::NT + tid, r = c / CPR, cc = c % CPR, col = n0 + cc * EPC;
        if (rbase + r < g.M && col < g.N) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(at(r, cc));
          epi.store(rbase + r, col, reinterpret_cast<const S*>(&v), min(EPC, g.N - col), prior[u]);
        }
      }
    }
    if (p == 0) barrier();
  }
}

template <typename T, class Epi, bool AMN, bool BMN>
__global__ __launch_bounds__(Wide::NT, 1) void gemm_wide_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                                Shape g, Epi epi) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[Wide::kLdsBytes];
  apply_bound(g, Wide::BK);
  const int nbm = (g.M + Wide::BM - 1) / Wide::BM, nbn = (g.N + Wide::BN - 1) / Wide::BN;
  const int tiles = nbm * nbn;
  const int KTall = (g.K + Wide::BK - 1) / Wide::BK;  // >= 1 (checked by the launcher)
  const int nsplit = auto_splits(tiles, KTall, g.ksplit);
  if ((int)blockIdx.x >= tiles * nsplit) return;  // uniform: past a device-side bound
  const int split = (int)blockIdx.x / tiles;
  int tm, tn;
  tile_of_block<Wide::GROUP_M>((int)blockIdx.x - split * tiles, nbm, nbn, &tm, &tn);
  const int m0 = tm * Wide::BM, n0 = tn * Wide::BN;
  int KT = KTall, kt0 = 0;
  if (nsplit > 1) {  // this split's stages (auto_splits keeps every split non-empty)
    const int per = (KTall + nsplit - 1) / nsplit;
    kt0 = split * per;
    KT = min(per, KTall - kt0);
  }
  const int64_t k0 = (int64_t)kt0 * Wide::BK;
  const T* const pa = AMN ? A + k0 * g.lda + m0 : A + m0 * g.lda + k0;
  const T* const pb = BMN ? B + k0 * g.ldb + n0 : B + n0 * g.ldb + k0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int S = Wide::kOpBytes;
  wide_core<T, AMN, BMN>(acc, lds_raw, lds_raw + S, lds_raw + 2 * S, lds_raw + 3 * S, pa, pb, g.lda, g.ldb,
                         min(Wide::BM, g.M - m0), min(Wide::BN, g.N - n0), KT, g.ka - (int)k0, g.kb - (int)k0, wave,
                         (int)threadIdx.x & 63);
  Epi e = epi;
  apply_split(e, split, nsplit, g.M, 0);
  wide_epilogue(acc, lds_raw, m0, n0, g, e);
}

}  // namespace gemm
}  // namespace hk
