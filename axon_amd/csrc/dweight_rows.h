// dWeight[v][h] = sum_t dl[t][v] * hT[h][t] over few tokens (up to 768).
//
// The weight gradient of a short call is as much writing as multiplying: 151936 x 4096 in bf16 are 1.24 GB, 180 us at the
// 6.9 TB/s that a fill reaches, 64 tokens more are 53 us of matrix work.  In 256 x 256 tiles (gemm_store_kernel) a tile
// of so short a reduction spends more time on its first loads and on its epilogue than on its products, one after the other.
//
// Here a wavefront keeps the fragments of its rows of hT over ALL tokens in registers for the whole kernel, and the
// workgroup walks the vocabulary: tiles of dl go through a ring of LDS slots, requested kRing - 1 tiles ahead, each is
// multiplied with the resident rows and leaves as bf16.  dl is read once per eight wavefronts' rows, hT once; the stores
// of a tile have until the ring comes round to drain, and a wave never waits for a load that is younger than its
// last tile's stores.  Each accumulator takes the same products in the same order as in DmaLoop: the same bits.
//
// Measured (us between events, 256 x 256 tiles / this kernel, both on one card), vocabulary 151936 x hidden 4096: 64 tokens
// 362 / 232, 128 398 / 282, 192 455 / 321, 256 508 / 366, 300 556 / 419, 384 604 / 500, 448 658 / 528, 512 715 / 585, 640 804 / 710,
// 700 860 / 819, 768 917 / 877; 100 x 2880 x 201088 346 / 284, 333 532 / 495, 500 629 / 570; 300 x 896 x 151936 128 / 109, 600
// 185 / 180; 500 x 2048 x 32768 78 / 69, of which a loop over that call gives back most (dHidden, which follows, 72 / 80).
// What bounds it: the stores and the products of a tile still add up in part (all CUs are in the same phase); beyond 320 tokens a
// fragment from LDS serves two MFMAs, and beyond 640 the tiles are 32 columns wide, with a barrier every 88 or 96 MFMAs.
// Beyond 768 tokens the rows no longer fit in the registers.  Tried: the barrier in the middle of a tile, so that the
// next one's fragments are read ahead (64 tokens 252, 700 860), half of the wavefronts storing a tile later (264, 856),
// non-temporal stores (64-byte pieces of rows: 372), four wavefronts with twice the registers (700 tokens 974).
#pragma once
#include "gemm_nt.h"

namespace axon {

constexpr int kDwRowsMaxK = 768, kDwRowsMaxHidden = 8192;
constexpr int kDwRowsCus = 256, kDwRowsWaves = 8;

// 16-row blocks of hT per wavefront for a reduction of kt k-tiles of 64 tokens: four are whole 128-byte lines of the
// result and halve the LDS reads per MFMA (64 tokens 300 us with two), two where four would not fit in the registers.
constexpr int dw_rows_mb(int kt) { return kt <= 5 ? 4 : 2; }
// 16-column blocks of a tile: as many as the registers and two slots in LDS allow: eight up to 128 tokens, two for 257 to
// 320 and beyond 640, else four (448 tokens 636 us with two, 574 with four).
constexpr int dw_rows_nb(int kt) { return kt <= 2 ? 8 : kt == 5 || kt > 10 ? 2 : 4; }
// Workgroups that share the rows of hT; each takes one of kDwRowsCus / groups parts of the vocabulary's tiles (up to 8192
// hidden at least 90 % of the compute units then have work).
constexpr int64_t dw_rows_groups(int64_t h, int kt) {
  return (h + kDwRowsWaves * dw_rows_mb(kt) * kBlk - 1) / (kDwRowsWaves * dw_rows_mb(kt) * kBlk);
}

template <int KT>
struct DwRows {
  static constexpr int K = 64 * KT, KS = 2 * KT;
  static constexpr int MB = dw_rows_mb(KT), NB = dw_rows_nb(KT), kRows = MB * kBlk;
  static constexpr int kCols = NB * kBlk, kPitch = kCols * 2;  // a tile's columns; a k-row of it in LDS
  static constexpr int kTileBytes = K * kPitch;
  static constexpr int kRing = kGemmLdsBytes / kTileBytes < 4 ? kGemmLdsBytes / kTileBytes : 4;
  static constexpr int kDmas = kTileBytes / 1024;  // DMA instructions of a tile
  static constexpr int kDeep = KT == 5 || KT > 10 ? 4 : 8;  // fragments on their way from LDS
  // k-steps of hT in VGPRs; the others lie in the accumulators' half, 128 registers with the accumulators.  (Were that
  // exceeded the compiler would move them there in front of each MFMA, without the wait states that it cannot count.)
  static constexpr int kInVgprs = (kDeep == 8 ? 72 : 88) / (4 * MB);
  static_assert(kRing >= 2 && (KS > kInVgprs ? KS - kInVgprs : 0) * 4 * MB + 4 * MB * NB <= 128, "");
  // vmcnt before a tile is read: what is younger than its loads are the stores of kRing - 1 tiles and the loads of
  // kRing - 2; a wavefront without rows stores nothing
  static constexpr int kYoungLoads = (kRing - 2) * (kDmas / kDwRowsWaves);
  static constexpr int kYoung = kYoungLoads + (kRing - 1) * NB * (MB / 2);
  static_assert(kYoung <= 63, "");
};

constexpr int vmcnt(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int lgkmcnt(int n) { return 0xC07F | (n << 8); }

// `groups`: the workgroups that share the rows of hT, each with a `ranges`-th of the vocabulary's tiles.
template <int KT>
__global__ __launch_bounds__(kDwRowsWaves * 64, 2) void dw_rows_kernel(GemmOperands g, __bf16* __restrict__ out,
                                                                       int64_t ld_out, int groups, int ranges) {
  typedef DwRows<KT> P;
  typedef DmaLoopT<false, true> D;
  constexpr int MB = P::MB, NB = P::NB, KS = P::KS;
  extern __shared__ __align__(16) char smem[];
  const LanePos lp;
  const int wave = __builtin_amdgcn_readfirstlane(lp.wave);
  const int lda2 = (int)g.lda * 2, ldb2 = (int)g.ldb * 2, ldo2 = (int)ld_out * 2;
  // consecutive workgroup ids land on different XCDs: an XCD takes 32 consecutive places, the groups of a range side by
  // side, so that they find its dlogits in one L2
  const int place = (blockIdx.x % 8) * (kDwRowsCus / 8) + blockIdx.x / 8;
  const int range = place / groups, group = place - range * groups;
  if (range >= ranges) return;
  const int m_tiles = (g.m_rows + P::kRows - 1) / P::kRows, n_tiles = (g.n_rows + P::kCols - 1) / P::kCols;
  const int mt = group * m_tiles / groups + wave;
  const bool mine = mt < (group + 1) * m_tiles / groups;  // else: loads and barriers only
  int t = (int)((int64_t)range * n_tiles / ranges);
  const int t_end = (int)((int64_t)(range + 1) * n_tiles / ranges);

  // the resident rows: row l16 of block i, eight tokens from 8 * lq of k-step s on (rows beyond the matrix: zeros)
  bf16x8 af[KS][MB];
  {
    const __amdgpu_buffer_rsrc_t ra = DmaSide<false>::rsrc_of(reinterpret_cast<const char*>(g.a), g.m_rows * lda2);
    const int at = (mt * P::kRows + lp.l16) * lda2 + lp.lq * 16;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        af[s][i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(ra, at + s * 64, i * kBlk * lda2, 0));
  }

  // A slot holds the tile's k-rows one after the other, the 32-byte units (16 columns) of k-row r permuted by xor with
  // unit(r): the eight k-rows that half a wavefront reads with one instruction (r % 4 and r / 8 % 2 free) then lie in
  // eight different 32-byte groups of the banks.
  constexpr int kLanes = P::kPitch / 16, kRowsPer = 64 / kLanes;  // lanes to a k-row, k-rows to a DMA instruction
  auto unit = [](int r) {
    return NB == 8 ? (r & 3) + 4 * ((r >> 3) & 1) : NB == 4 ? ((r >> 1) & 1) + 2 * ((r >> 3) & 1) : (r >> 3) & 1;
  };
  // (an instruction's rows begin at a multiple of kRowsPer = 4, 8 or 16, eight instructions apart for a wave)
  const int lr = lp.lane / kLanes, r8 = kRowsPer == 4 ? (wave & 2) * 4 : kRowsPer == 8 ? (wave & 1) * 8 : 0;
  const int vb = lr * ldb2 + (((lp.lane % kLanes) ^ (2 * unit(lr + r8))) << 4);
  // tiles past the range: a descriptor of no bytes, the slot fills with zeros and is never read.  A tile's columns
  // beyond the last one are dl's padding: values of rows that are not stored.
  auto dma_tile = [&](int tile, int slot) {
    const int n0 = tile * P::kCols;
    const __amdgpu_buffer_rsrc_t rb = DmaSide<false>::rsrc_of(reinterpret_cast<const char*>(g.b) + (int64_t)n0 * 2,
                                                              tile < t_end ? g.k * ldb2 - n0 * 2 : 0);
#pragma unroll
    for (int q = 0; q < (P::kDmas + kDwRowsWaves - 1) / kDwRowsWaves; ++q) {
      const int d = q * kDwRowsWaves + wave;
      if (P::kDmas % kDwRowsWaves == 0 || d < P::kDmas)
        D::dma16<0>(rb, vb, d * kRowsPer * ldb2, smem + slot * P::kTileBytes + d * 1024);
    }
  };
#pragma unroll
  for (int q = 0; q < P::kRing - 1; ++q) dma_tile(t + q, q);

  // block 0's fragment of k-step 0: k-row 8 lq + 4 h + l16 / 4, columns 4 (l16 % 4) ..+3; block j's lies at that address
  // xor j << 5, k-step s 32 k-rows on
  typedef __attribute__((address_space(3))) const char* LdsPtr;
  const uint32_t b0 = (uint32_t)(uintptr_t)(LdsPtr)smem + (8 * lp.lq + (lp.l16 >> 2)) * P::kPitch + 8 * (lp.l16 & 1) +
                      (((lp.l16 & 3) >> 1) << 4) + (unit(8 * lp.lq + (lp.l16 >> 2)) << 5);
  acc4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = acc4{0.f, 0.f, 0.f, 0.f};
  // Where this lane's sixteen bytes go: row l16 of a block of columns, and of a pair of row blocks the eight values that
  // the lane holds after the swap below.  Where the matrix has no such row: an offset that stays beyond the descriptor's
  // end (2 MB at most) for every block of columns, so that the store is dropped.
  int vo[MB / 2];
#pragma unroll
  for (int h = 0; h < MB / 2; ++h) {
    const int m = mt * P::kRows + 32 * h + 16 * (lp.lq & 1) + 8 * (lp.lq >> 1);
    vo[h] = m < g.m_rows ? lp.l16 * ldo2 + m * 2 : INT32_MIN;
  }
  __builtin_amdgcn_s_waitcnt(vmcnt(0));

  int slot = 0;
#pragma unroll 1
  for (; t < t_end; ++t) {
    // this wave's share of tile t has landed, then everybody's; the slot of tile t - 1 is free
    if (mine) __builtin_amdgcn_s_waitcnt(vmcnt(P::kYoung));
    else __builtin_amdgcn_s_waitcnt(vmcnt(P::kYoungLoads));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    dma_tile(t + P::kRing - 1, slot == 0 ? P::kRing - 1 : slot - 1);
    __builtin_amdgcn_sched_barrier(0);
    if (mine) {
      const uint32_t b = b0 + slot * P::kTileBytes;
      constexpr int kAll = KS * NB;
      i16x4 bf[P::kDeep][2];
      auto read_b = [&](int q) {
        constexpr int kNear = 65536 / (32 * P::kPitch) - 1;  // k-steps that the instruction's offset field reaches
        const int st = q / NB, far = st / kNear;
        uint32_t a;  // an instruction: the compiler would hoist the addresses of all blocks into registers of their own
        asm volatile("v_xor_b32 %0, %1, %2" : "=v"(a) : "n"((q % NB) << 5), "v"(far ? b + far * kNear * 32 * P::kPitch : b));
        bf[q % P::kDeep][0] = D::read_tr(a, (st - far * kNear) * 32 * P::kPitch);
        bf[q % P::kDeep][1] = D::read_tr(a, (st - far * kNear) * 32 * P::kPitch + 4 * P::kPitch);
      };
#pragma unroll
      for (int q = 0; q < P::kDeep; ++q) read_b(q);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < kAll; ++q) {
        // fragment q has arrived, the younger reads may be under way
        switch (kAll - 1 - q < P::kDeep - 1 ? kAll - 1 - q : P::kDeep - 1) {
          case 0: __builtin_amdgcn_s_waitcnt(lgkmcnt(0)); break;
          case 1: __builtin_amdgcn_s_waitcnt(lgkmcnt(2)); break;
          case 2: __builtin_amdgcn_s_waitcnt(lgkmcnt(4)); break;
          case 3: __builtin_amdgcn_s_waitcnt(lgkmcnt(6)); break;
          case 4: __builtin_amdgcn_s_waitcnt(lgkmcnt(8)); break;
          case 5: __builtin_amdgcn_s_waitcnt(lgkmcnt(10)); break;
          case 6: __builtin_amdgcn_s_waitcnt(lgkmcnt(12)); break;
          default: __builtin_amdgcn_s_waitcnt(lgkmcnt(14)); break;
        }
        __builtin_amdgcn_sched_barrier(0);
        const int s = q / NB, j = q % NB;
        const bf16x8 x = D::join(bf[q % P::kDeep][0], bf[q % P::kDeep][1]);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          if (s == 0) mfma_16x16x32_from_zero(acc[i][j], af[s][i], x);
          else if (s < P::kInVgprs) mfma_16x16x32(acc[i][j], af[s][i], x);
          else mfma_16x16x32_agpr(acc[i][j], af[s][i], x);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (q + P::kDeep < kAll) read_b(q + P::kDeep);
        __builtin_amdgcn_sched_barrier(0);
      }
      settle_acc();
      // the tile leaves: the two 16-row blocks of a pair trade halves so that a lane holds sixteen contiguous bytes.  The
      // rows of the last tile that the result does not have end at the descriptor; a block's offset is added to the
      // lane's, which is what the hardware compares with the descriptor's size whatever it does with a scalar one.
      const int n0 = t * P::kCols;
      const __amdgpu_buffer_rsrc_t ro = DmaSide<false>::rsrc_of(reinterpret_cast<const char*>(out + (int64_t)n0 * ld_out),
                                                                min(g.n_rows - n0, P::kCols) * ldo2);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int h = 0; h < MB / 2; ++h) {
          acc4 &x = acc[2 * h][j], &y = acc[2 * h + 1][j];
          pin_acc(x);
          pin_acc(y);
          uint32_t x0 = pack_bf16(x[0], x[1]), x1 = pack_bf16(x[2], x[3]);
          uint32_t y0 = pack_bf16(y[0], y[1]), y1 = pack_bf16(y[2], y[3]);
          asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3"
                       : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1));
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
          const u32x4 v = {x0, x1, y0, y1};
          int at;  // an instruction: the compiler would keep the offsets of all blocks in registers of their own
          asm volatile("v_add_u32 %0, %1, %2" : "=v"(at) : "s"(j * kBlk * ldo2), "v"(vo[h]));
          __builtin_amdgcn_raw_buffer_store_b128(v, ro, at, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    slot = slot + 1 == P::kRing ? 0 : slot + 1;
  }
  __builtin_amdgcn_s_waitcnt(vmcnt(0));  // loads past the range must not land in the next workgroup's LDS
}

// Whether that is the faster way.  A workgroup loads its rows (up to 32 KB per wavefront) and fills the ring before its
// first tile, which a long enough walk makes up for.  Its time is that of eight wavefronts also where some have no rows,
// while a tile of 256 x 256 whose rows end in its first half is computed as half a tile: the more rows are computed here
// than there (`mine`, `theirs`), the longer that takes.  Beyond 640 tokens little is gained, and nothing where rows are computed
// for nothing or compute units go without a part of the vocabulary.  256 x 256 tiles / this kernel, us, on the same buffers
// (between buffers at other addresses either differs by up to 5 %), by columns walked:
//   192 tokens: hidden 896 192 columns 22.6 / 21.2, 256 23.9 / 23.6; 576 (1024 rows for 640) 192 17.0 / 18.6, 256 23.2 / 20.6; 2880 256
//     26.8 / 25.7.
//   256 tokens: hidden 896 256 columns 27.0 / 27.8, 384 36.8 / 34.3; 2880 256 29.3 / 29.5, 384 40.1 / 36.7; 576 384 28.6 / 29.2, 512 36.9 / 35.1.
//   320 tokens: hidden 896 384 columns 41.0 / 40.8, 512 53.6 / 50.7; 2880 512 56.0 / 49.9; 576 768 55.6 / 56.6, 1024 76.0 / 73.8.
//   384 and 576 tokens: hidden 896 1024 columns 57.1 / 54.7 and 71.8 / 70.3 (768: 54.9 / 56.8 for 576); 288 1024 65.6 / 66.2 for 576.
//   640 tokens: 1024 columns, hidden 2880 (3072 rows for 2944) 81.6 / 79.4, 1056 (1280 for 1152) 77.6 / 75.8, 288 (512 for 384)
//     69.2 / 73.8; 896 (1024 for 896) 1536 113.3 / 116.7, 1600 118.6 / 112.6, 2004 149.2 / 138.2, 2374 177.6 / 167.8.
//   704 tokens, 151936 vocabulary rows: hidden 896 188 / 194, 1248 254 / 246, 1504 (252 of 256 compute units) 300 / 296, 2560 (250) 514 / 521,
//     2880 579 / 599, 3072 (252) 623 / 624, 3584 (252, fourteen groups) 713 / 728, 4096 862 / 819, 5120 (240) 1045 / 1083.  By columns: hidden
//     512 1536 146.1 / 146.7, 2048 192.9 / 190.0, but 1571, where the tiles are 6.14 rounds, 154.5 / 139.1 and 1187 (4.64) 112 / 111;
//     992 1600 (6.25 rounds) 145 / 137, 2004 171 / 167; 2048 1536 136.2 / 139.1, 2048 187.1 / 185.9.
constexpr bool dw_rows_worth(int64_t h, int64_t vc, int64_t k) {
  const int kt = (int)(k / 64);
  const int64_t groups = dw_rows_groups(h, kt);
  const int64_t mine = groups * kDwRowsWaves * dw_rows_mb(kt) * kBlk, theirs = (h + 127) / 128 * 128;
  const bool sparse = 2 * mine > 3 * theirs, over = 8 * mine > 9 * theirs;
  // half tiles of the other way, 512 to a round: its last round leaves a twentieth of all of them unused
  const int64_t halves = (vc + 255) / 256 * (theirs / 128), rounds = (halves + 511) / 512;
  const bool ends_empty = 100 * 512 * rounds > 105 * halves;
  const int64_t walk = kt <= 3    ? 256
                       : kt == 4  ? (sparse ? 512 : 384)
                       : kt == 5  ? (sparse ? 1024 : 512)
                       : kt <= 9  ? 1024
                       : kt == 10 ? (over ? 1600 : 1024)
                                  : (ends_empty ? 1024 : 2000);
  const bool full = mine == theirs && kDwRowsCus % groups <= (groups <= 12 ? 4 : 1);
  return vc >= walk * (kDwRowsCus / groups) && (kt <= 10 || full);
}

template <int KT>
int launch_dw_rows_of(const GemmOperands& g, __bf16* out, int64_t ld_out, hipStream_t st) {
  typedef DwRows<KT> P;
  constexpr int kLds = P::kRing * P::kTileBytes;
  const int groups = (int)dw_rows_groups(g.m_rows, KT);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(dw_rows_kernel<KT>), hipFuncAttributeMaxDynamicSharedMemorySize,
                          kLds) != hipSuccess)
    return AXON_ERR_LAUNCH;
  hipLaunchKernelGGL(dw_rows_kernel<KT>, dim3(kDwRowsCus), dim3(kDwRowsWaves * 64), kLds, st, g, out, ld_out, groups,
                     kDwRowsCus / groups);
  AXON_CHECK_LAUNCH();
  return AXON_OK;
}
// g.a: hT [m_rows][lda], zero beyond the last token up to k; g.b: dl [k][ldb]; k a multiple of 64, at most kDwRowsMaxK.
inline int launch_dw_rows(const GemmOperands& g, __bf16* out, int64_t ld_out, hipStream_t st) {
  switch (g.k / 64) {
    case 1: return launch_dw_rows_of<1>(g, out, ld_out, st);
    case 2: return launch_dw_rows_of<2>(g, out, ld_out, st);
    case 3: return launch_dw_rows_of<3>(g, out, ld_out, st);
    case 4: return launch_dw_rows_of<4>(g, out, ld_out, st);
    case 5: return launch_dw_rows_of<5>(g, out, ld_out, st);
    case 6: return launch_dw_rows_of<6>(g, out, ld_out, st);
    case 7: return launch_dw_rows_of<7>(g, out, ld_out, st);
    case 8: return launch_dw_rows_of<8>(g, out, ld_out, st);
    case 9: return launch_dw_rows_of<9>(g, out, ld_out, st);
    case 10: return launch_dw_rows_of<10>(g, out, ld_out, st);
    case 11: return launch_dw_rows_of<11>(g, out, ld_out, st);
    case 12: return launch_dw_rows_of<12>(g, out, ld_out, st);
    default: return AXON_ERR_SHAPE;
  }
}

}  // namespace axon
