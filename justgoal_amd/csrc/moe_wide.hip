// Wide-tile grouped GEMM2: 256 H columns per tile, eight waves that all fetch and all compute.
//
// What bounds it. The bf16 MFMAs of a step (128 x 256 x 128: 2048 cycles per SIMD) share the vector
// issue port with the e4m3 -> bf16 conversion of W2 and the s2 scale FMAs (MFMA pipes busy 0.45 of the
// cycles at DS-V3 T=14107 with 7130 pairs, 0.57 at T=16384 skewed), and on long segments the chip is
// power-limited: the skewed batch (69290 pairs) runs at 1.76 GHz and takes 1942 us, on all-zero data
// 1415. So the tile is chosen for the fewest instructions and LDS bytes per MFMA. A wave owns 64 rows x
// 64 columns (BM = 128: 2 x 4 waves), so it converts each W2 fragment once per 64 rows (one
// conversion per 64 FLOP-equal 32x32x16 MFMA pair, half of a 32-row wave tile), reads 24 KB of
// fragments per step against 32 KB for the same work in 32 x 64 wave tiles, and C is fetched once per
// 256 columns. With eight waves per CU there are 256 VGPRs per wave. The accumulators (64), both
// halves of the C fragments (64), the MFMA results awaiting their scale (32) and two sections of
// weights (raw 16, converted 32) take 208 of the 241 used; nothing is spilled.
// Against the 128 x 128 tiles with a producer wave that it replaced, GEMM2 stage, same process (pairs
// / active experts of each batch; DS-V3 expects T pairs, and a batch's routing bias decides): DS-V3
// T=2048 (1028 / 24) 96.6 -> 87.5 us, T=4096 (2084 / 28) 133 -> 113, T=6000 (3021 / 29) 172 -> 145,
// T=14107 (7130 / 29) 292 -> 262, T=16384 skewed (69290 / 22) 2412 -> 1890; Qwen3-style T=1024 210 ->
// 190, T=2048 345 -> 280. With the expected pairs: T=4096 (4072 / 28) 187 us, T=14107 (13958 / 28) 450.
//
// Pipeline. A K step (one 128-wide scale block) is cut into sections of 64 K values x 32 columns
// per wave (four for BM = 128, two for BM = 64, whose waves own 32 columns). A section issues its
// MFMAs on fragments that the section before read; meanwhile it converts the next section's W2
// fragments, reads those of the one after, applies the scale to the results of the half before, and
// refills by LDS DMA the part of the ring slot that the sections before have finished with. So
// there is no producer wave and no burst: two vector-memory instructions per section and wave.
// Barriers stand only where a section reads newly landed data or refills a part that other
// waves read: two per step. W2 rows are fetched 6 sections ahead with two slots (BM = 128), two
// steps ahead with three (BM = 64).
//
// LDS images: W2 rows of 128 bytes, C rows as two planes of 128 bytes (64 K values each), both with
// the 16-byte chunk permutation wblk_swz; a 32x32x16 fragment read (lane = row l & 31, 16 bytes) is
// conflict-free under it. Lane half hf = l >> 5 takes K values [16 (2u + hf) + 8v, +8) for MFMA
// 2u + v of the step, on both operands.
#include "moe_device.h"
#include "moe_kernels.h"

namespace jgmoe {

namespace {

constexpr int kWideWaves = 8;

template <int I>
struct Int {
  static constexpr int v = I;
};

template <int OFF>
__device__ __forceinline__ v4u ds_read16_at(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "16-bit offset field");
  v4u v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
// Lane l < 32: b becomes lane l + 32's a; lane l + 32: a becomes lane l's b.
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16f mfma_bf16_32x32x16(const v8bf& a, const v8bf& b, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <int BM, int D, bool NT>
__global__ __launch_bounds__(kWideWaves* kWave) void gemm2_wide_kernel(
    const uint16_t* __restrict__ C, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    const float* __restrict__ sorted_w, Gemm2Out dst, int H, int I, int E_l, int max_pairs,
    int sched) {
  static_assert((BM == 128 && D == 2) || (BM == 64 && D >= 3), "DMA schedules below");
  constexpr int WM = BM / 64, WN = kWideWaves / WM;
  constexpr int BN = 256, NN = BN / WN / 32;     // 32-column sub-tiles per wave
  constexpr int NSEC = 2 * NN;                   // sections per step
  constexpr int kPlane = BM * kBlock;            // one 64-wide K half of the C tile
  constexpr int ASZ = 2 * kPlane, BSZ = BN * kBlock;
  constexpr int AI = kPlane / 1024 / kWideWaves; // C DMA instructions per wave and half
  __shared__ __attribute__((aligned(16))) uint8_t aring[D][ASZ];  // [half][row][128 B]
  __shared__ __attribute__((aligned(16))) uint8_t bring[D][BSZ];  // [n][wave column][32 rows]
  __shared__ __attribute__((aligned(16))) float wsc[2][2][kBlock];     // [item parity][block]
  __shared__ __attribute__((aligned(16))) float rowmeta[2][2][BM];     // [parity][weight, dst]
  __shared__ TileMapLds tml;

  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int NNT = (H + BN - 1) / BN, NKB = I / kBlock;
  const int items = uniform(tml.build(counts, offsets, E_l, BM, w == 0)) * NNT;
  int it = uniform((int)blockIdx.x);
  if (it >= items) return;  // whole workgroup
  __syncthreads();
  const int stride = gridDim.x;

  struct Item {
    int e, m0, cnt, seg, h0;
  };
  auto scalars = [&](int item, Item& x) {
    int nt;
    x.e = uniform(map_item<BM>(tml, item, items, NNT, E_l, sched, x.m0, x.cnt, x.seg, nt));
    x.m0 = uniform(x.m0);
    x.cnt = uniform(x.cnt);
    x.seg = uniform(x.seg);
    x.h0 = uniform(nt * BN);
  };

  const int wm = w / WN, wn = w % WN;
  const int r32 = lane & 31, hf = lane >> 5;
  const uint32_t dma0 = wblk_dma_off(lane, 0, I), dma1 = wblk_dma_off(lane, 1, I);
  // C DMA instruction i of a half: tile rows 8 (AI w + i) + lane / 8, relative to the tile's row 0
  uint32_t aoff[AI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int row = 8 * (AI * w + i) + (lane >> 3);
    aoff[i] = (uint32_t)row * I * 2 + 16 * ((lane & 7) ^ wblk_swz(row));
  }
  const __amdgpu_buffer_rsrc_t wgtres = make_rsrc(sorted_w, (uint32_t)max_pairs * 4);
  const __amdgpu_buffer_rsrc_t dstres = make_rsrc(dst.pair_dst, (uint32_t)max_pairs * 4);
  const __amdgpu_buffer_rsrc_t s2res = make_rsrc(s2, (uint32_t)E_l * (H / kBlock) * NKB * 4);

  auto meta_scales = [&](const Item& x, int par) {
    if (w < 4) {
      const int half = w & 1, blk = w >> 1;
      // (all in the per-lane offset, which the range check covers)
      const int row = x.e * (H / kBlock) + x.h0 / kBlock + blk;
      dma4(s2res, &wsc[par][blk][half * kWave], 4u * (row * NKB + half * kWave + lane), 0);
    }
  };
  auto meta_rows = [&](const Item& x, int par) {
    if (w >= 4 && w < 4 + 2 * WM) {
      const int half = (w & 3) >> 1, what = w & 1;
      const int r = x.m0 + half * kWave + lane, last = x.cnt - 1;
      const uint32_t off = 4u * (x.seg + (r < last ? r : last));
      dma4(what ? dstres : wgtres, &rowmeta[par][what][half * kWave], off, 0);
    }
  };
  // Issue-side state: the item whose blocks the DMAs fetch.
  const uint16_t* ic = nullptr;
  const uint8_t* iw = nullptr;
  uint32_t ibytes = 0, wbytes = 0, irow = 0;
  auto enter = [&](const Item& x, bool live) {
    ic = uniform(C + (size_t)(x.seg + x.m0) * I);
    ibytes = live ? uniform((uint32_t)(x.cnt - x.m0) * I * 2) : 0u;
    iw = uniform(w2 + (size_t)x.e * H * I);
    wbytes = live ? (uint32_t)H * I : 0u;
    int row = x.h0 + (NN == 2 ? (w >> 1) * 64 + (w & 1) * 16 : w * 32);
    if (row >= H) row -= kBlock;  // the missing half of the last tile: any rows, never stored
    irow = uniform((uint32_t)row);
  };
  auto dma_w = [&](__amdgpu_buffer_rsrc_t r, void* b, uint32_t vo, uint32_t so) {
    if constexpr (NT)
      dma16_stream(r, b, vo, so);
    else
      dma16(r, b, vo, so);
  };
  // Weight rows of sub-tile n (NN = 2: 16 of its 128 rows; NN = 1: this wave's own 32 columns).
  auto issue_w = [&](int n, int kbi, int slot) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(uniform(iw), wbytes);
    const uint32_t so = uniform((irow + 32 * n) * (uint32_t)I + (uint32_t)kbi * kBlock);
    uint8_t* b = &bring[slot][n * (BSZ / 2) + w * (NN == 2 ? 2048 : 4096)];
    dma_w(r, b, dma0, so);
    dma_w(r, b + 1024, dma1, so);
    if constexpr (NN == 1) {
      dma_w(r, b + 2048, dma0, so + 16u * I);
      dma_w(r, b + 3072, dma1, so + 16u * I);
    }
  };
  auto issue_c = [&](int h, int kbi, int slot) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(uniform(ic), ibytes);
    uint8_t* b = &aring[slot][h * kPlane + w * (AI * 1024)];
    const uint32_t so = uniform((uint32_t)kbi * 2 * kBlock + h * kBlock);
#pragma unroll
    for (int i = 0; i < AI; ++i) dma16(r, b + i * 1024, aoff[i], so);
  };
  // The DMAs of section s, in this order everywhere: they refill slot `slot`, last read by the
  // sections before, with block kbi.
  auto issue = [&](auto S, int kbi, int slot) {
    constexpr int s = decltype(S)::v;
    if constexpr (NN == 2) {
      if constexpr (s % 2 == 0)
        issue_w(s / 2, kbi, slot);
      else
        issue_c(s / 2, kbi, slot);
    } else {
      if constexpr (s == 0) issue_w(0, kbi, slot);
      issue_c(s, kbi, slot);
    }
  };
  constexpr int kOps = 4 + 2 * AI;  // vector-memory operations per wave and step
  // Operations issued after the last one that section s's reads need (-1: nothing new, no barrier).
  constexpr int kLanded[4] = {NN == 2 ? 8 : 2 + 6 * (D - 2), NN == 2 ? -1 : 6 + 6 * (D - 2),
                              NN == 2 ? 8 : -1, -1};

  v4u raw[2][2];   // fp8 fragments of two sections
  v8bf bw[2][4];   // bf16 fragments of two sections
  v4u a[2][2][4];  // C fragments [row sub-tile][half][chunk]
  float swn;
  uint32_t ard[4], brd[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ard[j] = lds_addr(&aring[0][0]) + wm * 64 * kBlock + r32 * kBlock +
             16 * ((4 * (j >> 1) + 2 * hf + (j & 1)) ^ wblk_swz(r32));
    brd[j] = lds_addr(&bring[0][0]) + wn * 32 * kBlock + r32 * kBlock +
             16 * ((2 * j + hf) ^ wblk_swz(r32));
  }
  // The read addresses move to the next slot when the first read of the next block goes out.
  auto flip_a = [&](int d) {
    const uint32_t x = d + 1 == D ? (uint32_t)-((D - 1) * ASZ) : (uint32_t)ASZ;
#pragma unroll
    for (int j = 0; j < 4; ++j) ard[j] += x;
  };
  auto flip_b = [&](int d) {
    const uint32_t x = d + 1 == D ? (uint32_t)-((D - 1) * BSZ) : (uint32_t)BSZ;
#pragma unroll
    for (int j = 0; j < 4; ++j) brd[j] += x;
  };
  auto read_raw = [&](auto S) {
    constexpr int s = decltype(S)::v;
    raw[s & 1][0] = ds_read16_at<(s >> 1) * (BSZ / 2)>(brd[2 * (s & 1)]);
    raw[s & 1][1] = ds_read16_at<(s >> 1) * (BSZ / 2)>(brd[2 * (s & 1) + 1]);
  };
  auto read_a = [&](auto HI) {
    constexpr int h = decltype(HI)::v;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[0][h][j] = ds_read16_at<h * kPlane>(ard[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) a[1][h][j] = ds_read16_at<h * kPlane + 32 * kBlock>(ard[j]);
  };
  auto read_sw = [&](int kbn, int par) {
    swn = ds_read4f(lds_addr(&wsc[par][wn * 32 * NN / kBlock][0]) + 4 * kbn);
  };
  auto fence_raw = [&](int i) {
    lds_fence(raw[i][0]);
    lds_fence(raw[i][1]);
  };
  auto fence_a = [&](int h) {
#pragma unroll
    for (int ms = 0; ms < 2; ++ms)
#pragma unroll
      for (int j = 0; j < 4; ++j) lds_fence(a[ms][h][j]);
  };
  auto convert = [&](int i) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        v2bf p0, p1, p2, p3;
        fp8x4_to_bf16x4((int)raw[i][u][2 * v], p0, p1);
        fp8x4_to_bf16x4((int)raw[i][u][2 * v + 1], p2, p3);
        bw[i][2 * u + v] = v8bf{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
      }
  };
  // Completes the reads in flight at the end of a step: the second section's weights, the first
  // halves of the C fragments and the scale. It stands before every branch and loop edge: the
  // compiler takes the asm reads as complete and may copy their registers there (it did copy swn
  // at the K loop's edge, ahead of the wait). The next step's first section waits for nothing
  // else, so the wait costs nothing here.
  auto drain = [&] {
    lds_wait_all();
    fence_raw(1);
    fence_a(0);
    lds_fence(swn);
  };

  Item cur, nxt;
  scalars(it, cur);
  meta_scales(cur, 0);
  enter(cur, true);
#pragma unroll
  for (int k = 0; k < D; ++k) {
    issue(Int<0>{}, k, k);
    issue(Int<1>{}, k, k);
    if constexpr (NSEC == 4) {
      issue(Int<2>{}, k, k);
      issue(Int<3>{}, k, k);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  vm_wait<kOps*(D - 1)>();
  __builtin_amdgcn_s_barrier();
  read_raw(Int<0>{});
  read_raw(Int<1>{});
  read_a(Int<0>{});
  read_sw(0, 0);
  drain();
  fence_raw(0);
  convert(0);

  int slot = 0, par = 0;
  for (;;) {
    const int it_n = it + stride;
    const bool more = it_n < items;
    scalars(more ? it_n : it, nxt);
    meta_rows(cur, par);
    meta_scales(nxt, par ^ 1);

    v16f acc[NN][2];  // [32-column sub-tile][32-row sub-tile]
    v16f t[2];
    float sw = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t[1][i] = 0.f;
#pragma unroll
    for (int n = 0; n < NN; ++n) acc[n][0] = acc[n][1] = t[1];

    auto scale = [&](int ms, int n) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[n][ms][i] = fmaf(t[ms][i], sw, acc[n][ms][i]);
    };
    auto mma = [&](int ms, int h) {
      const v16f z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f,
                      0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c)
        t[ms] = mfma_bf16_32x32x16(bw[h][c], __builtin_bit_cast(v8bf, a[ms][h][c]),
                                   h == 0 && c == 0 ? z : t[ms]);
    };

    // One section: a wave's 64 rows x 32 columns (sub-tile s / 2) x 64 of K (half s % 2).
    auto section = [&](auto BUSY, auto S, int kbi, int kbn, int d, int parn) {
      constexpr bool B = decltype(BUSY)::v;
      constexpr int s = decltype(S)::v;
      if constexpr (B && s > 0) {  // (the first section's fragments: drain)
        lds_wait_all();
        fence_raw((s + 1) & 1);
        if constexpr (s == 1) fence_a(1);
      }
      if constexpr (kLanded[s] >= 0) {
        vm_wait<(kLanded[s] < 0 ? 0 : kLanded[s])>();
        __builtin_amdgcn_s_barrier();
      }
      if constexpr (s == NSEC - 2) flip_b(d);
      if constexpr (s == NSEC - 1) flip_a(d);
      if constexpr (B) {
        read_raw(Int<(s + 2) % NSEC>{});
        if constexpr (s == NSEC - 1) {
          read_a(Int<0>{});
          read_sw(kbn, parn);
        }
        if constexpr (s == 0) read_a(Int<1>{});
        __builtin_amdgcn_sched_barrier(0);
        mma(0, s & 1);
        __builtin_amdgcn_sched_barrier(0);
        issue(S, kbi, d);
        if constexpr (s % 2 == 0) {
          scale(1, s == 0 ? NN - 1 : 0);
          if constexpr (s == 0) sw = swn;
        } else {
          convert((s + 1) & 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        mma(1, s & 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (s % 2 == 0) {
          convert((s + 1) & 1);
        } else {
          scale(0, s >> 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      } else {
        issue(S, kbi, d);
      }
    };
    auto k_loop = [&](auto BUSY) {
      int kb = 0;
#pragma unroll 1
      for (int part = 0; part < 2; ++part) {
        const int end = part ? NKB : NKB - D;
        if (part) enter(nxt, more);  // the last D blocks' refills come from the next item
        int kbi = part ? 0 : D;
#pragma unroll 1
        for (; kb < end; ++kb, ++kbi) {
          const bool last = kb + 1 == NKB;
          const int kbn = last ? 0 : kb + 1, parn = last ? par ^ 1 : par;
          section(BUSY, Int<0>{}, kbi, kbn, slot, parn);
          section(BUSY, Int<1>{}, kbi, kbn, slot, parn);
          if constexpr (NSEC == 4) {
            section(BUSY, Int<2>{}, kbi, kbn, slot, parn);
            section(BUSY, Int<3>{}, kbi, kbn, slot, parn);
          }
          if constexpr (decltype(BUSY)::v) drain();
          slot = slot + 1 == D ? 0 : slot + 1;
        }
      }
    };
    // A wave whose 64 rows of the tile are all padding keeps the barriers and its share of the
    // DMAs, and then reads the next item's head, whose block is refilled only past the next barrier.
    if (WM > 1 && cur.m0 + wm * 64 >= cur.cnt) {
      k_loop(Int<0>{});
      read_raw(Int<0>{});
      read_raw(Int<1>{});
      read_a(Int<0>{});
      read_sw(0, par ^ 1);
      drain();
      fence_raw(0);
      convert(0);
    } else {
      k_loop(Int<1>{});
      scale(1, NN - 1);
      const int col = cur.h0 + wn * 32 * NN;
#pragma unroll
      for (int ms = 0; ms < 2; ++ms) {
        const int row = wm * 64 + ms * 32 + r32;
        if (cur.m0 + row < cur.cnt && col < H) {
          float wp = ds_read4f(lds_addr(&rowmeta[par][0][0]) + 4 * row);
          float dd = ds_read4f(lds_addr(&rowmeta[par][1][0]) + 4 * row);
          lds_wait_all();
          lds_fence(wp);
          lds_fence(dd);
          const int d = __float_as_int(dd);
          // A lane holds H columns 8 j + 4 hf + (0..3) of each 32-column sub-tile; exchanging
          // halves between lanes l and l + 32 leaves columns 16 q + 8 hf + (0..7), 16 bytes.
          uint16_t* orow =
              (d >= 0 ? dst.out + (size_t)d * H : dst.partial + (size_t)(-1 - d) * H) + col + 8 * hf;
#pragma unroll
          for (int n = 0; n < NN; ++n)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const v16f& x = acc[n][ms];
              uint32_t h[4];
#pragma unroll
              for (int i = 0; i < 4; ++i)
                h[i] = (uint32_t)float_to_bf16_bits(x[8 * q + 2 * i] * wp) |
                       ((uint32_t)float_to_bf16_bits(x[8 * q + 2 * i + 1] * wp) << 16);
              swap_halves(h[0], h[2]);
              swap_halves(h[1], h[3]);
              *(uint4*)(orow + 32 * n + 16 * q) = uint4{h[0], h[1], h[2], h[3]};
            }
        }
      }
    }
    if (!more) break;
    it = it_n;
    cur = nxt;
    par ^= 1;
  }
  vm_wait<0>();  // no DMA may still target this workgroup's LDS when it retires
}

}  // namespace

// Item order. With a multiple of 8 N-tiles the tile-major round-robin order keeps a W2 panel on one
// XCD for all of an expert's M-tiles. DS-V3 has 28: there XCD-contiguous bands of 4 M-tiles,
// N-tile-major inside a band, share W2 panels and C rows in an XCD's L2 instead (GEMM2 T=2048 87.5
// -> 81.9 us, T=4096 119.6 -> 113.0; T=14107 255.6 -> 259.6, T=16384 skewed 1925 -> 1937: the batches
// above; with the expected pairs T=2048 127.1 -> 126.7, T=3072 159.5 -> 152.9, T=4096 193.7 -> 186.9, T=6000
// 244.5 -> 236.2, T=14107 445.2 -> 450.3; the skewed call 4192 -> 4164, whose GEMM1 gains. For the
// Qwen3-style 16 N-tiles round-robin is ahead at T=2048, 312 against 320, level at T=1024, and behind
// at T=1536, 228 against 219).
constexpr int kXcds = 8;
constexpr int kSchedBands = 1 | (4 << 1);
// Below 144 expected rows most experts have one M-tile, so each W2 byte is read once: the
// non-temporal hint then keeps GEMM2's rows in the memory-side cache for the combine. Whole call
// without -> with it: DS-V3 T=3072 (1545 pairs) 285.2 -> 280.1 us, T=4096 (2084) 344.8 -> 341.3, Qwen3-style
// T=1536 553.4 -> 546.2; T=2048 level. Where half of the experts have a second M-tile it costs:
// DS-V3 T=4096 (4072 pairs) 460.5 -> 464.2, Qwen3-style T=2048 (128 rows, all even) 703.7 -> 722.6; and at
// T=14107 (13958) 1016 -> 1023, T=16384 skewed 4164 -> 4326.
constexpr int kSharedRows = 144;
// 64-row tiles with three slots (two steps, 64 KB of W2, in flight per CU) up to 43 expected rows,
// if the experts' tiles fill the chip at least five times over: with fewer rounds the
// 64 x 128 tiles of moe_big.hip lose less in the last one. Whole call, Qwen3-style (2048 tiles, eight
// rounds): T=256 441.8 -> 433.0 us, T=512 476.2 -> 462.2, T=640 487.8 -> 472.8; T=768 (48 rows) 522.3 ->
// 508.8, but 502.9 with the 128-row tiles. DS-V3 (896 tiles, 3.5 rounds; batches of about half the
// expected pairs): T=256 164.7 against 172.4, T=512 186.5 against 193.4, T=1024 203.6 against 205.4,
// T=1792 236.6 against 239.0.
constexpr int kShortRows = 44;
constexpr int kBigTileRows = 64;
constexpr int kMinRounds = 5;

static int wide_grid(long long max_items) {
  const int cus = device_cu_count();
  const long long g = cus < max_items ? cus : max_items;
  return g < 1 ? 1 : (int)g;
}

static inline long long wide_tiles(int max_pairs, int bm, int E_l) {
  return (max_pairs + bm - 1) / bm + (E_l < max_pairs ? E_l : max_pairs);
}

template <int BM, int D, bool NT>
static hipError_t launch_gemm2_wide_t(const uint16_t* C, const uint8_t* w2, const float* s2,
                                      const int32_t* counts, const int32_t* offsets,
                                      const float* sorted_w, Gemm2Out dst, int H, int I, int E_l,
                                      int max_pairs, hipStream_t stream) {
  constexpr int BN = 256;
  if (I / kBlock < D) return hipErrorNotSupported;
  const int nnt = (H + BN - 1) / BN;
  const int grid = wide_grid(wide_tiles(max_pairs, BM, E_l) * nnt);
  gemm2_wide_kernel<BM, D, NT><<<grid, kWideWaves * kWave, 0, stream>>>(
      C, w2, s2, counts, offsets, sorted_w, dst, H, I, E_l, max_pairs,
      nnt % kXcds == 0 ? 0 : kSchedBands);
  return hipGetLastError();
}

hipError_t launch_gemm2_wide(const uint16_t* C, const uint8_t* w2, const float* s2,
                             const int32_t* counts, const int32_t* offsets, const float* sorted_w,
                             Gemm2Out dst, int H, int I, int E_l, int max_pairs, int rows_hint,
                             hipStream_t stream) {
  const int nnt = (H + 255) / 256;
  if (rows_hint < kBigTileRows && E_l * nnt < kMinRounds * device_cu_count() && I / kBlock >= 3)
    return hipErrorNotSupported;  // left to the 64 x 128 tiles
  if (rows_hint < kShortRows) {
    const hipError_t e = launch_gemm2_wide_t<64, 3, true>(C, w2, s2, counts, offsets, sorted_w,
                                                          dst, H, I, E_l, max_pairs, stream);
    if (e != hipErrorNotSupported) return e;  // I = 256: three slots need three K blocks
  }
  if (rows_hint < kSharedRows)
    return launch_gemm2_wide_t<128, 2, true>(C, w2, s2, counts, offsets, sorted_w, dst, H, I, E_l,
                                             max_pairs, stream);
  return launch_gemm2_wide_t<128, 2, false>(C, w2, s2, counts, offsets, sorted_w, dst, H, I, E_l,
                                            max_pairs, stream);
}

}  // namespace jgmoe
