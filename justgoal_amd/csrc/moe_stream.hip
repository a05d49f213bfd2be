// Weight-streaming grouped GEMMs for small per-expert segments (decode-sized batches).
//
// When an expert holds a handful of pairs, every weight byte feeds at most one 16-row MFMA
// tile, so both GEMMs are HBM streams and the kernels are built around keeping the weight
// stream saturated:
//
// * Work items are per wave: (M-tile of 16*MT pairs, 16 output columns, full K). Each wave loops
//   over its items (persistent grid, items dealt wave-index major); there is no workgroup
//   synchronisation. GEMM1's items may instead belong to a workgroup, each of its four waves taking
//   a quarter of K, with a reduction through LDS at the end of an item.
// * Weight K-blocks (16 rows x 128 bytes per matrix) go global -> LDS by DMA into a per-wave ring
//   of D slots, two instructions per block, each fetching 8 rows as whole 128-byte lines
//   (register-staged MFMA operands would touch every line twice). The activation rows of the
//   block and its activation scales ride in a matching register ring.
// * The issue side runs D blocks ahead of the compute side and crosses item boundaries: the
//   last D blocks of an item are followed directly by the first D blocks of the wave's next
//   item, so the stream never drains between items. Item metadata (token rows, weight-scale
//   rows) is resolved one item ahead so no load is waited on at an item switch.
// * All waits are counted: each K step issues the same number of vector-memory operations, so
//   "slot d is complete" is vmcnt <= (D-1) * ops_per_step. Blocks past the end of the wave's
//   last item are still issued (to keep that count) but with an out-of-range offset, so they
//   return zeros without fetching anything.
//
// MFMA form: weights are the first operand, so lane l holds output column 4*(l>>4)+i for row
// (pair) l & 15. GEMM1 applies the activation scale (one per lane) times the weight scale of the
// K block after every fp8 MFMA and ends with SwiGLU into bf16 C; GEMM2 converts the fp8 weight
// block to bf16 in registers, runs four bf16 MFMAs per K block over the bf16 C rows, scales by
// the block's weight scale, and stores bf16 rows times the pair's routing weight at the pair's
// destination (the output row for a token's first local pair, else one of its partial rows).
// gemm2_token_kernel (below) is GEMM2 of a few tokens with the combine folded in.
#include "moe_device.h"
#include "moe_kernels.h"

namespace jgmoe {

namespace {

constexpr int kWavesPerGroup = 4;
constexpr int kWBlk = 16 * kBlock;  // one weight K-block image: 16 rows x 128 bytes

// First item of wave w of this workgroup; each wave then takes every (grid * 4)-th item. Wave
// index major: the grid is sized for the most items a batch could have, so when it has fewer
// (one per wave or less: a batch of a few tokens) they still spread over every CU instead of
// filling the first workgroups' four waves and leaving the last CUs idle (DS-V3 T=16: 768 items
// on 256 workgroups of 4 waves used 192 CUs). GEMM1 stage: T=8 30.6 -> 24.0 us, T=16 33.8 ->
// 32.6, T=32 58.7 -> 49.8 (whole call T=8 52.6 -> 46.7, T=32 92.5 -> 83.9).
__device__ __forceinline__ int first_item(int w) { return w * (int)gridDim.x + (int)blockIdx.x; }

// vmcnt holds 6 bits; deeper counts are clamped, which only makes a wait stricter.
constexpr int vm_depth(int n) { return n > 63 ? 63 : n; }

// A per-lane buffer offset past every buffer these kernels address (the API keeps each below
// 2^31 - 16): loads with it return zeros without a memory access.
constexpr uint32_t kNoFetch = 0x7ffffff0u;

// ---- GEMM1: C = SwiGLU(A W1^T, A W3^T) --------------------------------------------------------

template <int MT>
struct G1Slot {
  v8i a[MT];     // activation bytes [32g, 32g+32) of the block for row r16 of each sub-tile
  float sa[MT];  // activation scale of that row and block
};

template <int MT>
struct G1Item {
  const uint8_t* wbase;  // the expert's W13 [2I, H]
  uint32_t wsoff;        // c0 * H: first of the 16 X1 rows
  LaneScales sc1, sc2;   // weight scales of the X1 / X2 row block, per K block
  uint32_t aoff[MT];     // per lane: token * H + 32 g
  uint32_t saoff[MT];    // per lane: token * 4
  int m0, cnt, seg, c0;
};

// LDS of a gemm1_stream_kernel workgroup, which sets how many a CU holds: the rings and, with K
// split, the double-buffered partial sums. (Counted without the latter, five blocks per wave took two
// workgroups per CU where one fits, and half of the grid started over with empty rings when the
// other half ended. GEMM1 stage, 128 experts all local, I 1536: H 2560 8 tokens 67.2 -> 64.2 us, 64
// tokens 159.6 -> 154.6; H 5120 64 tokens 304.1 -> 298.0; H 7680 32 tokens 383.3 -> 379.6. Whole-K
// items take 69.4, 164.5, 305.1 and 406.6.)
template <int MT, int D, int KS>
constexpr int g1_stream_lds() {
  return kWavesPerGroup * D * 2 * kWBlk + (KS > 1 ? 2 * KS * 2 * MT * kWave * (int)sizeof(v4f) : 0);
}

template <int MT, int D, int KS>
__global__ __launch_bounds__(256) void gemm1_stream_kernel(
    const uint8_t* __restrict__ hs, const float* __restrict__ hs_scale,
    const uint8_t* __restrict__ w13, const float* __restrict__ s13,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ sorted_tok, uint16_t* __restrict__ C, int T, int H, int I,
    int E_l) {
  constexpr int BM = 16 * MT;
  constexpr int OPS = 3 * MT + 4;  // vector-memory operations per K step
  static_assert(KS == 1 || KS == kWavesPerGroup, "K is split over the workgroup's waves or not");
  __shared__ __attribute__((aligned(16))) uint8_t ring[kWavesPerGroup][D][2 * kWBlk];
  // KS > 1: partial sums of an item, double buffered by item parity
  __shared__ __attribute__((aligned(16))) v4f red[KS > 1 ? 2 : 1][KS > 1 ? KS : 1][2 * MT][kWave];
  static_assert(sizeof(ring) + (KS > 1 ? sizeof(red) : 0) == g1_stream_lds<MT, D, KS>(),
                "the launcher sizes the grid by this");

  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int r16 = lane & 15, g = lane >> 4;
  const int NCT = I / 16, NKB = H / kBlock;
  const int nkb = NKB / KS, kfirst = KS > 1 ? w * nkb : 0;  // this wave's K blocks
  TileMap tm;
  tm.init(counts, offsets, E_l, BM);
  const int items = tm.total * NCT;
  const int stride = KS > 1 ? gridDim.x : gridDim.x * kWavesPerGroup;
  int it = __builtin_amdgcn_readfirstlane(KS > 1 ? (int)blockIdx.x : first_item(w));
  if (it >= items) return;  // KS > 1: the whole workgroup

  const __amdgpu_buffer_rsrc_t ares = make_rsrc(hs, (uint32_t)T * H);
  const __amdgpu_buffer_rsrc_t sares = make_rsrc(hs_scale, (uint32_t)T * NKB * 4);
  const uint32_t dma0 = wblk_dma_off(lane, 0, H), dma1 = wblk_dma_off(lane, 1, H);
  const uint32_t rd0 = wblk_read_off(lane, 0), rd1 = wblk_read_off(lane, 1);
  uint8_t* my_ring = &ring[w][0][0];

  // Item metadata without the token-dependent offsets; loads the item's token ids into tok.
  auto meta = [&](int item, G1Item<MT>& x, int (&tok)[MT]) {
    item = __builtin_amdgcn_readfirstlane(item);  // keeps the item chain in SGPRs
    const int tile = item / NCT, ct = item % NCT;
    const int e = tm.find(tile, BM, x.m0, x.cnt, x.seg);
    x.c0 = ct * 16;
    x.m0 = uniform(x.m0);
    x.cnt = uniform(x.cnt);
    x.seg = uniform(x.seg);
    x.wbase = uniform(w13 + (size_t)e * 2 * I * H);
    x.wsoff = uniform((uint32_t)x.c0 * H);
    const float* srow = s13 + (size_t)e * (2 * I / kBlock) * NKB;
    x.sc1.load(srow + (size_t)(x.c0 / kBlock) * NKB, NKB);
    x.sc2.load(srow + (size_t)((I + x.c0) / kBlock) * NKB, NKB);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = x.m0 + mt * 16 + r16;
      tok[mt] = sorted_tok[x.seg + (r < x.cnt ? r : x.cnt - 1)];
    }
  };
  auto finish = [&](G1Item<MT>& x, const int (&tok)[MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      x.aoff[mt] = (uint32_t)tok[mt] * H + 32 * g;
      x.saoff[mt] = (uint32_t)tok[mt] * 4;
    }
  };

  G1Item<MT> cur, nxt, nn;
  int tok[MT];
  meta(it, cur, tok);
  finish(cur, tok);
  int it_n = it + stride;
  meta(it_n < items ? it_n : it, nxt, tok);
  finish(nxt, tok);

  G1Slot<MT> sl[D];
  // Issue this wave's K block kbl of item cur (or nxt when `second`) into slot d. After a wave's
  // last item there is no next item: those prefetches keep the step's operation count (the counted waits
  // rely on it) but use an out-of-range offset, so they return zeros and fetch nothing.
  auto issue = [&](bool second, int kbl, G1Slot<MT>& s, int d) {
    const bool dead = uniform(second && it_n >= items);
    const int kbi = kfirst + kbl;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint32_t ao = dead ? kNoFetch : second ? nxt.aoff[mt] : cur.aoff[mt];
      const uint32_t so = dead ? kNoFetch : second ? nxt.saoff[mt] : cur.saoff[mt];
      s.a[mt] = buf_load32(ares, ao, (uint32_t)kbi * kBlock);
      s.sa[mt] = __uint_as_float(buf_load32b(sares, so, (uint32_t)kbi * T * 4));
    }
    const __amdgpu_buffer_rsrc_t wres =
        make_rsrc(uniform(second ? nxt.wbase : cur.wbase), 2u * I * H);
    const uint32_t ws = uniform((second ? nxt.wsoff : cur.wsoff) + (uint32_t)kbi * kBlock);
    const uint32_t w0 = dead ? kNoFetch : dma0, w1 = dead ? kNoFetch : dma1;
    uint8_t* slot = my_ring + d * 2 * kWBlk;
    dma16_stream(wres, slot, w0, ws);
    dma16_stream(wres, slot + 1024, w1, ws);
    dma16_stream(wres, slot + kWBlk, w0, ws + (uint32_t)I * H);
    dma16_stream(wres, slot + kWBlk + 1024, w1, ws + (uint32_t)I * H);
  };

  // Prologue in issue order: the loop's wait counts assume every slot's loads went out
  // together, and the loop-entry state would otherwise carry a reordered prologue into them.
#pragma unroll
  for (int d = 0; d < D; ++d) {
    issue(false, d, sl[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  retire(nxt.sc1.v0);  // loop entry must not carry pending loads (see the K loop)
  retire(nxt.sc1.v1);
  retire(nxt.sc2.v0);
  retire(nxt.sc2.v1);

  int turn = 0;
  for (;;) {
    // Token ids and scales of the item after nxt, consumed one item from now.
    const int it_nn = it_n + stride;
    meta(it_nn < items ? it_nn : (it_n < items ? it_n : it), nn, tok);

    v4f acc1[MT], acc2[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc1[mt] = v4f{0.f, 0.f, 0.f, 0.f};
      acc2[mt] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    // do-while: the compiler must see that the trip (with its retires) runs at least once
    int kb0 = 0;
    do {
      const bool last = kb0 + D >= nkb;  // this trip's prefetches belong to the next item
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int kb = kb0 + d;
        vm_wait<vm_depth((D - 1) * OPS)>();
        const uint32_t base = lds_addr(my_ring + d * 2 * kWBlk);
        v4u x1l = ds_read16(base + rd0), x1h = ds_read16(base + rd1);
        v4u x2l = ds_read16(base + kWBlk + rd0), x2h = ds_read16(base + kWBlk + rd1);
        lds_wait(x1l, x1h, x2l, x2h);
        const v8i b1 = v8i{(int)x1l[0], (int)x1l[1], (int)x1l[2], (int)x1l[3],
                           (int)x1h[0], (int)x1h[1], (int)x1h[2], (int)x1h[3]};
        const v8i b2 = v8i{(int)x2l[0], (int)x2l[1], (int)x2l[2], (int)x2l[3],
                           (int)x2h[0], (int)x2h[1], (int)x2h[2], (int)x2h[3]};
        const float sw1 = cur.sc1.get(kfirst + kb), sw2 = cur.sc2.get(kfirst + kb);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const float f1 = sl[d].sa[mt] * sw1, f2 = sl[d].sa[mt] * sw2;
          const v4f p = mfma_f8_16x16x128(b1, sl[d].a[mt]);
          const v4f q = mfma_f8_16x16x128(b2, sl[d].a[mt]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            acc1[mt][i] = fmaf(p[i], f1, acc1[mt][i]);
            acc2[mt][i] = fmaf(q[i], f2, acc2[mt][i]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        issue(last, last ? kb + D - nkb : kb + D, sl[d], d);
        __builtin_amdgcn_sched_barrier(0);
      }
      // The next-but-one item's metadata loads are long complete here; retiring them now
      // keeps their registers' later reuse from waiting on the whole stream.
      retire(nn.sc1.v0);
      retire(nn.sc1.v1);
      retire(nn.sc2.v0);
      retire(nn.sc2.v1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) retire(tok[mt]);
      kb0 += D;
    } while (kb0 < nkb);

    // KS > 1: every wave leaves its partial sums in LDS, and after one barrier the waves in turn
    // (wave n % KS for the workgroup's n-th item) add them up in wave order and store. The buffer of
    // item n is written again for item n + 2, past the barrier of item n + 1.
    bool store = true;
    if constexpr (KS > 1) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        red[turn & 1][w][2 * mt][lane] = acc1[mt];
        red[turn & 1][w][2 * mt + 1][lane] = acc2[mt];
      }
      lds_wait_all();
      __builtin_amdgcn_s_barrier();  // (a bare one: a fence would wait for every DMA in flight)
      store = w == turn % KS;
      if (store) {
        v4u part[KS][2 * MT];
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
          for (int j = 0; j < 2 * MT; ++j)
            part[k][j] = ds_read16(lds_addr(&red[turn & 1][k][j][lane]));
        lds_wait_all();
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
          for (int j = 0; j < 2 * MT; ++j) {
            lds_fence(part[k][j]);
            v4f& acc = (j & 1) ? acc2[j / 2] : acc1[j / 2];
            const v4f v = __builtin_bit_cast(v4f, part[k][j]);
            acc = k == 0 ? v : acc + v;
          }
      }
      ++turn;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = cur.m0 + mt * 16 + r16;
      if (store && r < cur.cnt) {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x1 = acc1[mt][i], x2 = acc2[mt][i];
          h[i] = float_to_bf16_bits(x1 * (x2 / (1.0f + __expf(-x2))));
        }
        *(uint2*)(C + (size_t)(cur.seg + r) * I + cur.c0 + 4 * g) =
            uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
      }
    }
    if (it_n >= items) break;
    it = it_n;
    it_n = it_nn;
    cur = nxt;
    nxt = nn;
    finish(nxt, tok);
  }
  vm_wait<0>();  // no DMA may still target this workgroup's LDS when it retires
}

// ---- GEMM2: bf16((C W2^T) * routing weight) into the pair's destination row ---------------------

template <int MT>
struct G2Slot {
  uint4 a[MT][4];  // bf16 C values K [32g + 8c, +8) of the block, c < 4, for row r16
};

template <int MT>
struct G2Item {
  const uint8_t* wbase;  // the expert's W2 [H, I]
  uint32_t wsoff;        // h0 * I
  LaneScales sc;         // weight scales of the 128-row block holding h0, per K block
  uint32_t coff[MT];     // per lane: byte offset of C[pair][32 g]
  float wgt[MT];         // routing weight of the lane's pair
  int dst[MT];           // destination row code of the lane's pair (pair_dst)
  int m0, cnt, seg, h0;
};

template <int MT, int D>
__global__ __launch_bounds__(256) void gemm2_stream_kernel(
    const uint16_t* __restrict__ C, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    const float* __restrict__ sorted_w, Gemm2Out dst, int H, int I, int E_l, int max_pairs) {
  constexpr int BM = 16 * MT;
  constexpr int OPS = 4 * MT + 2;
  __shared__ __attribute__((aligned(16))) uint8_t ring[kWavesPerGroup][D][kWBlk];

  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int r16 = lane & 15, g = lane >> 4;
  const int NHT = H / 16, NKB = I / kBlock;
  TileMap tm;
  tm.init(counts, offsets, E_l, BM);
  const int items = tm.total * NHT;
  const int stride = gridDim.x * kWavesPerGroup;
  int it = __builtin_amdgcn_readfirstlane(first_item(w));
  if (it >= items) return;

  const __amdgpu_buffer_rsrc_t cres = make_rsrc(C, (uint32_t)max_pairs * I * 2);
  const uint32_t dma0 = wblk_dma_off(lane, 0, I), dma1 = wblk_dma_off(lane, 1, I);
  const uint32_t rd0 = wblk_read_off(lane, 0), rd1 = wblk_read_off(lane, 1);
  uint8_t* my_ring = &ring[w][0][0];

  auto meta = [&](int item, G2Item<MT>& x) {
    item = __builtin_amdgcn_readfirstlane(item);
    const int tile = item / NHT, ht = item % NHT;
    const int e = tm.find(tile, BM, x.m0, x.cnt, x.seg);
    x.h0 = ht * 16;
    x.m0 = uniform(x.m0);
    x.cnt = uniform(x.cnt);
    x.seg = uniform(x.seg);
    x.wbase = uniform(w2 + (size_t)e * H * I);
    x.wsoff = uniform((uint32_t)x.h0 * I);
    x.sc.load(s2 + ((size_t)e * (H / kBlock) + x.h0 / kBlock) * NKB, NKB);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = x.m0 + mt * 16 + r16;
      const int p = x.seg + (r < x.cnt ? r : x.cnt - 1);
      x.coff[mt] = ((uint32_t)p * I + 32 * g) * 2;
      x.wgt[mt] = sorted_w[p];
      x.dst[mt] = dst.pair_dst[p];
    }
  };

  G2Item<MT> cur, nxt, nn;
  meta(it, cur);
  int it_n = it + stride;
  meta(it_n < items ? it_n : it, nxt);

  G2Slot<MT> sl[D];
  // As in GEMM1, prefetches past a wave's last item use an out-of-range offset (no traffic).
  auto issue = [&](bool second, int kbi, G2Slot<MT>& s, int d) {
    const bool dead = uniform(second && it_n >= items);
    const __amdgpu_buffer_rsrc_t cr = cres;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const uint32_t co = dead ? kNoFetch : second ? nxt.coff[mt] : cur.coff[mt];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s.a[mt][c] = buf_load16(cr, co, 2 * (kbi * kBlock + 8 * c));
    }
    const __amdgpu_buffer_rsrc_t wres =
        make_rsrc(uniform(second ? nxt.wbase : cur.wbase), (uint32_t)H * I);
    const uint32_t ws = uniform((second ? nxt.wsoff : cur.wsoff) + (uint32_t)kbi * kBlock);
    uint8_t* slot = my_ring + d * kWBlk;
    dma16_stream(wres, slot, dead ? kNoFetch : dma0, ws);
    dma16_stream(wres, slot + 1024, dead ? kNoFetch : dma1, ws);
  };

  // Prologue in issue order: the loop's wait counts assume every slot's loads went out
  // together, and the loop-entry state would otherwise carry a reordered prologue into them.
#pragma unroll
  for (int d = 0; d < D; ++d) {
    issue(false, d, sl[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  retire(nxt.sc.v0);  // loop entry must not carry pending loads (see the K loop)
  retire(nxt.sc.v1);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    retire(nxt.wgt[mt]);
    retire(nxt.dst[mt]);
  }

  for (;;) {
    const int it_nn = it_n + stride;
    meta(it_nn < items ? it_nn : (it_n < items ? it_n : it), nn);

    v4f acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = v4f{0.f, 0.f, 0.f, 0.f};
    int kb0 = 0;
    do {
      const bool last = kb0 + D >= NKB;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int kb = kb0 + d;
        vm_wait<vm_depth((D - 1) * OPS)>();
        const uint32_t base = lds_addr(my_ring + d * kWBlk);
        v4u lo = ds_read16(base + rd0), hi = ds_read16(base + rd1);
        lds_wait(lo, hi);
        const uint32_t wv[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        v8bf bw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          v2bf p0, p1, p2, p3;
          fp8x4_to_bf16x4((int)wv[2 * c], p0, p1);
          fp8x4_to_bf16x4((int)wv[2 * c + 1], p2, p3);
          bw[c] = v8bf{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
        }
        const float sw = cur.sc.get(kb);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          v4f t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < 4; ++c)
            t = mfma_bf16_16x16x32(bw[c], __builtin_bit_cast(v8bf, sl[d].a[mt][c]), t);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mt][i] = fmaf(t[i], sw, acc[mt][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue(last, last ? kb + D - NKB : kb + D, sl[d], d);
        __builtin_amdgcn_sched_barrier(0);
      }
      retire(nn.sc.v0);
      retire(nn.sc.v1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        retire(nn.wgt[mt]);
        retire(nn.dst[mt]);
      }
      kb0 += D;
    } while (kb0 < NKB);

#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = cur.m0 + mt * 16 + r16;
      if (r < cur.cnt) {
        const float wp = cur.wgt[mt];
        const int d = cur.dst[mt];
        uint16_t* row = d >= 0 ? dst.out + (size_t)d * H : dst.partial + (size_t)(-1 - d) * H;
        const uint32_t h01 = (uint32_t)float_to_bf16_bits(acc[mt][0] * wp) |
                             ((uint32_t)float_to_bf16_bits(acc[mt][1] * wp) << 16);
        const uint32_t h23 = (uint32_t)float_to_bf16_bits(acc[mt][2] * wp) |
                             ((uint32_t)float_to_bf16_bits(acc[mt][3] * wp) << 16);
        *(uint2*)(row + cur.h0 + 4 * g) = uint2{h01, h23};
      }
    }
    if (it_n >= items) break;
    it = it_n;
    it_n = it_nn;
    cur = nxt;
    nxt = nn;
  }
  vm_wait<0>();
}

// ---- GEMM2 and combine of a few tokens ----------------------------------------------------------
//
// Up to 16 tokens fill one 16-row MFMA tile together, whatever experts they picked. A workgroup
// owns `cols` H columns (NB blocks of 16, the last one filled in part) and goes through all active
// experts, its four waves each a quarter of K: row r of the tile is token r, whose C row for the
// expert (if it picked it) is the MFMA operand, so the results add up per token in registers:
// w * (C W2^T) over the token's experts in ascending order, in fp32 and rounded once. No partial
// rows and no combine launch. Each wave keeps R experts of N K blocks in flight: weights in an LDS
// ring of D = R * N slots, the C fragments beside it in registers.
// Bound by HBM (the weights of the active experts, once); the launch that it saves is a fixed 2-4
// us. `cols` gives every CU one workgroup with an equal share of the columns: with 16 columns per
// workgroup DS-V3's 448 leave the CUs with one or two each, and the busiest one sets the time (16
// tokens 72.7 us, with 28 columns 67.1). R: three experts of 3 blocks instead of four 100.0 -> 97.2 us
// (H 4096, I 1536, 4 tokens); two of 4 blocks instead of three 237.0 -> 234.0 us (H 8192, I 2048).
//
// Where it is used: up to kTokenRows tokens and kTokenPairs expected pairs. Measured, call with
// GEMM2 and combine in two launches -> here:
//   DS-V3: 1 token 29.2 -> 26.4 us, 4 tokens 32.8 -> 30.6, 7 tokens 45.0 -> 43.3, 16 tokens
//   70.5 -> 67.1; H 4096, I 1536, 128 experts: 1 token 42.0 -> 39.1, 4 tokens 102.0 -> 97.2, 12 tokens
//   (96 pairs) 210.9 -> 207.4, but 16 tokens (128 pairs, 80 experts one after another) 237.8 -> 239.7;
//   H 6144, I 1536: 16 pairs 80.4 -> 76.7, 64 pairs 222.2 -> 218.1; H 8192, I 2048, 64 pairs
//   386.3 -> 375.3.
// From kTokenCols columns: narrower shares (H 2048: 8 columns) put the same search for an expert's
// rows on half the weights: H 2048, I 1024, 32 pairs 48.5 -> 52.1 us. The same for one K block per
// wave (I 512, H 4096): 4 tokens 52.8 -> 53.9 us, 16 tokens 93.4 -> 101.2.
constexpr int kTokenRows = 16;
constexpr int kTokenPairs = 96;
constexpr int kTokenCols = 16;

template <int NB, int N, int R>
__global__ __launch_bounds__(256) void gemm2_token_kernel(
    const uint16_t* __restrict__ C, const uint8_t* __restrict__ w2, const float* __restrict__ s2,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
    const float* __restrict__ topk_w, const int32_t* __restrict__ pair_of, int T, int K, int H,
    int I, int E_l, int max_pairs, int cols, uint16_t* __restrict__ out) {
  constexpr int D = N * R;
  constexpr int OPS = 4 + 2 * NB;  // C loads and weight DMAs per step
  __shared__ __attribute__((aligned(16))) uint8_t ring[kWavesPerGroup][D][NB * kWBlk];
  __shared__ __attribute__((aligned(16))) v4f red[kWavesPerGroup][NB][kWave];
  __shared__ __attribute__((aligned(16))) float scl[kWavesPerGroup][R][kWave];

  const int lane = threadIdx.x & (kWave - 1), w = wave_id();
  const int r16 = lane & 15, g = lane >> 4;
  const int NKB = N * kWavesPerGroup, kfirst = w * N;  // this wave's K blocks
  const int h0 = blockIdx.x * cols;
  const int hend = min(h0 + cols, H);
  const __amdgpu_buffer_rsrc_t cres = make_rsrc(C, (uint32_t)max_pairs * I * 2);
  const __amdgpu_buffer_rsrc_t wgtres = make_rsrc(topk_w, (uint32_t)T * K * 4);
  const __amdgpu_buffer_rsrc_t s2res = make_rsrc(s2, (uint32_t)E_l * (H / kBlock) * NKB * 4);
  const __amdgpu_buffer_rsrc_t pofres = make_rsrc(pair_of, (uint32_t)T * K * 4);
  uint32_t dma[NB][2];  // rows past this workgroup's columns are not fetched
  int sidx[NB];         // scl index of the first K block's scale for this lane's four columns
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 16 * b + 8 * h + (lane >> 3);
      dma[b][h] = h0 + row < hend ? (uint32_t)(16 * b) * I + wblk_dma_off(lane, h, I) : kNoFetch;
    }
    sidx[b] = min((h0 + 16 * b + 4 * g) / kBlock - h0 / kBlock, 1) * N;
  }
  const uint32_t rd0 = wblk_read_off(lane, 0), rd1 = wblk_read_off(lane, 1);
  uint8_t* my_ring = &ring[w][0][0];

  // Lane l holds expert l + 64 j's pair count and segment; active[j] has a bit per lane with pairs.
  int cnt[4], seg[4];
  unsigned long long active[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = j * kWave + lane;
    cnt[j] = e < E_l ? counts[e] : 0;
    seg[j] = e < E_l ? offsets[e] : 0;
    active[j] = __ballot(cnt[j] > 0);
  }
  int pk[kMaxTopK];  // pairs of token r16 and their routing weights
  float wk[kMaxTopK];
#pragma unroll
  for (int k = 0; k < kMaxTopK; ++k) {
    const uint32_t v = r16 < T && k < K ? 4u * (r16 * K + k) : kNoFetch;
    pk[k] = (int)buf_load32b(pofres, v, 0) | (v == kNoFetch ? -1 : 0);
    wk[k] = __uint_as_float(buf_load32b(wgtres, v, 0));
  }

  int left = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) left += __popcll(active[j]);
  left = uniform(left);

  struct Rows {
    float wgt;      // routing weight of row r16's pair
    uint32_t coff;  // its C row (kNoFetch: none)
  };
  // Issue side: the next active expert; past the last one nothing is fetched.
  const uint8_t* wbase = w2;
  int seg0 = 0, pairs = 0;
  auto next_expert = [&](int r) {
    int e = -1;
    pairs = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (e < 0 && active[j]) {
        const int l = __ffsll((long long)active[j]) - 1;
        active[j] &= active[j] - 1;
        e = j * kWave + l;
        pairs = __builtin_amdgcn_readlane(cnt[j], l);
        seg0 = __builtin_amdgcn_readlane(seg[j], l);
      }
    }
    const int x = e < 0 ? 0 : e;
    const int hb = h0 / kBlock + (lane >= N);
    const uint32_t so = (uint32_t)((x * (H / kBlock) + hb) * NKB + kfirst + lane - (lane >= N) * N);
    dma4(s2res, &scl[w][r][0],
         pairs > 0 && lane < 2 * N && hb < H / kBlock ? 4u * so : kNoFetch, 0);
    wbase = uniform(w2 + (size_t)x * H * I);
  };
  auto find_rows = [&]() {
    Rows x = {0.f, kNoFetch};
#pragma unroll
    for (int k = 0; k < kMaxTopK; ++k) {
      const bool in = (uint32_t)(pk[k] - seg0) < (uint32_t)pairs;
      x.coff = in ? ((uint32_t)pk[k] * I + 32 * g) * 2 : x.coff;
      x.wgt = in ? wk[k] : x.wgt;
    }
    return x;
  };
  uint4 a[D][4];
  auto issue_rows = [&](int d, const Rows& x) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      a[d][c] = buf_load16(cres, x.coff, 2 * ((kfirst + d % N) * kBlock + 8 * c));
  };
  auto issue_weights = [&](int d) {
    const int kb = kfirst + d % N;
    const __amdgpu_buffer_rsrc_t wres = make_rsrc(uniform(wbase), (uint32_t)H * I);
    const uint32_t ws = uniform((uint32_t)h0 * I + (uint32_t)kb * kBlock);
    uint8_t* slot = my_ring + d * NB * kWBlk;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      dma16_stream(wres, slot + b * kWBlk, pairs > 0 ? dma[b][0] : kNoFetch, ws);
      dma16_stream(wres, slot + b * kWBlk + 1024, pairs > 0 ? dma[b][1] : kNoFetch, ws);
    }
  };

  Rows rows[R];
  int seg_r[R], pairs_r[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {  // all weights first: they need no pair lookup
    next_expert(r);
    seg_r[r] = seg0, pairs_r[r] = pairs;
#pragma unroll
    for (int i = 0; i < N; ++i) issue_weights(r * N + i);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    seg0 = seg_r[r], pairs = pairs_r[r];
    rows[r] = find_rows();
#pragma unroll
    for (int i = 0; i < N; ++i) issue_rows(r * N + i, rows[r]);
  }
  __builtin_amdgcn_sched_barrier(0);
  v4f acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = v4f{0.f, 0.f, 0.f, 0.f};
  for (; left > 0; left -= R) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      vm_wait<vm_depth((D - 1) * OPS)>();
      float sc[NB][N];
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < N; ++i) sc[b][i] = ds_read4f(lds_addr(&scl[w][r][sidx[b] + i]));
      lds_wait_all();
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < N; ++i) lds_fence(sc[b][i]);
      const Rows cur = rows[r];
      next_expert(r);
      rows[r] = find_rows();
      v4f ae[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) ae[b] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int d = r * N + i;
        vm_wait<vm_depth((D - 1) * OPS)>();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const uint32_t base = lds_addr(my_ring + (d * NB + b) * kWBlk);
          v4u lo = ds_read16(base + rd0), hi = ds_read16(base + rd1);
          lds_wait(lo, hi);
          const uint32_t wv[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          v4f t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            v2bf p0, p1, p2, p3;
            fp8x4_to_bf16x4((int)wv[2 * c], p0, p1);
            fp8x4_to_bf16x4((int)wv[2 * c + 1], p2, p3);
            const v8bf bw = v8bf{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
            t = mfma_bf16_16x16x32(bw, __builtin_bit_cast(v8bf, a[d][c]), t);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) ae[b][q] = fmaf(t[q], sc[b][i], ae[b][q]);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue_rows(d, rows[r]);
        issue_weights(d);
        __builtin_amdgcn_sched_barrier(0);
      }
      // (rows without a pair are zero rows of the product: kept out, as 0 x NaN or 0 x inf is NaN)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          acc[b][q] = cur.coff != kNoFetch ? fmaf(ae[b][q], cur.wgt, acc[b][q]) : acc[b][q];
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) red[w][b][lane] = acc[b];
  vm_wait<0>();  // no DMA may still target this workgroup's LDS when it retires
  __syncthreads();
  if (w < NB && r16 < T && h0 + 16 * w + 4 * g < hend) {
    v4f s = red[0][w][lane];
#pragma unroll
    for (int k = 1; k < kWavesPerGroup; ++k) s += red[k][w][lane];
    const uint32_t h01 = (uint32_t)float_to_bf16_bits(s[0]) | ((uint32_t)float_to_bf16_bits(s[1]) << 16);
    const uint32_t h23 = (uint32_t)float_to_bf16_bits(s[2]) | ((uint32_t)float_to_bf16_bits(s[3]) << 16);
    *(uint2*)(out + (size_t)r16 * H + h0 + 16 * w + 4 * g) = uint2{h01, h23};
  }
}

}  // namespace

// Persistent grid: `per_cu` workgroups per CU, capped by the largest possible item count.
static int persistent_grid(int per_cu, long long max_items) {
  const int cus = device_cu_count();
  long long g = (long long)cus * per_cu;
  if (g > max_items) g = max_items;
  return g < 1 ? 1 : (int)g;
}

static inline long long max_m_tiles(int max_pairs, int bm, int E_l) {
  return (max_pairs + bm - 1) / bm + (E_l < max_pairs ? E_l : max_pairs);
}

// Workgroups per CU that fit its 160 KiB of LDS.
static inline int groups_per_cu(int lds_bytes) {
  const int n = (160 * 1024) / lds_bytes;
  return n < 1 ? 1 : n > 8 ? 8 : n;
}

// Ring depth: the largest power of two <= dmax that divides the K-block count, so an item's K
// steps split into whole trips.
static inline int ring_depth(int nkb, int dmax) {
  int d = dmax;
  while (d > 1 && nkb % d != 0) d >>= 1;
  return d;
}

constexpr int kG1StreamD = 8;
constexpr int kG2StreamD = 8;

// GEMM1 items split over the K quarters of a workgroup's four waves (KS = 4). A wave then fetches a
// contiguous quarter of each weight row, the four side by side, instead of 1 KiB windows of 16
// rows far from its neighbours': with the 4 KiB row pitch of H = 4096 the unsplit form keeps
// hitting few memory channels (Qwen3-style GEMM1 stage T=8 114 -> 98 us, T=16 177 -> 154, T=32 237 ->
// 208, T=64 270 -> 237: 6.8 TB/s, the rate of a plain non-temporal read). It also gives a
// batch of few items four times as many, so that no CU is left with one wave's loads in flight
// (DS-V3 T=1 call 33.3 -> 31.0 us), and evens out the last round (DS-V3 T=48 90.1 -> 88.1, T=128 126.4
// -> 125.0). From half to one and a half whole-K items per wave that the chip holds the split only
// adds its reduction (Qwen3-style T=1 43.9 against 44.6 us, T=2 62.1 against 64.2; DS-V3 T=7 46.6
// against 47.0), so there K stays whole. `expected` counts one expert for every expected pair up to
// all of them: an upper bound, since pairs share experts (7 DS-V3 tokens: 7 expected pairs, 3.6 experts).

hipError_t launch_gemm1_stream(const uint8_t* hs, const float* hs_scale, const uint8_t* w13,
                               const float* s13, const int32_t* counts, const int32_t* offsets,
                               const int32_t* sorted_tok, uint16_t* C, int T, int H, int I,
                               int E_l, int max_pairs, int pairs_hint, int mt,
                               hipStream_t stream) {
  const int nkb = H / kBlock;
  const long long expected = (long long)(pairs_hint < E_l ? pairs_hint : E_l) * (I / 16);
  const long long waves = (long long)kWavesPerGroup * device_cu_count();
  const bool split = 2 * expected < waves || 2 * expected > 3 * waves;
#define JG_G1S(MT, D, KS)                                                                      \
  {                                                                                            \
    const long long tiles = max_m_tiles(max_pairs, 16 * MT, E_l) * (I / 16);                   \
    const int grid = persistent_grid(groups_per_cu(g1_stream_lds<MT, D, KS>()),                \
                                     (tiles * KS + kWavesPerGroup - 1) / kWavesPerGroup);       \
    gemm1_stream_kernel<MT, D, KS><<<grid, kWavesPerGroup * kWave, 0, stream>>>(               \
        hs, hs_scale, w13, s13, counts, offsets, sorted_tok, C, T, H, I, E_l);                 \
    return hipGetLastError();                                                                  \
  }
  const int d = ring_depth(nkb, mt == 1 ? kG1StreamD : 4);
  if (mt == 1) {
    if (split && nkb % kWavesPerGroup == 0) {
      const int n = nkb / kWavesPerGroup;
      if (n % 8 == 0) JG_G1S(1, 8, 4)
      if (n % 7 == 0) JG_G1S(1, 7, 4)
      if (n % 6 == 0) JG_G1S(1, 6, 4)
      if (n % 5 == 0) JG_G1S(1, 5, 4)
      if (n % 4 == 0) JG_G1S(1, 4, 4)
    }
    if (d >= 8) JG_G1S(1, 8, 1)
    if (d == 4) JG_G1S(1, 4, 1)
    if (d == 2) JG_G1S(1, 2, 1)
    JG_G1S(1, 1, 1)
  }
  if (mt == 2) {
    if (d == 4) JG_G1S(2, 4, 1)
    if (d == 2) JG_G1S(2, 2, 1)
    JG_G1S(2, 1, 1)
  }
  if (d == 4) JG_G1S(4, 4, 1)
  if (d == 2) JG_G1S(4, 2, 1)
  JG_G1S(4, 1, 1)
#undef JG_G1S
}

hipError_t launch_gemm2_stream(const uint16_t* C, const uint8_t* w2, const float* s2,
                               const int32_t* counts, const int32_t* offsets,
                               const float* sorted_w, Gemm2Out dst, int H, int I, int E_l,
                               int max_pairs, int mt, hipStream_t stream) {
  const int nkb = I / kBlock;
#define JG_G2S(MT, D)                                                                          \
  {                                                                                            \
    const long long waves = max_m_tiles(max_pairs, 16 * MT, E_l) * (H / 16);                   \
    const int grid = persistent_grid(groups_per_cu(kWavesPerGroup * D * kWBlk),                \
                                     (waves + kWavesPerGroup - 1) / kWavesPerGroup);            \
    gemm2_stream_kernel<MT, D><<<grid, kWavesPerGroup * kWave, 0, stream>>>(                   \
        C, w2, s2, counts, offsets, sorted_w, dst, H, I, E_l, max_pairs);                  \
    return hipGetLastError();                                                                  \
  }
  const int d = ring_depth(nkb, mt == 1 ? kG2StreamD : mt == 2 ? 4 : 2);
  if (mt == 1) {
    if (d >= 8) JG_G2S(1, 8)
    if (d == 4) JG_G2S(1, 4)
    if (d == 2) JG_G2S(1, 2)
    JG_G2S(1, 1)
  }
  if (mt == 2) {
    if (d == 4) JG_G2S(2, 4)
    if (d == 2) JG_G2S(2, 2)
    JG_G2S(2, 1)
  }
  if (d == 2) JG_G2S(4, 2)
  JG_G2S(4, 1)
#undef JG_G2S
}

hipError_t launch_gemm2_token(const uint16_t* C, const uint8_t* w2, const float* s2,
                              const int32_t* counts, const int32_t* offsets, const float* topk_w,
                              const int32_t* pair_of, int T, int K, int H, int I, int E_l,
                              int max_pairs, int pairs_hint, uint16_t* out, hipStream_t stream) {
  const int cus = device_cu_count();
  const int cols = (H + 4 * cus - 1) / (4 * cus) * 4;
  if (T > kTokenRows || pairs_hint > kTokenPairs || cols < kTokenCols || E_l > 4 * kWave)
    return hipErrorNotSupported;
#define JG_G2T(NB, N, R)                                                                        \
  if (cols <= NB * 16 && I == N * kWavesPerGroup * kBlock) {                                    \
    gemm2_token_kernel<NB, N, R><<<(H + cols - 1) / cols, kWavesPerGroup * kWave, 0, stream>>>( \
        C, w2, s2, counts, offsets, topk_w, pair_of, T, K, H, I, E_l, max_pairs, cols, out);    \
    return hipGetLastError();                                                                   \
  }
  JG_G2T(1, 2, 4)
  JG_G2T(1, 3, 3)
  JG_G2T(1, 4, 2)
  JG_G2T(2, 2, 4)
  JG_G2T(2, 3, 3)
  JG_G2T(2, 4, 2)
#undef JG_G2T
  return hipErrorNotSupported;
}

}  // namespace jgmoe
