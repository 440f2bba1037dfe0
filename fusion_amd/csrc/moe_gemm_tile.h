// Grouped GEMM tiles for prefill (tens to thousands of rows per expert), gfx950: the block
// sizes 64, 128 and 256 of `glm52_moe_gemm*`, and o_proj from 17 rows.  Semantics are
// those of the other mappings: `moe_gateup_kernel` (`glm52/kernels/moe_gateup.py:34-148`) when
// gated, `moe_down_kernel` with MUL_ROUTED_WEIGHT (`glm52/kernels/moe_down_merge.py:66-169`)
// when weighted, `oproj_gemm_kernel` (`glm52/kernels/oproj_resadd.py:32-136`) for EPI 1-3.
//
// Tile.  A workgroup owns one layout block of MT tokens and NT rows of that expert's W (gated:
// the `gate` and `up` rows of NT / 2 consecutive outputs): a whole packed 512-row tile or half
// of one (the choice is at launch_tile_as).  Four waves: each holds 128 W rows, against all of
// the block's real 16-token groups (NT 512) or half of them (NT 256: 2 x 2 waves, so a
// part-filled block costs both token halves the same), in `v_mfma_f32_16x16x32_bf16` blocks
// with W as the first operand.
//
// Pipeline.  K advances in 32-k stages through a ring of LDS buffers (as many as 160 KB hold:
// five at 256 x 256) filled by direct global -> LDS loads.  While the MFMAs of stage s run on
// fragments already in registers, the wave reads the fragments of stage s + 1 and issues loads
// for the buffer that stage s left; the order is pinned.  What the loop may not contain was
// measured on the 256 x 256 tile's bare loop: 64
// MFMAs, 16 fragment reads, 8 loads and a barrier take 1060 cycles a stage (1024 for the MFMAs
// alone).  A branch per load (a cache-policy choice, a clamp past the last stage) and LDS
// addresses formed per read made it 1450, so the cache policy is a template argument, the
// loads past the last stage go through a descriptor of zero bytes (no memory access) and a
// stage has two LDS base addresses.  The 16x16x32 form runs 5-8 % above 32x32x16 at the
// board's power limit (the bare loop on all CUs: 537 against 584 us).
//
// Token rows are staged two stages at a time: a stage takes 64 bytes of a row, half of a
// 128-byte line, and the other half, asked for a stage later, was often fetched again.  The
// two halves are loaded by adjacent instructions (T = 4096, w13: 2732 -> 2410 us).  Row-major
// W is staged the same way.
//
// W tiles that only one item streams are loaded non-temporally, so that they do not evict the
// token rows and shared tiles that other workgroups of the XCD re-read from L2 (T = 8192 with
// skewed load: w13 3737 -> 3580 us).
//
// Order and dealing.  The kernel is persistent, one workgroup per CU.  Each XCD owns a contiguous
// share of the items, ordered expert by expert (a share may end inside an expert), and deals it
// from a counter of its own, then helps the other XCDs; the row blocks of an expert in groups of
// kRowGroup, so that the 32 workgroups of an XCD read 4 row blocks and 8 column tiles (or 8
// and 4) at a time (12 operand tiles for 32 products; column tile by column tile it was 33:
// o_proj at M = 8192 1941 -> 1352 us with nothing else changed).
//
// Between items.  The next item is decoded and the first stages that fill its ring (four to
// eight) are issued before the current item's epilogue, so their latency runs under it.
#pragma once

#include "moe_gemm.h"
#include "tile_range.h"

#include <atomic>
#include <type_traits>

namespace glm52 {
namespace {  // one copy per source file: each has its own counters and their sequence

// the kernel's lambdas share its state by reference, which stays in registers only inlined
#define GLM52_INLINE __attribute__((always_inline))

constexpr int kBK = 32;  // k per stage

// Counters the items are dealt from, a set per launch: XCD x's at 16 x, the exits at 128; the
// last workgroup out clears the set.  Two launches on one set would each run part of the items,
// so launches in flight together need sets of their own.  Every instance of the source file
// draws from the one sequence beside the array: an eager launch takes the next of kDealSets
// sets, so it shares one only with a launch a whole multiple of kDealSets before it; a captured
// launch takes the next of another kDealSets and keeps it in the graph, so eager launches never
// meet it (replays that overlap must be of graphs whose captured launches use different sets).
constexpr int kDealSets = 1024;
constexpr int kDealStride = 256;
__device__ __align__(256) int g_tile_deal[2 * kDealSets * kDealStride];
std::atomic<unsigned> g_next_eager{0}, g_next_captured{0};

int take_deal_set(hipStream_t st) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess) {
    (void)hipGetLastError();  // the launch reports its own error
    cap = hipStreamCaptureStatusNone;
  }
  const bool captured = cap != hipStreamCaptureStatusNone;
  std::atomic<unsigned>& next = captured ? g_next_captured : g_next_eager;
  const int set = (int)(next.fetch_add(1, std::memory_order_relaxed) % kDealSets);
  return note_item_set(captured ? kDealSets + set : set);
}

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>), unrolled at compile time.
template <int N, int I = 0, typename F>
GLM52_DEV void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

GLM52_DEV int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Raw buffer descriptor over `bytes` bytes at `base`: a load past them reads zero without
// touching memory.
GLM52_DEV u32x4_t make_srd(const void* base, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  u32x4_t r;
  r[0] = (uint32_t)uniform((int)(uint32_t)b);
  r[1] = (uint32_t)uniform((int)((uint32_t)(b >> 32) & 0xffffu));
  r[2] = (uint32_t)uniform((int)bytes);
  r[3] = 0x00020000u;
  return r;
}

// One direct 16-byte-per-lane load into LDS: lane l's 16 bytes at base + voff + soff land at
// byte `lds` + 16 l (lds and soff wave-uniform); ordered by explicit vmcnt waits, as dma16s.
template <bool NT>
GLM52_DEV void dma16b(const u32x4_t& srd, uint32_t voff, uint32_t soff, uint32_t lds) {
  const u32x4_t d = {(uint32_t)uniform((int)srd[0]), (uint32_t)uniform((int)srd[1]),
                     (uint32_t)uniform((int)srd[2]), (uint32_t)uniform((int)srd[3])};
  const int m = uniform((int)lds), so = uniform((int)soff);
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(m), "v"(voff), "s"(d), "s"(so)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(m), "v"(voff), "s"(d), "s"(so)
                 : "memory");
}

// Two fp32 as packed bf16, round to nearest even, as pack8 but for a NaN's bits (0xffc0 here).
GLM52_DEV uint32_t cvt_pk_bf16(float lo, float hi) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// Lanes 32-63 of `a` change places with lanes 0-31 of `b`.
GLM52_DEV void swap_halves(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
GLM52_DEV void swap_halves(float& a, float& b) {
  uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  swap_halves(x, y);
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}

// Every wave's LDS reads and direct loads are done, for all waves.
GLM52_DEV void drain_and_meet() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

// EPI (non-gated): 0 bf16 store; 1 bf16(acc + R); 2 C32 += acc (+ R); 3 C32 = acc (fp32
// partials); 4 the atomic expert merge, bf16 packed atomic adds into row tok / merge_topk.
template <int MT, int NT, bool GATED, bool WEIGHTED, bool PACKED, int EPI>
__global__ __launch_bounds__(256) void moe_gemm_tile_kernel(GemmArgs p) {
  constexpr int kWaveN = NT / 128, kWaveM = 4 / kWaveN;  // waves along W and along the tokens
  constexpr uint32_t kRowsBytes = NT * kBK * 2;  // W's part of a stage; the token rows follow
  constexpr uint32_t kStageBytes = (NT + MT) * kBK * 2;
  constexpr int kStages = 163840 / kStageBytes;
  constexpr int kWI = NT / 64;  // W load instructions per wave and stage
  constexpr int kAI = MT / 64;  // token-row load instructions per wave and stage
  constexpr int kQ = MT / kWave;
  // Row blocks of an expert per group of the item order.  An XCD's 32 workgroups read 12 operand
  // tiles at a time with groups of 4 (4 row blocks and 8 column tiles) and of 8 alike.  In o_proj
  // 8 stream B once, not twice, for 5 to 8 row blocks (M = 1536 369 -> 348 us, M = 2048 379 ->
  // 362; M = 8192 1278 -> 1272).  The expert GEMMs stay at 4: the T = 8192 block is the same
  // with 8 (6025, 5970 us, runs 1 % apart), and two of three blocks at T = 3000 - 4096 2-3 % slower.
  constexpr int kRowGroup = PACKED && !GATED && !WEIGHTED ? 8 : 4;
  const unsigned long long t_start = p.wg_trace ? __builtin_amdgcn_s_memrealtime() : 0ull;
  int n_run = 0;  // items this workgroup ran (the trace record)
  constexpr int NO = GATED ? NT / 2 : NT;    // outputs per tile; a packed tile has twice those
  __shared__ __attribute__((aligned(1024))) uint16_t ring[kStages * kStageBytes / 2];

  constexpr int kHalves = 512 / NT;  // tiles per packed 512-row tile

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wv = uniform(tid / kWave);
  const int wn = wv % kWaveN, wm = wv / kWaveN;
  const int r16 = lane & 15, g4 = lane >> 4;

  const int num_m = *p.ntp / MT;
  const int num_n = p.n_out / NO;
  const int items = num_m * num_n;
  const int nk = p.K / kBK;
  const int per_xcd = (items + 7) / 8;
  // the extra (shared) expert, packed weights only: its items follow each XCD's routed ones
  const bool has_x = PACKED && EPI == 0 && p.Wx && p.x_rows > 0;
  const int nbx = has_x ? (p.x_rows + MT - 1) / MT : 0;
  const int items_x = nbx * num_n;
  const int per_xcd_x = (items_x + 7) / 8;
  int* const deal = g_tile_deal + p.deal_set * kDealStride;
  const int wg_xcd = gridDim.x / 8;  // workgroups per XCD (the launcher rounds to 8)

  const uint32_t ring_base = lds_addr(ring);
  const char* const ring_c = reinterpret_cast<const char*>(ring);
  int* const slot = reinterpret_cast<int*>(ring);  // used between items only

  // ---- the item being staged ----------------------------------------------------------
  int xcd = blockIdx.x % 8;  // the XCD whose items this workgroup takes: its own first
  int tried = 1;
  int k = blockIdx.x / 8;    // its next item there
  bool xs = false;           // an item of the extra expert
  int krot = 0;              // its first stage
  bool w_once = false;       // no other item reads this W tile
  int n0 = 0, nv_rows = 0;   // its first output; its real rows, a prefix of the block
  int tq[kQ];                // the flat token of row q * 64 + lane
  u32x4_t srd_w, srd_a;
  uint32_t w_bytes = 0;
  uint32_t wvoff[PACKED ? 1 : kWI], avoff[kAI];

  auto fetch_now = [&]() GLM52_INLINE {  // the next index of XCD xcd's items, for the whole workgroup
    if (tid == 0)
      *slot = __hip_atomic_fetch_add(deal + xcd * 16, 1, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int v = uniform(wg_xcd + *slot);
    __syncthreads();
    return v;
  };

  // Decodes item k of XCD xcd (routed items first, then the extra expert's), going on to the
  // next XCDs' items once its own are taken and past blocks with no real row; false: none left.
  auto decode = [&]() GLM52_INLINE -> bool {
    for (;;) {
      const int n_r = max(0, min(per_xcd, items - xcd * per_xcd));
      const int n_local = n_r + max(0, min(per_xcd_x, items_x - xcd * per_xcd_x));
      if (k >= n_local) {
        if (tried == 8) return false;
        ++tried;
        xcd = (xcd + 1) % 8;
        k = fetch_now();
        continue;
      }
      xs = k >= n_r;
      int pid_n, row0, e;
      if (!xs) {
        // The expert's row blocks mb .. me - 1: the run of equal expert ids around block b,
        // from one load of the 64 ids around it (longer runs: block by block).
        const int L = xcd * per_xcd + k;
        const int b = L / num_n;
        const int bi = b - 32 + lane;
        const int ev = bi >= 0 && bi < num_m ? p.eids[bi] : -2;
        e = __builtin_amdgcn_readlane(ev, 32);
        const unsigned long long same = __ballot(ev == e);
        const uint32_t lo = ~(uint32_t)same, hi = ~(uint32_t)(same >> 32);
        const int below = lo ? __builtin_clz(lo) : 32, above = hi ? __builtin_ctz(hi) : 32;
        int mb = b - below, me = b + above;
        if (below == 32)
          while (mb > 0 && p.eids[mb - 1] == e) --mb;
        if (above == 32)
          while (me < num_m && p.eids[me] == e) ++me;
        mb = uniform(mb);
        const int cnt = uniform(me) - mb;
        w_once = cnt == 1;
        // groups of kRowGroup row blocks, column tile major inside a group
        const int local = L - mb * num_n;
        const int g0 = local / (kRowGroup * num_n) * kRowGroup;
        const int gs = min(kRowGroup, cnt - g0);
        const int in = local - g0 * num_n;
        pid_n = in / gs;
        row0 = (mb + g0 + in % gs) * MT;
      } else {
        const int Lx = xcd * per_xcd_x + (k - n_r);
        pid_n = Lx / nbx;
        row0 = (Lx % nbx) * MT;
        e = 0;
        w_once = nbx == 1;
      }
      const int nvalid = xs ? p.x_rows : p.num_valid;
      nv_rows = 0;
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int r = row0 + q * kWave + lane;
        tq[q] = xs ? min(r, p.x_rows) : p.sti[r];
      }
#pragma unroll
      for (int q = 0; q < kQ; ++q) nv_rows += __popcll(__ballot(tq[q] < nvalid));
      nv_rows = uniform(nv_rows);
      if (nv_rows == 0) {
        k = fetch_now();
        continue;
      }
      ++n_run;
      n0 = pid_n * NO;
      const int P = pid_n / kHalves, sub = pid_n % kHalves;

      // The item's first stage (its stages run from there, wrapping) in the expert GEMMs on 64-
      // and 128-token tiles.  There most W tiles are streamed by one item, the workgroups
      // advance in step, and with every item at the same stage the loads in flight sit a
      // multiple of 2 MB apart; starting each expert's packed tiles 16 stages apart spreads
      // them over the HBM channels (T = 1000 block 3262 -> 3237 us).  256-token tiles keep
      // stage 0: there the tiles of an expert share its token rows stage by stage (T = 8192,
      // w13 3857 -> 3973 us with the start).  It depends on the expert and the packed tile
      // only, so packed and in-place W, one launch or separate ones, and the atomic merge add
      // an output's products in one order.
      krot = MT <= 128 && (EPI == 0 || EPI == 4) ? ((e * (num_n / kHalves) + P) * 16) % nk : 0;
      // W: the wave's load instruction i fills slab wv * kWI + i (16 rows) of the stage
      if constexpr (PACKED) {
        const int64_t tile = packed_tile_elems(nk);
        w_bytes = (uint32_t)(tile * 2);
        srd_w = make_srd((xs ? p.Wx : p.Wp) + (int64_t)(e * (num_n / kHalves) + P) * tile, w_bytes);
        wvoff[0] = (uint32_t)(packed_slot_off(nk, sub * 16 + wv * kWI) * 2 + lane * 16);
      } else {
        w_bytes = kInPlaceBytes;
        srd_w = make_srd(p.W + (int64_t)e * p.swe, w_bytes);
#pragma unroll
        for (int i = 0; i < kWI; ++i) {
          const int slab = sub * 16 + wv * kWI + i;
          const int row = P * (kHalves * NO) + w512_row(GATED, p.gu_off, slab / 8, slab % 8, lane);
          wvoff[i] = (uint32_t)(((int64_t)row * p.swn + w512_chunk(lane) * 8) * 2);
        }
      }
      // token rows: instruction i fills rows wv * MT / 4 + i * 16 + lane / 4
      srd_a = make_srd(xs ? p.Ax : p.A, kTokenBytes);
      int tw = tq[0];
#pragma unroll
      for (int q = 1; q < kQ; ++q) tw = wv * (MT / 4) / kWave == q ? tq[q] : tw;
#pragma unroll
      for (int i = 0; i < kAI; ++i) {
        const int rl = wv * (MT / 4) + i * 16 + (lane >> 2);
        const int t = __shfl(tw, rl % kWave);
        avoff[i] = rl < nv_rows
                       ? (uint32_t)((xs ? t : t / p.a_div) * (int)(xs ? p.sax : p.sam) +
                                    w512_chunk(lane) * 8) * 2u
                       : kNowhere;
      }
      return true;
    }
  };

  // ---- the ring -------------------------------------------------------------------------
  // W: stage sw is next, at ring offset wo; token rows: the pair of stages sa, sa + 1
  int sw = 0, sa = 0;
  uint32_t wo = 0, ao = 0, so_w = 0, so_w1 = 0, so_a = 0, so_a1 = 0, lw = 0, lw1 = 0, la = 0, la1 = 0;
  auto next = [&](uint32_t o) GLM52_INLINE { return o == (kStages - 1) * kStageBytes ? 0u : o + kStageBytes; };
  constexpr int WS = PACKED ? kPackStride * 2 : kBK * 2;  // bytes from a stage of W to the next
  auto w_begin = [&]() GLM52_INLINE {  // packed: one stage; in place: a pair
    const StageLoad l = stage_load(sw, nk, krot, WS, w_bytes);
    srd_w[2] = l.bytes;
    so_w = l.off;
    so_w1 = l.off1;
    lw = ring_base + wo + (uint32_t)(wv * kWI * 1024);
    wo = next(wo);
    ++sw;
    if constexpr (!PACKED) {
      lw1 = ring_base + wo + (uint32_t)(wv * kWI * 1024);
      wo = next(wo);
      ++sw;
    }
  };
  auto a_begin = [&]() GLM52_INLINE {
    const StageLoad l = stage_load(sa, nk, krot, kBK * 2, kTokenBytes);
    srd_a[2] = l.bytes;
    so_a = l.off;
    so_a1 = l.off1;
    la = ring_base + ao + kRowsBytes + (uint32_t)(wv * kAI * 1024);
    ao = next(ao);
    la1 = ring_base + ao + kRowsBytes + (uint32_t)(wv * kAI * 1024);
    ao = next(ao);
    sa += 2;
  };
  constexpr int WN = PACKED ? kWI : 2 * kWI, AN = 2 * kAI;  // instructions of w_begin / a_begin
  auto w_one = [&](auto nt, int i) GLM52_INLINE {
    constexpr bool STREAM = decltype(nt)::value;
    if constexpr (PACKED)
      dma16b<STREAM>(srd_w, wvoff[0] + i * 1024, so_w, lw + i * 1024);
    else  // the two halves of a line by adjacent instructions
      dma16b<STREAM>(srd_w, wvoff[i / 2], (i % 2) ? so_w1 : so_w,
                     ((i % 2) ? lw1 : lw) + (i / 2) * 1024);
  };
  auto a_one = [&](int i) GLM52_INLINE {
    dma16b<false>(srd_a, avoff[i / 2], (i % 2) ? so_a1 : so_a,
                  ((i % 2) ? la1 : la) + (i / 2) * 1024);
  };
  // Stage s loads into the ring, N = kStages: W of stage s + N (packed), and in the stages of
  // parity kPA the pair s + N - 1, s + N of the token rows (and of W, in place).  later(odd):
  // the loads younger than the last of stage s + 1's at the start of an even / odd stage s.
  constexpr int kPA = kStages % 2 ? 0 : 1;
  auto later = [](bool odd) constexpr {
    const int pairs = kPA == 0 ? (kStages - 3) / 2 : odd ? (kStages - 4) / 2 : (kStages - 2) / 2;
    return PACKED ? (kStages - 2) * kWI + pairs * AN : pairs * (WN + AN);
  };
  // the loads younger than stage 0's at the end of the prologue, which issues what the stages
  // -N .. -1 would
  constexpr int kLater0 =
      later(true) + (PACKED ? WN + (kPA == 1 ? AN : 0) : (kPA == 1 ? WN + AN : 0));
  static_assert(kLater0 < 64 && later(false) < 64, "vmcnt range");
  auto prologue_nt = [&](auto nt) GLM52_INLINE {
    auto w_all = [&]() GLM52_INLINE {
      w_begin();
#pragma unroll
      for (int i = 0; i < WN; ++i) w_one(nt, i);
    };
    auto a_all = [&]() GLM52_INLINE {
      a_begin();
#pragma unroll
      for (int i = 0; i < AN; ++i) a_one(i);
    };
    static_for<kStages>([&](auto v) GLM52_INLINE {  // stage v - N
      constexpr bool pair = (decltype(v)::value + kStages) % 2 == kPA;
      if constexpr (pair) a_all();
      if constexpr (PACKED || pair) w_all();
    });
  };
  auto prologue = [&]() GLM52_INLINE {
    sw = sa = 0;
    wo = ao = 0;
    if (w_once) prologue_nt(std::true_type{});
    else prologue_nt(std::false_type{});
  };

  // lane (r, g) reads 16-byte chunk {0, 3, 1, 2}[g] of row r for both operands (a permutation
  // of the stage's k): with the staged rows' chunk c at c ^ ((r / 4) % 4), the 16 lanes that a
  // 128-bit LDS read serves together then read 16 distinct bank groups (in order they read 8)
  const uint32_t rd_lane =
      (uint32_t)(r16 * 64 + ((((0x2130 >> (4 * g4)) & 3) ^ ((r16 >> 2) & 3)) * 16));

  bool have = decode();
  if (have) prologue();
  while (have) {
    // this item, for its epilogue: the staging variables move on to the next item before it
    const bool c_xs = xs;
    const int c_nv = nv_rows, c_n0 = n0;
    const int nvalid = c_xs ? p.x_rows : p.num_valid;

    auto run = [&](auto nv_tag, auto nt) GLM52_INLINE {
      constexpr int NV = decltype(nv_tag)::value;  // 16-token groups per wave
      constexpr int NMF = 8 * NV;                  // MFMAs per stage
      constexpr int NRD = 8 + NV;                  // fragment reads per stage
      constexpr int RS = NV >= 4 ? 2 : 1;          // MFMAs from one read to the next
      // the lane's tokens (nvalid: none) and routing weights, for the epilogue
      int tok[NV];
      float wgt[NV];
#pragma unroll
      for (int t = 0; t < NV; ++t) {
        const int gr = wm * NV + t;
        int o = nvalid;
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
          const int v = __shfl(tq[q], (gr % 4) * 16 + r16);
          o = gr / 4 == q ? v : o;
        }
        tok[t] = gr * 16 + r16 < c_nv ? o : nvalid;
      }
      if (WEIGHTED) {
#pragma unroll
        for (int t = 0; t < NV; ++t)
          wgt[t] = !c_xs && tok[t] < nvalid ? p.topw[tok[t]] : 1.f;
      }
      // the next item's index, fetched while this one runs.  The address goes through a
      // register the compiler cannot prove uniform, or the atomic becomes a wave reduction
      // that waits for its result at once.
      int fetched = 0;
      if (tid == 0) {
        int z;
        asm volatile("v_mov_b32 %0, 0" : "=v"(z));
        fetched = __hip_atomic_fetch_add(deal + xcd * 16 + z, 1, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
      }

      floatx4_t acc[8][NV];
#pragma unroll
      for (int f = 0; f < 8; ++f)
#pragma unroll
        for (int t = 0; t < NV; ++t) acc[f][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
      uint4 fw[2][8], fa[2][NV];  // fragments of two stages

      const uint32_t rw = rd_lane + (uint32_t)(wn * 8 * 1024);
      const uint32_t ra = rd_lane + kRowsBytes + (uint32_t)(wm * NV * 1024);
      uint32_t rdo = 0;  // ring offset of the stage being read
      auto read = [&](auto q_tag, const char* bw, const char* ba, uint4 (&dw)[8], uint4 (&da)[NV]) GLM52_INLINE {
        constexpr int q = decltype(q_tag)::value;
        if constexpr (q == 0) dw[0] = *reinterpret_cast<const uint4*>(bw);
        else if constexpr (q <= NV) da[q - 1] = *reinterpret_cast<const uint4*>(ba + (q - 1) * 1024);
        else dw[q - NV] = *reinterpret_cast<const uint4*>(bw + (q - NV) * 1024);
      };

      auto stage = [&](auto par_tag) GLM52_INLINE {
        constexpr int PAR = decltype(par_tag)::value;
        constexpr int NA = PAR == kPA ? AN : 0;
        constexpr int NW = PACKED || PAR == kPA ? WN : 0;
        // this wave's reads of the stage are done (its buffer is refilled below) and its
        // loads of the next stage have landed, for every wave
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(later(PAR == 1)) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" : : : "memory");
        rdo = next(rdo);
        const char* const bw = ring_c + rdo + rw;
        const char* const ba = ring_c + rdo + ra;
        if constexpr (NA > 0) a_begin();
        if constexpr (NW > 0) w_begin();
        __builtin_amdgcn_sched_barrier(0);
        static_for<NMF>([&](auto m_tag) GLM52_INLINE {
          constexpr int m = decltype(m_tag)::value;
          constexpr int f = m / NV, t = m % NV;
          acc[f][t] = mfma16(fw[PAR][f], fa[PAR][t], acc[f][t]);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (m % RS == 0 && m / RS < NRD) {
            read(std::integral_constant<int, m / RS>{}, bw, ba, fw[1 - PAR], fa[1 - PAR]);
            __builtin_amdgcn_sched_barrier(0);
          }
          static_for<NA + NW>([&](auto o_tag) GLM52_INLINE {
            constexpr int o = decltype(o_tag)::value;
            if constexpr ((o * NMF) / (NA + NW) + (NA + NW <= NMF / 2) == m) {
              if constexpr (o < NA) a_one(o);
              else w_one(nt, o - NA);
              __builtin_amdgcn_sched_barrier(0);
            }
          });
        });
      };

      // stage 0 landed (the prologue's younger loads may be in flight), for every wave
      GLM52_WAIT_VMCNT(kLater0);
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
      static_for<NRD>([&](auto q) GLM52_INLINE { read(q, ring_c + rw, ring_c + ra, fw[0], fa[0]); });
#pragma unroll 1
      for (int kt = 0; kt < nk; kt += 2) {  // nk is even (the launcher checks K % 64)
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
      }

      // the ring is free; the next item's index from wave 0, its first stages on their way
      drain_and_meet();
      if (tid == 0) *slot = fetched;
      __syncthreads();
      k = uniform(wg_xcd + *slot);
      __syncthreads();
      have = decode();
      if (have) prologue();

      // Lane (r, g) holds the outputs 16 (g % 2) + 4 (g / 2) + 0..3 and those + 8 of each 32-row
      // group of the wave's W rows, for token r; after the exchange with lane (r, g ^ 2) the
      // eight from 16 (g % 2) + 8 (g / 2): one 16-byte store.
      const int og = (g4 & 1) * 16 + (g4 >> 1) * 8;
      if constexpr (EPI == 0) {
#pragma unroll
        for (int t = 0; t < NV; ++t) {
          uint16_t* const crow =
              (c_xs ? p.Cx + (int64_t)tok[t] * p.scx : p.C + (int64_t)tok[t] * p.scm) + c_n0 +
              wn * (GATED ? 64 : 128) + og;
#pragma unroll
          for (int q = 0; q < (GATED ? 2 : 4); ++q) {
            float ev[4], ov[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              if (GATED) {
                ev[i] = silu_mul(acc[2 * q][t][i], acc[4 + 2 * q][t][i]);
                ov[i] = silu_mul(acc[2 * q + 1][t][i], acc[5 + 2 * q][t][i]);
              } else {
                ev[i] = WEIGHTED ? acc[2 * q][t][i] * wgt[t] : acc[2 * q][t][i];
                ov[i] = WEIGHTED ? acc[2 * q + 1][t][i] * wgt[t] : acc[2 * q + 1][t][i];
              }
            }
            uint32_t e0 = cvt_pk_bf16(ev[0], ev[1]), e1 = cvt_pk_bf16(ev[2], ev[3]);
            uint32_t o0 = cvt_pk_bf16(ov[0], ov[1]), o1 = cvt_pk_bf16(ov[2], ov[3]);
            swap_halves(e0, o0);
            swap_halves(e1, o1);
            if (tok[t] < nvalid)
              *reinterpret_cast<uint4*>(crow + q * 32) = make_uint4(e0, e1, o0, o1);
          }
        }
      } else {
        // the residual rows are all loaded before the first store: one round trip, not one
        // per 16 bytes
        uint4 res[EPI == 1 || EPI == 2 ? NV : 1][4];
        if constexpr (EPI == 1 || EPI == 2) {
#pragma unroll
          for (int t = 0; t < NV; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              res[t][q] = make_uint4(0, 0, 0, 0);
              if (p.R && tok[t] < nvalid)
                res[t][q] = *reinterpret_cast<const uint4*>(p.R + (int64_t)tok[t] * p.srm + c_n0 +
                                                            wn * 128 + q * 32 + og);
            }
        }
#pragma unroll
        for (int t = 0; t < NV; ++t) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int col = c_n0 + wn * 128 + q * 32 + og;
            float v[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              v[i] = WEIGHTED ? acc[2 * q][t][i] * wgt[t] : acc[2 * q][t][i];
              v[4 + i] = WEIGHTED ? acc[2 * q + 1][t][i] * wgt[t] : acc[2 * q + 1][t][i];
              swap_halves(v[i], v[4 + i]);
            }
            if (tok[t] >= nvalid) continue;
            if constexpr (EPI == 1 || EPI == 2) {
              if (p.R) {
                float rf[8];
                unpack8(res[t][q], rf);
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = v[i] + rf[i];
              }
            }
            if constexpr (EPI == 2 || EPI == 3) {
              float4* const dst = reinterpret_cast<float4*>(p.C32 + (int64_t)tok[t] * p.scm + col);
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                float4 o = make_float4(v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]);
                if constexpr (EPI == 2) {
                  const float4 c = dst[h];
                  o = make_float4(c.x + o.x, c.y + o.y, c.z + o.z, c.w + o.w);
                }
                dst[h] = o;
              }
            } else if constexpr (EPI == 4) {
              uint16_t* const dst = p.C + (int64_t)(tok[t] / p.merge_topk) * p.scm + col;
#pragma unroll
              for (int h = 0; h < 4; ++h) atomic_add_bf16x2(dst + 2 * h, v[2 * h], v[2 * h + 1]);
            } else {
              *reinterpret_cast<uint4*>(p.C + (int64_t)tok[t] * p.scm + col) =
                  make_uint4(cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]),
                             cvt_pk_bf16(v[4], v[5]), cvt_pk_bf16(v[6], v[7]));
            }
          }
        }
      }
    };
    // An instance per 16-token group count, or per even one: a part-filled block then
    // multiplies up to 32 token rows of padding more.  Every count at 256 tokens with a bf16
    // store (the expert GEMMs, and o_proj without residual or K slices), where the matrix cores
    // and the power limit weigh most (T = 8192 block 6148 -> 6074 us).  With the odd counts the
    // 64- and 128-token tiles, which wait for their weights, and the other epilogues lose (T =
    // 1333 block 3222 -> 3313 us, o_proj at M = 256 131 -> 167 us, at M = 8192 1305 -> 1344).
    // o_proj's K slices at 256 rows have two instances only, 2 and 8: a tile's items all run at
    // once there, so a shorter last block ends no sooner, and its pace parts from that of the
    // block it shares W with (K = 32768: M = 400 226 -> 219 us, M = 256 139 -> 135; M = 300 216.5
    // -> 222; K = 16384: M = 700 202 -> 189).
    const int nvg = (c_nv + 16 * kWaveM - 1) / (16 * kWaveM);  // 16-token groups per wave
    auto pick = [&](auto nt) GLM52_INLINE {
      constexpr int MAXV = MT / (16 * kWaveM);
      if constexpr (MT == 256 && EPI == 0) {
        bool done = false;
        static_for<MAXV - 2>([&](auto v) GLM52_INLINE {  // the least of 2 .. MAXV that holds nvg
          constexpr int NV = decltype(v)::value + 2;
          if (!done && nvg <= NV) {
            run(std::integral_constant<int, NV>{}, nt);
            done = true;
          }
        });
        if (!done) run(std::integral_constant<int, MAXV>{}, nt);
      } else if (MAXV == 2 || nvg <= 2) run(std::integral_constant<int, 2>{}, nt);
      else if constexpr (MAXV == 8 && EPI == 3) run(std::integral_constant<int, MAXV>{}, nt);
      else if (MAXV == 4 || nvg <= 4) run(std::integral_constant<int, MAXV < 4 ? 2 : 4>{}, nt);
      else if constexpr (MAXV == 8) {
        if (nvg <= 6) run(std::integral_constant<int, 6>{}, nt);
        else run(std::integral_constant<int, 8>{}, nt);
      }
    };
    if (w_once) pick(std::true_type{});
    else pick(std::false_type{});
  }

  if (p.wg_trace && tid == 0) {  // start, end, items, XCD (hardware register XCC_ID)
    unsigned long long* rec = p.wg_trace + (int64_t)blockIdx.x * 4;
    rec[0] = t_start;
    rec[1] = __builtin_amdgcn_s_memrealtime();
    rec[2] = (unsigned long long)n_run;
    rec[3] = (unsigned long long)(__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15);
  }
  // the last workgroup out clears the set for the next launch that uses it
  if (tid == 0 && __hip_atomic_fetch_add(deal + 128, 1, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1) {
    for (int x = 0; x < 8; ++x)
      __hip_atomic_store(deal + x * 16, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(deal + 128, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <int MT, int NT, bool GATED, bool WEIGHTED, bool PACKED, int EPI>
int launch_tile_mt(const GemmArgs& a_in, int capacity, hipStream_t st) {
  GemmArgs a = a_in;
  a.deal_set = take_deal_set(st);
  a.wg_trace = item_trace();
  const int x_blocks = PACKED && a.Wx && a.x_rows > 0 ? (a.x_rows + MT - 1) / MT : 0;
  const int items_max = (capacity / MT + x_blocks) * (a.n_out / (GATED ? NT / 2 : NT));
  int grid = items_max < 256 ? items_max : 256;
  grid = ((grid + 7) / 8) * 8;
  moe_gemm_tile_kernel<MT, NT, GATED, WEIGHTED, PACKED, EPI><<<grid, 256, 0, st>>>(a);
  GLM52_RETURN_LAUNCH();
}

// W rows per tile: 512 (four waves along W) for the packed expert GEMMs at 64 and 128 tokens,
// which are weight streams: the token rows are staged half as often (T = 3000 block 3776 ->
// 3663 us).  256 elsewhere: in place the smaller stage leaves room for a deeper ring, and
// o_proj has the more items for its few row blocks (M = 64 85 -> 75 us).
template <int MT, bool GATED, bool WEIGHTED, bool PACKED, int EPI>
int launch_tile_as(const GemmArgs& a, int capacity, hipStream_t st) {
  constexpr int NT = MT <= 128 && PACKED && (EPI == 0 || EPI == 4) ? 512 : 256;
  return launch_tile_mt<MT, NT, GATED, WEIGHTED, PACKED, EPI>(a, capacity, st);
}

template <int MT, bool GATED, bool WEIGHTED, int EPI>
int launch_tile_w(const GemmArgs& a, int capacity, hipStream_t st) {
  return a.Wp ? launch_tile_as<MT, GATED, WEIGHTED, true, EPI>(a, capacity, st)
              : launch_tile_as<MT, GATED, WEIGHTED, false, EPI>(a, capacity, st);
}

}  // namespace

template <int MT>
int launch_tile_gated(const GemmArgs& a, int capacity, bool weighted, hipStream_t st) {
  return weighted ? launch_tile_w<MT, true, true, 0>(a, capacity, st)
                  : launch_tile_w<MT, true, false, 0>(a, capacity, st);
}
template <int MT>
int launch_tile_plain(const GemmArgs& a, int capacity, bool weighted, hipStream_t st) {
  return weighted ? launch_tile_w<MT, false, true, 0>(a, capacity, st)
                  : launch_tile_w<MT, false, false, 0>(a, capacity, st);
}
// o_proj's epilogues (packed B only) and the atomic expert merge (weighted w2 only)
template <int MT>
int launch_tile_epi(const GemmArgs& a, int capacity, bool weighted, hipStream_t st) {
  if (a.merge_topk > 0) {
    if (!weighted || a.epi != 0) return GLM52_EUNSUPPORTED;
    return launch_tile_w<MT, false, true, 4>(a, capacity, st);
  }
  if (weighted || !a.Wp) return GLM52_EUNSUPPORTED;
  if (a.epi == 1) return launch_tile_as<MT, false, false, true, 1>(a, capacity, st);
  if (a.epi == 2) return launch_tile_as<MT, false, false, true, 2>(a, capacity, st);
  return launch_tile_as<MT, false, false, true, 3>(a, capacity, st);
}
}  // namespace glm52
