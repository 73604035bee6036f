// Large-M q4 linear for gfx950: per-op calls of more than 32 rows and forwards of more than
// 64 (Dream's
// full canvas, BD3 prefix commits). At these sizes the contraction is MFMA
// bound, so the weights are dequantized once per work-group into fp16 MFMA
// operands (w = s * q + b, one fp16 rounding; backends/mlx_ops.py:97-130 for the
// linear, :43-60 for the MLX q4 g64 packing) instead of the per-group scaled
// accumulators of the weight-streaming kernels, whose two FMAs per output and
// group would cost as much VALU time as the MFMAs.
//
// A work-group of 4 waves (WVM x WVN) owns 128 rows x 256 columns (1 x 4 waves of
// 128 x 64) or 128 x 128 (2 x 2 of 64 x 64); two work-groups per CU hide each other's
// waits.
//   A (the ACT_F16P activation: hi and lo planes of [M][K]) is streamed per
//     64-k group straight into LDS (buffer loads to LDS, no registers held),
//     double buffered: 2 planes x 128 rows x 128 B per group. Rows are stored
//     unpadded with the 16-byte chunks of row r permuted (chunk c at position
//     c ^ (r & 7) ^ ((r >> 3) & 1)), so the MFMA fragment reads of 8 consecutive
//     rows hit 8 different 16-byte bank groups of a 128-byte row, and those of
//     16 consecutive rows 16 different ones of two rows (256 bytes): no bank
//     conflict whether the LDS serves 8 or 16 lanes of a 16-byte read per
//     cycle. Each MFMA step multiplies hi and lo by the same B. The two buffers
//     are separate arrays, so the compiler can tell the one being read from the
//     one being filled and waits for no load in flight.
//   B (q4 tile layout: per 32-column n-tile and 64-k group, 1 KiB of words and
//     32 scale|bias pairs) goes straight from global memory to registers and is
//     dequantized there, one k step at a time.
// k step t + 1's fragments are read, and its B dequantized a nibble pair at a time,
// between step t's MFMAs; so are the loads of group g + 2 issued, between the MFMAs of
// group g's last step, once group g + 1 is proven in LDS (in one batch ahead of the
// MFMAs the loads and the VALU work held the wave's MFMAs up).
// Split-K over blockIdx.z (KS slices) writes fp32 partial slices y + ks * M * N
// that a reduce pass sums (residual_norm_kernel).
// Split last round (tail.kt >= 2, one-dimensional grid): when the tiles fill the
// device's work-group slots (two per CU) a whole number of times with some left over,
// the first tail.full tiles run whole and each of the remaining ones is split into
// tail.kt K ranges on as many work-groups of one XCD, so the last round takes a
// fraction of a tile instead of leaving most CUs idle. The slices meet as in the
// split-K decode linears: each writes its partial tile, counts its arrival in that
// XCD's L2, and the last to arrive adds the slices in slice order and runs the epilogue.
// Epilogues run on 32-row pieces of the tile staged through LDS:
//   EPI_STORE : y (+ bias on slice 0)
//   EPI_SWIGLU: [gate 64 | up 64] column blocks -> silu(g) * u -> ACT_F16P
//   EPI_QKV   : (+ bias), q/k RMSNorm, RoPE, Q out / K,V into the tiled cache
//   EPI_LMSTAT: the LM head's softmax statistics per (row, 64-column block),
//               the logits themselves only on request
#include "fused.h"
#include "gemm_core.h"
#include "launch.h"

#include "linear_dev.h"
#include "lmstat.h"

namespace {

constexpr int BG_WM = 128;                        // rows per work-group
constexpr int BG_PLANE_BYTES = BG_WM * 128;       // one plane of one group: 128 rows x 64 halves
constexpr int BG_BUF_BYTES = 2 * BG_PLANE_BYTES;  // hi + lo planes of one group
// column of element c of row r in an epilogue piece (float4s permuted by row, so that
// reads down a column and along a row both hit distinct banks)
DRT_DEV int bg_col(int r, int c) { return c ^ ((r & 31) << 2); }
// s_waitcnt: no vector load and no LDS read in flight
constexpr int BG_WAIT = 0x0070;

typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// Nibble pair e of word wt of a k step (the lane's word t of the group holds the 8 k of
// step t in the ACT_F16P order (0,4,1,5,2,6,3,7)) as fp16 weights s * q + z: (1024 + q)
// halves by bit placement, then q * s + z in one fma.
DRT_DEV uint32_t dequant_q4_pair(uint32_t wt, int e, h2v s2, h2v z2, uint32_t mask) {
  const h2v k2 = {(_Float16)-1024.f, (_Float16)-1024.f};
  const h2v h = __builtin_bit_cast(h2v, ((wt >> (4 * e)) & mask) | 0x64006400u);
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(h + k2, s2, z2));
}

}  // namespace

struct BgTail {
  int full = 0;            // whole tiles (the first work-groups, dealt in XCD runs)
  int rest = 0;            // remaining tiles
  int kt = 0;              // K slices per remaining tile (0: the three-dimensional grid)
  float* part = nullptr;   // [remaining tiles][kt][rows * columns of a tile] partial tiles
  int* count = nullptr;    // [remaining tiles] arrival counters, zero on entry and exit
};
using drt::BG_TAIL_KT_MAX;

template <int EPI, int TM, int TN, int WVM, int WVN>
DRT_DEV void big_q4_tile(const FusedArgs& a, int KS, const BgTail& tail) {
  constexpr int BN = 32 * TN * WVN;
  static_assert(WVM * WVN == 4 && 32 * TM * WVM == BG_WM && TN == 2, "four waves over 128 rows");
  static_assert(WVM * 32 * BN * 4 == BG_BUF_BYTES, "an epilogue piece fills a buffer");
  __shared__ __align__(1024) char buf0[BG_BUF_BYTES];
  __shared__ __align__(1024) char buf1[BG_BUF_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: LDS bases in SGPRs
  const int wm = wave / WVN, wn = wave % WVN;
  const int M = a.M, N = a.N, K = a.K, G = K >> 6;
  // Tiles t = y + MT (x + NX z) (row tile y fastest), dealt to the XCDs in
  // contiguous runs: work-group b runs on XCD b % 8 and takes tile
  // (b % 8) * T8 / 8 + b / 8 (the last T - T8 tiles as they come), so an XCD's
  // L2 holds whole columns of row tiles: each weight tile is fetched by one XCD,
  // and a K slice of a split-K grid whose tiles fill an XCD's run stays on it.
  const int MT = (M + BG_WM - 1) / BG_WM, NX = (N + BN - 1) / BN;
  auto xcd_run = [](int b, int T) {
    const int T8 = T & ~7;
    return b < T8 ? (b & 7) * (T8 >> 3) + (b >> 3) : b;
  };
  int tile_x, tile_y, ks, tail_idx = -1;
  {
    const int T = (int)(gridDim.x * gridDim.y * gridDim.z);
    const int t = xcd_run((int)(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)), T);
    tile_y = t % MT;
    tile_x = (t / MT) % NX;
    ks = t / (MT * NX);
  }
  constexpr bool TAIL = EPI == EPI_SWIGLU || EPI == EPI_STORE;
  if (TAIL && tail.kt) {
    // work-group b: tile b (the first full tiles in XCD runs), or K slice of a
    // remaining tile; the slices of one remaining tile share b % 8, i.e. one
    // XCD (full % 8 == 0)
    const int b = blockIdx.x;
    int t = xcd_run(b, tail.full);
    ks = 0;
    KS = 1;
    if (b >= tail.full) {
      const int j = b - tail.full, q = j >> 3;
      tail_idx = (j & 7) + 8 * (q / tail.kt);
      ks = q % tail.kt;
      KS = tail.kt;
      t = tail.full + tail_idx;
      // the slices meet through this XCD's L2: a work-group found elsewhere
      // raises the placement error (the host then fails the forward)
      if (threadIdx.x == 0 && a.placement_err) {
        const int xcc = (int)(__builtin_amdgcn_s_getreg((31 << 11) | 20) & 0xf);  // HW_REG_XCC_ID
        const int r = drt::xcd_rotation(xcc, b, 8);
        if (r != a.placement_err[1])
          __hip_atomic_fetch_or(a.placement_err, 1 | drt::placement_bit(r), __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
      }
      if (tail_idx >= tail.rest) return;  // padding of the last eight tiles
    }
    tile_y = t % MT;
    tile_x = t / MT;
  }
  const int n0 = tile_x * BN, m0 = tile_y * BG_WM;
  const int g_lo = (int)((int64_t)G * ks / KS), g_hi = (int)((int64_t)G * (ks + 1) / KS);
  const int n_g = g_hi - g_lo;
  const int NT = N >> 5;
  // this wave's two n-tiles, clamped so that loads stay in bounds (columns
  // beyond N are computed from the last n-tile and never stored)
  const int nt0 = min((n0 >> 5) + TN * wn, NT - 1);
  const int nt1 = min((n0 >> 5) + TN * wn + 1, NT - 1);

  // A of a group: plane pl, 8-row block blk = wave + 4 i is one wave instruction
  // (lane l: row blk * 8 + (l >> 3), LDS position l & 7, which holds the row's chunk
  // (l & 7) ^ (l >> 3) ^ (blk & 1), blk & 1 being wave & 1), from a buffer per plane
  // that ends with row M - 1: rows past it read zeros.
  const uint32_t K2 = (uint32_t)K * 2u;
  const uint32_t rows_bytes = (uint32_t)min(BG_WM, M - m0) * K2;
  const char* act = (const char*)a.act + (size_t)m0 * K2;
  const __amdgpu_buffer_rsrc_t hi_buf =
      __builtin_amdgcn_make_buffer_rsrc((void*)act, 0, rows_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t lo_buf =
      __builtin_amdgcn_make_buffer_rsrc((void*)(act + (size_t)M * K2), 0, rows_bytes, 0x00020000);
  const uint32_t a_off = (uint32_t)(wave * 8 + (lane >> 3)) * K2 +
                         (uint32_t)(((lane & 7) ^ (lane >> 3) ^ (wave & 1)) * 16);
  // load d (0 .. 7: block d & 3 of plane d >> 2) of group gi (past the last one out of
  // the buffer's range: zeros without a memory access, and no branch between the MFMAs)
  auto issue_a = [&](int gi, char* dst, int d) {
    const int i = d & 3, pl = d >> 2;
    const uint32_t past = gi < n_g ? 0u : 0x80000000u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        pl ? lo_buf : hi_buf,
        (__attribute__((address_space(3))) void*)(dst + pl * BG_PLANE_BYTES + (wave + 4 * i) * 1024),
        16, a_off + ((uint32_t)(32 * i) * K2 + past), (g_lo + min(gi, n_g - 1)) * 128, 0, 0);
  };
  u32x4 wq[2][TN];
  uint32_t wsb[2][TN];
  auto issue_b = [&](int gi, int slot) {
    const int g = g_lo + min(gi, n_g - 1);
    wq[slot][0] = *q4_tile_words(a.qw, nt0, G, g, lane);
    wq[slot][1] = *q4_tile_words(a.qw, nt1, G, g, lane);
    wsb[slot][0] = q4_tile_sb(a.sb, nt0, G, g, lane);
    wsb[slot][1] = q4_tile_sb(a.sb, nt1, G, g, lane);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  // one k step's operands (A hi and lo fragments, the dequantised B fragments); steps
  // alternate between two sets
  struct Ops {
    f16x8 h[TM], l[TM];
    u32x4 b[TN];
  };
  uint32_t nib_mask = 0x000F000Fu;
  asm volatile("" : "+v"(nib_mask));  // in a register: v_and_or_b32 takes one constant
  h2v gs2[TN], gz2[TN];               // the current group's scale and bias pairs
  auto group_scales = [&](int slot) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const _Float16 sc = (_Float16)bf16_bits_to_float(wsb[slot][j] & 0xffffu);
      const _Float16 zb = (_Float16)bf16_bits_to_float(wsb[slot][j] >> 16);
      gs2[j] = h2v{sc, sc};
      gz2[j] = h2v{zb, zb};
    }
  };
  // this lane's fragment row within each 32-row m-tile is lane & 31; its k chunk at
  // step t is 4 * (lane >> 5) + t
  const uint32_t a_row = (uint32_t)(wm * TM * 4096 + (lane & 31) * 128);
  const uint32_t a_swz = (uint32_t)((lane & 7) ^ ((lane >> 3) & 1));
  auto load_h = [&](Ops& o, const char* src, int t) {
    const char* p = src + a_row + (((uint32_t)(4 * (lane >> 5) + t) ^ a_swz) * 16);
#pragma unroll
    for (int i = 0; i < TM; ++i) o.h[i] = *(const f16x8*)(p + i * 4096);
  };
  auto load_l = [&](Ops& o, const char* src, int t) {
    const char* p = src + a_row + (((uint32_t)(4 * (lane >> 5) + t) ^ a_swz) * 16);
#pragma unroll
    for (int i = 0; i < TM; ++i) o.l[i] = *(const f16x8*)(p + BG_PLANE_BYTES + i * 4096);
  };
  Ops X, Y;
#pragma unroll
  for (int d = 0; d < 8; ++d) issue_a(0, buf0, d);
  issue_b(0, 0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int d = 0; d < 8; ++d) issue_a(1, buf1, d);
  issue_b(1, 1);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70 | (8 + 2 * TN));  // group 0 has arrived
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  group_scales(0);
  load_h(X, buf0, 0);
  load_l(X, buf0, 0);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) X.b[j][e] = dequant_q4_pair(wq[0][j][0], e, gs2[j], gz2[j], nib_mask);
  // k step t of group gi (in `here`, B slot S = gi & 1) on `cur`, the next step's
  // operands into `nxt`; at the last step, once group gi + 1 is in LDS in every wave and
  // this wave's reads of `here` are done, group gi + 2 goes into `here` and slot S (past
  // the last group the operands read are unused)
  auto kstep = [&](Ops& cur, Ops& nxt, int gi, int t, auto slot, char* here, char* there) {
    constexpr int S = decltype(slot)::value, SN = 2 * TM;  // MFMA rows: hi, then lo
    if (t < 3) {
      load_h(nxt, here, t + 1);
    } else {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(BG_WAIT);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load_h(nxt, there, 0);
      group_scales(S ^ 1);
      if (gi + 2 < n_g) issue_b(gi + 2, S);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < SN; ++s) {
      const int i = s % TM;
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = mfma_f16(s < TM ? cur.h[i] : cur.l[i], __builtin_bit_cast(f16x8, cur.b[j]), acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      // (the lo fragments once the current hi ones are spent: 16 registers fewer)
      if (s == TM - 1) load_l(nxt, t < 3 ? here : there, (t + 1) & 3);
#pragma unroll
      for (int q = 0; q < 4 * TN / SN; ++q) {
        const int p = s * (4 * TN / SN) + q, j = p >> 2, e = p & 3;
        nxt.b[j][e] = dequant_q4_pair(t < 3 ? wq[S][j][t < 3 ? t + 1 : 0] : wq[S ^ 1][j][0], e, gs2[j],
                                      gz2[j], nib_mask);
      }
      if (t == 3) {
#pragma unroll
        for (int q = 0; q < 8 / SN; ++q) issue_a(gi + 2, here, s * (8 / SN) + q);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto group = [&](int gi, auto slot, char* here, char* there) {
    kstep(X, Y, gi, 0, slot, here, there);
    kstep(Y, X, gi, 1, slot, here, there);
    kstep(X, Y, gi, 2, slot, here, there);
    kstep(Y, X, gi, 3, slot, here, there);
  };
  int g = 0;
  for (; g + 1 < n_g; g += 2) {
    group(g, std::integral_constant<int, 0>{}, buf0, buf1);
    group(g + 1, std::integral_constant<int, 1>{}, buf1, buf0);
  }
  if (g < n_g) group(g, std::integral_constant<int, 0>{}, buf0, buf1);
  __builtin_amdgcn_s_waitcnt(BG_WAIT);  // the epilogue reuses the buffers
  // (the thread index made opaque: the epilogue's addresses are not computed ahead of
  // the main loop and kept, or spilled, across it)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));

  if (TAIL && tail_idx >= 0) {
    // a K slice of a remaining tile: store it as 16-byte chunks (chunk c = four
    // consecutive accumulators of thread t at (c * 256 + t) * 4), and let the
    // last slice to arrive add them all in slice order, two chunks of every
    // slice in flight at a time
    constexpr int TILE = BG_WM * BN;
    float* pt = tail.part + (size_t)tail_idx * tail.kt * TILE;
    f32x4* mine = (f32x4*)(pt + (size_t)ks * TILE) + tid;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          mine[((i * TN + j) * 4 + q) * 256] =
              f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    __shared__ int last_flag;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // every store of the work-group is in this XCD's L2
    if (tid == 0)
      last_flag = __hip_atomic_fetch_add(&tail.count[tail_idx], 1, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP) == tail.kt - 1;
    __syncthreads();
    if (!last_flag) return;
    const f32x4* pv = (const f32x4*)pt + tid;
#pragma unroll
    for (int c0 = 0; c0 < 4 * TM * TN; c0 += 2) {
      f32x4 v[2][BG_TAIL_KT_MAX];
#pragma unroll
      for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int k = 0; k < BG_TAIL_KT_MAX; ++k)  // every slice's chunk loaded first
          v[cc][k] = pv[(size_t)min(k, tail.kt - 1) * (TILE / 4) + (c0 + cc) * 256];
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        const int c = c0 + cc, i = c / (4 * TN), j = (c >> 2) % TN, q = c & 3;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float sum = 0.f;
#pragma unroll
          for (int k = 0; k < BG_TAIL_KT_MAX; ++k)
            if (k < tail.kt) sum += k == ks ? acc[i][j][4 * q + e] : v[cc][k][e];
          acc[i][j][4 * q + e] = sum;
        }
      }
    }
    if (tid == 0) tail.count[tail_idx] = 0;
    ks = 0;
  }

  // Epilogue through LDS in pieces: MFMA row tile p of every wave, 32 rows per wave row.
  float* e = (float*)buf0;  // [32 * WVM][BN]
  uint16_t* vbuf = (uint16_t*)buf1;
  const int row0 = a.desc ? a.desc->row0 : 0;
#pragma unroll
  for (int p = 0; p < TM; ++p) {
    if (m0 + 32 * p >= M) break;  // uniform
    __syncthreads();  // the last fragment reads, then the previous piece's, are done
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rr = mfma_row(r, tid & 63);
        e[(wm * 32 + rr) * BN + bg_col(rr, (wn * TN + j) * 32 + (tid & 31))] = acc[p][j][r];
      }
    __syncthreads();
    auto row_of = [&](int rr) { return m0 + ((rr >> 5) * TM + p) * 32 + (rr & 31); };
    if (EPI == EPI_STORE) {
      float* y = a.y + (int64_t)ks * M * N;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int c = tid + 256 * i;
        const int rr = c / (BN / 4), cc = c % (BN / 4) * 4, n = n0 + cc, m = row_of(rr);
        if (m < M && n < N) {
          f32x4 v = *(const f32x4*)(e + rr * BN + bg_col(rr, cc));
          if (a.bias && ks == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] += bf16_bits_to_float(a.bias[n + k]);
          }
          *(f32x4*)(y + (int64_t)m * N + n) = v;
        }
      }
    } else if (EPI == EPI_SWIGLU) {
      // output chunk q: block q >> 3 of [gate 64 | up 64], 8 outputs at (q & 7) * 8;
      // ACT_F16P hi plane, then the lo plane at + M * F
      const int F = N >> 1;
      bool over = false;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int c = tid + 256 * i;
        const int rr = c / (BN / 16), q = c % (BN / 16), blk = q >> 3, c8 = (q & 7) * 8;
        const int m = row_of(rr);
        if (m < M && n0 + blk * 128 < N) {
          const float* er = e + rr * BN;
          float gv[8], uv[8];
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            const f32x4 g4 = *(const f32x4*)(er + bg_col(rr, blk * 128 + c8 + 4 * hf));
            const f32x4 u4 = *(const f32x4*)(er + bg_col(rr, blk * 128 + 64 + c8 + 4 * hf));
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              gv[4 * hf + k] = g4[k];
              uv[4 * hf + k] = u4[k];
            }
          }
          _Float16 h[8], lo[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float y = gv[k] * (1.f / (1.f + expf(-gv[k]))) * uv[k];
            const _Float16 hk = (_Float16)y;
            h[f16p_index(k)] = hk;
            lo[f16p_index(k)] = f16_lo(y, hk);
            over = over || f16_overflows(y);
          }
          _Float16* dst = (_Float16*)a.act_out + (int64_t)m * F + (n0 >> 1) + blk * 64 + c8;
          *(u32x4*)dst = __builtin_bit_cast(u32x4, h);
          *(u32x4*)(dst + (int64_t)M * F) = __builtin_bit_cast(u32x4, lo);
        }
      }
      if (over) raise_range(a);
    } else if (EPI == EPI_LMSTAT) {
      // lane: row lane & 31 of its wave's piece, the 32 columns half of its wave's 64
      const int r = tid & 31, half = (tid >> 5) & 1;
      const int col0 = n0 + wn * 64 + half * 32, row = m0 + (wm * TM + p) * 32 + r;
      const bool valid = row < M && n0 + wn * 64 < N;  // (N % 64 == 0)
      const float temperature = a.desc ? a.desc->temperature : a.lm_temp;
      const uint64_t seed = a.desc ? a.desc->seed : a.lm_seed;
      const int step = a.desc ? a.desc->step : a.lm_step;
      const int excl = a.desc ? a.desc->exclude_col : a.lm_excl;
      float v[32];
      const float* src = e + (wm * 32 + r) * BN;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const f32x4 t4 = *(const f32x4*)(src + bg_col(r, wn * 64 + half * 32 + 4 * q));
#pragma unroll
        for (int k = 0; k < 4; ++k) v[4 * q + k] = t4[k];
      }
      if (a.lm_logits && valid) {
        f32x4* lp = (f32x4*)(a.lm_logits + (int64_t)row * N + col0);
#pragma unroll
        for (int q = 0; q < 8; ++q) lp[q] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
#pragma unroll
      for (int c = 0; c < 32; ++c) v[c] = col0 + c == excl ? -INFINITY : v[c];
      const bool samp = temperature > 0.f && row < M;
      const uint64_t rk = samp ? sampling_row_key(seed, step, a.lm_pos[row]) : 0ull;
      const LmRun32 mine = lm_run32(v, col0, samp, temperature, rk);
      LmRun32 other;
      other.mx = __shfl_xor(mine.mx, 32, 64);
      other.arg = __shfl_xor(mine.arg, 32, 64);
      other.se = __shfl_xor(mine.se, 32, 64);
      other.skey = __shfl_xor(mine.skey, 32, 64);
      other.sarg = __shfl_xor(mine.sarg, 32, 64);
      other.sl = __shfl_xor(mine.sl, 32, 64);
      if (half == 0 && valid)
        ((LmStat*)a.lm_stats)[(int64_t)row * (N >> 6) + (n0 >> 6) + wn] = lm_join64(mine, other);
    } else if (EPI == EPI_QKV) {
#pragma unroll
      for (int w = 0; w < WVM; ++w) {
        const int mp = m0 + (w * TM + p) * 32;
        if (mp >= M) break;  // uniform
        const int rows = min(32, M - mp);
#pragma unroll
        for (int hl = 0; hl < BN / 128; ++hl) {
          const int head = (n0 >> 7) + hl;
          if (head * 128 >= N) break;    // uniform
          if (w || hl) __syncthreads();  // the V tile buffer of the last head has been copied out
          auto get = [&](int m, int d) { return e[(w * 32 + m) * BN + bg_col(m, hl * 128 + d)]; };
          const QkvTables qt = qkv_tables(a, head, row0 + mp, rows);
          if (a.kv_bf16) qkv_epilogue<__bf16>(a, qt, head, mp, row0 + mp, rows, get, vbuf);
          else qkv_epilogue<_Float16>(a, qt, head, mp, row0 + mp, rows, get, vbuf);
        }
      }
    }
  }
}

// (the buffer resource type is not known to the host pass: the body is a device function)
template <int EPI, int TM, int TN, int WVM, int WVN>
__global__ __launch_bounds__(256, 2) void big_q4_kernel(const FusedArgs a, int KS, const BgTail tail) {
  big_q4_tile<EPI, TM, TN, WVM, WVN>(a, KS, tail);
}

// The QKV epilogue of a split-K q|k|v projection: work-group (head, 32-row
// block) sums the KS fp32 partial slices of its head's 128 columns (bias
// excluded, added by the epilogue) into LDS - every slice's loads issued before
// the first add - and runs the same per-head epilogue from there.
template <typename T>
__global__ __launch_bounds__(256) void big_qkv_epilogue_kernel(const FusedArgs a,
                                                               const float* __restrict__ part,
                                                               int KS) {
  __shared__ __align__(16) float tile[32][132];
  __shared__ __align__(16) uint16_t vbuf[4096];
  const int M = a.M, N = a.N;
  const int head = blockIdx.x, mp = blockIdx.y * 32;
  const int rows = min(32, M - mp);
  const int row0 = a.desc ? a.desc->row0 : 0;
  // 32 rows x 32 float4 per slice: thread t takes rows t >> 5 + 8j, float4 t & 31
  constexpr int KMAX = drt::BG_QKV_MAX_KS;
  const QkvTables qt = qkv_tables(a, head, row0 + mp, rows);
  f32x4 v[KMAX][4];
#pragma unroll
  for (int k = 0; k < KMAX; ++k)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = min((threadIdx.x >> 5) + 8 * j, rows - 1);
      v[k][j] = *(const f32x4*)(part + (int64_t)min(k, KS - 1) * M * N + (int64_t)(mp + m) * N +
                                head * 128 + (threadIdx.x & 31) * 4);
    }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 sum = v[0][j];
#pragma unroll
    for (int k = 1; k < KMAX; ++k)
      if (k < KS) sum += v[k][j];
    if (a.rnd_bf16) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = round_bf16(sum[e]);
    }
    *(f32x4*)&tile[(threadIdx.x >> 5) + 8 * j][(threadIdx.x & 31) * 4] = sum;
  }
  __syncthreads();
  auto get = [&](int m, int d) { return tile[m][d]; };
  qkv_epilogue<T>(a, qt, head, mp, row0 + mp, rows, get, vbuf);
}

// y = sum of the KS slices (slice order) + bias, 4 floats per thread, every slice's load
// issued before the first add (2 slices of 2048 x 3072, 75 MB: 12.6 -> 11.9 us, 2048 x 1024: 8.3 -> 5.4; always eight
// loads, the last slice's repeated, before).
template <int KS>
__global__ __launch_bounds__(256) void sum_slices_kernel(const float* __restrict__ part, int64_t n,
                                                         const uint16_t* __restrict__ bias, int N,
                                                         float* __restrict__ y, int rnd_bf16) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 v[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) v[k] = *(const f32x4*)(part + k * n + i);
  f32x4 sum = v[0];
#pragma unroll
  for (int k = 1; k < KS; ++k) sum += v[k];
  if (rnd_bf16) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[e] = round_bf16(sum[e]);
  }
  if (bias) {  // N % 4 == 0: the four columns are one row's
    const int c = (int)(i % N);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[e] += bf16_bits_to_float(bias[c + e]);
  }
  *(f32x4_e*)(y + i) = sum;
}

template __global__ void big_qkv_epilogue_kernel<_Float16>(const FusedArgs, const float*, int);
template __global__ void big_qkv_epilogue_kernel<__bf16>(const FusedArgs, const float*, int);

namespace drt {

// K slices the workspaces of a large-M q4 linear are sized for: enough work-groups for
// two per CU, at most max_ks and at least 6 groups of 64 k each.
int big_linear_splits(int M, int N, int K, int max_ks) {
  const int tiles = ((M + BG_WM - 1) / BG_WM) * ((N + 255) / 256);
  if (tiles >= 384) return 1;
  int ks = std::min(max_ks, std::max(1, 512 / tiles));
  ks = std::min(ks, std::max(1, (K / 64) / 6));
  return std::max(1, ks);
}

namespace {
// Estimated us of n work-groups of g groups of 64 k. Measured us per group for a few
// work-groups (the loads' latency), for one per CU, for a few CUs with two (the others
// wait for them) and for two on every CU: 128 x 256 tiles 1.22 / 1.70 / 2.55 / 3.35, 128 x
// 128 tiles 0.85 / 1.00 / 1.45 / 1.95; and about 4 us to start and store a round.
float bg_cost(bool wide, int n, float g, int n_cu) {
  const float few = wide ? 1.22f : 0.85f, one = wide ? 1.70f : 1.00f;
  const float over = wide ? 2.55f : 1.45f, two = wide ? 3.35f : 1.95f;
  const int rounds = n / (2 * n_cu), rest = n - rounds * 2 * n_cu;
  float us = rounds * (two * g + 4.f);
  if (rest > n_cu) us += (over + (two - over) * (rest - n_cu) / n_cu) * g + 4.f;
  else if (rest > 0) us += (few + (one - few) * rest / n_cu) * g + 4.f;
  return us;
}
}  // namespace

// The cheapest estimate over the two tiles and, for plain stores, the K slices (each at
// least four groups; reduce_us: what the reduce pass costs besides its bytes), and for
// unsplit stores and gate|up the split last round: the tiles past whole rounds of one
// or two work-groups per CU over at most one K slice per CU. part_floats bounds the
// slices and the split tiles' partials. Measured (hi + lo MFMA rates in brackets):
// 512 x 18944 x 3584, 296 wide tiles: 155 us as they are, 156 as 592 narrow ones, 119
// with the last 40 tiles in six slices (1165 TFLOP/s); 512 x 37888 x 3584: 294 and 232 (80
// tiles in three slices; 246 in six, the last slice's adding outweighing the shorter
// round); 41 x 18944 x 3584: 73 unsplit, 32 in three slices; 2048 x 1024 x 1024: 21 us in
// two slices of wide tiles (+ 5 to add them), 21 unsplit narrow.
BigQ4Plan big_q4_plan(int M, int N, int K, int kind, int max_ks, size_t part_floats,
                      float reduce_us, bool tail_ok) {
  const int n_cu = n_cu_of_current_device(), G = K / 64, MT = (M + BG_WM - 1) / BG_WM;
  BigQ4Plan best;
  float best_us = 1e30f;
  auto take = [&](float us, const BigQ4Plan& p) {
    if (us < best_us) {
      best_us = us;
      best = p;
    }
  };
  for (int w = 1; w >= 0; --w) {
    const bool wide = w == 1;
    const int bn = wide ? 256 : 128, T = MT * ((N + bn - 1) / bn);
    for (int ks = 1; ks <= max_ks; ++ks) {
      if (ks > 1 && (kind != FL_STORE || G / ks < 4 || (size_t)ks * M * N > part_floats)) break;
      float us = bg_cost(wide, T * ks, (float)((G + ks - 1) / ks), n_cu);
      if (ks > 1) us += reduce_us + (2 * ks + 1) * 0.5e-6f * M * N;  // 4 bytes each at 8 TB/s
      take(us, BigQ4Plan{wide, ks, 0, 0});
    }
    if (!tail_ok || (kind != FL_STORE && kind != FL_SWIGLU)) continue;
    for (int unit = 1; unit <= 2; ++unit) {
      const int full = T / (unit * n_cu) * (unit * n_cu), rest = T - full;
      if (rest == 0 || rest > BIG_TAIL_COUNTERS || full % 8) continue;
      const int kt = std::min({BG_TAIL_KT_MAX, n_cu / rest, G / 2});
      if (kt < 2 || (size_t)rest * kt * BG_WM * bn > part_floats) continue;
      const float whole = bg_cost(wide, full, (float)G, n_cu);
      // an odd round of one per CU leaves the slices the second slots
      const bool beside = full % (2 * n_cu) != 0;
      const float us = beside ? whole + bg_cost(wide, rest * kt, (float)G / kt, n_cu) * 0.2f + 5.f
                              : whole + bg_cost(wide, rest * kt, (float)G / kt, n_cu) + 4.f;
      take(us, BigQ4Plan{wide, 1, full, kt});
    }
  }
  return best;
}

// The plan that cuts a linear's sums along K by its shape alone: big_linear_splits slices,
// and with split_last the gate|up tiles past whole rounds of two per CU over the K slices that
// fill one more. The tile changes no sum: the cheaper one.
// For a canvas's forward, whose tokens are chosen from it directly: the estimates above, which
// cut more to the point there (512 x 37888 x 3584: 247 us, 279 here without split_last; a
// 512-token canvas 14.1 ms, 15.2 here), round the fp32 sums otherwise, and over 28 layers that
// moved the token of one row in a few thousand, whose two best logits were all but equal.
// For per-op calls that take slices: with fewer, or a split last round in their place, the
// fp32 chains are longer (error against 64 bits up to 1.7 times, 512 rows of 3584 x 18944
// 4.5e-7 and 6.3e-7), and the estimates miss by more than they gain (300 x 3584 x 3584: 55 us,
// 39 here; 700 x 3584 x 18944: 292 and 198; 2048 x 2048 x 1024: 31 and 37).
BigQ4Plan big_q4_shape_plan(int M, int N, int K, int kind, int max_ks, size_t part_floats,
                              bool split_last) {
  const int n_cu = n_cu_of_current_device(), G = K / 64, MT = (M + BG_WM - 1) / BG_WM;
  const int T = MT * ((N + 255) / 256), S = 2 * n_cu, full = T / S * S, rest = T - full;
  if (kind == FL_SWIGLU && split_last && full > 0 && rest > 0 && rest % 8 == 0 &&
      rest <= BIG_TAIL_COUNTERS) {
    const int kt = std::min({BG_TAIL_KT_MAX, S / rest, G});
    if (kt >= 2 && (size_t)rest * kt * BG_WM * 256 <= part_floats)
      return BigQ4Plan{true, 1, full, kt};
  }
  BigQ4Plan p;
  p.ks = kind == FL_STORE ? big_linear_splits(M, N, K, max_ks) : 1;
  const float g = (float)((G + p.ks - 1) / p.ks);
  p.wide = bg_cost(true, T * p.ks, g, n_cu) <=
           bg_cost(false, MT * ((N + 127) / 128) * p.ks, g, n_cu);
  return p;
}

bool big_linear_supported(const FusedArgs& a, int kind) {
  if (!a.qw || !a.sb || a.M <= 32 || a.N % 32 != 0 || a.K % 64 != 0) return false;
  if ((kind == FL_QKV || kind == FL_SWIGLU) && a.N % 128 != 0) return false;
  if (kind == FL_SWIGLU && a.act_fmt != ACT_F16P) return false;
  if (kind == FL_LMSTAT) return a.N % 64 == 0 && a.lm_stats != nullptr;
  return kind == FL_QKV || kind == FL_SWIGLU || kind == FL_STORE;
}

void big_linear(const FusedArgs& a, int kind, const BigQ4Plan& p, hipStream_t s, float* tail_part,
                int* tail_count) {
  require(big_linear_supported(a, kind), "large-M linear: unsupported shape or kind");
  const int KS = p.ks;
  const bool wide = p.wide;
  require(KS >= 1 && KS <= a.K / 64 && (KS == 1 || kind == FL_STORE),
          "large-M linear: split-K only for plain stores");
  const int bn = wide ? 256 : 128;
  dim3 grid((a.N + bn - 1) / bn, (a.M + BG_WM - 1) / BG_WM, KS);
  BgTail tail;
  if (p.kt > 0) {
    const int T = (int)(grid.x * grid.y);
    require(KS == 1 && (kind == FL_STORE || kind == FL_SWIGLU) && tail_part && tail_count &&
                !a.fenced && a.n_xcc == 8 && p.full % 8 == 0 && p.full < T && p.kt >= 2 &&
                p.kt <= BG_TAIL_KT_MAX && p.kt <= a.K / 64 && T - p.full <= BIG_TAIL_COUNTERS,
            "large-M linear: split last round");
    tail.full = p.full;
    tail.rest = T - p.full;
    tail.kt = p.kt;
    tail.part = tail_part;
    tail.count = tail_count;
    grid = dim3((unsigned)(p.full + (tail.rest + 7) / 8 * 8 * p.kt), 1, 1);
  }
  const double bytes = (double)a.N * a.K / 2 + (double)a.N * a.K / 16 + 2.0 * a.M * a.K +
                       (kind == FL_STORE ? 4.0 * KS : 2.0) * a.M * a.N;
#define DRT_BG(E)                                                                            \
  {                                                                                          \
    if (wide)                                                                                \
      DRT_LAUNCH(Profiler::GEMM, bytes, (big_q4_kernel<E, 4, 2, 1, 4>), grid, dim3(256), 0, s, \
                 a, KS, tail);                                                               \
    else                                                                                     \
      DRT_LAUNCH(Profiler::GEMM, bytes, (big_q4_kernel<E, 2, 2, 2, 2>), grid, dim3(256), 0, s, \
                 a, KS, tail);                                                               \
  }
  if (kind == FL_QKV) DRT_BG(EPI_QKV)
  else if (kind == FL_SWIGLU) DRT_BG(EPI_SWIGLU)
  else if (kind == FL_LMSTAT) DRT_BG(EPI_LMSTAT)
  else DRT_BG(EPI_STORE)
#undef DRT_BG
  DRT_HIP(hipGetLastError());
}

void sum_slices(const float* part, int KS, int64_t n, const uint16_t* bias, int N, float* y,
                hipStream_t s, bool rnd_bf16) {
  require(KS >= 1 && KS <= 8 && n % 4 == 0 && N % 4 == 0, "sum_slices: 1..8 slices of n % 4 == 0");
  const int64_t blocks = (n / 4 + 255) / 256;
#define DRT_SS(K)                                                                              \
  case K:                                                                                      \
    hipLaunchKernelGGL(sum_slices_kernel<K>, dim3((unsigned)blocks), dim3(256), 0, s, part, n, \
                       bias, N, y, (int)rnd_bf16);                                             \
    break;
  switch (KS) {
    DRT_SS(1) DRT_SS(2) DRT_SS(3) DRT_SS(4) DRT_SS(5) DRT_SS(6) DRT_SS(7)
    DRT_SS(8)
  }
#undef DRT_SS
  DRT_HIP(hipGetLastError());
}

void big_qkv(const FusedArgs& a, float* part, size_t part_floats, bool canvas, hipStream_t s) {
  // (the epilogue pass: its own launch and 6 us besides its bytes)
  const BigQ4Plan split =
      canvas ? big_q4_shape_plan(a.M, a.N, a.K, FL_STORE, BG_QKV_MAX_KS, 0, false)
             : big_q4_plan(a.M, a.N, a.K, FL_STORE, BG_QKV_MAX_KS, part ? part_floats : 0, 6.f, false);
  if (split.ks == 1 || !part || (size_t)split.ks * a.M * a.N > part_floats) {
    big_linear(a, FL_QKV, big_q4_plan(a.M, a.N, a.K, FL_QKV, 1, 0, 0.f, false), s);
    return;
  }
  FusedArgs g = a;
  g.bias = nullptr;  // the epilogue adds it
  g.y = part;
  big_linear(g, FL_STORE, split, s);
  qkv_epilogue_slices(a, part, split.ks, s);
}

void qkv_epilogue_slices(const FusedArgs& a, const float* part, int ks, hipStream_t s) {
  require(ks >= 1 && ks <= BG_QKV_MAX_KS && a.N % 128 == 0, "q|k|v epilogue: 1..8 slices");
  const dim3 grid(a.N / 128, (a.M + 31) / 32);
  if (a.kv_bf16)
    hipLaunchKernelGGL(big_qkv_epilogue_kernel<__bf16>, grid, dim3(256), 0, s, a, part, ks);
  else
    hipLaunchKernelGGL(big_qkv_epilogue_kernel<_Float16>, grid, dim3(256), 0, s, a, part, ks);
  DRT_HIP(hipGetLastError());
}

}  // namespace drt
