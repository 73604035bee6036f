// bf16-weight linear on shared operands for gfx950 (a model's forwards of more than 64 rows;
// per-op calls where no kernel for few rows is faster): y = bf16(x) @ W^T with fp32
// accumulation, rounded to bf16 like the reference's bf16 matmul output
// (backends/mlx_ops.py:122-125).
//
// At these sizes the contraction is MFMA bound, so both operands are shared
// through LDS: a work-group of WVM x WVN waves owns 32*TM*WVM rows x 32*TN*WVN
// columns, and every byte it loads feeds 128 or 256 rows / columns.
//   A (ACT_BF16, [M][K]) and B (the bf16 tile layout of bf16_linear.hip) are
//     loaded per 64-k stage straight into LDS (buffer loads to LDS), double buffered.
//     A rows (128 B per stage) are stored with the 16-byte chunks of row r permuted
//     (chunk c at position c ^ (r & 7) ^ ((r >> 3) & 1)): the MFMA fragment reads
//     of 8 or 16 consecutive rows hit distinct bank groups. B is already in
//     fragment order: every read is one contiguous KiB.
//   The two stage buffers are separate arrays, so the compiler can tell the one
//     being read from the one being filled and waits for no load in flight.
// k step t + 1's fragments are read while step t's MFMAs run; the stage after next
// is issued at the last step's barrier, a whole stage of MFMAs ahead of its use.
// Split-K (KS slices, the slowest index of the one-dimensional grid) writes fp32 partial
// slices y + ks * M * N that a reduce pass sums and rounds.
// Epilogues:
//   EPI_STORE : y = bf16(tile) (+ bias); slices of a split, or without rnd_bf16: the
//               fp32 sums
//   EPI_SWIGLU: [gate 64 | up 64] column blocks -> silu(g) * u -> ACT_BF16
//   EPI_QKV   : (+ bias), q/k RMSNorm, RoPE, Q out / K,V into the tiled cache
#include "fused.h"
#include "gemm_core.h"
#include "launch.h"

#include "linear_dev.h"

namespace {

// s_waitcnt immediate: at most n vector loads in flight (other counters free);
// masked, no LDS read in flight either
constexpr int vm_wait(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int VM_LDS_WAIT_MASK = 0xF0FF;

}  // namespace

// (a device function: the buffer resource type is not known to the host pass)
template <int EPI, int TM, int TN, int WVM, int WVN, int S>
DRT_DEV void big_bf16_tile(const FusedArgs& a, int KS, int col0, int NX) {
  constexpr int NW = WVM * WVN, BM = 32 * TM * WVM, BN = 32 * TN * WVN;
  constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128;  // one 64-k stage
  constexpr int A_LD = BM / 8 / NW, B_LD = BN / 8 / NW;  // 1 KiB loads per wave and stage
  static_assert(NW % 2 == 0 && BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "stage split over waves");
  // the stage buffers; an epilogue piece of wave row w lives in buffer w
  constexpr int ST_BYTES = A_BYTES + B_BYTES;
  __shared__ __align__(1024) char buf0[ST_BYTES];
  __shared__ __align__(1024) char buf1[ST_BYTES];
  __shared__ __align__(1024) char buf2[S > 2 ? ST_BYTES : 16];
  __shared__ __align__(1024) char buf3[S > 2 ? ST_BYTES : 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WVN, wn = wave % WVN;
  const int M = a.M, N = a.N, K = a.K, G = K >> 6;
  // Tiles t = y + MT (x + NX z) (row tile y fastest) dealt to the XCDs in
  // contiguous runs (work-group b runs on XCD b % 8): each weight tile is fetched
  // by one XCD's L2.
  const int MT = (M + BM - 1) / BM;
  int tile_x, tile_y, ks;
  {
    const int T = (int)gridDim.x, T8 = T & ~7, b = (int)blockIdx.x;
    const int t = b < T8 ? (b & 7) * (T8 >> 3) + (b >> 3) : b;
    tile_y = t % MT;
    tile_x = (t / MT) % NX;
    ks = t / (MT * NX);
  }
  const int n0 = col0 + tile_x * BN, m0 = tile_y * BM;
  const int g_lo = (int)((int64_t)G * ks / KS), g_hi = (int)((int64_t)G * (ks + 1) / KS);
  const int n_g = g_hi - g_lo;
  const int NT = N >> 5, KC = K >> 4;

  // Sources of this wave's loads, as buffers that end with the last valid row and
  // n-tile: rows past M and columns past N read zeros. A: 8-row block blk = wave +
  // NW * i, lane l row blk * 8 + (l >> 3), LDS position l & 7 holding chunk (l & 7) ^
  // (l >> 3) ^ (blk & 1) (blk & 1 == wave & 1). B: load i of this wave is KiB
  // wave * B_LD + i of the stage, k chunk & 3 of n-tile >> 2.
  const __amdgpu_buffer_rsrc_t a_buf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.act + (size_t)m0 * K * 2), 0,
      (uint32_t)min(BM, M - m0) * (uint32_t)(2 * K), 0x00020000);
  const __amdgpu_buffer_rsrc_t b_buf = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.wb + ((size_t)(n0 >> 5) * KC << 10)), 0,
      (uint32_t)min(BN / 32, NT - (n0 >> 5)) * ((uint32_t)KC << 10), 0x00020000);
  uint32_t a_off[A_LD], b_off[B_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i)
    a_off[i] = (uint32_t)((wave + NW * i) * 8 + (lane >> 3)) * (uint32_t)(2 * K) +
               (uint32_t)(((lane & 7) ^ (lane >> 3) ^ (wave & 1)) * 16);
#pragma unroll
  for (int i = 0; i < B_LD; ++i) {
    const int q = wave * B_LD + i;
    b_off[i] = (((uint32_t)(q >> 2) * KC + (q & 3)) << 10) + lane * 16;
  }
  // load d of stage gi: A first, then B (past the last stage out of the buffers' range:
  // zeros without a memory access, and no branch between the MFMAs). Buffer
  // instructions: the compiler counts a global_load_lds as a flat access and then
  // waits for every LDS read in flight where some of them would do.
  auto issue = [&](int gi, char* dst, int d) {
    const int gc = g_lo + min(gi, n_g - 1);
    const uint32_t past = gi < n_g ? 0u : 0x80000000u;
    if (d < A_LD)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          a_buf, (__attribute__((address_space(3))) void*)(dst + (wave + NW * d) * 1024), 16,
          a_off[d < A_LD ? d : 0] + past, gc * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          b_buf,
          (__attribute__((address_space(3))) void*)(dst + A_BYTES + (wave * B_LD + d - A_LD) * 1024),
          16, b_off[d < A_LD ? 0 : d - A_LD] + past, gc * 4096, 0, 0);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  const uint32_t a_row = (uint32_t)(wm * TM * 4096 + (lane & 31) * 128);
  const uint32_t a_swz = (uint32_t)((lane & 7) ^ ((lane >> 3) & 1));
  const uint32_t b_row = (uint32_t)(A_BYTES + wn * TN * 4096 + lane * 16);
  struct Ops {
    bf16x8 x[TM], w[TN];
  };
  auto load_ops = [&](Ops& o, const char* src, int t) {
    const char* ap = src + a_row + (((uint32_t)(2 * t + (lane >> 5)) ^ a_swz) * 16);
    const char* bp = src + b_row + t * 1024;
#pragma unroll
    for (int i = 0; i < TM; ++i) o.x[i] = *(const bf16x8*)(ap + i * 4096);
#pragma unroll
    for (int j = 0; j < TN; ++j) o.w[j] = *(const bf16x8*)(bp + j * 4096);
  };
  // Stage g lives in buffer g % S. Its loads go out as the MFMAs of stages g - S
  // (k step 3, the first H, once every wave has read that buffer's last operands)
  // and g - S + 1 (k step 0, the rest) run, PER after each row of MFMAs: issued in
  // one batch they held up the wave's MFMAs (113 against 100 us for 1000 x 16384 x
  // 3584 on 256 x 256 tiles).
  constexpr int LD = A_LD + B_LD, PER = (LD + 2 * TM - 1) / (2 * TM), H = TM * PER;
  Ops X, Y;
  auto stage_buf = [&](auto i) -> char* {
    constexpr int I = decltype(i)::value % S;
    return I == 0 ? buf0 : I == 1 ? buf1 : I == 2 ? buf2 : buf3;
  };
#define DRT_I(n) std::integral_constant<int, (n)>{}
#pragma unroll
  for (int d = 0; d < LD; ++d) issue(0, buf0, d);
  if (S > 2) {
#pragma unroll
    for (int d = 0; d < LD; ++d) issue(1, buf1, d);
#pragma unroll
    for (int d = 0; d < LD; ++d) issue(2, buf2, d);
  }
#pragma unroll
  for (int d = 0; d < H && d < LD; ++d) issue(S - 1, stage_buf(DRT_I(S - 1)), d);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(vm_wait((S - 2) * LD + (H < LD ? H : LD)));  // stage 0 has arrived
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  load_ops(X, buf0, 0);
  // k step t of stage gi on `cur`, the next step's operands into `nxt`; at the last
  // step, stage gi + 1 must be in LDS in every wave and this wave's reads of its own
  // buffer done (past the last stage the operands read are stale and unused)
  auto kstep = [&](Ops& cur, Ops& nxt, int gi, int t, char* here, char* there, char* prev) {
    if (t < 3) {
      load_ops(nxt, here, t + 1);
    } else {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(vm_wait((S - 2) * LD) & VM_LDS_WAIT_MASK);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load_ops(nxt, there, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma_bf16(cur.x[i], cur.w[j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int d = i * PER + q;
        if (t == 3 && d < LD) issue(gi + S, here, d);
        if (t == 0 && H + d < LD) issue(gi - 1 + S, prev, H + d);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto stage = [&](int gi, auto i) {
    constexpr int I = decltype(i)::value;
    char* here = stage_buf(DRT_I(I));
    char* there = stage_buf(DRT_I(I + 1));
    char* prev = stage_buf(DRT_I(I + S - 1));
    kstep(X, Y, gi, 0, here, there, prev);
    kstep(Y, X, gi, 1, here, there, prev);
    kstep(X, Y, gi, 2, here, there, prev);
    kstep(Y, X, gi, 3, here, there, prev);
  };
  int g = 0;
  for (; g + S <= n_g; g += S) {
    stage(g, DRT_I(0));
    stage(g + 1, DRT_I(1));
    if constexpr (S > 2) {
      stage(g + 2, DRT_I(2));
      stage(g + 3, DRT_I(3));
    }
  }
  if (g < n_g) {
    stage(g, DRT_I(0));
    if constexpr (S > 2) {
      if (g + 1 < n_g) {
        stage(g + 1, DRT_I(1));
        if (g + 2 < n_g) stage(g + 2, DRT_I(2));
      }
    }
  }
#undef DRT_I
  __builtin_amdgcn_s_waitcnt(vm_wait(0));  // the epilogue reuses the buffers

  if (EPI == EPI_STORE) {
    // a lane holds one column of 16 rows per MFMA tile: each store instruction
    // writes two whole 128-byte lines
    const bool part = KS > 1 || !a.rnd_bf16;
    float* y = a.y + (int64_t)ks * M * N;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
      if (n >= N) continue;
      const float bias = a.bias && !part ? bf16_bits_to_float(a.bias[n]) : 0.f;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + (wm * TM + i) * 32 + mfma_row(r, lane);
          const float v = acc[i][j][r];
          if (m < M) y[(int64_t)m * N + n] = part ? v : round_bf16(v) + bias;
        }
    }
    return;
  }
  // 32-row pieces through LDS: MFMA row tile p of both wave rows at a time
  constexpr int EROW = BN + 4;
  static_assert(EPI == EPI_STORE ||
                    (WVM == 2 && 32 * EROW * 4 + (EPI == EPI_QKV ? 8192 : 0) <= ST_BYTES),
                "epilogue piece (+ V tile) must fit a stage buffer");
  constexpr int V_OFF = (32 * EROW * 4 + 15) / 16 * 16;
  const int row0 = a.desc ? a.desc->row0 : 0;
#pragma unroll
  for (int p = 0; p < TM; ++p) {
    __syncthreads();  // the stage buffers, then the previous piece, have been read
    float* e = (float*)(wm ? buf1 : buf0);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        e[mfma_row(r, lane) * EROW + (wn * TN + j) * 32 + (lane & 31)] = round_bf16(acc[p][j][r]);
    __syncthreads();
    if (EPI == EPI_SWIGLU) {
      // each wave row's threads turn its own piece into 8-output chunks
      const int mp = m0 + (wm * TM + p) * 32, F = N >> 1;
      constexpr int CPR = BN / 16;  // chunks per row
#pragma unroll
      for (int i = 0; i < 32 * CPR / (64 * WVN); ++i) {
        const int c = (wn * 64 + lane) + 64 * WVN * i;
        const int r = c / CPR, q = c % CPR, blk = q >> 3, c8 = (q & 7) * 8;
        if (mp + r < M && n0 + blk * 128 < N) {
          const float* gp = e + r * EROW + blk * 128 + c8;
          uint16_t o[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float g = gp[k], u = gp[64 + k];
            o[k] = float_to_bf16_bits(g * (1.f / (1.f + expf(-g))) * u);
          }
          *(u32x4*)((uint16_t*)a.act_out + (int64_t)(mp + r) * F + (n0 >> 1) + blk * 64 + c8) =
              __builtin_bit_cast(u32x4, o);
        }
      }
    } else if (EPI == EPI_QKV) {
      // all threads take the two pieces' heads in turn (256 threads, one head wide)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const int mp = m0 + (w * TM + p) * 32;
        if (mp >= M) break;  // uniform
        const int rows = min(32, M - mp), head = n0 >> 7;
        char* piece = w ? buf1 : buf0;
        const float* ew = (const float*)piece;
        uint16_t* vbuf = (uint16_t*)(piece + V_OFF);
        auto get = [&](int m, int d) { return ew[m * EROW + d]; };
        const QkvTables qt = qkv_tables(a, head, row0 + mp, rows);
        if (a.kv_bf16) qkv_epilogue<__bf16>(a, qt, head, mp, row0 + mp, rows, get, vbuf);
        else qkv_epilogue<_Float16>(a, qt, head, mp, row0 + mp, rows, get, vbuf);
      }
    }
  }
}

template <int EPI, int TM, int TN, int WVM, int WVN, int S>
__global__ __launch_bounds__(64 * WVM * WVN, S > 2 ? 1 : 2) void big_bf16_kernel(
    const FusedArgs a, int KS, int col0, int NX) {
  big_bf16_tile<EPI, TM, TN, WVM, WVN, S>(a, KS, col0, NX);
}

namespace drt {
namespace {

// The tile shapes, with what they measured (K = 3584, us per 64-k stage and round of
// work-groups, 1000 rows; the second figure with at most one work-group per CU):
//   T256: 256 x 256, 8 waves, one per CU: 1.74 (1.27 on 40 CUs); 97 us and 1206
//         TFLOP/s for 1000 x 16384 x 3584
//   T128: 128 x 128, 4 waves, two per CU: 1.03 for 512 work-groups, 0.74 for <= 256
//   D128: T128 with four stage buffers, one per CU: 0.59 (0.50)
//   D64 : 64 x 128, four stage buffers, one per CU: 0.35 (0.29)
// Per output a larger tile moves fewer bytes through LDS and L2; a smaller one, and a
// deeper pipeline, wins where the tiles do not fill the chip (the loads' latency then
// sets a stage's time) or would leave most of a round empty.
enum Tile : int { T256 = 0, T128 = 1, D128 = 2, D64 = 3 };
struct TileCost { int bm, bn, slots_per_cu; float one, full; };
constexpr TileCost TILES[] = {{256, 256, 1, 1.27f, 1.74f},
                              {128, 128, 2, 0.74f, 1.03f},
                              {128, 128, 1, 0.50f, 0.59f},
                              {64, 128, 1, 0.29f, 0.35f}};

// Estimated us of `groups` work-groups of g stages each.
float tile_cost(int t, int groups, float g, int n_cu) {
  const TileCost& c = TILES[t];
  const int slots = c.slots_per_cu * n_cu;
  const int rounds = groups / slots, rest = groups - rounds * slots;
  float us = rounds * (c.full * g + 1.5f);
  // the last round: up to one work-group per CU, less while part of the chip idles
  if (rest > n_cu) us += c.full * g + 1.5f;
  else if (rest > 0)
    us += g * (c.slots_per_cu > 1 ? c.one : c.one + (c.full - c.one) * rest / n_cu) + 1.5f;
  return us;
}

int bb_tiles(int t, int M, int N) {
  const TileCost& c = TILES[t];
  return ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
}

}  // namespace

// The cheapest estimate over the tile shapes, the split-K slice counts (plain stores
// only: each at least four stages, the slices within part_floats) and, unsplit, a
// whole number of rounds of 256 x 256 tiles with the last columns on 128 x 128 ones
// (a second launch: 1000 x 18944 x 3584, 296 large tiles on 256 CUs, 168 us all
// large, 154 all small). reduce_us: what a slice pass costs besides its bytes;
// split_us: the least a split call can take (the host's part of a second launch).
BigBf16Plan big_bf16_plan(int M, int N, int K, int kind, int max_ks, size_t part_floats,
                          float reduce_us, float split_us) {
  const int n_cu = n_cu_of_current_device(), G = K / 64;
  BigBf16Plan best;
  float best_us = 1e30f;
  const int lo = kind == FL_QKV ? T128 : T256, hi = kind == FL_QKV ? D128 : D64;
  for (int t = lo; t <= hi; ++t) {
    const int tiles = bb_tiles(t, M, N);
    for (int ks = 1; ks <= max_ks; ++ks) {
      if (ks > 1 && (kind != FL_STORE || G / ks < 4 || (size_t)ks * M * N > part_floats)) break;
      float us = tile_cost(t, tiles * ks, (float)((G + ks - 1) / ks), n_cu);
      if (ks > 1) us += reduce_us + (ks + 1) * 4e-6f * M * N / 4.f;  // 4 TB/s
      us = std::max(us, ks > 1 ? split_us : 0.f);
      if (us < best_us) {
        best_us = us;
        best = BigBf16Plan{t, ks, 0};
      }
    }
  }
  if (kind != FL_QKV) {
    const int MT = (M + 255) / 256, cols = (N + 255) / 256;
    const int c1 = (int)((int64_t)MT * cols / n_cu * n_cu / MT);  // column tiles of whole rounds
    if (c1 > 0 && c1 < cols) {
      const int n1 = c1 * 256;
      for (int t = T128; t <= D128; ++t) {
        const float us = tile_cost(T256, MT * c1, (float)G, n_cu) +
                         tile_cost(t, bb_tiles(t, M, N - n1), (float)G, n_cu) + 3.f;
        if (us < best_us) {
          best_us = us;
          best = BigBf16Plan{t, 1, n1};
        }
      }
    }
  }
  return best;
}

bool big_bf16_supported(const FusedArgs& a, int kind) {
  // (16-byte loads straight into LDS: aligned operands only)
  if ((((uintptr_t)a.wb | (uintptr_t)a.act) & 15) != 0) return false;
  if (!a.wb || a.qw || !a.act || a.M < 1 || a.N % 32 || a.K % 64 || a.K < 64) return false;
  if (kind == FL_SWIGLU) return a.N % 128 == 0 && a.act_fmt == ACT_BF16;
  if (kind == FL_QKV) return a.N % 128 == 0;
  return kind == FL_STORE;
}

void big_bf16_linear(const FusedArgs& a, int kind, const BigBf16Plan& p, hipStream_t s) {
  require(big_bf16_supported(a, kind), "large-M bf16 linear: unsupported shape or kind");
  require(p.ks >= 1 && p.ks <= a.K / 64 && (p.ks == 1 || kind == FL_STORE),
          "large-M bf16 linear: split-K only for plain stores");
  const double all = 2.0 * a.N * a.K + 2.0 * a.M * a.K +
                     (kind == FL_STORE ? 4.0 * p.ks : 2.0) * a.M * a.N;
#define DRT_BB(E, TM, TN, WM, WN, S)                                                          \
  DRT_LAUNCH(Profiler::GEMM, all * n / a.N, (big_bf16_kernel<E, TM, TN, WM, WN, S>),          \
             dim3((unsigned)(MT * NX * p.ks)), dim3(64 * WM * WN), 0, s, a, p.ks, col0, NX)
#define DRT_BB_T(E)                                                                           \
  switch (t) {                                                                                \
    case T256: DRT_BB(E, 4, 2, 2, 4, 2); break;                                               \
    case T128: DRT_BB(E, 2, 2, 2, 2, 2); break;                                               \
    case D128: DRT_BB(E, 2, 2, 2, 2, 4); break;                                               \
    default: DRT_BB(E, 1, 2, 2, 2, 4); break;                                                 \
  }
  // columns [col0, col0 + n) on tile shape t
  auto launch = [&](int t, int col0, int n) {
    const int MT = (a.M + TILES[t].bm - 1) / TILES[t].bm, NX = (n + TILES[t].bn - 1) / TILES[t].bn;
    if (kind == FL_STORE) {
      DRT_BB_T(EPI_STORE)
    } else if (kind == FL_SWIGLU) {
      DRT_BB_T(EPI_SWIGLU)
    } else if (t == T128) {
      DRT_BB(EPI_QKV, 2, 2, 2, 2, 2);
    } else {
      DRT_BB(EPI_QKV, 2, 2, 2, 2, 4);
    }
    DRT_HIP(hipGetLastError());
  };
  require(kind != FL_QKV || p.tile == T128 || p.tile == D128, "q|k|v needs one-head tiles");
  if (p.n256 > 0) launch(T256, 0, p.n256);
  launch(p.tile, p.n256, a.N - p.n256);
#undef DRT_BB_T
#undef DRT_BB
}

// q|k|v: one-head tiles with the epilogue fused, or (where they leave CUs idle) K
// slices into `part` and the epilogue as a pass of its own.
void big_bf16_qkv(const FusedArgs& a, float* part, size_t part_floats, hipStream_t s) {
  const BigBf16Plan whole = big_bf16_plan(a.M, a.N, a.K, FL_QKV, 1, 0, 0.f);
  const BigBf16Plan split =
      big_bf16_plan(a.M, a.N, a.K, FL_STORE, BG_QKV_MAX_KS, part ? part_floats : 0, 6.f);
  if (split.ks == 1) {
    big_bf16_linear(a, FL_QKV, whole, s);
    return;
  }
  FusedArgs g = a;
  g.bias = nullptr;  // the epilogue rounds the sum and adds it
  g.rnd_bf16 = 0;
  g.y = part;
  big_bf16_linear(g, FL_STORE, split, s);
  qkv_epilogue_slices(a, part, split.ks, s);
}

}  // namespace drt
