// sgemm_kwave.hip — tiles of C from 32 x 32 to 128 x 64 whose K the four waves
// of a workgroup share, for launches with too few 256 x 256 tiles to fill the
// chip (a layer's forward and backward over a batch, a Gram matrix, small and
// middle-sized products).
//
// Same contract as the other tile kernels: C = alpha * op(A) * op(B) + beta * C
// with FP32 matrix instructions (v_mfma_f32_32x32x2_f32), the optional bias /
// ReLU epilogue, only in-range C elements stored, no operand padding read into
// a result. Any m, n and K >= 8.
//
//   * A wave owns the whole 32*MB x 32*NB tile for every fourth slot of K (a
//     slot is 8*KP k values of both operands) and streams those slots into a
//     private LDS ring with buffer_load_dwordx4 ... lds, R - 1 slots ahead, as
//     the ring kernels do: the K loop has no barrier. What bounded these
//     launches before was parallelism (a 256 x 128 tile per workgroup leaves
//     most CUs without one, and cutting K over workgroups instead costs a
//     partial's store, its read and a second dispatch for each range) and,
//     for ragged ones, predicated loads: here every wave of the chip has work
//     from 256 small tiles on, at a quarter of K each.
//   * The four waves' sums meet in the LDS after the loop and are added in wave
//     order; the columns go out as whole 16-byte vectors.
//   * Neighbouring slots go to different waves, so the waves of a workgroup
//     read neighbouring pieces of a k-contiguous line at about the same time.
//     Each load takes 32*KP bytes of a line (KP = 2 or 4: 64 or 128 bytes; at
//     KP = 1 every 128-byte line is fetched four times, 3001 x 2047 x 4099 T/N
//     in 436 us against 388; N/T has no such lines, and there KP = 1 with four
//     workgroups a CU hides most of a shallow tile's prologue and epilogue:
//     4096 x 4096 x 256 in 82 us against 94).
//   * A launch may also split K over workgroups (p.splits > 1: raw sums to the
//     partials, splitk_reduce_kernel adds them), which the rule in
//     sgemm_launch.hpp takes when the tiles alone do not fill the chip.
//   * Precision: the sum of an element is cut into at least four chains (one a
//     wave). Where the large kernels' rules would cut the element's K into
//     shorter ranges than a wave's quarter, the wave adds its accumulators into
//     a second set every so many k values, so no chain is longer than there.
//
// Measured on device memory, before (256 x 128 tiles and split K) -> now, us a
// launch: 1024^3 41.7 -> 20.0; 128^3 15.8 -> 3.6; 3001 x 2047 x 4099 T/N 474 ->
// 377, N/T 555 -> 363; 16384 x 4 x 16384 T/N 551 -> 190 (5.7 TB/s); 4096 x 256 x
// 4096 T/N 97.4 -> 63.7; 4096 x 300 x 16384 N/N 453 -> 327; 500 x 500 x 60000
// T/N 292 -> 224; and, from launches of many tiles whose K is shallow or no
// multiple of the ring kernels' step, 3712 x 4590 x 503 N/T 313 -> 140, 6379 x
// 2968 x 32 N/T 67 -> 34. Bound by: MFMA issue from about 64 x 64 tiles on
// (120-140 TFLOP/s; 95 % of the cycles a CU is busy, the rest the last round),
// HBM for n up to 32, the launch itself below 256^3. No LDS bank conflicts.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "sgemm_device.hpp"
#include "sgemm_launch.hpp"

namespace xvram::kernels {
namespace {

using namespace device;

constexpr int kThreads = 256;
constexpr int kWaves = 4;

// k values of one wave between folds, of tiles inside rows [0, rows) x columns
// [0, cols) and of the others.
struct Folds {
  int inside, edge, rows, cols;
};

template <int N> using Int = std::integral_constant<int, N>;

// Workgroup id -> (tile_m, tile_n), returning its K range index: split_coords
// with each XCD's run of ids also where their number is not a multiple of 8.
template <int kGroupM>
__device__ __forceinline__ int kwave_coords(const Params& p, int& tm, int& tn) {
  const int tiles = p.tiles_m * p.tiles_n;
  const int total = tiles * p.splits;
  constexpr int kXcds = 8;
  const int xcd = blockIdx.x % kXcds, place = blockIdx.x / kXcds;
  const int per = total / kXcds, more = total % kXcds;
  int id = xcd * per + min(xcd, more) + place;
  const int split = id / tiles;
  id -= split * tiles;
  const int span = kGroupM * p.tiles_n;
  const int group = id / span;
  const int first_m = group * kGroupM;
  const int rows = min(p.tiles_m - first_m, kGroupM);
  const int in_group = id - group * span;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
  return split;
}

// Waits until at most kLoads * `after` vector loads are outstanding (after < 4).
template <int kLoads>
__device__ __forceinline__ void wait_slots(int after) {
  static_assert(3 * kLoads <= 63, "the counts fit vmcnt");
  if (after >= 3) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(3 * kLoads) : "memory");
  else if (after == 2) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(2 * kLoads) : "memory");
  else if (after == 1) asm volatile("s_waitcnt vmcnt(%0)" :: "i"(kLoads) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// A k-contiguous half in a ring slot: block i's 32 lines one after another,
// 2 * KP pieces of 16 bytes each; piece g of line lrow lies at this place of
// its line's run, so that the fragment reads (the same piece of consecutive
// lines) hit distinct banks in every group of 8 and of 16 lanes.
template <int KP>
__device__ __forceinline__ int piece_place(int lrow, int g) {
  if constexpr (KP == 4) return g ^ (lrow & 7) ^ ((lrow >> 3) & 1);
  else if constexpr (KP == 2) return g ^ ((lrow >> 1) & 3) ^ ((lrow >> 3) & 1);
  else return g ^ (((lrow >> 2) ^ (lrow >> 3)) & 1);
}

// Tile 32*MB x 32*NB; slots of 8*KP k values, R of them in each wave's ring;
// kPerCu workgroups share a CU (their LDS and registers fit); kRegions: tiles past
// folds.rows or folds.cols fold at another depth (instances of their own: the
// choice costs the others 1 to 2 %, 500 x 500 x 60000 T/N 227.4 -> 231.6 us).
//
// A slot's halves in its ring place: an extent-contiguous half (op-N A, op-T
// B) row-major 8*KP x extent as loaded, a k-contiguous one as piece_place says.
// MFMA row r of row block i is tile row MB*r + i (columns alike), and lane half
// h supplies k value 8t + 4h + s in k-step s of the slot's t-th eight, for both
// operands. Step (j, t) multiplies eight k values from registers; in its first
// half it issues the next kGroup loads of the slot R ahead, into the ring place
// of the slot whose last fragments are in registers, and in its middle it reads
// the next step's fragments (after waiting for their slot when it is a new one).
template <bool kAKC, bool kBKC, int MB, int NB, int KP, int R, int kPerCu, bool kFold, bool kRegions>
__global__ __launch_bounds__(kThreads, kPerCu) void sgemm_kwave_kernel(Params p, Folds folds) {
  constexpr int TM = 32 * MB, TN = 32 * NB;
  constexpr int kGroup = MB + NB;         // wave loads of 1 KiB per 8 k values
  constexpr int kLoads = kGroup * KP;     // ... per slot
  constexpr int kSlot = 256 * kLoads;     // floats per slot
  constexpr int kSlotK = 8 * KP;
  constexpr int kUnroll = KP % 2 == 0 || R % 2 == 0 ? R : 2 * R;
  // Columns of the tile whose sums go through the LDS at once (every wave's).
  constexpr int kAccFloats = TM * TN;
  constexpr int kPasses = kAccFloats <= R * kSlot || NB == 1 ? 1 : 2;
  constexpr int kPassFloats = kAccFloats / kPasses;
  constexpr int kWaveLds = R * kSlot > kPassFloats ? R * kSlot : kPassFloats;
  static_assert(kWaves * kWaveLds * 4 * kPerCu <= 160 * 1024, "the rings fit the LDS");
  __shared__ __attribute__((aligned(16))) float lds[kWaves * kWaveLds];

  int tile_m, tile_n;
  const int split = kwave_coords<8>(p, tile_m, tile_n);
  const Params whole = p;
  if (p.splits > 1) narrow_to_split(p, split, kAKC, kBKC);
  const int m0 = tile_m * TM, n0 = tile_n * TN;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;

  float16_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // Sums of whole runs of `fold` k values of this wave.
  float16_t total[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) total[i][j] = acc[i][j];
  auto fold_acc = [&] {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        total[i][j] += acc[i][j];
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
      }
  };

  const int slots = (p.k + kSlotK - 1) / kSlotK;
  const int mine = (slots - wave + kWaves - 1) / kWaves; // slots wave, wave + 4, ...
  const int a_lines = min(TM, p.m - m0), b_lines = min(TN, p.n - n0);
  const auto rsrc = [&](const float* x, int64_t ld, int e0, bool kc, int lines) {
    // A k-contiguous line is stored to a multiple of 4 values (its tail is masked).
    return kc ? panel_rsrc(x + (int64_t)e0 * ld, (uint32_t)(((lines - 1) * ld + ((p.k + 3) & ~3)) * 4))
              : panel_rsrc(x + e0, (uint32_t)(((int64_t)p.k * ld - e0) * 4));
  };
  const __amdgpu_buffer_rsrc_t rs_a = rsrc(p.a, p.lda, m0, kAKC, a_lines);
  const __amdgpu_buffer_rsrc_t rs_b = rsrc(p.b, p.ldb, n0, kBKC, b_lines);
  // Byte offset of this lane's 16 bytes in load `load` of a half's first slot;
  // rows, columns and lines past the operand are clamped to its last (they
  // feed only elements past C).
  const auto voff = [&](int64_t ld, int blocks, int load, bool kc, int lines) {
    if (kc) {
      const int lr = (load % KP) * (32 / KP) + lane / (2 * KP);
      const int line = min(blocks * lr + load / KP, lines - 1);
      return (uint32_t)((line * ld + 4 * piece_place<KP>(lr, lane % (2 * KP))) * 4);
    }
    const int u = 4 * (64 * load + lane), extent = 32 * blocks;
    return (uint32_t)(((u / extent) * ld + min(u % extent, ((lines + 3) & ~3) - 4)) * 4);
  };
  uint32_t vo_a[MB * KP], vo_b[NB * KP];
#pragma unroll
  for (int i = 0; i < MB * KP; ++i) vo_a[i] = voff(p.lda, MB, i, kAKC, a_lines);
#pragma unroll
  for (int i = 0; i < NB * KP; ++i) vo_b[i] = voff(p.ldb, NB, i, kBKC, b_lines);
  const uint32_t adv_a = kAKC ? kSlotK * 4 : (uint32_t)(kSlotK * 4 * p.lda);
  const uint32_t adv_b = kBKC ? kSlotK * 4 : (uint32_t)(kSlotK * 4 * p.ldb);
  float* ring = lds + wave * kWaveLds;
  const uint32_t ring_lds = lds_byte_addr(ring);

  // Load L of slot j into ring slot S: A's MB * KP, then B's.
  auto issue = [&]<int S, int L>(int j, Int<S>, Int<L>) {
    constexpr int off = (S * kSlot + L * 256) * 4;
    const uint32_t q = (uint32_t)(wave + kWaves * j);
    if constexpr (L < MB * KP)
      load_lds16<off>(ring_lds, vo_a[L], rs_a, __builtin_amdgcn_readfirstlane(adv_a * q));
    else
      load_lds16<off>(ring_lds, vo_b[L - MB * KP], rs_b, __builtin_amdgcn_readfirstlane(adv_b * q));
  };
  // fa[set][block][k-step].
  float fa[2][MB][4], fb[2][NB][4];
  auto read_half = [&]<int N, bool kc>(const float* half, int t, float (&f)[N][4], Int<N>,
                                       std::bool_constant<kc>) {
    if constexpr (kc) {
      const int unit = lrow * 2 * KP + piece_place<KP>(lrow, 2 * t + lhalf);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float4 v = *reinterpret_cast<const float4*>(half + 256 * KP * i + 4 * unit);
        f[i][0] = v.x;
        f[i][1] = v.y;
        f[i][2] = v.z;
        f[i][3] = v.w;
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float* row = half + (8 * t + 4 * lhalf + s) * 32 * N + N * lrow;
        if constexpr (N == 4) {
          const float4 v = *reinterpret_cast<const float4*>(row);
          f[0][s] = v.x;
          f[1][s] = v.y;
          f[2][s] = v.z;
          f[3][s] = v.w;
        } else if constexpr (N == 2) {
          const float2 v = *reinterpret_cast<const float2*>(row);
          f[0][s] = v.x;
          f[1][s] = v.y;
        } else {
          f[0][s] = row[0];
        }
      }
    }
  };
  // Fragments of k values 8t .. 8t+7 of slot j (in ring slot S).
  auto read_frag = [&]<int S, int F>(int j, int t, Int<S>, Int<F>) {
    const float* slot = ring + S * kSlot;
    read_half(slot, t, fa[F], Int<MB>{}, std::bool_constant<kAKC>{});
    read_half(slot + 256 * MB * KP, t, fb[F], Int<NB>{}, std::bool_constant<kBKC>{});
    const int k0 = (wave + kWaves * j) * kSlotK + 8 * t;
    if (k0 + 8 > p.k) { // the K tail: zeros past it in both operands
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bool in = k0 + 4 * lhalf + s < p.k;
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[F][i][s] = in ? fa[F][i][s] : 0.f;
#pragma unroll
        for (int i = 0; i < NB; ++i) fb[F][i][s] = in ? fb[F][i][s] : 0.f;
      }
    }
  };
  auto mfma_one = [&]<int F, int X>(Int<F>, Int<X>) {
    constexpr int s = X / (MB * NB), i = (X / NB) % MB, j = X % NB;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[F][i][s], fb[F][j][s], acc[i][j], 0, 0, 0);
  };

  auto issue_range = [&]<int S, int kFrom, int kTo>(int j, Int<S>, Int<kFrom>, Int<kTo>) {
    [&]<int... L>(std::integer_sequence<int, L...>) {
      (issue(j, Int<S>{}, Int<kFrom + L>{}), ...);
    }(std::make_integer_sequence<int, kTo - kFrom>{});
  };
  // Before slot j + 1 is read: slots j + 2 .. j + R - 1 and the first group of
  // slot j + R may be outstanding.
  static_assert((R - 2) * kLoads + kGroup <= 63, "outstanding loads fit the vmcnt counter");
  auto wait_next = [&]<bool kTail>(int j, std::bool_constant<kTail>) {
    if (!kTail || j + R < mine)
      asm volatile("s_waitcnt vmcnt(%0)" :: "i"((R - 2) * kLoads + kGroup) : "memory");
    else
      wait_slots<kLoads>(min(j + R - 1, mine - 1) - (j + 1));
  };
  if (mine > 0) {
    [&]<int... S>(std::integer_sequence<int, S...>) {
      ((S < mine ? (issue_range(S, Int<S>{}, Int<0>{}, Int<kLoads>{}), 0) : 0), ...);
    }(std::make_integer_sequence<int, R - 1>{});
    if (R - 1 < mine) issue_range(R - 1, Int<R - 1>{}, Int<0>{}, Int<kGroup>{});
    wait_next(-1, std::true_type{});
    read_frag(0, 0, Int<0>{}, Int<0>{});

    constexpr int kMfmas = 4 * MB * NB;
    constexpr int kSpace = kMfmas / 2 / kGroup > 0 ? kMfmas / 2 / kGroup : 1;
    constexpr int kReadAt = kMfmas / 2;
    static_assert((kGroup - 1) * kSpace < kReadAt, "a step's loads are issued before its wait");
    // Eight k values of slot j: J = j % kUnroll, t of KP.
    auto step = [&]<int J, int T, bool kTail>(int j, Int<J>, Int<T>, std::bool_constant<kTail> tail) {
      constexpr int cur = (J * KP + T) & 1, nxt = cur ^ 1;
      constexpr bool kLast = T == KP - 1;
      // The last eight k values of slot j are in registers: its ring slot
      // starts to take slot j + R; the rest of those loads follow in the
      // steps of slot j + 1.
      const int into = kLast ? j + R : j - 1 + R;
      constexpr int ring_slot = kLast ? J % R : (J + R - 1) % R;
      const bool load = !kTail || into < mine;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      [&]<int... X>(std::integer_sequence<int, X...>) {
        (([&] {
           if constexpr (X % kSpace == 0 && X / kSpace < kGroup) {
             if (load) {
               __builtin_amdgcn_sched_barrier(0);
               issue(into, Int<ring_slot>{}, Int<(kLast ? 0 : (T + 1) * kGroup) + X / kSpace>{});
               __builtin_amdgcn_sched_barrier(0);
             }
           }
           if constexpr (X == kReadAt) {
             __builtin_amdgcn_sched_barrier(0);
             if constexpr (!kLast) {
               read_frag(j, T + 1, Int<J % R>{}, Int<nxt>{});
             } else if (!kTail || j + 1 < mine) {
               wait_next(j, tail);
               read_frag(j + 1, 0, Int<(J + 1) % R>{}, Int<nxt>{});
             }
             __builtin_amdgcn_sched_barrier(0);
           }
           mfma_one(Int<cur>{}, Int<X>{});
         }()),
         ...);
      }(std::make_integer_sequence<int, kMfmas>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    auto slot_steps = [&]<int J, bool kTail>(int j, Int<J>, std::bool_constant<kTail> tail) {
      [&]<int... T>(std::integer_sequence<int, T...>) {
        (step(j, Int<J>{}, Int<T>{}, tail), ...);
      }(std::make_integer_sequence<int, KP>{});
    };
    int j = 0;
    // Blocks of kUnroll slots whose loads all exist, in runs of `fold` k values
    // (a multiple of the block's), then the rest.
    const int last = mine - kUnroll - R;
    const auto blocks = [&](int to) {
      for (; j <= to; j += kUnroll) {
        [&]<int... J>(std::integer_sequence<int, J...>) {
          (slot_steps(j + J, Int<J>{}, std::false_type{}), ...);
        }(std::make_integer_sequence<int, kUnroll>{});
      }
    };
    // Slots per run: a multiple of kUnroll.
    const bool inside = !kRegions || (m0 + TM <= folds.rows && n0 + TN <= folds.cols);
    const int run = (inside ? folds.inside : folds.edge) / kSlotK;
    int from = 0;                  // first slot of the current run
    if constexpr (kFold) {
      for (int to = run - kUnroll; ; to += run) {
        blocks(min(to, last));
        if (to > last) break;
        fold_acc();
        from = j;
      }
    } else {
      blocks(last);
    }
    for (; j < mine; j += kUnroll) {
      if (kFold && min(j + kUnroll, mine) - from > run) {
        fold_acc();
        from = j;
      }
      [&]<int... J>(std::integer_sequence<int, J...>) {
        ((j + J < mine ? (slot_steps(j + J, Int<J>{}, std::true_type{}), 0) : 0), ...);
      }(std::make_integer_sequence<int, kUnroll>{});
    }
  }

  if constexpr (kFold) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] += total[i][j];
  }
  // Sums of the four waves, in wave order, through the LDS.
  constexpr int kUnits = TM / 4; // float4s per column
  const bool raw = whole.splits > 1;
  float* out = raw ? whole.partial + (int64_t)split * partial_ld(whole.m) * whole.n : whole.c;
  const int64_t ldo = raw ? partial_ld(whole.m) : whole.ldc;
  constexpr int kNJ = NB / kPasses; // column blocks per pass
  // C past the L2 from 1 MiB on (2048 x 2048 x 256 N/T 24.0 -> 20.8 us; on a C of
  // 34 KB waiting for memory costs 0.3 us more than the L2).
  const bool stream = (int64_t)whole.m * whole.n >= (1 << 18);
  static_assert(kPasses == 1 || NB % kPasses == 0, "whole column blocks per pass");
#pragma unroll
  for (int pass = 0; pass < kPasses; ++pass) {
    if (pass > 0) __syncthreads(); // the pass before has been read
#pragma unroll
    for (int jj = 0; jj < kNJ; ++jj) {
      const int j = pass * kNJ + jj;
      // Column 32*jj + lrow of the pass; its float4s are permuted among eight so
      // that eight lanes' stores hit distinct banks.
      float* col = ring + (32 * jj + lrow) * TM;
#pragma unroll
      for (int g = 0; g < 4 * MB; ++g) {
        // Four consecutive rows 4*u .. 4*u+3 of the column.
        float4 v;
        int u;
        if constexpr (MB == 4) {
          v = make_float4(acc[0][j][g], acc[1][j][g], acc[2][j][g], acc[3][j][g]);
          u = 8 * (g >> 2) + 4 * lhalf + (g & 3);
        } else if constexpr (MB == 2) {
          v = make_float4(acc[0][j][2 * g], acc[1][j][2 * g], acc[0][j][2 * g + 1], acc[1][j][2 * g + 1]);
          u = (2 * (8 * (g >> 1) + 4 * lhalf + 2 * (g & 1))) / 4;
        } else {
          v = make_float4(acc[0][j][4 * g], acc[0][j][4 * g + 1], acc[0][j][4 * g + 2], acc[0][j][4 * g + 3]);
          u = 2 * g + lhalf;
        }
        *reinterpret_cast<float4*>(col + 4 * (u ^ (lrow & 7))) = v;
      }
    }
    __syncthreads();
    constexpr int kPerThread = kUnits * 32 * kNJ / kThreads;
    static_assert(kUnits * 32 * kNJ % kThreads == 0, "whole units per thread");
#pragma unroll
    for (int t = 0; t < kPerThread; ++t) {
      const int unit = t * kThreads + tid;
      const int pc = unit / kUnits, u = unit % kUnits;
      const int row = m0 + 4 * u, colm = n0 + NB * (pc % 32) + pass * kNJ + pc / 32;
      const float* src = lds + pc * TM + 4 * (u ^ (pc & 7));
      float4 s = *reinterpret_cast<const float4*>(src);
#pragma unroll
      for (int w = 1; w < kWaves; ++w) {
        const float4 x = *reinterpret_cast<const float4*>(src + w * kWaveLds);
        s.x += x.x;
        s.y += x.y;
        s.z += x.z;
        s.w += x.w;
      }
      if (row >= whole.m || colm >= whole.n) continue;
      if (raw) *reinterpret_cast<float4*>(out + (int64_t)colm * ldo + row) = s;
      else if (stream) store_quad<true>(whole, s, row, colm);
      else store_quad<false>(whole, s, row, colm);
    }
  }
}

template <bool AK, bool BK>
hipError_t launch_form(const Params& p, int tile, const Folds& folds, hipStream_t s, hipEvent_t e0,
                       hipEvent_t e1) {
  const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits)), block(kThreads);
  const bool regions = folds.edge != folds.inside;
  const auto go = [&](auto kernel) {
    hipExtLaunchKernelGGL(kernel, grid, block, 0, s, e0, e1, 0, p, folds);
    return hipGetLastError();
  };
  // kKwaveTiles (sgemm_launch.hpp) in its order.
  switch (tile) {
  case 0: return regions ? go(sgemm_kwave_kernel<AK, BK, 1, 1, 2, 2, 4, true, true>)
                         : go(sgemm_kwave_kernel<AK, BK, 1, 1, 2, 2, 4, true, false>);
  case 1: return regions ? go(sgemm_kwave_kernel<AK, BK, 2, 1, 2, 2, 3, true, true>)
                         : go(sgemm_kwave_kernel<AK, BK, 2, 1, 2, 2, 3, true, false>);
  case 2: return regions ? go(sgemm_kwave_kernel<AK, BK, 2, 2, 2, 2, 2, true, true>)
                         : go(sgemm_kwave_kernel<AK, BK, 2, 2, 2, 2, 2, true, false>);
  case 3: return regions ? go(sgemm_kwave_kernel<AK, BK, 4, 1, 2, 2, 2, true, true>)
                         : go(sgemm_kwave_kernel<AK, BK, 4, 1, 2, 2, 2, true, false>);
  case 4: return regions ? go(sgemm_kwave_kernel<AK, BK, 1, 1, 4, 4, 1, true, true>)
                         : go(sgemm_kwave_kernel<AK, BK, 1, 1, 4, 4, 1, true, false>);
  case 5:
    if constexpr (!AK && !BK) return go(sgemm_kwave_kernel<AK, BK, 4, 2, 1, 3, 2, false, false>);
    break;
  case 6:
    if constexpr (!AK && !BK) return go(sgemm_kwave_kernel<AK, BK, 2, 2, 1, 2, 4, false, false>);
  }
  return hipErrorInvalidValue;
}

} // namespace

hipError_t launch_splitk_reduce(const device::Params& p, hipStream_t stream, hipEvent_t stop);

// Launches `plan` (kwave_plan_for) of `p`; start / stop (optional) are recorded
// by the dispatches.
hipError_t launch_kwave(const Params& p0, const KwavePlan& plan, bool a_kcontig, bool b_ncontig,
                        hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  const KwaveTile& t = kKwaveTiles[plan.tile];
  Params p = p0;
  p.tiles_m = (p.m + 32 * t.mb - 1) / (32 * t.mb);
  p.tiles_n = (p.n + 32 * t.nb - 1) / (32 * t.nb);
  p.splits = plan.splits;
  p.split_depth = plan.depth;
  const Folds folds{plan.fold, plan.edge_fold, static_cast<int>(plan.rows), static_cast<int>(plan.cols)};
  hipEvent_t last = p.splits > 1 ? nullptr : stop;
  hipError_t e;
  if (!a_kcontig && !b_ncontig) e = launch_form<false, true>(p, plan.tile, folds, stream, start, last);
  else if (!a_kcontig && b_ncontig) e = launch_form<false, false>(p, plan.tile, folds, stream, start, last);
  else if (a_kcontig && !b_ncontig) e = launch_form<true, true>(p, plan.tile, folds, stream, start, last);
  else e = launch_form<true, false>(p, plan.tile, folds, stream, start, last);
  if (e != hipSuccess || p.splits <= 1) return e;
  return launch_splitk_reduce(p, stream, stop);
}

} // namespace xvram::kernels
