// sgemm_device.hpp — device-side pieces shared by the tile kernels
// (sgemm_kwave.hip: tiles of 32 x 32 to 128 x 64 whose K the waves share;
// sgemm_mfma.hip: 256 x 128 tiles, two workgroups per CU; sgemm_wide.hip:
// kernels of 256 x 256 tiles, one workgroup per CU). Compiled only by hipcc.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace xvram::kernels::device {

typedef float float16_t __attribute__((ext_vector_type(16)));

// One launch, canonical column-major form (see sgemm_launch.hpp).
struct Params {
  const float* a;
  const float* b;
  float* c;
  int64_t lda, ldb, ldc;
  int m, n, k;
  float alpha, beta;
  int tiles_m, tiles_n;
  const float* bias_row; // per-row bias (nullptr = none)
  const float* bias_col; // per-column bias (nullptr = none)
  int relu;
  // Second K panel (ring kernel only): k rows [k_split, k) of A and B come
  // from a2 / b2 (same leading dimensions) instead of a / b; nullptr = none.
  const float* a2;
  const float* b2;
  int k_split;
  // Split K: splits > 1 cuts K into ranges of split_depth; blockIdx.x covers
  // tiles x splits and each workgroup stores its range's raw sums to partial
  // `split` (column-major, ld = m rounded up to 4; partial_target).
  int splits;
  int split_depth;
  float* partial;
};

__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }

// Four consecutive elements of a line starting at `first`; elements at or
// beyond `limit` (and the whole vector when !line_ok) read as 0.
__device__ __forceinline__ float4 load4(const float* __restrict__ line, int first, int limit,
                                        bool line_ok) {
  if (!line_ok || first >= limit) return zero4();
  float4 v = *reinterpret_cast<const float4*>(line + first);
  if (first + 4 > limit) {
    const int left = limit - first;
    if (left < 4) v.w = 0.f;
    if (left < 3) v.z = 0.f;
    if (left < 2) v.y = 0.f;
  }
  return v;
}

// Raw buffer descriptor (no stride, 32-bit data format word) over `bytes`
// bytes from `base`; reads at or past `bytes` return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t panel_rsrc(const float* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// One wave-wide direct load: lane l's 16 bytes at rsrc.base + soff + voff land
// at LDS byte address lds_base + kOff + 16*l (lds_base wave-uniform). Counted
// by vmcnt only: the caller waits on vmcnt before the data is read (and, when
// other waves read it, before the barrier that publishes it).
template <int kOff>
__device__ __forceinline__ void load_lds16(uint32_t lds_base, uint32_t voff,
                                           __amdgpu_buffer_rsrc_t rsrc, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds_base), "v"(voff), "s"(rsrc), "s"(soff), "i"(kOff)
               : "memory", "m0", "scc");
}

__device__ __forceinline__ uint32_t lds_byte_addr(const float* p) {
  return __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}

// Linear workgroup id -> (tile_m, tile_n): undo the round-robin XCD dispatch
// so XCD x owns ids [x*per, (x+1)*per), then walk tiles in kGroupM-row groups
// (column-major inside a group).
template <int kGroupM>
__device__ __forceinline__ void tile_coords(const Params& p, int& tm, int& tn) {
  const int total = p.tiles_m * p.tiles_n;
  int id = blockIdx.x;
  constexpr int kXcds = 8;
  if ((total % kXcds) == 0) {
    const int per = total / kXcds;
    id = (id % kXcds) * per + id / kXcds;
  }
  const int span = kGroupM * p.tiles_n;
  const int group = id / span;
  const int first_m = group * kGroupM;
  const int rows = min(p.tiles_m - first_m, kGroupM);
  const int in_group = id - group * span;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

// Split-K launches: workgroup -> (tile_m, tile_n), returning its K range
// index. Ids are remapped per XCD as in tile_coords; the ids of one range are
// consecutive, so each XCD works on whole ranges and keeps their A and B
// K-slices in its own L2.
template <int kGroupM>
__device__ __forceinline__ int split_coords(const Params& p, int& tm, int& tn) {
  const int tiles = p.tiles_m * p.tiles_n;
  const int total = tiles * p.splits;
  int id = blockIdx.x;
  constexpr int kXcds = 8;
  if ((total % kXcds) == 0) {
    const int per = total / kXcds;
    id = (id % kXcds) * per + id / kXcds;
  }
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

// The launch parameters of K range `split` of a split launch: operand bases
// moved to the range's first k (k-contiguous operands by k elements, the
// others by k lines), K = the range's depth.
__device__ __forceinline__ void narrow_to_split(Params& p, int split, bool a_kcontig,
                                                bool b_kcontig) {
  const int k0 = split * p.split_depth;
  p.a += a_kcontig ? (int64_t)k0 : (int64_t)k0 * p.lda;
  p.b += b_kcontig ? (int64_t)k0 : (int64_t)k0 * p.ldb;
  p.k = min(p.split_depth, p.k - k0);
}

// Leading dimension of the partials of a split launch (sgemm_launch.hpp's
// split_partial_ld): m rounded up to 4, so every column is 16-byte aligned.
__host__ __device__ __forceinline__ int64_t partial_ld(int m) { return ((int64_t)m + 3) / 4 * 4; }

// Where a workgroup of a split launch stores its raw sums: its range's
// partial (ld = partial_ld(m)) with alpha 1, beta 0 and no epilogue (1 * x
// is exact).
__device__ __forceinline__ Params partial_target(const Params& p, int split) {
  Params o = p;
  o.ldc = partial_ld(p.m);
  o.c = p.partial + (int64_t)split * o.ldc * p.n;
  o.alpha = 1.f;
  o.beta = 0.f;
  o.bias_row = nullptr;
  o.bias_col = nullptr;
  o.relu = 0;
  return o;
}

// Writes one wave's accumulators: acc[i][j] holds MFMA block (row block i,
// column block j) of v_mfma_f32_32x32x2f32; element v of this lane sits at
// MFMA row 8*(v/4) + 4*lhalf + v%4 and MFMA column lrow, i.e. tile row
// row0 + 4*(that) + i and tile column col0 + kNJ*lrow + j (row blocks and
// column blocks interleaved so one float4 covers four consecutive rows).
// C = alpha*acc + beta*C (C not read when beta == 0), then + bias_row[i] +
// bias_col[j], then ReLU (NaN kept: v < 0 is false). Only in-range elements
// are touched.
//
// A wave whose whole 128 x 32*kNJ region lies inside C takes the interior path:
// no per-element bounds, and the loads of old C (beta != 0), of the column
// biases and of the row biases are issued in batches before any is used, so
// the wave waits for memory once per kBatch columns of its lane instead of
// once per float4 (a serial chain of 16*kNJ round trips that every workgroup of
// a launch would otherwise run at the same moment). Same arithmetic, in the
// same order, as the general path. Row biases are loaded ahead only with
// kRowBiasAhead (64 more registers: the 256 x 256 kernels have them, the
// 256 x 128 kernel at two workgroups per CU does not). One column of a lane per
// batch: with two the kernels, which compile the general path as well, spill.
template <int kNJ, bool kRowBiasAhead>
__device__ __forceinline__ void store_c_interior(const Params& p, const float16_t (&acc)[4][kNJ],
                                                 int row0, int col0, int lrow, int lhalf) {
  const bool read_c = p.beta != 0.f;
  const bool extra = p.bias_row != nullptr || p.bias_col != nullptr || p.relu != 0;
  const auto row_of = [&](int v) { return row0 + 4 * (8 * (v >> 2) + 4 * lhalf + (v & 3)); };
  float brow[16][4];
  if (kRowBiasAhead && p.bias_row != nullptr) {
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int t = 0; t < 4; ++t) brow[v][t] = p.bias_row[row_of(v) + t];
  }
  const auto finish = [&](float v, int vi, int t, float bias_c) {
    if (p.bias_row != nullptr) v += kRowBiasAhead ? brow[vi][t] : p.bias_row[row_of(vi) + t];
    v += bias_c;
    return (p.relu != 0 && v < 0.f) ? 0.f : v;
  };
#pragma unroll
  for (int j = 0; j < kNJ; ++j) {
    const int col = col0 + kNJ * lrow + j;
    float* cline = p.c + (int64_t)col * p.ldc;
    const float bias_c = p.bias_col != nullptr ? p.bias_col[col] : 0.f;
    float4 old[16];
    if (read_c) {
#pragma unroll
      for (int v = 0; v < 16; ++v) old[v] = *reinterpret_cast<const float4*>(cline + row_of(v));
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      float4 r;
      if (read_c) {
        r.x = p.alpha * acc[0][j][v] + p.beta * old[v].x;
        r.y = p.alpha * acc[1][j][v] + p.beta * old[v].y;
        r.z = p.alpha * acc[2][j][v] + p.beta * old[v].z;
        r.w = p.alpha * acc[3][j][v] + p.beta * old[v].w;
      } else {
        r.x = p.alpha * acc[0][j][v];
        r.y = p.alpha * acc[1][j][v];
        r.z = p.alpha * acc[2][j][v];
        r.w = p.alpha * acc[3][j][v];
      }
      if (extra) {
        r.x = finish(r.x, v, 0, bias_c);
        r.y = finish(r.y, v, 1, bias_c);
        r.z = finish(r.z, v, 2, bias_c);
        r.w = finish(r.w, v, 3, bias_c);
      }
      *reinterpret_cast<float4*>(cline + row_of(v)) = r;
    }
  }
}

typedef float float4_t __attribute__((ext_vector_type(4)));

// Four consecutive floats of C. kStream: past the L2 (a workgroup's C is not
// read again by its launch, and what the L2 still holds dirty is written back
// when the launch ends, with every CU idle).
template <bool kStream>
__device__ __forceinline__ void store4(float* dst, float x, float y, float z, float w) {
  const float4_t v = {x, y, z, w};
  if constexpr (kStream) __builtin_nontemporal_store(v, reinterpret_cast<float4_t*>(dst));
  else *reinterpret_cast<float4_t*>(dst) = v;
}

// C(row .. row+3, col) from the sums of four consecutive rows (row a multiple
// of 4 below m): alpha, beta, biases and ReLU in store_c_tile's arithmetic and
// order; only rows inside C are touched.
template <bool kStream>
__device__ __forceinline__ void store_quad(const Params& p, const float4& sum, int row, int col) {
  float* cp = p.c + (int64_t)col * p.ldc + row;
  const bool extra = p.bias_row != nullptr || p.bias_col != nullptr || p.relu != 0;
  const float bias_c = p.bias_col != nullptr ? p.bias_col[col] : 0.f;
  const auto finish = [&](float v, int r) {
    if (p.bias_row != nullptr) v += p.bias_row[r];
    v += bias_c;
    return (p.relu != 0 && v < 0.f) ? 0.f : v;
  };
  if (row + 4 <= p.m) {
    float r[4] = {p.alpha * sum.x, p.alpha * sum.y, p.alpha * sum.z, p.alpha * sum.w};
    if (p.beta != 0.f) {
      const float4 old = *reinterpret_cast<const float4*>(cp);
      r[0] = p.alpha * sum.x + p.beta * old.x;
      r[1] = p.alpha * sum.y + p.beta * old.y;
      r[2] = p.alpha * sum.z + p.beta * old.z;
      r[3] = p.alpha * sum.w + p.beta * old.w;
    }
    if (extra) {
#pragma unroll
      for (int t = 0; t < 4; ++t) r[t] = finish(r[t], row + t);
    }
    store4<kStream>(cp, r[0], r[1], r[2], r[3]);
    return;
  }
  const float v[4] = {sum.x, sum.y, sum.z, sum.w};
  for (int t = 0; t < 4 && row + t < p.m; ++t) {
    const float val = p.alpha * v[t];
    const float out = p.beta != 0.f ? val + p.beta * cp[t] : val;
    cp[t] = extra ? finish(out, row + t) : out;
  }
}

template <int kNJ, bool kRowBiasAhead>
__device__ __forceinline__ void store_c_tile(const Params& p, const float16_t (&acc)[4][kNJ],
                                             int row0, int col0, int lrow, int lhalf) {
  if (row0 + 128 <= p.m && col0 + 32 * kNJ <= p.n) {
    store_c_interior<kNJ, kRowBiasAhead>(p, acc, row0, col0, lrow, lhalf);
    return;
  }
  const bool read_c = p.beta != 0.f;
  const bool extra = p.bias_row != nullptr || p.bias_col != nullptr || p.relu != 0;
  const auto finish = [&](float v, int r, float bias_c) {
    if (p.bias_row != nullptr) v += p.bias_row[r];
    v += bias_c;
    return (p.relu != 0 && v < 0.f) ? 0.f : v;
  };
#pragma unroll
  for (int j = 0; j < kNJ; ++j) {
    const int col = col0 + kNJ * lrow + j;
    if (col >= p.n) continue;
    float* cline = p.c + (int64_t)col * p.ldc;
    const float bias_c = p.bias_col != nullptr ? p.bias_col[col] : 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int mrow = 8 * (v >> 2) + 4 * lhalf + (v & 3);
      const int row = row0 + 4 * mrow;
      if (row >= p.m) continue;
      const float out[4] = {acc[0][j][v], acc[1][j][v], acc[2][j][v], acc[3][j][v]};
      if (row + 4 <= p.m) {
        float4* dst = reinterpret_cast<float4*>(cline + row);
        float4 r;
        if (read_c) {
          const float4 old = *dst;
          r.x = p.alpha * out[0] + p.beta * old.x;
          r.y = p.alpha * out[1] + p.beta * old.y;
          r.z = p.alpha * out[2] + p.beta * old.z;
          r.w = p.alpha * out[3] + p.beta * old.w;
        } else {
          r.x = p.alpha * out[0];
          r.y = p.alpha * out[1];
          r.z = p.alpha * out[2];
          r.w = p.alpha * out[3];
        }
        if (extra) {
          r.x = finish(r.x, row, bias_c);
          r.y = finish(r.y, row + 1, bias_c);
          r.z = finish(r.z, row + 2, bias_c);
          r.w = finish(r.w, row + 3, bias_c);
        }
        *dst = r;
      } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (row + t < p.m) {
            const float val = p.alpha * out[t];
            const float sum = read_c ? val + p.beta * cline[row + t] : val;
            cline[row + t] = extra ? finish(sum, row + t, bias_c) : sum;
          }
        }
      }
    }
  }
}

// Between LDS accesses of one wave by which its lanes hand each other values: the
// compiler keeps the accesses before it before those after it, also where it could
// prove their per-lane addresses apart. No instruction: the LDS serves a wave's
// accesses in order.
__device__ __forceinline__ void lanes_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same for the ring kernels' waves (kNJ = 4), through 16 KiB of the wave's
// own LDS: column block j of the accumulators (every fourth column) goes in as
// the MFMAs left it and comes out with 32 lanes on 128 consecutive rows of a
// column, so C is read and written in runs of 512 bytes instead of 16. Written
// as 16-byte pieces of 64 columns at once, a 256-tile launch spent about 12 us
// of its last round on its C (4096 x 4096 x 256 N/T: 80 us for 55 us of MFMAs, now 71; 8192 x 8192 x 128
// 207 -> 165; 4096^3 920 -> 907; 8192^3 7227 -> 7180).
// No other wave's LDS is touched and the LDS serves a wave in order, so there
// is no barrier; lanes_exchange keeps the compiler to that order too. A lane's
// four rows stay the same, and so does its row bias.
template <bool kEdge, bool kStream>
__device__ __forceinline__ void store_c_ring(const Params& p, const float16_t (&acc)[4][4], float* lds,
                                             int row0, int col0, int lane) {
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int row = row0 + 4 * lrow; // of this lane's C
  const bool read_c = p.beta != 0.f;
  float4 bias_r = zero4();
  if (p.bias_row != nullptr) {
    if (!kEdge || row + 4 <= p.m) {
      bias_r = make_float4(p.bias_row[row], p.bias_row[row + 1], p.bias_row[row + 2], p.bias_row[row + 3]);
    } else {
      if (row < p.m) bias_r.x = p.bias_row[row];
      if (row + 1 < p.m) bias_r.y = p.bias_row[row + 1];
      if (row + 2 < p.m) bias_r.z = p.bias_row[row + 2];
    }
  }
  const bool row_bias = p.bias_row != nullptr;
  const auto finish = [&](float v, float br, float bc) {
    if (row_bias) v += br;
    v += bc;
    return (p.relu != 0 && v < 0.f) ? 0.f : v;
  };
  const bool extra = row_bias || p.bias_col != nullptr || p.relu != 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    // MFMA column lrow, rows 4*u .. 4*u+3; float4s permuted among eight so that
    // eight lanes' stores hit distinct banks.
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int u = 8 * (v >> 2) + 4 * lhalf + (v & 3);
      *reinterpret_cast<float4*>(lds + 128 * lrow + 4 * (u ^ (lrow & 7))) =
          make_float4(acc[0][j][v], acc[1][j][v], acc[2][j][v], acc[3][j][v]);
    }
    lanes_exchange();
    // Columns in batches of 8 per lane, a batch's old C loaded before its use.
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float4 old[8];
      if (read_c) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int col = col0 + 4 * (16 * b + 2 * t + lhalf) + j;
          if (!kEdge || (row + 4 <= p.m && col < p.n))
            old[t] = *reinterpret_cast<const float4*>(p.c + (int64_t)col * p.ldc + row);
        }
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int pc = 16 * b + 2 * t + lhalf;
        const int col = col0 + 4 * pc + j;
        const float4 s = *reinterpret_cast<const float4*>(lds + 128 * pc + 4 * (lrow ^ (pc & 7)));
        if (kEdge && (row >= p.m || col >= p.n)) continue;
        float* dst = p.c + (int64_t)col * p.ldc + row;
        const float bias_c = p.bias_col != nullptr ? p.bias_col[col] : 0.f;
        if (!kEdge || row + 4 <= p.m) {
          float4 r = make_float4(p.alpha * s.x, p.alpha * s.y, p.alpha * s.z, p.alpha * s.w);
          if (read_c) {
            r.x = p.alpha * s.x + p.beta * old[t].x;
            r.y = p.alpha * s.y + p.beta * old[t].y;
            r.z = p.alpha * s.z + p.beta * old[t].z;
            r.w = p.alpha * s.w + p.beta * old[t].w;
          }
          if (extra) {
            r.x = finish(r.x, bias_r.x, bias_c);
            r.y = finish(r.y, bias_r.y, bias_c);
            r.z = finish(r.z, bias_r.z, bias_c);
            r.w = finish(r.w, bias_r.w, bias_c);
          }
          store4<kStream>(dst, r.x, r.y, r.z, r.w);
        } else {
          const float sv[3] = {s.x, s.y, s.z}, br[3] = {bias_r.x, bias_r.y, bias_r.z};
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            if (row + i >= p.m) continue;
            const float val = p.alpha * sv[i];
            const float out = read_c ? val + p.beta * dst[i] : val;
            dst[i] = extra ? finish(out, br[i], bias_c) : out;
          }
        }
      }
    }
    if (j < 3) lanes_exchange(); // the next block goes over this one
  }
}

} // namespace xvram::kernels::device
