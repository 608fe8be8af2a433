// kernels_u16_whole.hip -- step two over uint16 step-one sums, a tile's rows all
// in LDS.
//
// The sums of kernels_u16_staged.hip (exact integers, equal to the reference's
// sequential float sum, include/Dedispersion.hpp:155-176), in another order.
// There the rows of a tile pass through LDS a few at a time, so a tile takes a
// load's latency per group of rows, and its outputs leave together at its end:
// all tiles take the same time, the workgroups of the chip store at the same
// time, and neither hides the other.  Here all rows of a tile are staged at once,
// and then each wavefront sums one DM after another and stores it: one latency
// per tile, and the stores spread over the sums.
//
//  * Lane l owns the sample pairs t0 + 2 l + 128 k, one dword of a row each.  Rows
//    are kept in two copies, copy 1 shifted down by one element, so that a DM's
//    pairs are dwords of copy (offset & 1): conflict-free ds_read2st64_b32.
//  * Up to four rows are added as 16-bit pairs (exact while four subband sums stay
//    below 2^16); of the results, the sum of the dwords and that of their upper
//    halves are kept, 32 bits each.
//  * A workgroup takes a run of sample tiles of one beam and coarse DM: the rows'
//    places, and the DMs' places in them, are the same for all of them.
//
// Measured on MI355X, 16 uneven beams of 1536 channels (0.51e9 outputs from 32
// subbands): 0.805 ms against 0.884 for the general kernel, each at its best shape;
// 40 such beams 1.98 against 2.22.  Its parts by themselves: the sums 0.53 (LDS
// reads, 2 bytes per addition at 128 B/clk/CU), staging 0.26, loads and stores alone
// 0.60 (3 GB).  Tried and slower: rows added in pairs before the DMs read them (54
// windows for 32 rows leave room for 256 samples per tile only: 0.826), the next
// tile's loads held in registers through the sums (0.819).
#include "staged_common.hpp"

namespace ddamd {
namespace {

using namespace staged;

template <int RUN> __device__ __forceinline__ void whole_tile(const RowSumF32Params &p, uint32_t logical, uint32_t *lds) {
  constexpr int TS = 64 * RUN;  // samples per tile
  constexpr int ND = RUN / 2;   // dwords (sample pairs) per lane, row and DM
  constexpr int HELD = 5;       // staging chunks in flight per thread
  typedef float f32x2 __attribute__((ext_vector_type(2)));

  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t nwaves = blockDim.x >> 6;
  const uint32_t TD = p.tile_dms;
  const Tile tile = tile_split(logical, p.n_tiles_x, p.n_tiles_y);
  const uint32_t first_tile = tile.x * p.tiles_per_run;
  const uint32_t n_tiles = min(p.tiles_per_run, (p.n_samples + TS - 1) / TS - first_tile);
  const uint32_t t0 = first_tile * TS;
  const uint32_t d0 = tile.y * TD;
  const uint32_t n_dms = min(TD, p.n_dms - d0);
  const uint32_t coarse = tile.z % p.n_coarse;
  const uint32_t sbeam = tile.z / p.n_coarse;
  const uint32_t NR = p.n_rows;
  const uint32_t WE = p.win_floats;  // uint16 elements per window (multiple of 8)
  const uint32_t WD = WE / 2;        // dwords per window copy
  const uint32_t NCH = WE / 8;       // 16-byte chunks per window

  // LDS: windows [NR][2 copies][WD] | rows [NR] | DM addresses [TD][NR]
  u32x4 *rows = reinterpret_cast<u32x4 *>(lds + 2 * NR * WD);
  uint32_t *meta = lds + 2 * NR * WD + 4 * NR;

  // A row's entry: the byte offset of its window in the input, at a multiple of
  // 16, its delay, and what a DM's shift is less by to give its element.
  int past = 0;  // staging loads reach past the input's end
  for (uint32_t r = threadIdx.x; r < NR; r += blockDim.x) {
    const uint32_t in_beam = p.map[(uint64_t)(p.first_sbeam + sbeam) * p.map_pitch + r];
    const float tab = p.table[r];
    const uint32_t shift = shift_of(p.first_dm, p.dm_step, d0, tab);
    const uint64_t off = (uint64_t)in_beam * p.in_beam_pitch + (uint64_t)coarse * p.in_coarse_pitch +
                         (uint64_t)r * p.in_row_pitch + t0 + shift;
    const uint64_t at = off & ~uint64_t(7);
    past |= at + (uint64_t)(n_tiles - 1) * TS + WE + 2 > p.in_floats;
    rows[r] = u32x4{(uint32_t)(2 * at), (uint32_t)(at >> 31), __builtin_bit_cast(uint32_t, tab),
                    shift - (uint32_t)(off - at)};
  }
  past = __syncthreads_or(past);

  // the DMs' LDS byte addresses in the rows
  for (uint32_t d = wave; d < n_dms; d += nwaves) {
    const float dm = __fadd_rn(p.first_dm, __fmul_rn((float)(d0 + d), p.dm_step));
    for (uint32_t r = lane; r < NR; r += 64) {
      const u32x4 e = rows[r];
      const uint32_t bits = e[2];  // through a scalar: a bit cast of a vector's element reads element 0 (hipcc 7.2)
      const uint32_t o = (uint32_t)__fmul_rn(dm, __builtin_bit_cast(float, bits)) - e[3];
      meta[d * NR + r] = 4 * ((2 * r + (o & 1)) * WD + (o >> 1));
    }
  }

  const char *in = reinterpret_cast<const char *>(p.in);
  auto store_chunk = [&](uint32_t r, uint32_t m, const u32x4 &v, uint32_t next) {
    uint32_t *w = lds + 2 * r * WD + 4 * m;
    const u32x4 h = {__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16),
                     __builtin_amdgcn_alignbit(v[3], v[2], 16), __builtin_amdgcn_alignbit(next, v[3], 16)};
    *reinterpret_cast<u32x4 *>(w) = v;
    *reinterpret_cast<u32x4 *>(w + WD) = h;
  };
  // every thread takes chunks blockDim.x apart, HELD of them in flight
  const uint32_t total = NR * NCH;
  auto stage = [&](uint32_t tile_bytes) {
    for (uint32_t x0 = threadIdx.x; x0 < total; x0 += HELD * blockDim.x) {
      u32x4 v[HELD];
      uint32_t next[HELD], r[HELD], m[HELD];
#pragma unroll
      for (int i = 0; i < HELD; ++i) {
        const uint32_t x = min(x0 + i * blockDim.x, total - 1);
        r[i] = __umulhi(x, p.chunk_magic);
        m[i] = x - r[i] * NCH;
        const u32x4 e = rows[r[i]];
        const char *src = in + (((uint64_t)e[1] << 32) | e[0]) + tile_bytes + 16 * m[i];
        v[i] = *reinterpret_cast<const u32x4 *>(src);
        next[i] = *reinterpret_cast<const uint32_t *>(src + 16);
      }
#pragma unroll
      for (int i = 0; i < HELD; ++i)
        if (x0 + i * blockDim.x < total) store_chunk(r[i], m[i], v[i], next[i]);
    }
  };
  // dword by dword, zeros past the end
  auto stage_past = [&](uint32_t tile_bytes) {
    const uint64_t end = (2 * p.in_floats + 3) & ~uint64_t(3);
    for (uint32_t x = threadIdx.x; x < total; x += blockDim.x) {
      const uint32_t r = x / NCH, m = x - r * NCH;
      const u32x4 e = rows[r];
      const uint64_t at = (((uint64_t)e[1] << 32) | e[0]) + tile_bytes + 16 * m;
      uint32_t d[5];
      for (int i = 0; i < 5; ++i) d[i] = at + 4 * i < end ? *reinterpret_cast<const uint32_t *>(in + at + 4 * i) : 0;
      store_chunk(r, m, u32x4{d[0], d[1], d[2], d[3]}, d[4]);
    }
  };

  const char *lane_base = reinterpret_cast<const char *>(lds) + 4 * lane;
  const uint32_t combine = p.combine_rows;
  // The sum of DM d's rows: of the dwords, and of their upper halves.
  auto sum_dm = [&](uint32_t d, uint32_t (&acc)[ND], uint32_t (&upper)[ND]) {
#pragma unroll
    for (int k = 0; k < ND; ++k) acc[k] = upper[k] = 0;
    for (uint32_t r0 = 0; r0 < NR; r0 += 64) {
      // the addresses of 64 rows with one read, taken from their lanes
      const uint32_t some = min(64u, NR - r0);
      const uint32_t words = meta[d * NR + r0 + min(lane, some - 1)];
      auto load = [&](uint32_t r, uint32_t (&x)[ND]) {
        const char *src = lane_base + (uint32_t)__builtin_amdgcn_readlane((int)words, (int)r);
#pragma unroll
        for (int k = 0; k < ND; ++k) x[k] = *reinterpret_cast<const uint32_t *>(src + 256 * k);
      };
      auto add = [&](uint32_t v, int k) {
        acc[k] += v;
        upper[k] += v >> 16;
      };
      uint32_t r = 0;
      if (combine >= 4)
        for (; r + 4 <= some; r += 4) {
          uint32_t x[4][ND];
#pragma unroll
          for (int i = 0; i < 4; ++i) load(r + i, x[i]);
#pragma unroll
          for (int k = 0; k < ND; ++k) add(x[0][k] + x[1][k] + x[2][k] + x[3][k], k);
        }
      if (combine >= 2)
        for (; r + 2 <= some; r += 2) {
          uint32_t x[2][ND];
#pragma unroll
          for (int i = 0; i < 2; ++i) load(r + i, x[i]);
#pragma unroll
          for (int k = 0; k < ND; ++k) add(x[0][k] + x[1][k], k);
        }
      for (; r < some; ++r) {
        uint32_t x[ND];
        load(r, x);
#pragma unroll
        for (int k = 0; k < ND; ++k) add(x[k], k);
      }
    }
  };

  float *out = p.out + (uint64_t)sbeam * p.out_beam_pitch + ((uint64_t)coarse * p.n_dms + d0) * p.out_dm_pitch;
  for (uint32_t k = 0; k < n_tiles; ++k) {
    if (past) stage_past(2 * TS * k);
    else stage(2 * TS * k);
    __syncthreads();
    for (uint32_t d = wave; d < n_dms; d += nwaves) {
      uint32_t acc[ND], upper[ND];
      sum_dm(d, acc, upper);
      float *orow = out + (uint64_t)d * p.out_dm_pitch;
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        const uint32_t t = t0 + TS * k + 2 * lane + 128 * i;
        const f32x2 f = {(float)(acc[i] - (upper[i] << 16)), (float)upper[i]};
        if (p.vec_store && t + 1 < p.n_samples) {
          if (p.nontemporal) __builtin_nontemporal_store(f, reinterpret_cast<f32x2 *>(orow + t));
          else *reinterpret_cast<f32x2 *>(orow + t) = f;
        } else {
          if (t < p.n_samples) orow[t] = f[0];
          if (t + 1 < p.n_samples) orow[t + 1] = f[1];
        }
      }
    }
    __syncthreads();
  }
}

// Persistent form over (beam, tile) descriptors (see rowsum_u8_batch).
template <int RUN>
__global__ void __launch_bounds__(512) rowsum_u16_whole_batch(const RowSumF32Params *__restrict__ beams, const TileQueues q) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  __shared__ uint32_t claimed;
  QueueCursor cur;
  for (;;) {
    const uint32_t t = cur.next(q, &claimed);
    if (t == kNoTile) break;
    const TileDesc d = q.tiles[t];
    whole_tile<RUN>(beams[d.job], d.tile, lds);
  }
}

// One workgroup per listed (job, tile) descriptor, in XCD-aware order.
template <int RUN>
__global__ void __launch_bounds__(512)
rowsum_u16_whole_list(const RowSumF32Params *__restrict__ jobs, const TileDesc *__restrict__ tiles, uint32_t n) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  const TileDesc d = tiles[xcd_logical(blockIdx.x, n)];
  whole_tile<RUN>(jobs[d.job], d.tile, lds);
}

template <typename F> hipError_t dispatch(const Geometry &g, F &&f) {
  switch (g.items_d0) {
  case 4: return f(std::integral_constant<int, 4>{});
  case 8: return f(std::integral_constant<int, 8>{});
  case 16: return f(std::integral_constant<int, 16>{});
  default: return hipErrorInvalidValue;
  }
}

} // namespace

hipError_t launch_rowsum_u16_whole_batch(const RowSumF32Params *d_jobs, const TileQueues &q, const Geometry &g,
                                         uint32_t workgroups, hipStream_t stream) {
  return dispatch(g, [&](auto run) {
    hipLaunchKernelGGL((rowsum_u16_whole_batch<run.value>), dim3(workgroups), dim3(64 * g.threads_d1), g.lds_bytes, stream,
                       d_jobs, q);
    return hipGetLastError();
  });
}

hipError_t launch_rowsum_u16_whole_list(const RowSumF32Params *d_jobs, const TileDesc *d_tiles, uint32_t n,
                                        const Geometry &g, hipStream_t stream) {
  return dispatch(g, [&](auto run) {
    hipLaunchKernelGGL((rowsum_u16_whole_list<run.value>), dim3(n), dim3(64 * g.threads_d1), g.lds_bytes, stream, d_jobs,
                       d_tiles, n);
    return hipGetLastError();
  });
}

hipError_t rowsum_u16_whole_batch_occupancy(const Geometry &g, int *per_cu) {
  return dispatch(g, [&](auto run) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rowsum_u16_whole_batch<run.value>,
                                                        (int)(64 * g.threads_d1), (size_t)g.lds_bytes);
  });
}

} // namespace ddamd
