// kernels_f32_staged.hip -- pipelined shifted row sums over float rows.
//
// Same operation and arithmetic as kernels_f32.hip: step two
// (include/Dedispersion.hpp:155-176), and the single step and step one over
// float input (:70-153 with I = float).  A slice's rows (subbands, or live
// channels) are added in order into float accumulators that start at 0,
// bit-identical to the reference's sequential float sum for any input.
//
//  * Lane l owns the sample quads t0 + 4l + 256k, each read with one
//    ds_read_b128.  A DM's offset into a row's window is any sample and a 16-byte
//    read wants 16-byte alignment (190 B/clk/CU against 16 without it, and 120 of
//    the 4- and 8-byte reads that any offset allows), so a row is kept in four
//    copies, copy c shifted down by c samples.
//  * The copies are four loads of the input, each a sample further, that go to LDS
//    without passing through registers (global_load_lds), a group of `unroll`
//    rows ahead of the sums, into the other of two buffers.
//  * A row's integer shifts for the tile's DMs are computed once, by the
//    wavefront that stages it, and published through LDS as byte addresses.
//  * Workgroups are ordered XCD-aware (staged_common.hpp).
//
// Tiles of few DMs in large grids run kernels_f32_narrow.hip, one copy of a row.
//
// Bound by the LDS reads, 4 bytes per addition, at 16 bytes per lane.  Measured on
// MI355X against one copy per row read 4 bytes at a time (us, one to the other, the
// same inputs and tile shape; then each at its best shape): 768 channels x 512 DMs x
// 12288 samples 1648 -> 538, best 381 -> 328; 256 x 2048 x 24576 best 690 -> 586
// (22e12 additions per second); step one, 32 channels x 32 coarse DMs x 20000
// samples x 32 subbands, best 64.2 -> 51.6; step two, 32 subbands x 2048 DMs x
// 24576, 124 -> 114 (its loads and stores alone take 100, its sums 73).
#include "staged_common.hpp"

namespace ddamd {
namespace {

using namespace staged;

// One (slice, DM tile, sample tile) block: logical tile index `logical` of
// the launch described by p (DM tile fastest).
// MANY: a slice may have more rows than kF32Rows, and they are listed in LDS that
// many at a time (a loop that costs 5-10 registers: a wavefront per SIMD at RUN 8 and
// 4 DMs, 231 against 201 us over both steps of 1536 channels x 2048 DMs x 24576).
template <int RUN, int DPW, bool MANY>
__device__ __forceinline__ void f32_tile(const RowSumF32Params &p, uint32_t logical, float *ldsf) {
  constexpr int TS = 64 * RUN;
  constexpr int NQ = RUN / 4;       // sample quads per lane
  constexpr int SPW = kStagedSlotsPerWave;
  constexpr int CPL = RUN / 4 + 1;  // 16-byte staging loads per lane, copy and row

  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t nwaves = blockDim.x >> 6;
  const uint32_t TD = nwaves * DPW;
  const Tile tile = tile_split(logical, p.n_tiles_x, p.n_tiles_y);
  const uint32_t t0 = tile.x * TS;
  const uint32_t d0 = tile.y * TD;
  const uint32_t dw = wave * DPW;
  // a wavefront whose DMs all lie past the last DM (a partial DM tile) only stages rows
  const bool busy = d0 + dw < p.n_dms;
  const uint32_t inner = tile.z % p.n_coarse;
  const uint32_t outer = tile.z / p.n_coarse;
  const uint32_t G = uniform(p.unroll);
  const uint32_t WF = p.win_floats;  // floats per copy of a window (multiple of 4)
  const uint32_t NCH = WF / 4;
  const uint32_t dmax = p.n_dms - 1;
  const uint32_t *list = p.rows ? p.rows + (uint64_t)inner * p.rows_pitch : nullptr;
  const uint32_t nrows = list ? uniform(p.rows_count[inner]) : p.n_rows;
  const uint32_t most = list ? p.rows_pitch : p.n_rows;
  const uint32_t slots = MANY ? min(most, kF32Rows) : most;  // row entries in LDS

  // LDS: windows [2][G][4 copies][WF] | rows [slots] | DM addresses [2][G][TD]
  uint32_t *lds = reinterpret_cast<uint32_t *>(ldsf);
  u32x4 *rows = reinterpret_cast<u32x4 *>(lds + 8 * G * WF);
  uint32_t *meta = lds + 8 * G * WF + 4 * slots;

  // A row's entry: its window's byte offset in the input (its top bit: the
  // copies reach past the input's end), its delay and its shift at the first DM.
  auto list_rows = [&](uint32_t first, uint32_t n) {
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
      const uint32_t row = list ? list[first + k] : first + k;
      const uint32_t in_beam = p.map ? p.map[(uint64_t)(p.first_sbeam + outer) * p.map_pitch + row] : outer;
      const float tab = p.table[row];
      const uint32_t shift = shift_of(p.first_dm, p.dm_step, d0, tab);
      const uint64_t off = (uint64_t)in_beam * p.in_beam_pitch + (uint64_t)inner * p.in_coarse_pitch +
                           (uint64_t)row * p.in_row_pitch + t0 + shift;
      const uint32_t past = off + WF + 3 > p.in_floats ? 0x80000000u : 0u;
      rows[k] = u32x4{(uint32_t)(4 * off), (uint32_t)(off >> 30) | past, __builtin_bit_cast(uint32_t, tab), shift};
    }
    __syncthreads();
  };

  // ---- staging: wavefront w sends for rows w and w + nwaves of a group.  The
  // loads are written in assembly because the compiler, which knows only that
  // they write LDS, would wait for them before any LDS read; they have no output
  // registers, and `arrived` waits for them. ----
  const float dm_value = __fadd_rn(p.first_dm, __fmul_rn((float)min(d0 + lane, dmax), p.dm_step));
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)lds;
  auto arrived = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  auto send_for = [&](uint32_t buf, uint32_t k0, uint32_t nn) {
    u32x4 e[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) e[s] = rows[k0 + min(wave + s * nwaves, nn - 1)];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      const uint32_t g = wave + s * nwaves;
      if (g < nn) {
        const uint32_t at = 4 * (buf * G + g) * WF;  // the row's copies, in floats
        const bool past = (int)uniform(e[s][1]) < 0;
        const uint64_t first = ((uint64_t)uniform(e[s][1] & 0x7FFFFFFFu) << 32) | uniform(e[s][0]);
        if (!past) {
          const char *src = reinterpret_cast<const char *>(p.in) + first + 16 * lane;
#pragma unroll
          for (int c = 0; c < CPL; ++c)
            if (lane + 64 * c < NCH) {
#pragma unroll
              for (int copy = 0; copy < 4; ++copy)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(
                                 uniform(lds_base + 4 * (at + copy * WF) + 1024 * c)),
                             "v"(src + 4 * copy + 1024 * c)
                             : "memory", "m0");
            }
        } else {  // sample by sample, zeros past the end
          const __amdgpu_buffer_rsrc_t rsrc =
              make_rsrc(reinterpret_cast<const char *>(p.in) + first, records_from_floats(p.in_floats, first / 4));
          for (uint32_t x = lane; x < 4 * WF; x += 64)
            lds[at + x] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, 4 * (x % WF + x / WF), 0, 0);
        }
        // the DM's LDS byte address: copy (offset & 3), quad offset >> 2
        const uint32_t bits = e[s][2];  // through a scalar: a bit cast of a vector's element reads element 0 (hipcc 7.2)
        const uint32_t o = (uint32_t)__fmul_rn(dm_value, __builtin_bit_cast(float, bits)) - e[s][3];
        if (lane < TD) meta[(buf * G + g) * TD + lane] = 4 * (at + (o & 3) * WF) + 16 * (o >> 2);
      }
    }
  };

  f32x4 acc[DPW][NQ];
#pragma unroll
  for (int j = 0; j < DPW; ++j)
#pragma unroll
    for (int k = 0; k < NQ; ++k) acc[j][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // DM after DM and row after row; the quads of the next DM (of the next row
  // after the last) are read before a DM's are added, and a row's addresses
  // while the row before it is.  The order is kept as written.
  const char *lane_base = reinterpret_cast<const char *>(lds) + 16 * lane;
  auto compute = [&](uint32_t buf, uint32_t n) {
    const uint32_t *words = meta + buf * G * TD + dw;  // broadcast reads
    constexpr int NB = DPW > 1 ? 2 : 1;
    f32x4 x[NB][NQ];
    uint32_t w[DPW], wn[DPW];
    auto fetch = [&](uint32_t g, uint32_t (&a)[DPW]) {
#pragma unroll
      for (int j = 0; j < DPW; ++j) a[j] = words[g * TD + j];
    };
    auto load = [&](uint32_t word, f32x4 (&v)[NQ]) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) v[k] = *reinterpret_cast<const f32x4 *>(lane_base + word + 1024 * k);
    };
    fetch(0, wn);
    if constexpr (NB > 1) load(wn[0], x[0]);
    for (uint32_t g = 0; g < n; ++g) {
#pragma unroll
      for (int j = 0; j < DPW; ++j) w[j] = wn[j];
      fetch(min(g + 1, n - 1), wn);
#pragma unroll
      for (int j = 0; j < DPW; ++j) {
        if constexpr (NB == 1) load(w[j], x[0]);
        else if (j + 1 < DPW) load(w[j + 1], x[(j + 1) % NB]);
        else load(wn[0], x[0]);
#pragma unroll
        for (int k = 0; k < NQ; ++k)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[j][k][e] += x[j % NB][k][e];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  uint32_t cur = 0;
  auto sum_rows = [&](uint32_t first, uint32_t n) {
    list_rows(first, n);
    if (n > 0) {
      send_for(cur, 0, min(G, n));
      arrived();
    }
    __syncthreads();
    for (uint32_t s0 = 0; s0 < n; s0 += G) {
      const uint32_t sn = s0 + G;
      if (sn < n) send_for(cur ^ 1, sn, min(G, n - sn));
      if (busy) compute(cur, min(G, n - s0));
      arrived();
      __syncthreads();
      cur ^= 1;
    }
  };
  if constexpr (MANY) {
    for (uint32_t first = 0; first < nrows; first += kF32Rows) sum_rows(first, min(nrows - first, kF32Rows));
  } else {
    sum_rows(0, nrows);
  }
  if (!busy) return;

#pragma unroll
  for (int j = 0; j < DPW; ++j) {
    const uint32_t dm = d0 + dw + j;
    if (dm >= p.n_dms) continue;
    float *orow = p.out + (uint64_t)outer * p.out_beam_pitch + (uint64_t)inner * p.out_inner_pitch +
                  (uint64_t)dm * p.out_dm_pitch;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const uint32_t t = t0 + 4 * lane + 256 * k;
      if (p.vec_store && t + 3 < p.n_samples) {
        if (p.nontemporal) __builtin_nontemporal_store(acc[j][k], reinterpret_cast<f32x4 *>(orow + t));
        else *reinterpret_cast<f32x4 *>(orow + t) = acc[j][k];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (t + e < p.n_samples) orow[t + e] = acc[j][k][e];
      }
    }
  }
}

template <int RUN, int DPW, bool MANY>
__global__ void __launch_bounds__(512) rowsum_f32_staged(const RowSumF32Params p) {
  extern __shared__ __attribute__((aligned(16))) float ldsf[];
  f32_tile<RUN, DPW, MANY>(p, xcd_logical(blockIdx.x, p.n_tiles), ldsf);
}

// Persistent form over (beam, tile) descriptors (see rowsum_u8_batch).
template <int RUN, int DPW, bool MANY>
__global__ void __launch_bounds__(512) rowsum_f32_batch(const RowSumF32Params *__restrict__ beams,
                                                          const TileQueues q) {
  extern __shared__ __attribute__((aligned(16))) float ldsf[];
  __shared__ uint32_t claimed;
  QueueCursor cur;
  for (;;) {
    const uint32_t t = cur.next(q, &claimed);
    if (t == kNoTile) break;
    const TileDesc d = q.tiles[t];
    f32_tile<RUN, DPW, MANY>(beams[d.job], d.tile, ldsf);
  }
}

// One workgroup per listed (job, tile) descriptor, in XCD-aware order.
template <int RUN, int DPW, bool MANY>
__global__ void __launch_bounds__(512) rowsum_f32_list(const RowSumF32Params *__restrict__ jobs, const TileDesc *__restrict__ tiles,
                                                      uint32_t n) {
  extern __shared__ __attribute__((aligned(16))) float ldsf[];
  const TileDesc d = tiles[xcd_logical(blockIdx.x, n)];
  f32_tile<RUN, DPW, MANY>(jobs[d.job], d.tile, ldsf);
}

// Calls f(RUN, DPW, MANY) with the compile-time constants of geometry g.
template <typename F> hipError_t dispatch(const Geometry &g, F &&shaped) {
  auto f = [&](auto run, auto dpw) -> hipError_t {
    return g.many ? shaped(run, dpw, std::true_type{}) : shaped(run, dpw, std::false_type{});
  };
  auto by_dpw = [&](auto run) -> hipError_t {
    switch (g.items_d1) {
    case 1: return f(run, std::integral_constant<int, 1>{});
    case 2: return f(run, std::integral_constant<int, 2>{});
    case 4: return f(run, std::integral_constant<int, 4>{});
    case 8: return f(run, std::integral_constant<int, 8>{});
    default: return hipErrorInvalidValue;
    }
  };
  switch (g.items_d0) {
  case 4: return by_dpw(std::integral_constant<int, 4>{});
  case 8: return by_dpw(std::integral_constant<int, 8>{});
  case 16: return by_dpw(std::integral_constant<int, 16>{});
  default: return hipErrorInvalidValue;
  }
}

} // namespace

hipError_t launch_rowsum_f32_staged(const RowSumF32Params &p, const Geometry &g, hipStream_t stream) {
  if (g.narrow) return launch_rowsum_f32_narrow(p, g, stream);
  return dispatch(g, [&](auto run, auto dpw, auto many) {
    hipLaunchKernelGGL((rowsum_f32_staged<run.value, dpw.value, many.value>), dim3(p.n_tiles), dim3(64 * g.threads_d1),
                       g.lds_bytes, stream, p);
    return hipGetLastError();
  });
}

hipError_t launch_rowsum_f32_batch(const RowSumF32Params *d_jobs, const TileQueues &q, const Geometry &g,
                                   uint32_t workgroups, hipStream_t stream) {
  if (g.narrow) return launch_rowsum_f32_narrow_batch(d_jobs, q, g, workgroups, stream);
  return dispatch(g, [&](auto run, auto dpw, auto many) {
    hipLaunchKernelGGL((rowsum_f32_batch<run.value, dpw.value, many.value>), dim3(workgroups), dim3(64 * g.threads_d1),
                       g.lds_bytes, stream, d_jobs, q);
    return hipGetLastError();
  });
}

hipError_t launch_rowsum_f32_list(const RowSumF32Params *d_jobs, const TileDesc *d_tiles, uint32_t n, const Geometry &g,
                                  hipStream_t stream) {
  if (g.narrow) return launch_rowsum_f32_narrow_list(d_jobs, d_tiles, n, g, stream);
  return dispatch(g, [&](auto run, auto dpw, auto many) {
    hipLaunchKernelGGL((rowsum_f32_list<run.value, dpw.value, many.value>), dim3(n), dim3(64 * g.threads_d1), g.lds_bytes, stream,
                       d_jobs, d_tiles, n);
    return hipGetLastError();
  });
}

hipError_t rowsum_f32_batch_occupancy(const Geometry &g, int *per_cu) {
  if (g.narrow) return rowsum_f32_narrow_batch_occupancy(g, per_cu);
  return dispatch(g, [&](auto run, auto dpw, auto many) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, rowsum_f32_batch<run.value, dpw.value, many.value>,
                                                        (int)(64 * g.threads_d1), (size_t)g.lds_bytes);
  });
}

// Zeroes the claim counters of the work queues (a kernel rather than a
// memset so that the reset can sit in a captured graph).
__global__ void clear_words(uint32_t *words, uint32_t n) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) words[i] = 0;
}

hipError_t launch_clear_words(uint32_t *d_words, uint32_t n, hipStream_t stream) {
  hipLaunchKernelGGL(clear_words, dim3(1), dim3(256), 0, stream, d_words, n);
  return hipGetLastError();
}

} // namespace ddamd
