// kernels_u8_matrix.hip -- shifted row sums over uint8 rows on the matrix
// cores (single-step dedispersion, include/Dedispersion.hpp:70-109, and step
// one, :111-153).
//
// The tile and its results are those of kernels_u8_staged.hip.  The summation
// is a product of small integer matrices: write sample t of a tile as
// t = 8 c + p (column c, phase p) and take two DMs d at a time.  Then
//     out[(d, p)][c] = sum over rows r and k < 32 of
//                      A_r[(d, p)][k] * in[r][base_r + 8 c + k],
// where A_r[(d, p)][k] is 1 at k = shift(r, d) - base_r + p and 0 elsewhere:
// one v_smfmac_i32_16x16x128_i8 adds four rows to 2 DMs x 128 samples.  Its A
// operand is 2:4 sparse, which a matrix with one 1 per 32 always is, so the
// unit works on 128 values of k in the time of 64.  base_r is the first DM's
// shift rounded down to 8 samples, so every B operand is two 8-byte LDS reads
// of consecutive bytes and no lane needs its own alignment: the rows are
// staged once, not in four shifted copies.  A row whose shifts reach past the
// 32 samples (shift spread over the wavefront's DMs + 14 >= 32) takes further
// windows of 32.
//
// Sums are exact in 32 bits.  The unit multiplies signed bytes, so byte rows
// are staged with their top bit flipped (x - 128) and the accumulators start
// at 128 x rows; packed samples are at most 15 and need neither.
//
// Measured, 1459 rows, 2048 DMs x 24576 samples: 1.08 ms against 1.96 for the
// vector form (68 T additions/s against 37); 1024 DMs x 12288 2-bit samples: 0.39
// ms against 0.69.  Bounds, by the counters of the larger: the matrix cores are busy 43%
// of the cycles, VALU issue 44% and LDS reads 60%, at two wavefronts per SIMD (128 sums
// per lane).  A product of 16 cycles starts every 37, a fifth of which is staging; the
// rest is the vector instructions that build the A operands (a v_smfmac holds up its
// own wavefront's) and the reads.  The 32x32x64 shape overlaps better but draws so much
// power that the clock falls to 1.5 GHz (24 ns for the work that two of these do in 17).
#include "staged_common.hpp"
#include "u8_unpack.hpp"

namespace ddamd {
namespace {

using namespace staged;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr uint32_t kNoPosition = 0x40000000u;  // offset of the DMs of a row that is missing

template <int RUN, int DPW, bool PACKED, bool WIDE>
__device__ __forceinline__ void u8_matrix_tile(const RowSumU8Params &p, uint32_t logical, uint32_t *lds) {
  constexpr int NT = RUN / 2;   // 16-column (128-sample) blocks of the tile
  constexpr int MT = DPW / 2;   // blocks of two DMs of the wavefront
  constexpr int TS = 64 * RUN;  // samples per tile
  constexpr int SPW = kStagedSlotsPerWave;
  constexpr int CPL = kU8StagedChunks;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t nwaves = blockDim.x >> 6;
  const uint32_t TD = nwaves * DPW;
  const Tile tile = tile_split(logical, p.n_tiles_x, p.n_tiles_y);
  const uint32_t t0 = tile.x * TS;
  const uint32_t d0 = tile.y * TD;
  const uint32_t dw = wave * DPW;  // first DM of this wavefront, relative to d0
  // a wavefront whose DMs all lie past the last DM (a partial DM tile) only stages rows
  const bool busy = d0 + dw < p.n_dms;
  const uint32_t group = tile.z % p.n_groups;
  const uint32_t beam = tile.z / p.n_groups;
  const uint32_t nlive = uniform(p.live_count[group]);
  const uint32_t *live = p.live + (uint64_t)group * p.live_pitch;
  const uint32_t G = uniform(p.unroll);
  const uint32_t NCH = p.win_bytes / 16;                             // 16-byte chunks per window
  const uint32_t WD = (p.win_bytes + kU8MatrixReach) / 4;            // dwords between windows
  const uint32_t lf = PACKED ? p.in_log2f : 0u;                      // log2 of samples per input byte
  const uint32_t dmax = p.n_dms - 1;

  // LDS: raw windows [G][WD] | rows [live_pitch] | windows [2][G][WD] | words
  // [2][G + 1][TD + nwaves] and two rows more: the offset of every DM from its wavefront's base,
  // then every wavefront's base
  const uint32_t rows_off = G * WD, win_off = rows_off + 4 * p.live_pitch;
  u32x4 *rows = reinterpret_cast<u32x4 *>(lds + rows_off);
  uint32_t *windows = lds + win_off;
  uint32_t *meta = windows + 2 * G * WD;
  const uint32_t MW = TD + nwaves, MB = (((G + 3) & ~3u) + 4) * MW;

  // A row's window starts at the dword that holds its first sample; packed
  // rows hold 1 << lf samples per byte.  Entry: the window's byte offset in the
  // input (its top bit: the window reaches past the input's end), the row's
  // delay and, negated, the window's first sample relative to t0.
  const uint32_t raw_chunks = ((16 * NCH >> lf) + 15) / 16;  // 16-byte pieces of a window in the input
  const uint64_t in_end = (p.in_bytes + 3) & ~uint64_t(3);   // the dword holding the last byte is safe to read
  for (uint32_t k = threadIdx.x; k < nlive; k += blockDim.x) {
    const uint32_t row = live[k];
    const uint32_t in_beam = p.map ? p.map[(uint64_t)(p.first_sbeam + beam) * p.map_pitch + row] : beam;
    const float tab = p.table[row];
    const uint32_t shift = shift_of(p.first_dm, p.dm_step, d0, tab), x = t0 + shift;
    const uint64_t off = (uint64_t)in_beam * p.in_beam_pitch + (uint64_t)row * p.in_row_pitch + (x >> lf);
    const uint64_t a0 = off & ~uint64_t(3);
    const uint32_t slop = ((uint32_t)(off & 3) << lf) + (x & ((1u << lf) - 1));
    const uint32_t past = a0 + 16 * raw_chunks > in_end ? 0x80000000u : 0u;
    rows[k] = u32x4{(uint32_t)a0, (uint32_t)(a0 >> 32) | past, __builtin_bit_cast(uint32_t, tab), shift - slop};
  }
  __syncthreads();

  // ---- staging: wavefront w stages rows w and w + nwaves of a group.  The
  // input goes to the raw windows without passing through registers
  // (global_load_lds); a group later, when it has arrived, the wavefront turns
  // it into signed bytes in the group's windows and sends for the next group.
  // The load is written in assembly because the compiler, which knows only
  // that it writes LDS, would wait for it before any LDS read; it has no
  // output registers, and `arrived` waits for it. ----
  const float dm_value = __fadd_rn(p.first_dm, __fmul_rn((float)min(d0 + lane, dmax), p.dm_step));
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint32_t *)lds;
  auto arrived = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  const uint32_t lane_dst = uniform(lds_base + 4 * wave * WD);
  auto send_for = [&](uint32_t k0, uint32_t nn) {
    u32x4 e[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) e[s] = rows[k0 + min(wave + s * nwaves, nn - 1)];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      // a window that reaches past the input's end is read when it is due
      if (wave + s * nwaves < nn && (int)uniform(e[s][1]) >= 0) {
        const uint8_t *src = p.in + (((uint64_t)e[s][1] << 32) | e[s][0]) + 16 * lane;
        const uint32_t dst = lane_dst + 4 * s * nwaves * WD;
        if (lane < raw_chunks)
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory", "m0");
        if (lane + 64 < raw_chunks)
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst + 1024), "v"(src + 1024)
                       : "memory", "m0");
      }
    }
  };
  auto stage = [&](uint32_t buf, uint32_t k0, uint32_t nn) {
    // everything that is read first, for both rows
    u32x4 e[SPW], v[SPW][CPL];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      const uint32_t g = min(wave + s * nwaves, nn - 1);
      e[s] = rows[k0 + g];
      const uint32_t *raw = lds + g * WD;
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const uint32_t m = lane + 64 * c;
        if (m < NCH) {
          if (!PACKED || lf == 0) {
            v[s][c] = *reinterpret_cast<const u32x4 *>(raw + 4 * m);
          } else {  // the dwords that hold the chunk's 16 samples
            const uint32_t pd = (16 * m >> lf) / 4;
            v[s][c][0] = raw[pd];
            if (lf == 1) v[s][c][1] = raw[pd + 1];
          }
        }
      }
    }
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      if ((int)uniform(e[s][1]) < 0) {
        const uint64_t a0 = ((uint64_t)uniform(e[s][1] & 0x7FFFFFFFu) << 32) | uniform(e[s][0]);
        const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(p.in + a0, records_from(p.in_bytes, a0));
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const uint32_t m = lane + 64 * c;
          const uint32_t pd = PACKED ? (16 * m >> lf) / 4 : 4 * m;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[s][c][q] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, 4 * (pd + q), 0, 0);
        }
      }
    }
    // every DM's offset from its wavefront's base, which is the first DM's
    // offset rounded down to 8
    uint32_t o[SPW], base[SPW];
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      const uint32_t bits = e[s][2];  // through a scalar: a bit cast of a vector's element reads element 0 (hipcc 7.2)
      o[s] = (uint32_t)__fmul_rn(dm_value, __builtin_bit_cast(float, bits)) - e[s][3];
      base[s] = (uint32_t)__builtin_amdgcn_ds_swizzle((int)o[s], 31 & ~(DPW - 1)) & ~7u;
    }
#pragma unroll
    for (int s = 0; s < SPW; ++s) {
      const uint32_t g = wave + s * nwaves;
      uint32_t *words = meta + buf * MB + g * MW;
      if (g < nn) {
        const uint32_t at = (buf * G + g) * WD;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const uint32_t m = lane + 64 * c;
          if (m < NCH) {
            u32x4 x = v[s][c] ^ 0x80808080u;
            if constexpr (PACKED) {
              if (lf != 0) {
                uint32_t u[4] = {}, next;
                if (lf == 1) unpack_group<1>(v[s][c], m, u, next);
                else if (lf == 2) unpack_group<2>(v[s][c], m, u, next);
                else unpack_group<3>(v[s][c], m, u, next);
                x = u32x4{u[0], u[1], u[2], u[3]};
              }
            }
            *reinterpret_cast<u32x4 *>(windows + at + 4 * m) = x;
          }
        }
        if (lane < TD) words[lane] = o[s] - base[s];
        if (lane < TD && lane % DPW == 0) words[TD + lane / DPW] = 4 * (win_off + at) + base[s];
      }
    }
    // the rows that are missing to whole sets of four: no position is in any window
    for (uint32_t g = nn + wave; g < ((nn + 3) & ~3u); g += nwaves) {
      uint32_t *words = meta + buf * MB + g * MW;
      if (lane < TD) words[lane] = kNoPosition;
      if (lane < nwaves) words[TD + lane] = 4 * win_off;
    }
  };

  // ---- accumulation: lane l holds column l % 16 and, for A, row l % 16 of
  // the block: DM l / 8 % 2, phase l % 8, of staged row l / 16 of the four ----
  v4i acc[MT][NT];
  const int bias = lf == 0 ? 128 * (int)nlive : 0;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = bias;

  // B operands: lanes 0-31 hold rows 0 and 2 of the four, lanes 32-63 rows 1
  // and 3.  Of a row's 32 samples, the even 16 lanes read the 8-byte chunks 0
  // and 2, the odd ones 1 and 3 (one ds_read2_b64: chunks side by side would be
  // merged into 16-byte reads at 8-byte alignment, 16 against 120 B/clk/CU); the
  // A operand has its chunks in the same order.
  const uint32_t phase = lane & 7, quarter = lane >> 4;
  const char *lane_base = reinterpret_cast<const char *>(lds) + 8 * (lane & 15) + 8 * (quarter & 1);

  // The A operand for a 1 at position `pos` of the row's 32 (none past 31).
  // Of each four k, two bytes are stored, with the two k that they stand for:
  // (q, 3) and the 1 in the first byte for q = pos % 4 < 3, (2, 3) and the
  // second byte for q = 3.  Bytes u = pos % 8 of the tables hold the bit of
  // the 1 in its dword and the index pairs of two groups of four.
  auto one_hot = [&](uint32_t pos, v4i &a, int &idx) {
    const uint32_t u = pos & 7, w = pos >> 3;
    const uint32_t v = 1u << __builtin_amdgcn_perm(0x18101010u, 0x08000000u, u);
    const uint32_t pair = __builtin_amdgcn_perm(0xEEEEDDCCu, 0xEEEEDDCCu, u);
    idx = (int)__builtin_amdgcn_perm(pair, pair, 0u);
    a[0] = w == 0 ? (int)v : 0;
    a[1] = w == 2 ? (int)v : 0;
    a[2] = w == 1 ? (int)v : 0;
    a[3] = w == 3 ? (int)v : 0;
  };
  auto load = [&](const char *r0, const char *r1, int j) {
    const u32x2 x0 = *reinterpret_cast<const u32x2 *>(r0 + 128 * j);
    const u32x2 x1 = *reinterpret_cast<const u32x2 *>(r0 + 128 * j + 16);
    const u32x2 y0 = *reinterpret_cast<const u32x2 *>(r1 + 128 * j);
    const u32x2 y1 = *reinterpret_cast<const u32x2 *>(r1 + 128 * j + 16);
    return v8i{(int)x0[0], (int)x0[1], (int)x1[0], (int)x1[1], (int)y0[0], (int)y0[1], (int)y1[0], (int)y1[1]};
  };
  // One window of four rows: the positions in it and the A operands, and where
  // it starts in this lane's two rows.
  struct Set {
    uint32_t pos[MT];
    v4i a[MT];
    int idx[MT];
    const char *src0, *src1;
  };
  // B operands in registers: this block's and those read ahead (the largest
  // shape has room for fewer beside packed rows or further windows)
  constexpr int NB = NT < 4 ? NT : MT * NT == 32 && (PACKED || WIDE) ? 2 : 4;
  auto compute = [&](uint32_t buf, uint32_t n) {
    // this lane's words of the next four rows: MT offsets and two bases
    const uint32_t *words = meta + buf * MB + quarter * MW + dw + ((lane >> 3) & 1);
    const uint32_t *bases = meta + buf * MB + (quarter >> 1) * MW + TD + wave;
    uint32_t off[MT], at0, at1;
    auto fetch = [&]() {
#pragma unroll
      for (int i = 0; i < MT; ++i) off[i] = words[2 * i];
      at0 = bases[0];
      at1 = bases[2 * MW];
      words += 4 * MW;
      bases += 4 * MW;
    };
    // Opens what follows set c in x -- the next window of its rows when they
    // have one (the last DMs' positions are the furthest; a missing row's stays
    // above kNoPosition / 2 over the at most 66 windows of a row, a position that
    // has been passed wraps to the top), else the first window of the next four rows, whose
    // successors' words it fetches.  No branches, which would have the compiler
    // copy the fetched words and wait for them here (past the last rows, it
    // opens them again).
    uint32_t left = (n + 3) / 4;  // sets not yet opened
    auto open = [&](const Set &c, Set &x) {
      const bool on = WIDE && __ballot(c.pos[MT - 1] >= 32 && c.pos[MT - 1] < kNoPosition / 2) != 0;
      x.src0 = on ? c.src0 + 32 : lane_base + at0;
      x.src1 = on ? c.src1 + 32 : lane_base + at1;
#pragma unroll
      for (int i = 0; i < MT; ++i) x.pos[i] = on ? c.pos[i] - 32 : off[i] + phase;
      const uint32_t back = on || left <= 1 ? 4 * MW : 0;
      words -= back;
      bases -= back;
      fetch();
      const bool more = on || left > 0;
      left -= on || left == 0 ? 0 : 1;
      return more;
    };
    // The products of window c, block after block of columns; in between, which
    // depend on neither, the A operands of the window after it are built and its
    // first B operands read.  The order is kept as written (the scheduler would
    // move the reads next to their uses and wait for each).
    v8i b[NB];
    auto step = [&](Set &c, Set &x) {
      bool more = false;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (j == 0) more = open(c, x);
        b[(j + NB - 1) % NB] = j + NB - 1 < NT ? load(c.src0, c.src1, j + NB - 1) : load(x.src0, x.src1, j + NB - 1 - NT);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if (j == ((i + 1) * NT > MT ? (i + 1) * NT / MT - 1 : 0)) one_hot(x.pos[i], x.a[i], x.idx[i]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[i][j] = __builtin_amdgcn_smfmac_i32_16x16x128_i8(c.a[i], b[j % NB], acc[i][j], c.idx[i], 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      return more;
    };
    Set u, v;
    fetch();
    v.pos[MT - 1] = 0;  // no set before the first
    v.src0 = v.src1 = lane_base;
    open(v, u);
#pragma unroll
    for (int j = 0; j < NB - 1; ++j) b[j] = load(u.src0, u.src1, j);
#pragma unroll
    for (int i = 0; i < MT; ++i) one_hot(u.pos[i], u.a[i], u.idx[i]);
    while (step(u, v) && step(v, u)) {
    }
  };

  // ---- pipeline over groups of rows ----
  uint32_t cur = 0;
  if (nlive > 0) {
    send_for(0, min(G, nlive));
    arrived();
    stage(0, 0, min(G, nlive));
    if (G < nlive) send_for(G, min(G, nlive - G));
  }
  __syncthreads();
  // Wavefronts w and w + 4 share a SIMD: one stages before its products and the
  // other after them, so that either's staging runs beside the other's products
  // (staged by all at the end, it held the matrix units back for a sixth of the
  // time).
  const bool early = wave >= 4;
  for (uint32_t k0 = 0; k0 < nlive; k0 += G) {
    const uint32_t k1 = k0 + G, k2 = k1 + G;
    auto next_group = [&]() {
      arrived();
      stage(cur ^ 1, k1, min(G, nlive - k1));
      if (k2 < nlive) send_for(k2, min(G, nlive - k2));
    };
    if (early && k1 < nlive) next_group();
    if (busy) compute(cur, min(G, nlive - k0));
    if (!early && k1 < nlive) next_group();
    __syncthreads();
    cur ^= 1;
  }
  if (!busy) return;

  // register e of a block: DM lane / 32, sample 8 (lane % 16) + 4 (lane / 16 % 2) + e
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const uint32_t dm = d0 + dw + 2 * i + (lane >> 5);
    if (dm >= p.n_dms) continue;
    const uint64_t row = (uint64_t)beam * p.out_beam_pitch + (uint64_t)group * p.out_group_pitch +
                         (uint64_t)dm * p.out_dm_pitch;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const uint32_t t = t0 + 128 * j + 8 * (lane & 15) + 4 * (quarter & 1);
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (uint32_t)acc[i][j][e];
      if (p.out_u16) {
        // compact output: the four sums as uint16 (each below 2^16)
        uint16_t *orow = reinterpret_cast<uint16_t *>(p.out) + row;
        if (p.vec_store && t + 3 < p.n_samples) {
          *reinterpret_cast<u32x2 *>(orow + t) = u32x2{v[0] | (v[1] << 16), v[2] | (v[3] << 16)};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t + e < p.n_samples) orow[t + e] = (uint16_t)v[e];
        }
      } else {
        float *orow = p.out + row;
        if (p.vec_store && t + 3 < p.n_samples) {
          const f32x4 f = {(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
          if (p.nontemporal) __builtin_nontemporal_store(f, reinterpret_cast<f32x4 *>(orow + t));
          else *reinterpret_cast<f32x4 *>(orow + t) = f;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t + e < p.n_samples) orow[t + e] = (float)v[e];
        }
      }
    }
  }
}

template <int RUN, int DPW, bool PACKED, bool WIDE>
__global__ void __launch_bounds__(512) rowsum_u8_matrix(const RowSumU8Params p) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  u8_matrix_tile<RUN, DPW, PACKED, WIDE>(p, xcd_logical(blockIdx.x, p.n_tiles), lds);
}

// Persistent form over (job, tile) descriptors (see rowsum_u8_batch).
template <int RUN, int DPW, bool PACKED, bool WIDE>
__global__ void __launch_bounds__(512)
rowsum_u8_matrix_batch(const RowSumU8Params *__restrict__ jobs, const TileQueues q) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  __shared__ uint32_t claimed;
  QueueCursor cur;
  for (;;) {
    const uint32_t t = cur.next(q, &claimed);
    if (t == kNoTile) break;
    const TileDesc d = q.tiles[t];
    u8_matrix_tile<RUN, DPW, PACKED, WIDE>(jobs[d.job], d.tile, lds);
  }
}

// One workgroup per listed (job, tile) descriptor, in XCD-aware order.
template <int RUN, int DPW, bool PACKED, bool WIDE>
__global__ void __launch_bounds__(512)
rowsum_u8_matrix_list(const RowSumU8Params *__restrict__ jobs, const TileDesc *__restrict__ tiles, uint32_t n) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  const TileDesc d = tiles[xcd_logical(blockIdx.x, n)];
  u8_matrix_tile<RUN, DPW, PACKED, WIDE>(jobs[d.job], d.tile, lds);
}

// Calls f(RUN, DPW, PACKED, WIDE) with the compile-time constants of geometry
// g; PACKED kernels also read packed rows, WIDE ones take more than one window
// of 32 samples per row.
template <typename F> hipError_t dispatch(const Geometry &g, F &&f) {
  auto by_dpw = [&](auto run, auto pk, auto wd) -> hipError_t {
    switch (g.items_d1) {
    case 4: return f(run, std::integral_constant<int, 4>{}, pk, wd);
    case 8: return f(run, std::integral_constant<int, 8>{}, pk, wd);
    default: return hipErrorInvalidValue;
    }
  };
  auto by_run = [&](auto pk, auto wd) -> hipError_t {
    switch (g.items_d0) {
    case 4: return by_dpw(std::integral_constant<int, 4>{}, pk, wd);
    case 8: return by_dpw(std::integral_constant<int, 8>{}, pk, wd);
    case 16: return by_dpw(std::integral_constant<int, 16>{}, pk, wd);
    default: return hipErrorInvalidValue;
    }
  };
  if (g.packed) return g.wide ? by_run(std::true_type{}, std::true_type{}) : by_run(std::true_type{}, std::false_type{});
  return g.wide ? by_run(std::false_type{}, std::true_type{}) : by_run(std::false_type{}, std::false_type{});
}

} // namespace

hipError_t launch_rowsum_u8_matrix(const RowSumU8Params &p, const Geometry &g, hipStream_t stream) {
  return dispatch(g, [&](auto run, auto dpw, auto pk, auto wd) {
    hipLaunchKernelGGL((rowsum_u8_matrix<run.value, dpw.value, pk.value, wd.value>), dim3(p.n_tiles), dim3(64 * g.threads_d1),
                       g.lds_bytes, stream, p);
    return hipGetLastError();
  });
}

hipError_t launch_rowsum_u8_matrix_batch(const RowSumU8Params *d_jobs, const TileQueues &q, const Geometry &g,
                                         uint32_t workgroups, hipStream_t stream) {
  return dispatch(g, [&](auto run, auto dpw, auto pk, auto wd) {
    hipLaunchKernelGGL((rowsum_u8_matrix_batch<run.value, dpw.value, pk.value, wd.value>), dim3(workgroups),
                       dim3(64 * g.threads_d1), g.lds_bytes, stream, d_jobs, q);
    return hipGetLastError();
  });
}

hipError_t launch_rowsum_u8_matrix_list(const RowSumU8Params *d_jobs, const TileDesc *d_tiles, uint32_t n,
                                        const Geometry &g, hipStream_t stream) {
  return dispatch(g, [&](auto run, auto dpw, auto pk, auto wd) {
    hipLaunchKernelGGL((rowsum_u8_matrix_list<run.value, dpw.value, pk.value, wd.value>), dim3(n), dim3(64 * g.threads_d1),
                       g.lds_bytes, stream, d_jobs, d_tiles, n);
    return hipGetLastError();
  });
}

hipError_t rowsum_u8_matrix_batch_occupancy(const Geometry &g, int *per_cu) {
  return dispatch(g, [&](auto run, auto dpw, auto pk, auto wd) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu,
                                                        rowsum_u8_matrix_batch<run.value, dpw.value, pk.value, wd.value>,
                                                        (int)(64 * g.threads_d1), (size_t)g.lds_bytes);
  });
}

} // namespace ddamd
