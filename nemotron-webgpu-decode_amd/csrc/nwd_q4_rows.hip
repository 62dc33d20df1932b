// nwd_q4_rows.hip — the 4-bit projections of several activation rows at once
// on the matrix cores (gfx950).
//
// nwd_q4.hip runs one workgroup column per activation row: every row streams
// and unpacks all the weights again. Here a weight is read and unpacked once
// for up to 64 rows, as the B operand of v_mfma_f32_16x16x32_f16 (one 32-
// weight block along K is one MFMA's depth):
//   B  the exact integers nib - zp of one block of 16 columns, in fp16;
//   A  16 activation rows, each scaled by a power of two so that its largest
//      magnitude lies in [2^14, 2^15) and carried as fp16 high and low parts
//      (hi = fp16(x), lo = fp16(x - hi)), two MFMAs onto one accumulator;
//   D  the block's sums, multiplied by the block's scale into fp32 sums.
// At the end a row's sums are multiplied by its power of two. Against 64 bits
// the results are closer than those of the one-row kernels (2-norm of the
// error over the result, K = 3136 and 5120: 1.1e-7 and 1.2e-7 against 2.2e-7
// and 2.5e-7): the products are exact, and the zero points come off the
// weights exactly instead of as a difference of two large sums.
//
// The parts hold x within 2^-23 of its magnitude, and never closer than 2^-25
// after the scaling, where the low part is at the end of fp16's range. A row
// with a block whose largest magnitude is more than 15 binades below the
// row's (an activation of 10^6 beside ordinary ones) would lose bits there
// that a weight of zero at the large element brings to light: such a row is
// "wide", and its sums are taken in fp32 from the activations themselves, by
// the same wavefronts over the weights in LDS (wide_sums) or by a wide pick's
// merge. So every x is held within 2^-23 of the largest magnitude of its
// block, at least.
//
// Two launches per call: q4_rows_kernel converts the activation rows into
// the A operands' lane order in the context's workspace, q4_product_kernel
// multiplies; picks add the merge of their records. A workgroup of the product
// kernel stages the weights of 16 or 32 columns, all of K, in LDS with copies
// of whole runs of a column (reading 4 blocks at a time straight into the
// MFMA's lane order touched 3 cache lines for 84 useful bytes of a column and
// took twice as long), its 8 or 4 wavefronts split K and read the A operands
// of their part from L2.
#include "nwd_argmax.h"
#include "nwd_common.h"
#include "nwd_internal.h"

#include <atomic>

namespace nwd {

namespace {

// Cells (columns) of up to three projections side by side, the argument block
// of the kernels.
struct RowsArgs {
  Q4Mat m[3];
  int n_mats;
  int cols;               // all columns
  int n_blocks;
  int rows;               // activation rows of this launch
  const float* x;         // activations [rows][32 n_blocks]
  const u32x4* a;         // A operands (q4_rows_kernel)
  const float* factor;    // [rows] power of two of each row (kWideRow, NaN)
  // where the results go
  int epilogue;           // Q4Epilogue (plain projections)
  float* y;               // [rows][cols]
  void* q_out;            // q/k/v: queries and caches
  f16* k_cache;
  f16* v_cache;
  const int32_t* pos;
  int n_kv, head_dim, cap, q16;
  int64_t cache_size;     // elements of one cache
  Q4Scratch scratch;      // for the checked build's bounds and its status word
  unsigned long long* records;  // greedy pick
  int per_row;
  unsigned long long* wide_best;  // [rows] picks of wide rows, and the arrivals
  int* wide_tickets;              // (q4_pick_merge_kernel); zeros from q4_rows_kernel
  int red_offset;  // of the workgroup's sums in LDS
};

enum RowsKind { kRowsPlain = 0, kRowsQkv = 1, kRowsArgmax = 2 };

// Lane offset of a read that is not to happen: at or past every descriptor's
// byte count (below 2^31), it returns zeros without a memory access. Only the
// lane offset is compared with the byte count as it stands: the range check
// subtracts the scalar offset from the count first, so a scalar offset stays
// inside the buffer whatever the lane offset is.
constexpr uint32_t kNoRead = 0x80000000u;

// The matrix that columns col0 .. col0 + 15 lie in (a 16-column tile never
// straddles two of them: their widths are multiples of 16), col0 made
// relative to it.
__device__ inline Q4Mat matrix_of(const RowsArgs& p, int& col0) {
  Q4Mat m = p.m[0];
  if (p.n_mats > 1 && col0 >= p.m[0].n) {
    col0 -= p.m[0].n;
    m = p.m[1];
    if (col0 >= p.m[1].n) {
      col0 -= p.m[1].n;
      m = p.m[2];
    }
  }
  return m;
}

// The checked build's test of a store of n bytes into the workspace.
__device__ inline bool in_scratch(const Q4Scratch& s, const void* at, int64_t n) {
  return in_bounds(static_cast<const char*>(at) - static_cast<const char*>(s.base), n, (int64_t)s.bytes, s.status);
}

__device__ inline f16x2 twice(uint32_t h) {  // the low half in both
  const f16x2 v = __builtin_bit_cast(f16x2, h);
  return __builtin_shufflevector(v, v, 0, 0);
}
__device__ inline f16x2 and_or(uint32_t v, uint32_t mask, uint32_t bits) {
  uint32_t r;  // one instruction: hipcc makes two of an AND and an OR with literals
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(bits));
  return __builtin_bit_cast(f16x2, r);
}

// Eight nibbles less their zero point z as fp16, exactly, in the order
// 0, 4, 1, 5, 2, 6, 3, 7: a nibble in the low mantissa bits of 1024, or in
// the next four of 64, is 1024 + n or 64 + n. (The nibbles alone are fp16
// subnormals, n 2^-24 and n 2^-20, but the MFMAs align such products by
// their nominal exponent: 4.5e-6 of error against 1.1e-7.)
__device__ inline f16x8 unpack(uint32_t t, uint32_t z) {
  constexpr uint32_t k1024 = 0x64006400u, k64 = 0x54005400u;
  const f16x2 z1024 = twice(z | 0x6400u), z64 = twice(z << 4 | 0x5400u);
  const uint32_t u = t >> 8;
  const f16x2 p04 = and_or(t, 0x000F000Fu, k1024) - z1024;
  const f16x2 p15 = and_or(t, 0x00F000F0u, k64) - z64;
  const f16x2 p26 = and_or(u, 0x000F000Fu, k1024) - z1024;
  const f16x2 p37 = and_or(u, 0x00F000F0u, k64) - z64;
  return f16x8{p04[0], p04[1], p15[0], p15[1], p26[0], p26[1], p37[0], p37[1]};
}

// ----------------------------------------------------------------- results

// One value of a plain or q/k/v projection to its place (row < p.rows, col
// < p.cols).
template <int kKind>
__device__ inline void put(const RowsArgs& p, int row, int col, float v) {
  if constexpr (kKind == kRowsPlain) {
    const int64_t at = (int64_t)row * p.cols + col;
    if (!in_bounds(at, 1, (int64_t)p.rows * p.cols, p.scratch.status)) return;
    float* y = p.y + at;
    if (p.epilogue == kQ4Relu2) {
      const float t = fmaxf(v, 0.f);
      v = t * t;
    } else if (p.epilogue == kQ4Accumulate) {
      v = *y + v;  // H[i] = H[i] + B[i]
    }
    *y = v;
  } else if constexpr (kKind == kRowsQkv) {
    if (col < p.m[0].n) {
      const int64_t at = (int64_t)row * p.m[0].n + col;
      if (!in_bounds(at, 1, (int64_t)p.rows * p.m[0].n, p.scratch.status)) return;
      if (p.q16)
        static_cast<f16*>(p.q_out)[at] = (f16)v;
      else
        static_cast<float*>(p.q_out)[at] = v;
      return;
    }
    // kv_append (kernels/kv_append.wgsl:12-18), rounded to fp16, at pos[row];
    // a position outside the cache writes nothing and is reported.
    col -= p.m[0].n;
    const bool is_k = col < p.m[1].n;
    if (!is_k) col -= p.m[1].n;
    const int t = p.pos[row];
    if (t < 0 || t >= p.cap) {
      if (col == 0) atomicOr(p.scratch.status, kStatusBadPos);
      return;
    }
    const int64_t at = cache_index_d(row, t, col / p.head_dim, col % p.head_dim, p.n_kv, p.cap, p.head_dim);
    if (!in_bounds(at, 1, p.cache_size, p.scratch.status)) return;
    (is_k ? p.k_cache : p.v_cache)[at] = (f16)v;
  }
}

// A logit of a greedy pick, where they are asked for, and a record.
__device__ inline void put_logit(const RowsArgs& p, int row, int col, float v) {
  const int64_t at = (int64_t)row * p.cols + col;
  if (p.y && in_bounds(at, 1, (int64_t)p.rows * p.cols, p.scratch.status)) p.y[at] = v;
}
__device__ inline void put_record(const RowsArgs& p, int row, int i, unsigned long long v) {
  unsigned long long* at = p.records + (int64_t)row * p.per_row + i;
  if (in_scratch(p.scratch, at, 8)) *at = v;
}

// ------------------------------------------------------------ activation rows

// One workgroup per activation row: its power of two, and its high and low
// parts in the lane order of the MFMA A operand. Tile layout (1 KB = 64 lanes
// of 8 halves): [tile of 16 rows][block][hi, lo], lane (row, g) holding
// elements 8g .. 8g + 7 of the block in unpack()'s order; packed (up to 8
// rows), [block] with the high parts as rows 0-7 and the low parts as rows
// 8-15, one MFMA for both.
// A row that holds an infinity or a NaN gets the factor NaN: the one-row
// kernels' sums (nib x - zp x per block) give NaN for such a row too. A wide
// row gets the factor kWideRow, which no power of two here is.
constexpr int kRowsThreads = 256;
constexpr float kWideRow = 0.f;
constexpr uint32_t kWideBinades = 15;  // a block's largest is then at least 2^-1, the parts' step 2^-24
constexpr int kRowsRuns = kQ4MaxBlocks * 4 / kRowsThreads;  // 8-element runs per thread

__global__ __launch_bounds__(kRowsThreads) void q4_rows_kernel(const float* __restrict__ x,
                                                               int n_blocks, int packed,
                                                               u32x4* __restrict__ a,
                                                               float* __restrict__ factor,
                                                               unsigned long long* __restrict__ wide_best,
                                                               int* __restrict__ wide_tickets,
                                                               const Q4Scratch scratch) {
  __shared__ uint32_t wave_max[kRowsThreads / 64], wave_low[kRowsThreads / 64];
  const int row = blockIdx.x, t = threadIdx.x, runs = n_blocks * 4;
  const f32x4* xr = reinterpret_cast<const f32x4*>(x + (int64_t)row * n_blocks * 32);
  f32x4 v[kRowsRuns][2];
  uint32_t m = 0, low = 0xFFFFFFFFu;  // largest magnitudes: of the row, and of its smallest block not all zeros
#pragma unroll
  for (int j = 0; j < kRowsRuns; ++j) {
    const int i = t + j * kRowsThreads;
    if (i < runs) {
      v[j][0] = xr[2 * i];
      v[j][1] = xr[2 * i + 1];
    }
  }
#pragma unroll
  for (int j = 0; j < kRowsRuns; ++j) {
    if (t + j * kRowsThreads < runs) {  // the same in the 4 lanes of a block
      uint32_t b = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) b = max(b, __float_as_uint(v[j][e >> 2][e & 3]) & 0x7FFFFFFFu);
      b = max(b, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, kDppQuadXor1, 0xF, 0xF, false));
      b = max(b, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, kDppQuadXor2, 0xF, 0xF, false));
      m = max(m, b);
      low = min(low, b - 1u);  // zeros wrap to the top
    }
  }
#pragma unroll
  for (int s = 32; s >= 4; s >>= 1) {
    m = max(m, (uint32_t)__shfl_xor((int)m, s, 64));
    low = min(low, (uint32_t)__shfl_xor((int)low, s, 64));
  }
  if ((t & 63) == 0) {
    wave_max[t >> 6] = m;
    wave_low[t >> 6] = low;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kRowsThreads / 64; ++w) {
    m = max(m, wave_max[w]);
    low = min(low, wave_low[w]);
  }
  // 2^e brings the largest magnitude's exponent to 14; e stays where 2^e and
  // 2^-e are normal numbers.
  const bool finite = m < 0x7F800000u;
  const bool wide = m != 0 && (m >> 23) - ((low + 1u) >> 23) > kWideBinades;
  const int e = min(141 - (int)(m >> 23), 126);
  const float up = finite ? __uint_as_float((uint32_t)(e + 127) << 23) : 0.f;
  if (t == 0) {
    if (in_bounds(row, 1, reinterpret_cast<unsigned long long*>(wide_tickets) - wide_best, scratch.status))
      wide_best[row] = 0ull;
    if (row == 0 && in_scratch(scratch, wide_tickets, 4)) *wide_tickets = 0;
    if (in_bounds(row, 1, reinterpret_cast<float*>(wide_best) - factor, scratch.status))
      factor[row] = !finite ? __uint_as_float(0x7FC00000u)
                            : (wide ? kWideRow : __uint_as_float((uint32_t)(127 - e) << 23));
  }
#pragma unroll
  for (int j = 0; j < kRowsRuns; ++j) {
    const int i = t + j * kRowsThreads;
    if (i >= runs) break;
    f16x8 hi, lo;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int src = (k >> 1) + (k & 1) * 4;  // 0, 4, 1, 5, 2, 6, 3, 7
      const float f = finite ? v[j][src >> 2][src & 3] * up : 0.f;
      hi[k] = (f16)f;
      lo[k] = (f16)(f - (float)hi[k]);
    }
    const int blk = i >> 2, g = i & 3;
    if (packed) {
      u32x4* o = a + (int64_t)blk * 64 + g * 16 + row;
      if (!in_bounds(o - a, 9, reinterpret_cast<u32x4*>(factor) - a, scratch.status)) continue;
      o[0] = __builtin_bit_cast(u32x4, hi);
      o[8] = __builtin_bit_cast(u32x4, lo);
    } else {
      const int64_t at = (int64_t)(row >> 4) * n_blocks + blk;
      u32x4* o = a + at * 128 + g * 16 + (row & 15);
      if (!in_bounds(o - a, 65, reinterpret_cast<u32x4*>(factor) - a, scratch.status)) continue;
      o[0] = __builtin_bit_cast(u32x4, hi);
      o[64] = __builtin_bit_cast(u32x4, lo);
    }
  }
}

// The factor of a row's sums: a wide row's are not scaled.
__device__ inline float sum_factor(float factor) { return factor == kWideRow ? 1.f : factor; }

// Lane l's factor of row row0 + l, of n <= 64 rows.
__device__ inline float lane_factor(const RowsArgs& p, int row0, int n) {
  const int lane = threadIdx.x & 63;
  return lane < n && row0 + lane < p.rows ? p.factor[row0 + lane] : 1.f;
}

// One block of a wide row: its 32 activations times the weights less their
// zero point, which are exact in fp16.
__device__ inline float wide_dot(const f32x4* __restrict__ x, u32x4 q, uint32_t z) {
  float d = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const f16x8 b = unpack(q[w], z);
    const f32x4 v[2] = {x[2 * w], x[2 * w + 1]};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int src = (k >> 1) + (k & 1) * 4;  // 0, 4, 1, 5, 2, 6, 3, 7
      d = fmaf((float)b[k], v[src >> 2][src & 3], d);
    }
  }
  return d;
}

// The sums of the wide rows among a wavefront's, in place of its products'.
// Lane (column l % 16, quarter l / 16) holds sums acc[mt][c][r] of row
// 16 mt + 4 (l / 16) + r (packed: rows 8 up hold the low parts' sums, here
// zeros). The four quarters share a row's blocks; block(c, blk, x) is the
// lane's column's block blk of column tile c. K = 3136, 7168 columns, 16 rows:
// 11.0 us, with one wide row 14.6, with 16 71 (one-row kernels 55).
template <int kMt, int kCols, bool kPacked, typename Block>
__device__ inline void wide_sums(const RowsArgs& p, uint64_t wide, int row0, int first, int end,
                                 f32x4 (&acc)[kMt][kCols], const Block& block) {
  const int quarter = (threadIdx.x >> 4) & 3;
  while (wide) {
    const int at = __builtin_ctzll(wide);
    wide &= wide - 1;
    const f32x4* x = reinterpret_cast<const f32x4*>(p.x + (int64_t)(row0 + at) * p.n_blocks * 32);
    float sum[kCols];
#pragma unroll
    for (int c = 0; c < kCols; ++c) sum[c] = 0.f;
#pragma unroll 1
    for (int blk = first + quarter; blk < end; blk += 4) {
#pragma unroll
      for (int c = 0; c < kCols; ++c) sum[c] += block(c, blk, x + 8 * blk);
    }
#pragma unroll
    for (int c = 0; c < kCols; ++c) sum[c] = sum_xor32(sum_xor16(sum[c]));
#pragma unroll
    for (int mt = 0; mt < kMt; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (at >> 4 == mt && (at & 3) == r) {
#pragma unroll
          for (int c = 0; c < kCols; ++c) {
            if (quarter == ((at >> 2) & 3)) acc[mt][c][r] = sum[c];
            if (kPacked && quarter == ((at >> 2) & 3) + 2) acc[mt][c][r] = 0.f;
          }
        }
  }
}

// -------------------------------------------------------------- the products

// A workgroup owns kCols tiles of 16 columns, whose weights, all of K, it
// stages in LDS at once, and walks row groups of kTiles row tiles (0:
// packed). Its wavefronts split the blocks of K.
// LDS of a 16-column tile, in cells (column, block): columns at an odd
// stride, so that the 16 columns' reads of one block fall on distinct banks.
__host__ __device__ inline int tile_cells(int n_blocks) { return 16 * (n_blocks | 1); }
constexpr int kCellBytes = 16 + 4;  // nibbles, scale
constexpr int kRedPad = 4;
constexpr int red_floats(int waves, int cols) { return waves * 16 * (cols * 16 + kRedPad); }

template <int kTiles, int kCols, int kWaves, int kKind>
__global__ __launch_bounds__(kWaves * 64, kTiles == 4 ? 2 : 4) void q4_product_kernel(const RowsArgs p) {
  constexpr int kThreads = kWaves * 64;
  constexpr int kPolicy = kKind == kRowsArgmax ? kStreamPolicy : 0;
  constexpr int kMt = kTiles ? kTiles : 1;                           // row tiles
  constexpr int kParts = kTiles ? 2 : 1;                             // A operands per tile and block
  constexpr int kHeld = 8 / (kMt * kParts) < 2 ? 2 : 8 / (kMt * kParts);  // blocks of A operands in flight
  constexpr int kWgCols = kCols * 16;
  constexpr int kRows = kTiles ? 16 : 8;  // rows of a tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, nb = p.n_blocks;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int stride = nb | 1, cells = tile_cells(nb), col_base = blockIdx.x * kWgCols;
  u32x4* lds_q = reinterpret_cast<u32x4*>(smem);
  float* lds_s = reinterpret_cast<float*>(smem + kCols * cells * 16);
  float* red = reinterpret_cast<float*>(smem + p.red_offset);

  // ---- the weights: nibbles and scales of 64 blocks of a column per copy
  __amdgpu_buffer_rsrc_t rz[kCols];
  int zcell[kCols], zlast[kCols];
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    int col0 = min(col_base + c * 16, p.cols - 1);
    const Q4Mat m = matrix_of(p, col0);
    const int n_cells = m.n * nb;  // 16 * n_cells < 2^31 (q4_rows_shape)
    const auto rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m.quant), 0, n_cells * 16, kBufferWord3);
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(m.scales), 0, n_cells * 4, kBufferWord3);
    for (int b = 0; b < nb; b += 64) {
      if (b + lane >= nb) break;
#pragma unroll
      for (int i = 0; i < 16 / kWaves; ++i) {
        const int cc = i * kWaves + wave;
        if (col0 + cc < m.n) {
          const int cell = (col0 + cc) * nb + b, at = c * cells + cc * stride + b;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (lds_void*)(lds_q + at), 16, lane * 16, cell * 16, 0, kPolicy);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(lds_s + at), 4, lane * 4, cell * 4, 0, 0);
        }
      }
    }
    rz[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m.zp), 0, (n_cells + 1) / 2, kBufferWord3);
    zcell[c] = min(col0 + (lane & 15), m.n - 1) * nb;
    zlast[c] = (n_cells + 1) / 2 - 8;
  }

  // ---- row groups
  const int first = wave * nb / kWaves, end = (wave + 1) * nb / kWaves;
  const int last = max(end - 1, 0);  // requests past the part's blocks repeat its last one's
  const int groups = (p.rows + kRows * kMt - 1) / (kRows * kMt);
  const int cell0 = (lane & 15) * stride, g = (lane >> 4) & 3;
  bool staged = false;
  for (int group = blockIdx.y; group < groups; group += gridDim.y) {
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<u32x4*>(p.a + (int64_t)group * kMt * nb * kParts * 64), 0, kMt * nb * kParts * 1024, kBufferWord3);
    f16x8 a[kHeld][kMt][kParts];
    const auto load_a = [&](f16x8 (&dst)[kMt][kParts], int blk) __attribute__((always_inline)) {
      const int b = min(blk, last);
#pragma unroll
      for (int mt = 0; mt < kMt; ++mt)
#pragma unroll
        for (int part = 0; part < kParts; ++part)
          dst[mt][part] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(
              ra, lane * 16, ((mt * nb + b) * kParts + part) * 1024, 0));
    };
    f32x4 acc[kMt][kCols];
#pragma unroll
    for (int mt = 0; mt < kMt; ++mt)
#pragma unroll
      for (int c = 0; c < kCols; ++c) acc[mt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    // The lane's column's zero points of 8 blocks from blk on: one 8-byte
    // read from any nibble offset, moved back where it would pass the end.
    const auto load_z = [&](u32x2 (&dst)[kCols], int blk) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < kCols; ++c)
        dst[c] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(
            rz[c], min((zcell[c] + blk) >> 1, zlast[c]), 0, 0));
    };
    const auto nibbles = [&](const u32x2& v, int c, int blk) __attribute__((always_inline)) {
      const int byte = (zcell[c] + blk) >> 1;
      return (uint32_t)(__builtin_bit_cast(uint64_t, v) >>
                        ((byte - min(byte, zlast[c])) * 8 + ((zcell[c] + blk) & 1) * 4));
    };
    // Block blk, the i-th of the zero points in z.
    const auto block = [&](const f16x8 (&av)[kMt][kParts], int blk, const uint32_t (&z)[kCols], int i) __attribute__((always_inline)) {
      f16x8 bv[kCols];
      float s[kCols];
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        const int cell = c * cells + cell0 + blk;
        s[c] = lds_s[cell];
        bv[c] = unpack(reinterpret_cast<const uint32_t*>(lds_q)[cell * 4 + g], (z[c] >> (4 * i)) & 15u);
      }
      f32x4 d[kMt][kCols];
#pragma unroll
      for (int part = 0; part < kParts; ++part)
#pragma unroll
        for (int mt = 0; mt < kMt; ++mt)
#pragma unroll
          for (int c = 0; c < kCols; ++c)
            d[mt][c] = mfma16x16x32(av[mt][part], bv[c], part ? d[mt][c] : f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int mt = 0; mt < kMt; ++mt)
#pragma unroll
        for (int c = 0; c < kCols; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[mt][c][r] = fmaf(s[c], d[mt][c][r], acc[mt][c][r]);
    };
#pragma unroll
    for (int i = 0; i < kHeld; ++i) load_a(a[i], first + i);
    u32x2 zv[kCols];
    load_z(zv, first);
    if (!staged) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the copies into LDS
      __syncthreads();
      staged = true;
    }
    for (int blk = first; blk < end; blk += 8) {
      uint32_t z[kCols];
#pragma unroll
      for (int c = 0; c < kCols; ++c) z[c] = nibbles(zv[c], c, blk);
      load_z(zv, blk + 8);
      if (blk + 8 <= end) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          block(a[i % kHeld], blk + i, z, i);
          load_a(a[i % kHeld], blk + i + kHeld);
          // One block at a time: with the next ones' reads hoisted, the 64-
          // row forms spilled (K = 3136, 5120 columns, 512 rows: 108.7 us
          // against 73.0).
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (blk + i < end) block(a[i % kHeld], blk + i, z, i);
          if (kHeld < 8 && blk + i + kHeld < end) load_a(a[i % kHeld], blk + i + kHeld);
        }
      }
    }

    // What follows counts from an opaque copy of the thread, so that none of its
    // addresses is held, or spilled, across the products (q/k/v of K = 3136, 64
    // rows 20.8 us against 21.9 to 22.5).
    int et = threadIdx.x;
    asm volatile("" : "+v"(et));
    const int elane = et & 63;
    const float factors = lane_factor(p, group * kMt * kRows, kMt * kRows);
    const uint64_t wide = __ballot(factors == kWideRow);
    if (wide)
      wide_sums<kMt, kCols, !kTiles>(p, wide, group * kMt * kRows, first, end, acc, [&](int c, int blk, const f32x4* x) __attribute__((always_inline)) {
        const int cell = c * cells + cell0 + blk, zat = zcell[c] + blk;
        const uint32_t z = __builtin_amdgcn_raw_buffer_load_b8(rz[c], zat >> 1, 0, 0) >> (4 * (zat & 1)) & 15u;
        return lds_s[cell] * wide_dot(x, lds_q[cell], z);
      });

    // The wavefronts' sums, added in wavefront order, one row tile at a time.
#pragma unroll
    for (int mt = 0; mt < kMt; ++mt) {
      __syncthreads();
#pragma unroll
      for (int c = 0; c < kCols; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          red[(wave * 16 + (elane >> 4) * 4 + r) * (kWgCols + kRedPad) + c * 16 + (elane & 15)] = acc[mt][c][r];
      __syncthreads();
#pragma unroll
      for (int e = 0; e < kRows * kWgCols; e += kThreads) {
        const int r = (e + et) / kWgCols, cc = (e + et) % kWgCols;
        const int row = (group * kMt + mt) * kRows + r, cl = col_base + cc;
        const bool live = r < kRows && row < p.rows && cl < p.cols;
        float v = 0.f;
        if (r < kRows) {
#pragma unroll
          for (int k = 0; k < kWaves; ++k) {
            v += red[(k * 16 + r) * (kWgCols + kRedPad) + cc];
            if constexpr (!kTiles) v += red[(k * 16 + r + 8) * (kWgCols + kRedPad) + cc];
          }
        }
        v *= sum_factor(__shfl(factors, mt * kRows + (r < kRows ? r : 0), 64));
        if constexpr (kKind == kRowsArgmax) {  // one record per row and workgroup
          if (live) put_logit(p, row, cl, v);
          unsigned long long best = live ? argmax_enc(v, cl, argmax_shape(p.cols)) : 0ull;
#pragma unroll
          for (int m = kWgCols / 2; m >= 1; m >>= 1) {
            const unsigned long long o = __shfl_xor(best, m, 64);
            best = o > best ? o : best;
          }
          if (cc == 0 && r < kRows && row < p.rows) put_record(p, row, blockIdx.x, best);
        } else {
          if (live) put<kKind>(p, row, cl, v);
        }
      }
    }
  }
}

// ------------------------------------------------------- wide greedy picks

// lm_head with the pick (pick_wide says which): one persistent workgroup per
// CU. Its 8 wavefronts split K and hold their part of one row tile's A operands
// in registers for the whole launch (read per 32 columns, as above, they were
// more L2 traffic than the weights); the weights of the next 32 columns, one
// run of memory, lie in the other LDS buffer and those after it are on their
// way in registers. Row tiles share the workgroups out, side by side over the
// same columns, so that L2 and the Infinity Cache serve the weights' second
// reading. A thread keeps the best of its logits of a row; one record per row
// and workgroup. 131072 x 3136, us per call, the kernel above against this: 4
// rows 98 against 68, 16 rows 118 against 75, 32 rows 171 against 135. Its
// products alone take 44 of the 75, its reads 55 (4.8 TB/s).
constexpr int kPickWaves = 8;
constexpr int kPickThreads = kPickWaves * 64;
constexpr int kPickCols = 32;
constexpr int kPickBlocks = 13;                  // of K per wavefront, at most
constexpr int kPickMaxBlocks = 8 * kPickBlocks;  // 104: K <= 3328
constexpr int kPickLoads = kPickCols * kPickMaxBlocks / kPickThreads + 1;
static_assert((kPickBlocks + 3) / 4 * 2 >= kPickLoads, "two requests beside every four blocks");
constexpr int kPickRed = kPickWaves * 16 * (kPickCols + kRedPad);  // floats
constexpr int pick_lds(int n_blocks) { return 2 * kPickCols * (n_blocks | 1) * kCellBytes + kPickRed * 4; }

template <int kTiles>
__global__ __launch_bounds__(kPickThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void q4_pick_kernel(
    const RowsArgs p, int row_tiles) {
  constexpr int kParts = kTiles ? 2 : 1;
  constexpr int kRows = kTiles ? 16 : 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, nb = p.n_blocks;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = blockIdx.x % row_tiles, slot = blockIdx.x / row_tiles;
  const int slots = gridDim.x / row_tiles;  // workgroups of a row tile
  const int groups = (p.cols + kPickCols - 1) / kPickCols;
  const int stride = nb | 1, buffer = kPickCols * stride * kCellBytes;
  float* red = reinterpret_cast<float*>(smem + 2 * buffer);
  const Q4Mat m = p.m[0];
  const int n_cells = m.n * nb;  // 16 * n_cells < 2^31 (q4_rows_shape)
  const auto rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m.quant), 0, n_cells * 16, kBufferWord3);
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(m.scales), 0, n_cells * 4, kBufferWord3);
  const auto rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(m.zp), 0, (n_cells + 1) / 2, kBufferWord3);
  const int zlast = (n_cells + 1) / 2 - 8;
  const int first = wave * nb / kPickWaves, end = (wave + 1) * nb / kPickWaves;

  // Cell tid + 512 i of a group's run of 32 nb cells, and where it goes.
  int to[kPickLoads];
  const int cells = kPickCols * nb;
#pragma unroll
  for (int i = 0; i < kPickLoads; ++i) {
    const int idx = tid + i * kPickThreads, c = idx / nb;
    to[i] = idx < cells ? c * stride + idx - c * nb : -1;
  }
  u32x4 wq[kPickLoads];
  float ws[kPickLoads];
  u32x2 zn[2][2];     // [column tile][blocks first .. + 7, first + 8 .. + 15]
  uint32_t zv[2][2], znext[2][2];  // zero points of those blocks, a nibble each
  // Requests i and i + 1 of a group's, the zero points with the last. A
  // group's requests do not fit the memory path's queues at once: issued
  // together they held the wavefronts up for as long as the products take.
  const auto load_w = [&](int group, int first_i) __attribute__((always_inline)) {
    const int base = group * cells;  // past the last column: no read
#pragma unroll
    for (int i = first_i; i < first_i + 2; ++i) {
      if (i >= kPickLoads) break;
      const int cell = base + tid + i * kPickThreads;
      const bool in = to[i] >= 0 && cell < n_cells;
      wq[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
          rq, in ? cell * 16 : kNoRead, 0, kStreamPolicy));
      ws[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, in ? cell * 4 : kNoRead, 0, 0));
    }
    if (first_i + 2 < kPickLoads) return;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int cell = min(group * kPickCols + c * 16 + (lane & 15), m.n - 1) * nb + first + 8 * h;
        zn[c][h] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(
            rz, group < groups && first + 8 * h < end ? min(cell >> 1, zlast) : kNoRead, 0, 0));
      }
  };
  const auto load_all = [&](int group) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kPickLoads; i += 2) load_w(group, i);
  };
  const auto store_w = [&](int buf, int group) __attribute__((always_inline)) {
    u32x4* q = reinterpret_cast<u32x4*>(smem + buf * buffer);
    float* s = reinterpret_cast<float*>(smem + buf * buffer + kPickCols * stride * 16);
#pragma unroll
    for (int i = 0; i < kPickLoads; ++i)
      if (to[i] >= 0) {
        q[to[i]] = wq[i];
        s[to[i]] = ws[i];
      }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int cell = min(group * kPickCols + c * 16 + (lane & 15), m.n - 1) * nb + first + 8 * h, byte = cell >> 1;
        znext[c][h] = (uint32_t)(__builtin_bit_cast(uint64_t, zn[c][h]) >>
                                 ((byte - min(byte, zlast)) * 8 + (cell & 1) * 4));
      }
  };

  f16x8 a[kPickBlocks][kParts];
  const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(p.a + (int64_t)tile * nb * kParts * 64), 0,
                                                    nb * kParts * 1024, kBufferWord3);
  load_all(slot);
#pragma unroll
  for (int b = 0; b < kPickBlocks; ++b)
#pragma unroll
    for (int part = 0; part < kParts; ++part)
      a[b][part] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(
          ra, first + b < end ? lane * 16 : kNoRead, first + b < end ? ((first + b) * kParts + part) * 1024 : 0, 0));
  // The thread's logit of a group: row tid / 32 of the tile, column tid % 32.
  const int r = tid / kPickCols, cc = tid % kPickCols, row = tile * kRows + r;
  const bool live_row = r < kRows && row < p.rows;
  const float factor = live_row ? p.factor[row] : 0.f;
  const ArgmaxShape shape = argmax_shape(p.cols);
  unsigned long long best = 0ull;
  const auto step_z = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) zv[c][h] = znext[c][h];
  };
  store_w(0, slot);
  step_z();
  load_all(slot + slots);
  __syncthreads();

  int buf = 0;
  for (int group = slot; group < groups; group += slots, buf ^= 1) {
    store_w(buf ^ 1, group + slots);  // requested an iteration ago
    const uint32_t* q = reinterpret_cast<const uint32_t*>(smem + buf * buffer);
    const float* s = reinterpret_cast<const float*>(smem + buf * buffer + kPickCols * stride * 16);
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const auto block = [&](int b) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int cell = (c * 16 + (lane & 15)) * stride + first + b;
        const f16x8 bv = unpack(q[cell * 4 + (lane >> 4)], (zv[c][b / 8] >> (4 * (b % 8))) & 15u);
        f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int part = 0; part < kParts; ++part) d = mfma16x16x32(a[b][part], bv, d);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[c][e] = fmaf(s[cell], d[e], acc[c][e]);
      }
    };
    // four blocks to a branch, so that their reads and products overlap
#pragma unroll
    for (int b = 0; b < kPickBlocks; b += 4) {
      load_w(group + 2 * slots, b / 2);
      __builtin_amdgcn_sched_barrier(0);
      if (b + 4 <= kPickBlocks && first + b + 4 <= end) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (b + i < kPickBlocks) block(b + i);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (b + i < kPickBlocks && first + b + i < end) block(b + i);
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        red[(wave * 16 + (lane >> 4) * 4 + e) * (kPickCols + kRedPad) + c * 16 + (lane & 15)] = acc[c][e];
    step_z();
    __syncthreads();
    const int cl = group * kPickCols + cc;
    if (r < kRows) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < kPickWaves; ++k) {
        v += red[(k * 16 + r) * (kPickCols + kRedPad) + cc];
        if constexpr (!kTiles) v += red[(k * 16 + r + 8) * (kPickCols + kRedPad) + cc];
      }
      v *= factor;
      if (live_row && cl < p.cols) {
        put_logit(p, row, cl, v);
        const unsigned long long e = argmax_enc(v, cl, shape);
        best = e > best ? e : best;
      }
    }
    __syncthreads();  // the sums are read
  }
#pragma unroll
  for (int i = kPickCols / 2; i >= 1; i >>= 1) {
    const unsigned long long o = __shfl_xor(best, i, 64);
    best = o > best ? o : best;
  }
  if (cc == 0 && live_row) put_record(p, row, slot, best);
}

// The picks of q4_pick_kernel's records, a workgroup per row; and the wide
// rows, whose logits and records there are void: all workgroups share their
// columns out, 16 lanes to a column, and the last to arrive writes the picks.
// (In q4_pick_kernel, code for them in its walk or after it cost every call
// 3 to 5%.) 131072 x 3136, 16 rows: 78 us, with one wide row 158, with 16 931
// (one-row kernels 592).
constexpr int kPickMergeGrid = 512;
constexpr int kPickMergeThreads = 256;
constexpr int kWideLanes = 16;
constexpr int kWideIters = (kPickMaxBlocks + kWideLanes - 1) / kWideLanes;
constexpr int kWideStride = 36;  // floats of an activation block in LDS: 16 lanes' reads on distinct banks

__global__ __launch_bounds__(kPickMergeThreads) void q4_pick_merge_kernel(const RowsArgs p,
                                                                          uint32_t* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float x[kPickMaxBlocks * kWideStride];
  __shared__ unsigned long long best;
  __shared__ int last;
  const int tid = threadIdx.x, nb = p.n_blocks;
  const ArgmaxShape shape = argmax_shape(p.cols);
  uint64_t wide = __ballot(lane_factor(p, 0, p.rows) == kWideRow);  // at most 48 rows
  if ((int)blockIdx.x < p.rows && !((wide >> blockIdx.x) & 1)) {
    if (tid == 0) best = 0ull;
    __syncthreads();
    const unsigned long long* rec = p.records + (int64_t)blockIdx.x * p.per_row + tid;
    const unsigned long long e = wave_max_u64(tid < p.per_row && in_scratch(p.scratch, rec, 8) ? *rec : 0ull);
    if ((tid & 63) == 0) atomicMax(&best, e);
    __syncthreads();
    if (tid == 0) out[blockIdx.x] = argmax_decode(best, shape);
  }
  if (!wide) return;
  const Q4Mat m = p.m[0];
  const int part = tid % kWideLanes, group = tid / kWideLanes;
  for (uint64_t left = wide; left; left &= left - 1) {
    const int row = __builtin_ctzll(left);
    const float* xr = p.x + (int64_t)row * nb * 32;
    __syncthreads();
    if (tid == 0) best = 0ull;
    for (int i = tid; i < nb * 32; i += kPickMergeThreads) x[i / 32 * kWideStride + i % 32] = xr[i];
    __syncthreads();
    unsigned long long e = 0ull;
    for (int col = blockIdx.x * (kPickMergeThreads / kWideLanes) + group; col < p.cols;
         col += gridDim.x * (kPickMergeThreads / kWideLanes)) {
      u32x4 q[kWideIters];
      float s[kWideIters];
      uint32_t z[kWideIters];
#pragma unroll
      for (int i = 0; i < kWideIters; ++i) {  // past the last block: its weights again, times zero
        const int blk = part + i * kWideLanes;
        const int64_t cell = (int64_t)col * nb + min(blk, nb - 1);
        q[i] = *reinterpret_cast<const u32x4*>(m.quant + cell * 16);
        s[i] = m.scales[cell];
        z[i] = m.zp[cell >> 1] >> (4 * (cell & 1)) & 15u;
      }
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < kWideIters; ++i) {
        const int blk = part + i * kWideLanes;
        const float d = s[i] * wide_dot(reinterpret_cast<const f32x4*>(x + min(blk, nb - 1) * kWideStride), q[i], z[i]);
        v += blk < nb ? d : 0.f;
      }
      v = sum8(v);
      v += dpp_mov<kDppRowMirror>(v);
      if (part == 0) {
        put_logit(p, row, col, v);
        const unsigned long long c = argmax_enc(v, col, shape);
        e = c > e ? c : e;
      }
    }
    if (e) atomicMax(&best, e);
    __syncthreads();
    if (tid == 0 && in_scratch(p.scratch, p.wide_best + row, 8))
      __hip_atomic_fetch_max(p.wide_best + row, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (tid == 0)
    last = __hip_atomic_fetch_add(p.wide_tickets, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
  __syncthreads();
  if (last && tid < p.rows && ((wide >> tid) & 1))
    out[tid] = argmax_decode(__hip_atomic_load(p.wide_best + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), shape);
}

// ------------------------------------------------------------------- launch

constexpr int kPackedRows = 8;

// Row tiles (0: packed), column tiles and wavefronts of a workgroup, and the
// workgroups that share a column range's row groups.
struct RowsPlan {
  int tiles, cols, waves, split;
};

// Row tiles: as few as hold the rows, up to 4 (64 rows: a wavefront's sums,
// operands and products then fill its 256 registers). Two column tiles halve
// what a workgroup reads of the A operands per column, which L2 bounds with 4
// row tiles, where the workgroups still fill half the chip: us per call, one
// tile against two, K = 3136, 64 rows, 7168 columns 27.1 against 19.8. With fewer row
// tiles two workgroups of one column tile to a CU overlap better, unless K is
// short and each has little to do: 131072 columns, K = 256, 8 and 32 rows 52.4
// against 40.8 and 55.5 against 51.1; K = 896 53.7 against 45.9 and 67.8
// against 61.1; but K = 2048 71.5 against 70.2 and 132.5 against 167.9, K =
// 3136, 16 rows 114.7 against 123.9, K = 4096, 8 rows 117.4 against 142.7,
// and at 16384 columns K = 256, 16 rows 10.3 against 10.9.
// Wavefronts: 8, or 4 where two such workgroups of 64 rows then fit a CU (by
// their LDS) and the launch has them: 512 rows, K = 3136, 5120 columns 66.5
// against 76.6; one workgroup per CU loses with 4 (K = 5120, 3136 columns
// 88.5 against 76.1, 1024 columns 27.3 against 25.0).
// Split: the launch takes rounds of as many workgroups as fit the chip; the
// split with the fewest rounds times row groups (and half a group for the
// weights) wins. 512 rows, 8 wavefronts, split 8 / 4 / 2: K = 3136, 5120
// columns 76.6 / 80.0 / 99.2 us; K = 5120, 3136 columns 90.5 / 82.5 / 76.1;
// K = 3136, 1024 columns 25.0 / 34.9 / 55.8.
RowsPlan rows_plan(int cols, int n_blocks, int rows) {
  constexpr int kCus = 256, kWide = 32768, kShort = 48;
  RowsPlan r;
  r.tiles = rows <= kPackedRows ? 0 : (rows <= 16 ? 1 : (rows <= 32 ? 2 : 4));
  const int per = r.tiles ? 16 * r.tiles : kPackedRows, groups = (rows + per - 1) / per;
  const int64_t pairs = (cols + 31) / 32;
  const bool two = r.tiles == 4 ? n_blocks <= 160 && pairs * groups >= kCus / 2 : n_blocks <= kShort && cols >= kWide;
  r.cols = two ? 2 : 1;
  const int64_t wgs = r.cols == 2 ? pairs : (cols + 15) / 16;
  r.waves = r.cols == 2 && r.tiles == 4 && n_blocks <= 100 && wgs * groups >= 2 * kCus ? 4 : 8;
  const int64_t slots = r.waves == 4 ? 2 * kCus : kCus;
  r.split = 1;
  double best = 0;
  for (int s = 1; s <= groups && s <= 64; ++s) {
    const double t = (double)((wgs * s + slots - 1) / slots) * ((groups + s - 1) / s + 0.5);
    if (s == 1 || t < best) {
      best = t;
      r.split = s;
    }
  }
  return r;
}

// The wide pick: its grid, which picks it takes, and its records per row
// (one per workgroup of a row tile). The limit of K is its registers'. Each
// further row tile has it read and unpack the weights again: past 32 rows it
// wins only near its longest K, where the other kernel's 64-row form has one
// workgroup per CU, and with many columns. 131072 columns, the other kernel
// against this, us: K = 3136, 16 rows 118 against 75, 32 rows 171 against 135,
// 48 rows 203 against 195, 64 rows 211 against 252; K = 3328, 48 rows 241
// against 202; K = 2560, 48 rows 168 against 170; K = 896, 32 rows 93 against
// 79, 48 rows 96 against 113; 32768 columns, K = 3136, 48 rows 62 against 63.
constexpr int kPickGrid = 256;
bool pick_wide(int cols, int n_blocks, int rows) {
  return cols >= 16384 && n_blocks <= kPickMaxBlocks &&
         (rows <= 32 || (rows <= 48 && n_blocks > 96 && cols > 32768));
}
int pick_tiles(int rows) { return rows <= kPackedRows ? 1 : (rows + 15) / 16; }
int records_per_row(int cols, int n_blocks, int rows) {
  if (pick_wide(cols, n_blocks, rows)) return kPickGrid / pick_tiles(rows);
  const int wg_cols = 16 * rows_plan(cols, n_blocks, rows).cols;
  return (cols + wg_cols - 1) / wg_cols;
}
static_assert(pick_lds(kPickMaxBlocks) <= 160 * 1024, "the weights of two groups and the sums fit a CU");

// Scratch of a launch: the A operands (whole row groups, which the products
// read), each row's factor, the wide rows' picks and their tickets, and for
// greedy picks the records, a workgroup's one per row.
struct RowsLayout {
  size_t factor, best, tickets, records, bytes;
};
RowsLayout rows_layout(int cols, int n_blocks, int rows, bool pick) {
  const int tiles = rows <= 16 ? 1 : (rows <= 32 ? 2 : (rows + 63) / 64 * 4);
  RowsLayout l;
  l.factor = (size_t)n_blocks * (rows <= kPackedRows ? 1024 : tiles * (size_t)2048);
  l.best = l.factor + (size_t)((rows + 3) / 4) * 16;
  l.tickets = l.best + (size_t)((rows + 1) / 2) * 16;
  l.records = l.tickets + 16;
  l.bytes = l.records;
  if (pick) l.bytes += (size_t)rows * records_per_row(cols, n_blocks, rows) * 8;
  return l;
}

// Rows per launch within the scratch: all of them, a multiple of 64, or what
// fewer row tiles hold.
int rows_per_launch(int cols, int n_blocks, int rows, bool pick, size_t scratch) {
  const auto fits = [&](int r) { return rows_layout(cols, n_blocks, r, pick).bytes <= scratch; };
  if (fits(rows)) return rows;
  const size_t operands = scratch / ((size_t)n_blocks * 128);  // rows whose operands alone fit
  for (int r = (operands < (size_t)rows ? (int)operands : rows - 1) / 64 * 64; r >= 64; r -= 64)
    if (fits(r)) return r;
  for (int r : {32, 16, kPackedRows})
    if (r < rows && fits(r)) return r;
  return 0;
}

// The dynamic LDS exceeds the 64 KB default: raises the kernel's limit once
// per device (the attribute is per device).
template <auto kKernel>
hipError_t raise_lds_limit() {
  static std::atomic<uint64_t> attr_set{0};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (attr_set.load() & bit) return hipSuccess;
  e = hipFuncSetAttribute(reinterpret_cast<const void*>(kKernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          160 * 1024);
  if (e == hipSuccess) attr_set.fetch_or(bit);
  return e;
}

template <int kKind>
hipError_t launch_rows(RowsArgs p, const float* x, Q4Scratch scratch, uint32_t* out, hipStream_t stream) {
  const int rows = p.rows, nb = p.n_blocks;
  const RowsLayout at = rows_layout(p.cols, nb, rows, kKind == kRowsArgmax);
  p.x = x;
  p.scratch = scratch;
  p.scratch.bytes = at.bytes;
  char* base = static_cast<char*>(scratch.base);
  p.a = reinterpret_cast<const u32x4*>(base);
  float* factor = reinterpret_cast<float*>(base + at.factor);
  p.factor = factor;
  p.wide_best = reinterpret_cast<unsigned long long*>(base + at.best);
  p.wide_tickets = reinterpret_cast<int*>(base + at.tickets);
  p.records = reinterpret_cast<unsigned long long*>(base + at.records);
  p.per_row = kKind == kRowsArgmax ? records_per_row(p.cols, nb, rows) : 0;
  if constexpr (kKind == kRowsArgmax) {
    if (pick_wide(p.cols, nb, rows)) {
      const bool packed = rows <= kPackedRows;
      const int tiles = pick_tiles(rows);
      q4_rows_kernel<<<rows, kRowsThreads, 0, stream>>>(x, nb, packed ? 1 : 0, reinterpret_cast<u32x4*>(base), factor,
                                                        p.wide_best, p.wide_tickets, p.scratch);
      hipError_t e = hipGetLastError();
      if (e == hipSuccess) e = packed ? raise_lds_limit<q4_pick_kernel<0>>() : raise_lds_limit<q4_pick_kernel<1>>();
      if (e != hipSuccess) return e;
      if (packed)
        q4_pick_kernel<0><<<tiles * p.per_row, kPickThreads, pick_lds(nb), stream>>>(p, tiles);
      else
        q4_pick_kernel<1><<<tiles * p.per_row, kPickThreads, pick_lds(nb), stream>>>(p, tiles);
      if ((e = hipGetLastError()) != hipSuccess) return e;
      q4_pick_merge_kernel<<<kPickMergeGrid, kPickMergeThreads, 0, stream>>>(p, out);
      return hipGetLastError();
    }
  }
  const RowsPlan plan = rows_plan(p.cols, nb, rows);
  q4_rows_kernel<<<rows, kRowsThreads, 0, stream>>>(x, nb, plan.tiles == 0 ? 1 : 0, reinterpret_cast<u32x4*>(base),
                                                    factor, p.wide_best, p.wide_tickets, p.scratch);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int wg_cols = plan.cols * 16, wg_rows = plan.tiles ? 16 * plan.tiles : kPackedRows;
  const int groups = (rows + wg_rows - 1) / wg_rows, split = groups < plan.split ? groups : plan.split;
  const dim3 grid((p.cols + wg_cols - 1) / wg_cols, split);
  // The sums may overwrite the weights where no other row group follows.
  const int weights = plan.cols * tile_cells(nb) * kCellBytes, sums = red_floats(plan.waves, plan.cols) * 4;
  p.red_offset = split == groups ? 0 : weights;
  const int lds = split == groups ? (weights > sums ? weights : sums) : weights + sums;
#define NWD_ROWS_CASE(T, C, W)                                                                \
  if (plan.tiles == T && plan.cols == C && plan.waves == W) {                                 \
    if ((e = raise_lds_limit<q4_product_kernel<T, C, W, kKind>>()) != hipSuccess) return e;   \
    q4_product_kernel<T, C, W, kKind><<<grid, W * 64, lds, stream>>>(p);                      \
    if ((e = hipGetLastError()) != hipSuccess || kKind != kRowsArgmax) return e;              \
    return launch_argmax_merge(p.records, p.per_row, p.cols, out, rows, stream);              \
  }
  NWD_ROWS_CASE(0, 1, 8) NWD_ROWS_CASE(0, 2, 8) NWD_ROWS_CASE(1, 1, 8) NWD_ROWS_CASE(1, 2, 8)
  NWD_ROWS_CASE(2, 1, 8) NWD_ROWS_CASE(2, 2, 8) NWD_ROWS_CASE(4, 1, 8) NWD_ROWS_CASE(4, 2, 8)
  NWD_ROWS_CASE(4, 2, 4)
#undef NWD_ROWS_CASE
  return hipErrorInvalidValue;
}

RowsArgs rows_args(const Q4Mat* m, int n_mats, int n_blocks) {
  RowsArgs p{};
  p.n_mats = n_mats;
  for (int i = 0; i < n_mats; ++i) {
    p.m[i] = m[i];
    p.cols += m[i].n;
  }
  p.n_blocks = n_blocks;
  return p;
}

// Estimates of a call on either kind of kernel, us, of which the less decides
// (q4_rows_shape). The one-row kernels stream their columns' weights once per
// row, at any size; a workgroup here takes a row group through all of K,
// however few workgroups there are, so that few columns with a long K leave
// most of the chip idle for that long. One-row against matrix-core, us: K =
// 8192, 64 columns, 96 rows 9.5 against 31.6, 512 columns, 17 rows 13.5
// against 18.8, 2048 columns, 3 rows 11.3 against 12.5; K = 3136, 256
// columns, 64 rows 10.3 against 16.6; K = 5120, 100 columns, 96 rows 12.0
// against 24.2, 16 columns, 4000 rows 60 against 129; with the pick, 131072
// columns, 2 rows, K = 896 31 against 43, K = 2048 56 against 59. Over K of 32 to
// 8192, 16 to 131072 columns and 2 to 4000 rows (picks: 4096 columns up, 2 to
// 64 rows), 2100 shapes past the bound of q4_rows_shape, the choice lost more
// than 7% against the one-row kernels at one (14%: K = 8192, 48 columns, 2000
// rows) and more than 13% against the matrix cores at one (18%: K = 8192, 100
// columns, 256 rows).
double one_row_us(int cols, int n_blocks, int rows, bool pick) {
  const double nb = n_blocks;
  // lm_head's form (128-thread workgroups, K in registers), per column and row
  if (pick && cols >= 16384) return 8 + 1e-3 * rows * cols * (0.03 + (0.0016 + 0.0000118 * nb) * nb);
  // per 16 columns and row, by the wavefronts that share K (q4_split)
  const double unit = nb < 64 ? 1.8 + 0.038 * nb : (nb < 128 ? 2.6 + 0.0475 * nb : 4.8 + 0.052 * nb);
  return (pick ? 8 : 3) + 1e-3 * rows * ((cols + 15) / 16) * unit;
}
double several_rows_us(int cols, int n_blocks, int rows, bool pick) {
  const double nb = n_blocks;
  if (pick && pick_wide(cols, n_blocks, rows)) return 11.5 + 1e-3 * pick_tiles(rows) * cols * (0.15 + 0.0036 * nb);
  const RowsPlan p = rows_plan(cols, n_blocks, rows);
  // a round of workgroups, and its row groups' time per block of K, by row
  // tiles (packed, 1, 2, 4) and column tiles
  constexpr double kRound[2] = {0.9, 1.9}, kGroup[2][4] = {{0.0195, 0.026, 0.046, 0.092}, {0.017, 0.025, 0.046, 0.114}};
  const int wg_rows = p.tiles ? 16 * p.tiles : kPackedRows, groups = (rows + wg_rows - 1) / wg_rows;
  const int64_t wgs = (cols + 16 * p.cols - 1) / (16 * p.cols) * (int64_t)p.split;
  const int64_t slots = p.waves == 4 ? 512 : 256, rounds = (wgs + slots - 1) / slots;
  const double operands = 1e-3 * rows * nb;  // written and read once, past L2 where many
  return (pick ? 10 : 6) + (0.1 + 0.0001 * operands) * operands +
         rounds * (kRound[p.cols - 1] + kGroup[p.cols - 1][p.tiles == 4 ? 3 : p.tiles] * nb *
                                            ((groups + p.split - 1) / p.split) * (p.waves == 4 ? 2 : 1));
}

}  // namespace

bool q4_rows_shape(int n, int narrowest, int n_blocks, int rows, bool pick, Q4Scratch scratch) {
  const int64_t cells = (int64_t)n * n_blocks;
  if (rows < 2 || cells * rows < (pick && n >= 16384 ? 6000000 : 1500000)) return false;
  if ((int64_t)narrowest * n_blocks < 16 || cells * 16 >= ((int64_t)1 << 31) - (1 << 20)) return false;
  const int per = rows_per_launch(n, n_blocks, rows, pick, scratch.bytes);
  if (per == 0) return false;
  const int rest = rows % per;
  double several = rows / per * several_rows_us(n, n_blocks, per, pick);
  if (rest) several += several_rows_us(n, n_blocks, rest, pick);
  return several < one_row_us(n, n_blocks, rows, pick);
}

hipError_t launch_q4_rows_gemv(const float* x, const Q4Mat& w, int n_blocks, float* y, int rows,
                               int epilogue, Q4Scratch scratch, hipStream_t stream) {
  const int per = rows_per_launch(w.n, n_blocks, rows, false, scratch.bytes);
  for (int r = 0; r < rows; r += per) {
    RowsArgs p = rows_args(&w, 1, n_blocks);
    p.rows = rows - r < per ? rows - r : per;
    p.epilogue = epilogue;
    p.y = y + (int64_t)r * w.n;
    const hipError_t e = launch_rows<kRowsPlain>(p, x + (int64_t)r * n_blocks * 32, scratch, nullptr, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_q4_rows_qkv(const Shape& s, const float* x, const Q4Mat& wq, const Q4Mat& wk,
                              const Q4Mat& wv, int n_blocks, void* q_out, void* k_cache,
                              void* v_cache, const int32_t* pos, int batch, Q4Scratch scratch, hipStream_t stream) {
  const Q4Mat m[3] = {wq, wk, wv};
  const int per = rows_per_launch(wq.n + wk.n + wv.n, n_blocks, batch, false, scratch.bytes);
  const int64_t seq = (int64_t)s.n_kv * s.cap * s.head_dim;  // cache elements per sequence
  for (int r = 0; r < batch; r += per) {
    RowsArgs p = rows_args(m, 3, n_blocks);
    p.rows = batch - r < per ? batch - r : per;
    p.q_out = static_cast<char*>(q_out) + (int64_t)r * wq.n * (s.q16 ? 2 : 4);
    p.k_cache = static_cast<f16*>(k_cache) + r * seq;
    p.v_cache = static_cast<f16*>(v_cache) + r * seq;
    p.pos = pos + r;
    p.n_kv = s.n_kv;
    p.head_dim = s.head_dim;
    p.cap = s.cap;
    p.q16 = s.q16;
    p.cache_size = p.rows * seq;
    const hipError_t e = launch_rows<kRowsQkv>(p, x + (int64_t)r * n_blocks * 32, scratch, nullptr, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_q4_rows_argmax(const float* x, const Q4Mat& w, int n_blocks, float* logits,
                                 uint32_t* out, int batch, Q4Scratch scratch, hipStream_t stream) {
  const int per = rows_per_launch(w.n, n_blocks, batch, true, scratch.bytes);
  for (int r = 0; r < batch; r += per) {
    RowsArgs p = rows_args(&w, 1, n_blocks);
    p.rows = batch - r < per ? batch - r : per;
    p.y = logits ? logits + (int64_t)r * w.n : nullptr;
    const hipError_t e = launch_rows<kRowsArgmax>(p, x + (int64_t)r * n_blocks * 32, scratch, out + r, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace nwd
