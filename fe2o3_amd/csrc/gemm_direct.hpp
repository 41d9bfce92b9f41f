// gemm_direct.hpp -- GEMMs with too few output tiles for the pipelined tile
// (gemm_pipe.hpp) to fill the device: a decoding step's few activation rows,
// small outputs, and operands at any alignment with any K.
//
// C[m][n] = A[m][k] B[n][k]^T, both operands k-contiguous.  A workgroup of 8
// waves owns an output block of 16 MB x 16 NB and splits K over its waves:
// wave w takes the 128-byte units w, w + 8, ... of every row, so that no wave
// waits for another until the partial sums meet in LDS at the end.  A unit
// comes to registers D units ahead of its use, eight adjacent lanes per
// 128-byte row piece, and passes through LDS of the wave's own (no barrier)
// to reach the lanes that the MFMA wants it in.  Loads are 16 bytes per lane
// at the operand's own alignment (gfx950 global loads take any).
//
// Loading straight into the MFMA's lanes, without LDS, puts adjacent lanes on
// different rows: the CU then loads 16 bytes a clock instead of 64
// (bf16 16 x 4096 x 14336: 34.1 us against 24.7; 128 x 4096 x 4096: 23.9
// against 13.6).
//
// The in-order form gives every wave an output block of its own and all of K
// instead: C's bits are then those of the pipelined tile, for the calls that
// would take the tile if their operands could be read in place or copied.
//
// What bounds it: with one block row (m <= 16 MB) the weights' HBM stream,
// else the 64 bytes a clock that a CU loads (16 (MB + NB) rows of K per
// block).  bf16 16 x 4096 x 4096 runs at 4.4 TB/s, fp8 32 x 8192 x 8192 at 5.4;
// the 128 x 128 tiles they took before occupy 32 and 64 CUs.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "gemm_pipe.hpp"
#include "internal.hpp"

namespace gemm_direct {

using namespace fe2o3;

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr uint32_t kUnit = 128;  // bytes of k per row and step

typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));

// One 16-row block's unit, two 16-byte pieces per lane.  As loaded: of rows
// l / 8 (words 0-3) and 8 + l / 8 (words 4-7) the piece l % 8.  As an MFMA
// operand: of row l % 16 the pieces l / 16 (words 0-3) and 4 + l / 16 (words
// 4-7); both operands use the same assignment, so every k meets its own.  (In
// the in-order form the pieces that the pipelined tile's MFMA takes from that
// lane: for fp8 2 (l / 16) and the next.)
typedef u32x8_t Frag;

struct Bf16 {
  static constexpr uint32_t kBytes = 2;  // per element
  static constexpr bool kScaled = false;
  static constexpr int kDeep = 3;  // units in flight of the widest forms
  static FE2O3_DEVICE uint32_t tile_piece(uint32_t g, uint32_t h) { return 4u * h + g; }
  static FE2O3_DEVICE void mma(const Frag& b, const Frag& a, f32x4_t& acc) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const u32x4_t bw = {b[4 * h], b[4 * h + 1], b[4 * h + 2], b[4 * h + 3]};
      const u32x4_t aw = {a[4 * h], a[4 * h + 1], a[4 * h + 2], a[4 * h + 3]};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, bw),
                                                    __builtin_bit_cast(bf16x8_t, aw), acc, 0, 0, 0);
    }
  }
};

// OCP e4m3: the unscaled 16x16x128 MFMA, as in gemm_pipe::Fp8Mma16
struct Fp8 {
  static constexpr uint32_t kBytes = 1;
  static constexpr bool kScaled = true;
  static constexpr int kDeep = 2;
  static FE2O3_DEVICE uint32_t tile_piece(uint32_t g, uint32_t h) { return 2u * g + h; }
  static FE2O3_DEVICE void mma(const Frag& b, const Frag& a, f32x4_t& acc) {
    acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
        __builtin_bit_cast(i32x8_t, b), __builtin_bit_cast(i32x8_t, a), acc, 0, 0, 0, 0, 0, 0);
  }
};

FE2O3_DEVICE u32x4_t load16(const uint8_t* p) {
  return *reinterpret_cast<const u32x4_any_t*>(p);
}

// A wave-uniform address that stays in scalar registers (the empty asm keeps
// the compiler from folding it into a 64-bit address per lane and load, which
// would cost two registers each): the lane adds a 32-bit offset.
struct ScalarBase {
  uint64_t p;
  explicit FE2O3_DEVICE ScalarBase(const uint8_t* q) : p((uint64_t)q) { asm("" : "+s"(p)); }
  template <class Off>
  FE2O3_DEVICE u32x4_t load16(Off off) const {
    typedef __attribute__((address_space(1))) const uint8_t* Global;
    typedef __attribute__((address_space(1))) const u32x4_any_t* Global16;
    return *(Global16)((Global)p + off);
  }
};

// A 16-byte piece shifted down by `bits` (0 .. 127), zeros shifted in; 128 and
// more leave it anyhow.
FE2O3_DEVICE u32x4_t shift_down(u32x4_t v, uint32_t bits) {
  uint64_t lo = v[0] | (uint64_t)v[1] << 32, hi = v[2] | (uint64_t)v[3] << 32;
  if (bits >= 64u) {
    lo = hi >> (bits & 63u);
    hi = 0;
  } else if (bits != 0u) {
    lo = lo >> bits | hi << (64u - bits);
    hi >>= bits;
  }
  return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// The 16-byte piece at byte `at` of a row of `bytes` bytes, zeros past its
// end.  Nothing past the row is read: a piece that straddles the end comes
// from the row's last 16 bytes, shifted down; a row shorter than that is read
// element by element.
template <uint32_t ELEM, class Off>
FE2O3_DEVICE u32x4_t load_end(const uint8_t* row, Off at, Off bytes) {
  if (at >= bytes) return u32x4_t{0, 0, 0, 0};
  if (bytes - at >= 16u) return load16(row + at);
  const uint32_t left = (uint32_t)(bytes - at);
  if (bytes >= 16u) return shift_down(load16(row + (bytes - 16u)), 8u * (16u - left));
  uint64_t lo = 0, hi = 0;
  // at most 15 bytes of a whole row: independent loads, no load waits
#pragma unroll
  for (uint32_t i = 0; i < 16u; i += ELEM) {
    if (i >= left) continue;
    uint64_t v;
    if constexpr (ELEM == 2) v = *reinterpret_cast<const uint16_t*>(row + at + i);
    else v = row[at + i];
    if (i < 8u) lo |= v << (8u * i);
    else hi |= v << (8u * i - 64u);
  }
  return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// HIP refuses a grid of 2^32 threads or more in one dimension, so the ids of a
// list of workgroups continue in y from kGridX on; the last row of the grid
// may run past the list.
constexpr uint32_t kGridX = 1u << 22;
inline dim3 list_grid(uint64_t workgroups) {
  return dim3((unsigned)(workgroups < kGridX ? workgroups : kGridX),
              (unsigned)((workgroups + kGridX - 1u) / kGridX));
}
FE2O3_DEVICE uint32_t list_id() { return blockIdx.y * kGridX + blockIdx.x; }

// Output block (tm, tn) of workgroup `id`: each XCD takes a contiguous run of
// the list (as tile_plan::xcd_tile_order does), block rows fastest, so that
// the blocks that read the same rows of B run together behind one L2.
FE2O3_DEVICE void block_of(uint32_t id, uint32_t tiles_m, uint32_t tiles_n, uint32_t xcds,
                           uint32_t* tm, uint32_t* tn) {
  const uint32_t total = tiles_m * tiles_n;
  if (xcds > 1u && total % xcds == 0u) id = (id % xcds) * (total / xcds) + id / xcds;
  *tm = id % tiles_m;
  *tn = id / tiles_m;
}

// One output block per workgroup, or (IN_ORDER) per wave.  T: Bf16 or Fp8.  D:
// units in flight per wave.  smem: kWaves * max(MB * NB, 2 (MB + NB)) KiB.  c:
// m x n bf16, rows n apart.  Off: of byte offsets within the block's rows
// (uint32_t while 64 rows of K fit it).
template <class T, int MB, int NB, int D, class Off = uint32_t, bool IN_ORDER = false>
FE2O3_DEVICE void block(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                        uint16_t* __restrict__ c, uint32_t m, uint32_t n, uint32_t k, float scale,
                        uint32_t xcds, uint8_t* smem) {
  const uint32_t lane = threadIdx.x & 63u, lr = lane & 15u, g = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tiles_m = (m - 1u) / (16u * MB) + 1u, tiles_n = (n - 1u) / (16u * NB) + 1u;
  // IN_ORDER: a workgroup's waves take neighbouring blocks of the list, and
  // share nothing, so a wave past its end just leaves
  const uint32_t id = IN_ORDER ? list_id() * kWaves + wave : list_id();
  if (id >= tiles_m * tiles_n) return;
  uint32_t tm, tn;
  block_of(id, tiles_m, tiles_n, IN_ORDER ? 1u : xcds, &tm, &tn);
  const uint32_t row0 = tm * 16u * MB, col0 = tn * 16u * NB;
  const Off kbytes = (Off)k * T::kBytes;
  // this lane's rows as offsets from the block's first; rows past the end
  // repeat the last, whose products reach no stored output
  const uint8_t* a0 = a + (uint64_t)row0 * kbytes;
  const uint8_t* b0 = b + (uint64_t)col0 * kbytes;
  const uint32_t pr = lane >> 3, pc = lane & 7u;  // piece: row (of 8) and place in the unit
  Off ao[2 * MB], bo[2 * NB];
#pragma unroll
  for (int i = 0; i < 2 * MB; ++i) ao[i] = min(8u * i + pr, m - 1u - row0) * kbytes + 16u * pc;
#pragma unroll
  for (int j = 0; j < 2 * NB; ++j) bo[j] = min(8u * j + pr, n - 1u - col0) * kbytes + 16u * pc;
  // the wave's LDS: 16 rows of 128 bytes per block, piece c of row r at place
  // c ^ swz(r), where neither the writes nor the reads conflict
  using G = gemm_pipe::Geo<128>;
  uint8_t* own = smem + wave * (uint32_t)(MB + NB) * 2048u;
  const uint32_t wr0 = pr * 128u + ((pc ^ G::swz(pr)) << 4);
  const uint32_t wr1 = (8u + pr) * 128u + ((pc ^ G::swz(8u + pr)) << 4);
  auto piece = [&](uint32_t h) { return IN_ORDER ? T::tile_piece(g, h) : 4u * h + g; };
  const uint32_t rd0 = lr * 128u + ((piece(0) ^ G::swz(lr)) << 4);
  const uint32_t rd1 = lr * 128u + ((piece(1) ^ G::swz(lr)) << 4);

  f32x4_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t af[D][2 * MB], bf[D][2 * NB];
  constexpr uint32_t kStride = IN_ORDER ? 1u : kWaves;  // units between the wave's own
  const uint32_t first_unit = IN_ORDER ? 0u : wave;
  // the wave's unit u into set s
  auto load = [&](int s, uint32_t u) {
    __builtin_amdgcn_sched_barrier(0);  // not before the set's last use: it has no second one
    const uint64_t at = ((uint64_t)u * kStride + first_unit) * kUnit;
    const ScalarBase pa(a0 + at), pb(b0 + at);
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j) bf[s][j] = pb.load16(bo[j]);
#pragma unroll
    for (int i = 0; i < 2 * MB; ++i) af[s][i] = pa.load16(ao[i]);
  };
  auto put = [&](uint32_t blk, u32x4_t lo, u32x4_t hi) {
    *reinterpret_cast<u32x4_t*>(own + blk * 2048u + wr0) = lo;
    *reinterpret_cast<u32x4_t*>(own + blk * 2048u + wr1) = hi;
  };
  auto get = [&](uint32_t blk) {
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(own + blk * 2048u + rd0);
    const u32x4_t hi = *reinterpret_cast<const u32x4_t*>(own + blk * 2048u + rd1);
    return Frag(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // set s through LDS into the sums.  A wave's LDS operations run in order,
  // so its reads see its writes and the next writes wait for these reads; the
  // fences only keep the compiler from reordering them (it sees one lane's
  // addresses, not the wave's).
  auto mma = [&](int s) {
#pragma unroll
    for (int j = 0; j < NB; ++j) put(MB + j, bf[s][2 * j], bf[s][2 * j + 1]);
#pragma unroll
    for (int i = 0; i < MB; ++i) put(i, af[s][2 * i], af[s][2 * i + 1]);
    asm volatile("" ::: "memory");
    Frag fb[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) fb[j] = get(MB + j);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const Frag fa = get(i);
#pragma unroll
      for (int j = 0; j < NB; ++j) T::mma(fb[j], fa, acc[i][j]);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  const uint32_t units = (uint32_t)(kbytes / kUnit);  // whole ones
  const uint32_t mine =
      units > first_unit ? (units - first_unit + kStride - 1u) / kStride : 0u;
  if (mine >= (uint32_t)D) {
#pragma unroll
    for (int s = 0; s < D; ++s) load(s, s);
    uint32_t u = D;
    for (; u + D <= mine; u += D)
#pragma unroll
      for (int s = 0; s < D; ++s) {
        mma(s);
        load(s, u + s);
      }
    const uint32_t rest = mine - u;  // below D
#pragma unroll
    for (int s = 0; s < D; ++s)
      if ((uint32_t)s < rest) {
        mma(s);
        load(s, u + s);
      }
#pragma unroll
    for (int s = 0; s < D; ++s)
      if ((uint32_t)s >= rest) mma(s);
#pragma unroll
    for (int s = 0; s < D; ++s)
      if ((uint32_t)s < rest) mma(s);
  } else {
#pragma unroll
    for (int s = 0; s < D; ++s)
      if ((uint32_t)s < mine) load(s, s);
#pragma unroll
    for (int s = 0; s < D; ++s)
      if ((uint32_t)s < mine) mma(s);
  }
  if (kbytes % kUnit != 0u && units % kStride == first_unit) {  // the partial last unit
    const Off at = (Off)units * kUnit + 16u * pc;
    if (kbytes >= 16u) {
      // a piece that the row's end cuts (or that lies past it) is read 16
      // bytes before it and shifted down, zeros shifted in: every load at once
      const Off from = min(at, kbytes - 16u);
      const uint32_t past = (uint32_t)min(at - from, (Off)16u);
      auto load_last = [&](const uint8_t* base, Off row) {
        return load16(base + (row - 16u * pc) + from);
      };
      auto cut = [&](u32x4_t v) { return past < 16u ? shift_down(v, 8u * past) : u32x4_t{}; };
#pragma unroll
      for (int j = 0; j < 2 * NB; ++j) bf[0][j] = load_last(b0, bo[j]);
#pragma unroll
      for (int i = 0; i < 2 * MB; ++i) af[0][i] = load_last(a0, ao[i]);
#pragma unroll
      for (int j = 0; j < 2 * NB; ++j) bf[0][j] = cut(bf[0][j]);
#pragma unroll
      for (int i = 0; i < 2 * MB; ++i) af[0][i] = cut(af[0][i]);
    } else {  // rows shorter than a piece
#pragma unroll
      for (int j = 0; j < 2 * NB; ++j)
        bf[0][j] = load_end<T::kBytes>(b0 + (bo[j] - 16u * pc), at, kbytes);
#pragma unroll
      for (int i = 0; i < 2 * MB; ++i)
        af[0][i] = load_end<T::kBytes>(a0 + (ao[i] - 16u * pc), at, kbytes);
    }
    mma(0);
  }

  const bool vec = n % 4u == 0u && ((uintptr_t)c & 7u) == 0u;
  // lane l's 4 columns of 16 x 16 block blk (i * NB + j)
  auto store = [&](uint32_t blk, uint32_t l, f32x4_t sum) {
    const uint32_t row = row0 + 16u * (blk / NB) + (l & 15u);
    const uint32_t col = col0 + 16u * (blk % NB) + 4u * (l >> 4);
    if (row >= m || col >= n) return;
    uint16_t* out = c + (uint64_t)row * n + col;
    if constexpr (T::kScaled)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] *= scale;
    if (vec) {
      *reinterpret_cast<u32x2_t*>(out) =
          u32x2_t{pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < n) out[e] = bf16_bits_from_f32(sum[e]);
    }
  };
  if constexpr (IN_ORDER) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) store(i * NB + j, lane, acc[i][j]);
    return;
  }
  __syncthreads();  // the partial sums take the LDS of all waves' units
  // partial sums [wave][block][lane], then one thread per 4 columns of a row
  // adds the waves' in order
  f32x4_t* part = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) part[(wave * MB * NB + i * NB + j) * 64u + lane] = acc[i][j];
  __syncthreads();
#pragma unroll
  for (uint32_t t = threadIdx.x; t < MB * NB * 64u; t += kThreads) {
    f32x4_t sum = part[t];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += part[w * MB * NB * 64u + t];
    store(t >> 6, t & 63u, sum);
  }
}

// ---- forms -----------------------------------------------------------------------------
// MB x NB of a workgroup and the units in flight (registers: 8 (MB + NB) D
// fragments and 4 MB NB sums).  The light forms leave room for two workgroups
// per CU (128 registers), the wide ones for one.
struct Form {
  uint32_t mb, nb;
  bool wide;
};
constexpr Form kForms[] = {{1, 1, false}, {1, 2, false}, {2, 1, false}, {2, 2, false},
                           {1, 4, true},  {4, 1, true},  {2, 4, true},  {4, 2, true}};
constexpr int kNumForms = sizeof(kForms) / sizeof(kForms[0]);

inline uint64_t grid_of(const Form& f, uint32_t m, uint32_t n) {
  return ((uint64_t)m + 16u * f.mb - 1u) / (16u * f.mb) *
         (((uint64_t)n + 16u * f.nb - 1u) / (16u * f.nb));
}
// What a form costs: the 16-row blocks of operand that the busiest CU loads.
inline uint64_t cost_of(const Form& f, uint32_t m, uint32_t n, uint32_t cus) {
  return (grid_of(f, m, n) + cus - 1u) / cus * (f.mb + f.nb);
}
// The cheapest form; of equals the larger block, which reads less in all.
inline int choose(uint32_t m, uint32_t n, uint32_t cus, uint64_t* cost = nullptr) {
  int best = 0;
  for (int i = 1; i < kNumForms; ++i)
    if (cost_of(kForms[i], m, n, cus) <= cost_of(kForms[best], m, n, cus)) best = i;
  if (cost) *cost = cost_of(kForms[best], m, n, cus);
  return best;
}

// Whether the direct kernel takes a GEMM that the pipelined tile could run
// too.  The tile's time hardly depends on the output while that is at most
// one round of 128 x 128 tiles; the direct kernel's grows with the cost, and
// passes it between 10 and 12 (us, tile against direct):
//   bf16 16 x 4096 x 4096   21.4 |  7.7     fp8 32 x 8192 x 8192  22.9 | 12.4
//   bf16 64 x 4096 x 4096   24.3 |  9.6     fp8 64 x 8192 x 8192  24.7 | 16.4
//   bf16 128 x 4096 x 4096  22.5 | 13.6     fp8 128 x 4096 x 8192 22.8 | 13.7
//   bf16 128 x 8192 x 4096  23.5 | 25.4     fp8 128 x 8192 x 2048  8.7 | 10.1
// (the last line costs 12).  Where the tile needs its operands repacked first,
// the lines cross between 18 and 24 (256 x 4096 x 4097: 58.1 | 36.2, 320: 58.0 |
// 52.9, 512 x 4096 x 4090: 42.7 | 77.4).  At most 32 rows or columns (of K from
// eight units on, one a wave) stream the other operand, and stream_prefer
// decides.  The rules look at sizes only, so that a misaligned operand gives
// the aligned one's bits.
//
// stream_prefer: `rows` of the streamed operand, the other's at most 32; tall:
// it is A, and C has few columns.  Up to a round of tiles the line lies at the
// cost again, and past it once the tiles fill most CUs and no longer stream
// faster for being more.  Beyond a round the direct kernel's smaller blocks
// spread better, unless K is so short that its merge shows more than the
// tile's stores (of a tall C they cost most).  Tile against direct, us, the
// streamed operand from HBM and (in brackets) from the last-level cache, which
// a program that streams its weights does not see:
//   bf16 16 x 14336 x 4096  36.5 | 24.5 (23.3 | 19.5)   cost 5, 112 tiles
//   bf16 16 x 20000 x 512    8.3 |  7.1  (6.1 |  4.7)   cost 9, 157 tiles
//   bf16 16 x 20000 x 4096  40.8 | 37.8 (26.6 | 34.3)
//   bf16 32 x 20000 x 4096  42.3 | 44.8 (28.5 | 34.1)   cost 12
//   bf16 16 x 28672 x 1024  13.5 | 15.0 (12.1 | 12.9)   cost 10, 224 tiles
//   bf16 16 x 28672 x 4096  46.5 | 43.9 (34.5 | 36.9)
//   bf16 32 x 28672 x 1024  13.3 | 16.4 (11.9 | 13.8)   cost 12
//   bf16 32 x 28672 x 4096  53.3 | 48.9 (36.3 | 38.6)
//   bf16 16 x 40000 x 512   15.9 | 13.3 (13.6 | 10.0)   cost 15, 313 tiles
//   bf16 16 x 65536 x 1024  30.1 | 31.8 (26.9 | 26.5)   cost 20, 512 tiles
//   bf16 65536 x 16 x 1024  38.5 | 31.5 (34.7 | 25.8)
//   bf16 16 x 65536 x 4096 131.2 | 97.8                 fp8 69.8 | 58.9 (47.2 | 44.2)
inline bool stream_prefer(uint32_t rows, bool tall, uint64_t kbytes, uint64_t cost,
                          uint32_t cus) {
  const uint64_t tiles = ((uint64_t)rows + 127u) / 128u;
  if (tiles > cus) return tall || kbytes >= 4096u || 2u * tiles <= 3ull * cus;
  if (kbytes < 4096u) return cost <= (tall ? 10u : 9u);
  return cost <= 10u || 4u * tiles >= 3ull * cus;
}
inline bool prefer(uint32_t m, uint32_t n, uint32_t k, uint32_t elem_bytes, uint32_t cus) {
  const uint64_t kbytes = (uint64_t)k * elem_bytes;
  uint64_t cost = 0;
  choose(m, n, cus, &cost);
  if ((m <= 32u || n <= 32u) && kbytes >= kWaves * kUnit)
    return kbytes % 16u != 0u || stream_prefer(m > n ? m : n, m > n, kbytes, cost, cus);
  return cost <= (kbytes % 16u == 0u ? 10u : 18u);
}
// Operands that the pipelined tiles cannot read in place are taken up to 65535
// blocks of 64 rows of A; more are a shape error.
inline bool rows_ok(uint32_t m) { return ((uint64_t)m + 63u) / 64u <= 65535u; }

// A call past prefer's line whose operands the tile cannot read in place, but
// could at these sizes at another alignment or after a copy: its C has the
// tile's bits on every way there.
//   tile_sizes: outputs from 128 x 128 on (any K, copied into rows of whole
//     pieces), and smaller ones whose rows are whole pieces.
//   repack: they are copied into scratch for the tile; small ones only when
//     K is long and the call is not captured into a graph, else the in-order
//     form, which also serves without scratch (us, copies and tile against
//     in order: bf16 100 x 8192 x 4096 53 | 114, fp8 38 | 59; bf16 127 x 9000 x
//     1024 29 | 31, fp8 29 | 17; bf16 16 x 40000 x 256 25 | 10).
constexpr uint32_t kRepackMin = 128;
constexpr uint32_t kShortK = 2048;  // bytes, 16 units
inline bool tile_sizes(uint32_t m, uint32_t n, uint32_t k, uint32_t elem_bytes) {
  const uint64_t kbytes = (uint64_t)k * elem_bytes, padded = (kbytes + 15u) / 16u * 16u;
  return 256ull * padded < (1ull << 31) &&
         (padded == kbytes || (m >= kRepackMin && n >= kRepackMin));
}
inline bool repack(uint32_t m, uint32_t n, uint32_t k, uint32_t elem_bytes, hipStream_t s) {
  return tile_sizes(m, n, k, elem_bytes) &&
         ((m >= kRepackMin && n >= kRepackMin) ||
          ((uint64_t)k * elem_bytes > kShortK && rows_ok(m) && !fe2o3_host::capturing(s)));
}
// The in-order form also takes the short K of sizes that no tile runs: at most
// two units a wave do not pay for the split's merge.  Split | in order, us:
//   bf16 100000 x 5 x 65 21 | 8   40001 x 33 x 75 23 | 9   20000 x 100 x 401 33 | 25
//   fp8 20000 x 100 x 1601 48 | 44   past the line: bf16 20000 x 100 x 1601 55 | 73
inline bool in_order(uint32_t m, uint32_t n, uint32_t k, uint32_t elem_bytes) {
  return tile_sizes(m, n, k, elem_bytes) || (uint64_t)k * elem_bytes <= kShortK;
}

// 64 rows of K within 32-bit byte offsets, as the chosen forms need
inline bool k_fits(uint32_t k, uint32_t elem_bytes) { return 64ull * k * elem_bytes < (1ull << 32); }

constexpr uint32_t smem_of(uint32_t mb, uint32_t nb) {
  return kWaves * 1024u * (mb * nb > 2u * (mb + nb) ? mb * nb : 2u * (mb + nb));
}
// Launches of the light kernel or the wide one, which also holds the last three
// (in the light one they would cost its forms registers).
constexpr int kAnyK = kNumForms, kInOrder = kNumForms + 1, kFill = kNumForms + 2;
struct Launch {
  int form;
  bool wide;
  uint64_t grid;
  uint32_t smem;
};
inline Launch plan(uint32_t m, uint32_t n, uint32_t k, uint32_t elem_bytes, uint32_t cus) {
  const int form = k_fits(k, elem_bytes) ? choose(m, n, cus) : kAnyK;
  const Form f = form < kNumForms ? kForms[form] : Form{1, 4, true};
  return {form, f.wide, grid_of(f, m, n), smem_of(f.mb, f.nb)};
}
// 2 x 2 blocks, one per wave; their ids are 32-bit, so more of them stay a grid
// that the launch refuses
inline Launch plan_in_order(uint32_t m, uint32_t n) {
  const uint64_t blocks = grid_of(Form{2, 2, false}, m, n);
  return {kInOrder, true, blocks > 0x7fffffffu ? blocks : (blocks + kWaves - 1u) / kWaves,
          smem_of(2, 2)};
}
// K = 0: C is all +0 (an empty sum, whatever the scales).  A grid-stride fill
// rather than a memset node, so a caller may capture it, and rather than the
// blocks' walk over nothing (8192 x 8192: 235 us).
inline Launch plan_fill(uint64_t c_len) {
  const uint64_t groups = (c_len / 8u + kThreads - 1u) / kThreads;
  return {kFill, true, groups < 2048u ? (groups ? groups : 1u) : 2048u, 0u};
}

constexpr int kLightSmem = (int)smem_of(2, 2), kWideSmem = (int)smem_of(4, 2);

FE2O3_DEVICE void fill(uint16_t* __restrict__ c, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * kThreads;
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x, pieces = n / 8u;
  for (uint64_t i = t; i < pieces; i += stride)
    *reinterpret_cast<u32x4_any_t*>(c + 8u * i) = u32x4_t{0, 0, 0, 0};
  if (t < n % 8u) c[8u * pieces + t] = 0;
}

// A launch's workgroup on form `form` (an index of kForms, or one of the forms
// past it).
template <class T, bool WIDE>
FE2O3_DEVICE void run_form(int form, const uint8_t* a, const uint8_t* b, uint16_t* c, uint32_t m,
                           uint32_t n, uint32_t k, float scale, uint32_t xcds, uint8_t* smem) {
#define FE2O3_DIRECT(MB, NB, D) return block<T, MB, NB, D>(a, b, c, m, n, k, scale, xcds, smem)
  if constexpr (!WIDE) {
    switch (form) {
      case 0: FE2O3_DIRECT(1, 1, 4);
      case 1: FE2O3_DIRECT(1, 2, 3);
      case 2: FE2O3_DIRECT(2, 1, 3);
      default: FE2O3_DIRECT(2, 2, 2);
    }
  } else {
    switch (form) {
      case 4: FE2O3_DIRECT(1, 4, 3);
      case 5: FE2O3_DIRECT(4, 1, 3);
      case 6: FE2O3_DIRECT(2, 4, T::kDeep);
      case 7: FE2O3_DIRECT(4, 2, T::kDeep);
      case kInOrder:
        return block<T, 2, 2, 2, uint32_t, true>(a, b, c, m, n, k, scale, xcds, smem);
      case kFill: return fill(c, (uint64_t)m * n);
      default: return block<T, 1, 4, 1, uint64_t>(a, b, c, m, n, k, scale, xcds, smem);
    }
  }
#undef FE2O3_DIRECT
}

}  // namespace gemm_direct
