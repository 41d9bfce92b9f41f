// softmax.hip -- stable row softmax for gfx950.
//
// Semantics (examples/row_softmax_v1/src/kernel.rs:13-42 for the arithmetic,
// examples/row_softmax_v1/src/numerical_contract.rs:130-199 for the mask):
//   max over active elements, w_i = exp(x_i - max) in f32 (OCML expf, as the
//   reference's DeviceMath::exp_f32), sum of w, out_i = w_i / sum (correctly
//   rounded f32 division); masked elements -> +0.  A row without an active
//   element is written as all +0.
//   Non-finite input: the reference's contract rejects a row holding a NaN
//   or an infinity anywhere, masked elements included
//   (examples/row_softmax_v1/src/numerical_contract.rs:145-151).  Such a row
//   is written as all quiet NaN (0x7fc00000) and the device's contract-status
//   word is marked, so the host's next synchronize reports
//   FE2O3_ERR_NONFINITE; other rows are unaffected.  The check is one FMA per
//   element folded into the pass that already holds the row.
//
// Rows of 4 .. 8192 columns, any width and any 4-byte alignment, live in
// registers (softmax_reg_kernel): each row is read from HBM once and written
// once, so the kernel is HBM-bound at 8 bytes per element (9 with a mask).
// Other widths take a strided three-pass path (max, sum, write) per lane.
#include "common.hpp"
#include "internal.hpp"
#include "profiles.hpp"

namespace {

using namespace fe2o3;

constexpr int ROWS_PER_BLOCK = 4;  // 4 waves, one row each

// 16 bytes at 4-byte alignment: gfx950 global accesses of four dwords need no
// more, and a wave's 1 KiB then touches at most one cache line extra.
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32_any_t __attribute__((aligned(1)));

// Reductions over the LANES lanes of one row.
template <int LANES>
FE2O3_DEVICE float row_max(float v) {
#pragma unroll
  for (int o = 1; o < LANES; o <<= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
template <int LANES>
FE2O3_DEVICE float row_sum(float v) {
#pragma unroll
  for (int o = 1; o < LANES; o <<= 1) v = v + __shfl_xor(v, o, 64);
  return v;
}

// One row of 4 <= cols <= 4 * LANES * NV columns on LANES lanes (64 / LANES
// rows per wave): lane l, chunk j holds the four columns from c = 4 (LANES j
// + l) on.  The last TAIL chunks may pass the row's end (the others do not:
// cols >= 4 LANES (NV - TAIL)).  There the lane whose four would pass it takes
// the row's last four instead, of which the ones from column c on are its
// own: it counts those only, and stores all four, since the lane it shares
// the others with stores the same bits.  Lanes past the end load those four
// too and store nothing, so no load is guarded and none leaves the row.
//
// Bound by HBM for wide rows, by the exponential and the division (about 40
// VALU instructions an element) for rows that the caches hold.  Against three
// passes over the row with 4-byte accesses and two exponentials per element,
// which every width but 256 x a power of two took: 32768 x 1000 with a mask
// 155.4 -> 45.9 us (6.4 TB/s), 32768 x 1001 124.3 -> 46.5, 30388 x 7168 898 ->
// 312 (5.6 TB/s), 100000 x 64 27.6 -> 10.8, 64 x 8000 76 -> 10.3.
template <int LANES, int NV, int TAIL, bool MASK>
FE2O3_DEVICE void softmax_row_regs(const float* __restrict__ in, float* __restrict__ out,
                                   const uint8_t* __restrict__ mask, uint64_t rows, uint32_t cols,
                                   uint32_t* __restrict__ status) {
  constexpr uint32_t kRowsPerWave = 64 / LANES, kChunk = 4u * LANES;
  if constexpr (TAIL == 0) cols = kChunk * NV;
  // Long rows take their exponentials and divisions chunk by chunk, and their
  // addresses from scalar registers: interleaved, they need registers that
  // cost a wave per SIMD (65536 x 4096: 370.6 -> 365.2 us).  Whole rows of
  // 8192 and the shorter ones run 1-2% faster without.
  constexpr bool in_order = NV > 8 && !(NV == 32 && TAIL == 0);
  const uint32_t lane = threadIdx.x & 63u, l = lane % LANES;
  const uint32_t w = threadIdx.x >> 6, wave = in_order ? __builtin_amdgcn_readfirstlane(w) : w;
  const uint64_t row =
      ((uint64_t)blockIdx.x * ROWS_PER_BLOCK + wave) * kRowsPerWave + lane / LANES;
  if (row >= rows) return;
  const float* src = in + row * cols;
  f32x4_t x[NV];
  uint32_t act[NV];
  // where this lane's four of chunk j are in a row (whole chunks at constant
  // distances, so that their addresses share registers), and how many of the
  // four belong to the lane before it (4 and more: all of them)
  auto at = [&](auto* base, int j) {
    return j < NV - TAIL ? base + 4u * l + kChunk * j : base + min(kChunk * j + 4u * l, cols - 4u);
  };
  auto shared = [&](int j) {
    const uint32_t c = kChunk * j + 4u * l;
    return c - min(c, cols - 4u);
  };
#pragma unroll
  for (int j = 0; j < NV; ++j)
    x[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_any_t*>(at(src, j)));
  if (MASK) {
    const uint8_t* msrc = mask + row * cols;
#pragma unroll
    for (int j = 0; j < NV; ++j) act[j] = *reinterpret_cast<const u32_any_t*>(at(msrc, j));
  }
  auto active = [&](int j, int e) -> bool {
    return !MASK || ((act[j] >> (8 * e)) & 0xffu) != 0u;
  };
  float mx = -INFINITY;
  f32x4_t probe = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < NV; ++j) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      probe[e] = finite_probe(probe[e], x[j][e]);
      if (active(j, e)) mx = fmaxf(mx, x[j][e]);
    }
  }
  mx = row_max<LANES>(mx);
  const float pr = (probe[0] + probe[1]) + (probe[2] + probe[3]);
  const uint64_t bad = __ballot(pr != pr);
  const bool rejected =
      LANES == 64 ? bad != 0ull
                  : ((bad >> (lane - l)) & ((1ull << (LANES & 63)) - 1ull)) != 0ull;
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (in_order) __builtin_amdgcn_sched_barrier(0);
    f32x4_t own;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[j][e] = active(j, e) ? expf(x[j][e] - mx) : 0.0f;
      own[e] = j < NV - TAIL || shared(j) <= (uint32_t)e ? x[j][e] : 0.0f;
    }
    sum += (own[0] + own[1]) + (own[2] + own[3]);
  }
  sum = row_sum<LANES>(sum);
  const bool any = mx != -INFINITY;
  float* dst = out + row * cols;
  auto store = [&](int j, f32x4_t y) {
    if (j < NV - TAIL || shared(j) < 4u)
      __builtin_nontemporal_store(f32x4_any_t(y), reinterpret_cast<f32x4_any_t*>(at(dst, j)));
  };
  if (rejected) {
    if (l == 0) mark_nonfinite(status);
    const float nan = quiet_nan();
#pragma unroll
    for (int j = 0; j < NV; ++j) store(j, f32x4_t{nan, nan, nan, nan});
    return;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (in_order) __builtin_amdgcn_sched_barrier(0);
    f32x4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = any ? x[j][e] / sum : 0.0f;
    store(j, y);
  }
}

// Rows per wave: rows of at most 64 columns take a quarter of a wave, rows of
// at most 256 half of one (131072 x 256: 47.4 -> 42.6 us against one row per
// wave).
FE2O3_HD uint32_t rows_per_wave(uint64_t cols) { return cols <= 64 ? 4u : cols <= 256 ? 2u : 1u; }

// Rows of at most 256 NV columns (and, NV > 4, more than 128 NV), by their
// number of 256-column chunks: one form per chunk up to 16, every second one
// up to 32.  Whole rows of 256 NV columns have no tail, and WHOLE kernels of
// their own where the tail forms would cost them waves.  Forms are unrolled
// over exactly their chunks: one form per NV that branches around the chunks
// past the row took 1.24x the time of the whole-row form at 65536 x 2048 (149
// registers instead of 58).
template <int NV, bool MASK, bool WHOLE>
__global__ void __launch_bounds__(256) softmax_reg_kernel(const float* __restrict__ in,
                                                          float* __restrict__ out,
                                                          const uint8_t* __restrict__ mask,
                                                          uint64_t rows, uint32_t cols,
                                                          uint32_t* __restrict__ status) {
#define FE2O3_SOFTMAX_FORM(LANES, CHUNKS, TAIL) \
  return softmax_row_regs<LANES, CHUNKS, TAIL, MASK>(in, out, mask, rows, cols, status)
#define FE2O3_SOFTMAX_TAIL_FORM(CHUNKS, TAIL) \
  if (cols <= 256u * (CHUNKS)) FE2O3_SOFTMAX_FORM(64, (CHUNKS), TAIL)
  if constexpr (WHOLE) {
    FE2O3_SOFTMAX_FORM(64, NV, 0);
  } else if constexpr (NV == 4) {
    if (cols == 256u) FE2O3_SOFTMAX_FORM(32, 2, 0);
    if (cols == 512u) FE2O3_SOFTMAX_FORM(64, 2, 0);
    if (cols == 1024u) FE2O3_SOFTMAX_FORM(64, 4, 0);
    if (rows_per_wave(cols) == 4u) FE2O3_SOFTMAX_FORM(16, 1, 1);
    if (cols <= 128u) FE2O3_SOFTMAX_FORM(32, 1, 1);
    if (rows_per_wave(cols) == 2u) FE2O3_SOFTMAX_FORM(32, 2, 1);
    FE2O3_SOFTMAX_TAIL_FORM(2, 1);
    FE2O3_SOFTMAX_TAIL_FORM(3, 1);
    FE2O3_SOFTMAX_FORM(64, 4, 1);
  } else {
    constexpr int H = NV / 2, T = NV == 32 ? 2 : 1;  // forms H + T, H + 2T, ... NV
    if constexpr (NV == 8) {
      if (cols == 2048u) FE2O3_SOFTMAX_FORM(64, 8, 0);
    } else {
      FE2O3_SOFTMAX_TAIL_FORM(H + T, T);
      FE2O3_SOFTMAX_TAIL_FORM(H + 2 * T, T);
      FE2O3_SOFTMAX_TAIL_FORM(H + 3 * T, T);
      FE2O3_SOFTMAX_TAIL_FORM(H + 4 * T, T);
    }
    FE2O3_SOFTMAX_TAIL_FORM(NV - 3 * T, T);
    FE2O3_SOFTMAX_TAIL_FORM(NV - 2 * T, T);
    FE2O3_SOFTMAX_TAIL_FORM(NV - T, T);
    FE2O3_SOFTMAX_FORM(64, NV, T);
  }
#undef FE2O3_SOFTMAX_TAIL_FORM
#undef FE2O3_SOFTMAX_FORM
}

__global__ void __launch_bounds__(256) softmax_strided_kernel(const float* __restrict__ in,
                                                              float* __restrict__ out,
                                                              const uint8_t* __restrict__ mask,
                                                              uint64_t rows, uint64_t cols,
                                                              uint32_t* __restrict__ status) {
  const uint64_t row = (uint64_t)blockIdx.x * ROWS_PER_BLOCK + (threadIdx.x >> 6);
  if (row >= rows) return;
  fe2o3_profiles::softmax_row(in + row * cols, out + row * cols,
                              mask ? mask + row * cols : nullptr, cols, status);
}

template <int NV, bool WHOLE>
void launch_reg(const float* in, float* out, const uint8_t* mask, uint64_t rows, uint32_t cols,
                dim3 grid, uint32_t* status, hipStream_t s) {
  if (mask)
    softmax_reg_kernel<NV, true, WHOLE><<<grid, 256, 0, s>>>(in, out, mask, rows, cols, status);
  else
    softmax_reg_kernel<NV, false, WHOLE><<<grid, 256, 0, s>>>(in, out, mask, rows, cols, status);
}

// exact_profile: the one-row profile, whose bits are those of the code
// object that runs softmax_row too.
int32_t row_softmax(const float* input, uint64_t input_len, float* output, uint64_t output_len,
                    const uint8_t* mask, uint64_t mask_len, uint64_t rows, uint64_t cols,
                    bool exact_profile, void* stream) {
  if (cols == 0) return FE2O3_ERR_SHAPE;
  if (rows > UINT64_MAX / cols) return FE2O3_ERR_OVERFLOW;
  const uint64_t n = rows * cols;
  if (input_len != n || output_len != n || (mask && mask_len != n)) return FE2O3_ERR_LENGTH;
  if (n == 0) return FE2O3_OK;
  if (!input || !output) return FE2O3_ERR_NULL;
  if ((rows + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK > 0x7fffffffu) return FE2O3_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  uint32_t* status = fe2o3_host::status_word();
  if (status == nullptr) return (int32_t)hipErrorInvalidSymbol;
  const bool regs = cols >= 4 && cols <= 256 * 32 && !exact_profile;
  const uint64_t per_block = ROWS_PER_BLOCK * (regs ? rows_per_wave(cols) : 1u);
  const dim3 grid((unsigned)((rows + per_block - 1) / per_block));
  const uint32_t c = (uint32_t)cols;
  if (!regs)
    softmax_strided_kernel<<<grid, 256, 0, s>>>(input, output, mask, rows, cols, status);
  else if (c <= 1024)
    launch_reg<4, false>(input, output, mask, rows, c, grid, status, s);
  else if (c <= 2048)
    launch_reg<8, false>(input, output, mask, rows, c, grid, status, s);
  else if (c < 4096)
    launch_reg<16, false>(input, output, mask, rows, c, grid, status, s);
  else if (c == 4096)
    launch_reg<16, true>(input, output, mask, rows, c, grid, status, s);
  else if (c < 8192)
    launch_reg<32, false>(input, output, mask, rows, c, grid, status, s);
  else
    launch_reg<32, true>(input, output, mask, rows, c, grid, status, s);
  return fe2o3_host::after_launch();
}

// kernels behind each entry point (fe2o3_kernel_resources)
const fe2o3_host::KernelRegistrar kRegistered[] = {
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax_v1", "softmax_strided_kernel", (const void*)softmax_strided_kernel, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<4>", (const void*)softmax_reg_kernel<4, false, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<4, mask>", (const void*)softmax_reg_kernel<4, true, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<8>", (const void*)softmax_reg_kernel<8, false, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<8, mask>", (const void*)softmax_reg_kernel<8, true, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<16>", (const void*)softmax_reg_kernel<16, false, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<16, mask>", (const void*)softmax_reg_kernel<16, true, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<16, whole>", (const void*)softmax_reg_kernel<16, false, true>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<16, mask, whole>", (const void*)softmax_reg_kernel<16, true, true>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<32>", (const void*)softmax_reg_kernel<32, false, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<32, mask>", (const void*)softmax_reg_kernel<32, true, false>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<32, whole>", (const void*)softmax_reg_kernel<32, false, true>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_reg_kernel<32, mask, whole>", (const void*)softmax_reg_kernel<32, true, true>, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_row_softmax", "softmax_strided_kernel", (const void*)softmax_strided_kernel, 256, 0})};

}  // namespace

extern "C" {

int32_t fe2o3_row_softmax_v1(const float* input, uint64_t input_len, float* output,
                             uint64_t output_len, void* stream) {
  FE2O3_ENTRY("fe2o3_row_softmax_v1");
  // examples/row_softmax_v1: exactly one 64-element row.
  if (input_len != 64 || output_len != 64) return FE2O3_ERR_LENGTH;
  return row_softmax(input, input_len, output, output_len, nullptr, 0, 1, 64, true, stream);
}

int32_t fe2o3_row_softmax(const float* input, uint64_t input_len, float* output,
                          uint64_t output_len, const uint8_t* mask, uint64_t mask_len,
                          uint64_t rows, uint64_t cols, void* stream) {
  FE2O3_ENTRY("fe2o3_row_softmax");
  return row_softmax(input, input_len, output, output_len, mask, mask_len, rows, cols, false,
                     stream);
}

}  // extern "C"
