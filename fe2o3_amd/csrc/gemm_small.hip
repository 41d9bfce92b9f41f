// gemm_small.hip -- the reference's fixed-profile and general GEMM kernels,
// rebuilt for gfx950:
//   * tiled_gemm_lds_slice1 / moe_expert_gemm_bf16_m16_n16_k16: one 16x16x16
//     bf16 tile, one wave64, LDS staging, one v_mfma_f32_16x16x32_bf16 with
//     the upper K half zero;
//   * tiled_gemm_general_v1: any m, n, k, strides, alpha/beta; the pipelined
//     tiles of gemm_pipe.hpp, or 64x64 tiles through registers for small
//     outputs and operands of any alignment; unfused alpha/beta epilogue.  The
//     reference's two global-transfer schedules
//     (crates/dialect-schedule/src/general_gemm.rs:13-38) are two entry points
//     to the same kernels;
//   * scalar_gemm_v1: f32, the reference's per-output sequential unfused
//     recurrence, LDS-tiled and register-blocked (4x4 outputs per thread),
//     bit-identical to the scalar oracle.
#include "common.hpp"
#include "gemm_core.hpp"
#include "gemm_direct.hpp"
#include "gemm_pipe.hpp"
#include "internal.hpp"

namespace {

using namespace fe2o3;

// ---- 16x16x16 bf16 tile ------------------------------------------------------------
// A row-major [16 rows][16 k]; B row-major [16 k][16 n]; C row-major f32.
// LDS holds A as [row][k] and B transposed as [n][k] so both MFMA operands
// are one 16-byte read: lane l < 32 reads row/col l%16, k-chunk l/16 (8 k
// values); lanes 32..63 feed zeros for the unused upper K half.  The output
// fragment of lane l is column l%16, rows 4*(l/16)+i (i = 0..3), i.e. the
// reference's Blocked<Index1D,16,4> ownership
// (crates/fe2o3-device/src/thread.rs:569-600) of the row-major C tile.
__global__ void __launch_bounds__(64) tile16_bf16_kernel(const uint16_t* __restrict__ a,
                                                         const uint16_t* __restrict__ b,
                                                         float* __restrict__ c) {
  __shared__ __attribute__((aligned(16))) uint16_t a_lds[16 * 16];
  __shared__ __attribute__((aligned(16))) uint16_t bt_lds[16 * 16];
  const int l = threadIdx.x;
  // stage: lane l owns elements 4l..4l+3 of each operand
  {
    const uint2 av = *reinterpret_cast<const uint2*>(a + 4 * l);
    *reinterpret_cast<uint2*>(a_lds + 4 * l) = av;
    const uint2 bv = *reinterpret_cast<const uint2*>(b + 4 * l);
    const int kk = l >> 2, n0 = (l & 3) * 4;
    bt_lds[(n0 + 0) * 16 + kk] = (uint16_t)(bv.x & 0xffffu);
    bt_lds[(n0 + 1) * 16 + kk] = (uint16_t)(bv.x >> 16);
    bt_lds[(n0 + 2) * 16 + kk] = (uint16_t)(bv.y & 0xffffu);
    bt_lds[(n0 + 3) * 16 + kk] = (uint16_t)(bv.y >> 16);
  }
  __syncthreads();
  bf16x8_t af = {}, bf = {};
  if (l < 32) {
    const int rc = l & 15, chunk = l >> 4;
    af = *reinterpret_cast<const bf16x8_t*>(a_lds + rc * 16 + chunk * 8);
    bf = *reinterpret_cast<const bf16x8_t*>(bt_lds + rc * 16 + chunk * 8);
  }
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, acc, 0, 0, 0);
  const int col = l & 15, row0 = (l >> 4) * 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) c[(row0 + i) * 16 + col] = acc[i];
}

// ---- exact-tile multi-tile GEMM (tiled_gemm_v1 plan) ---------------------------------
// C[M,N] f32 = A[M,K] bf16 (row-major) * B[K,N] bf16 (row-major), M, N, K
// multiples of 16.  One wave64 per 16x16 output tile, as the reference's plan
// assigns (examples/tiled_gemm_v1/src/contract.rs:387-427); workgroup id ->
// (tile column, tile row) = (id % tile_cols, id / tile_cols).  Each
// v_mfma_f32_16x16x32_bf16 consumes two 16-deep reduction tiles; with an odd
// count the last MFMA's upper half is zero.  Operand lanes: A row l%16 and
// B column l%16, k chunk 8*(l/16) .. +7 of the 32-deep step, read straight
// from global memory (a chunk lies wholly inside or wholly past K).  The
// output lane map is tile16_bf16_kernel's.
__global__ void __launch_bounds__(64) tiled_v1_kernel(const uint16_t* __restrict__ a,
                                                      const uint16_t* __restrict__ b,
                                                      float* __restrict__ c, uint32_t n,
                                                      uint32_t k, uint32_t tile_cols) {
  const uint32_t l = threadIdx.x;
  const uint32_t tr = blockIdx.x / tile_cols, tc = blockIdx.x % tile_cols;
  const uint32_t rc = l & 15u, chunk = l >> 4;
  const uint16_t* arow = a + (uint64_t)(tr * 16u + rc) * k;
  const uint16_t* bcol = b + tc * 16u + rc;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (uint32_t kk = 0; kk < k; kk += 32u) {
    const uint32_t k0 = kk + 8u * chunk;
    bf16x8_t af = {}, bf = {};
    if (k0 < k) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        af[i] = __builtin_bit_cast(__bf16, arow[k0 + i]);
        bf[i] = __builtin_bit_cast(__bf16, bcol[(uint64_t)(k0 + i) * n]);
      }
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, acc, 0, 0, 0);
  }
  float* ctile = c + (uint64_t)(tr * 16u + 4u * chunk) * n + tc * 16u + rc;
#pragma unroll
  for (int i = 0; i < 4; ++i) ctile[(uint64_t)i * n] = acc[i];
}

// +0 fill of the plan's K = 0 case (a kernel rather than a memset, so the
// call can sit inside a captured graph).
__global__ void __launch_bounds__(256) zero_fill_kernel(float* __restrict__ c, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u)
    c[i] = 0.0f;
}

// ---- scalar f32 GEMM (sequential, unfused) -----------------------------------------
// Workgroup tile 16x16, 256 threads, one output per thread, whose accumulator
// follows acc = acc + a*b over t = 0..k-1 in order.  One output per thread
// (rather than a register block) spreads a 256^3 problem over 256 workgroups;
// the k loop runs in LDS chunks of 256, so k <= 256 waits for global memory
// once.
constexpr int S_BM = 16, S_BN = 16, S_BK = 256;

__global__ void __launch_bounds__(256) scalar_gemm_kernel(const float* __restrict__ a,
                                                          const float* __restrict__ b,
                                                          float* __restrict__ c, uint32_t m,
                                                          uint32_t n, uint32_t k) {
#pragma clang fp contract(off)
  // Both tiles k-contiguous per row (B transposed on the way in), rows padded
  // to 260 floats: 16-byte reads of 4 consecutive depths, conflict-free.
  constexpr int LD = S_BK + 4;
  __shared__ __attribute__((aligned(16))) float a_lds[S_BM][LD];   // [row][depth]
  __shared__ __attribute__((aligned(16))) float bt_lds[S_BN][LD];  // [col][depth]
  const int t = threadIdx.x;
  const int tr = t >> 4, tc = t & 15;  // thread owns output (row0 + tr, col0 + tc)
  // linear workgroup id over (row tile, column tile), column tiles fastest
  const uint32_t tiles_n = (uint32_t)(((uint64_t)n + S_BN - 1) / S_BN);
  const uint64_t row0 = (uint64_t)(blockIdx.x / tiles_n) * S_BM;
  const uint64_t col0 = (uint64_t)(blockIdx.x % tiles_n) * S_BN;
  float acc = 0.0f;
  for (uint64_t k0 = 0; k0 < k; k0 += S_BK) {
    // A tile 16 rows x 256 depths and B tile 256 depths x 16 cols, 16 values each per thread
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int i = t + 256 * e;
      const int ar = i >> 8, ad = i & 255;
      const uint64_t gr = row0 + ar, gd = k0 + ad;
      a_lds[ar][ad] = (gr < m && gd < k) ? a[gr * k + gd] : 0.0f;
      const int bd = i >> 4, bc = i & 15;
      const uint64_t gbd = k0 + bd, gc = col0 + bc;
      bt_lds[bc][bd] = (gbd < k && gc < n) ? b[gbd * n + gc] : 0.0f;
    }
    __syncthreads();
    const int depth = (k - k0) < (uint64_t)S_BK ? (int)(k - k0) : S_BK;
    if (depth == S_BK) {
#pragma unroll 16
      for (int d = 0; d < S_BK; d += 4) {
        const f32x4_t av = *reinterpret_cast<const f32x4_t*>(&a_lds[tr][d]);
        const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(&bt_lds[tc][d]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p = av[e] * bv[e];
          acc = acc + p;
        }
      }
    } else {
      for (int d = 0; d < depth; ++d) {
        const float p = a_lds[tr][d] * bt_lds[tc][d];
        acc = acc + p;
      }
    }
    __syncthreads();
  }
  const uint64_t gr = row0 + tr, gc = col0 + tc;
  if (gr < m && gc < n) c[gr * n + gc] = acc;
}

bool aligned(const void* p, uintptr_t bytes) { return ((uintptr_t)p & (bytes - 1)) == 0; }

int32_t tile16(const uint16_t* a, uint64_t a_len, const uint16_t* b, uint64_t b_len, float* c,
               uint64_t c_len, void* stream) {
  if (a_len != 256 || b_len != 256 || c_len != 256) return FE2O3_ERR_LENGTH;
  if (!a || !b || !c) return FE2O3_ERR_NULL;
  if (!aligned(a, 8) || !aligned(b, 8) || !aligned(c, 4)) return FE2O3_ERR_ALIGNMENT;
  tile16_bf16_kernel<<<1, 64, 0, (hipStream_t)stream>>>(a, b, c);
  return fe2o3_host::after_launch();
}

// kernels behind each entry point (fe2o3_kernel_resources)
const fe2o3_host::KernelRegistrar kRegistered[] = {
    fe2o3_host::KernelRegistrar({"fe2o3_tiled_gemm_lds_slice1_v1", "tile16_bf16_kernel", (const void*)tile16_bf16_kernel, 64, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_moe_expert_gemm_bf16_m16_n16_k16_v1", "tile16_bf16_kernel", (const void*)tile16_bf16_kernel, 64, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_tiled_gemm_v1", "tiled_v1_kernel", (const void*)tiled_v1_kernel, 64, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_tiled_gemm_v1", "zero_fill_kernel", (const void*)zero_fill_kernel, 256, 0}),
    fe2o3_host::KernelRegistrar({"fe2o3_scalar_gemm_v1", "scalar_gemm_kernel", (const void*)scalar_gemm_kernel, 256, 0})};

}  // namespace

extern "C" {

int32_t fe2o3_tiled_gemm_lds_slice1_v1(const uint16_t* a, uint64_t a_len, const uint16_t* b,
                                       uint64_t b_len, float* c, uint64_t c_len, void* stream) {
  FE2O3_ENTRY("fe2o3_tiled_gemm_lds_slice1_v1");
  return tile16(a, a_len, b, b_len, c, c_len, stream);
}

int32_t fe2o3_moe_expert_gemm_bf16_m16_n16_k16_v1(const uint16_t* activations,
                                                  uint64_t activations_len,
                                                  const uint16_t* weights, uint64_t weights_len,
                                                  float* output, uint64_t output_len,
                                                  void* stream) {
  FE2O3_ENTRY("fe2o3_moe_expert_gemm_bf16_m16_n16_k16_v1");
  return tile16(activations, activations_len, weights, weights_len, output, output_len, stream);
}

int32_t fe2o3_tiled_gemm_v1(const uint16_t* a, uint64_t a_len, const uint16_t* b, uint64_t b_len,
                            float* c, uint64_t c_len, uint32_t m, uint32_t n, uint32_t k,
                            void* stream) {
  FE2O3_ENTRY("fe2o3_tiled_gemm_v1");
  // ShapeV1::checked (contract.rs:145-179): an empty output needs no
  // operand buffers; otherwise byte extents of A, B, C in that order
  if (m == 0 || n == 0) {
    if (a_len != 0 || b_len != 0 || c_len != 0) return FE2O3_ERR_LENGTH;
    return FE2O3_OK;  // NoDispatchEmptyOutput
  }
  const uint64_t ea = (uint64_t)m * k, eb = (uint64_t)k * n, ec = (uint64_t)m * n;
  if (ea > UINT64_MAX / 2 || eb > UINT64_MAX / 2 || ec > UINT64_MAX / 4) return FE2O3_ERR_OVERFLOW;
  if (a_len != ea || b_len != eb || c_len != ec) return FE2O3_ERR_LENGTH;
  // plan_v1 (contract.rs:387-427), in its order
  if (m % 16u != 0) return FE2O3_ERR_M_TAIL;
  if (n % 16u != 0) return FE2O3_ERR_N_TAIL;
  if (k != 0 && k % 16u != 0) return FE2O3_ERR_K_TAIL;
  if ((uint64_t)(n / 16u) * 64u > UINT32_MAX) return FE2O3_ERR_OVERFLOW;  // AQL grid x
  if (!c || (k != 0 && (!a || !b))) return FE2O3_ERR_NULL;
  hipStream_t s = (hipStream_t)stream;
  if (k == 0) {  // HostFillPositiveZero
    const uint64_t blocks = (ec + 255u) / 256u;
    zero_fill_kernel<<<(unsigned)(blocks < 4096u ? blocks : 4096u), 256, 0, s>>>(c, ec);
    return fe2o3_host::after_launch();
  }
  const uint64_t tiles = (uint64_t)(m / 16u) * (n / 16u);
  if (tiles > 0x7fffffffu) return FE2O3_ERR_SHAPE;
  tiled_v1_kernel<<<(unsigned)tiles, 64, 0, s>>>(a, b, c, n, k, n / 16u);
  return fe2o3_host::after_launch();
}

}  // extern "C"

namespace {

// ---- general GEMM on the pipelined tile ----------------------------------------------
// The same contract on the 256x256 MFMA tile of gemm_pipe.hpp: A's rows
// (lda apart) are k-contiguous as the tile wants; B is stored [k][n], so its
// 64-k stages arrive as 64 rows of 256 columns and the MFMA fragments are
// read with the transposing LDS read (gemm_pipe::Bf16MmaKN).  Rows past m
// and columns past n repeat the last valid ones and are not stored.  Each
// accumulator receives the same 16x16x32 MFMAs over the same k slices in the
// same order as in gemm_general_kernel, so both give the same bits.  The
// epilogue is that kernel's: alpha * sum and beta * C rounded separately,
// then added.
constexpr int kGpRowBytes = 128, kGpStages = 2;
constexpr int kGpSmem = kGpStages * 2 * gemm_pipe::Geo<kGpRowBytes>::kTileBytes;  // 128 KiB

// C = alpha * acc + beta * C over one tile of TN columns (rows x cols valid),
// accumulators Acc16T<RB, CB> of waves holding RPW rows by CPW columns.  Per
// 16-row block: every C load of the lane first (one wait), then the products
// and stores.  A lane's 4 columns move as one access of 16 bytes at C's own
// 4-byte alignment (gfx950 global accesses of four dwords need no more).  In
// a tile that the last column cuts, the group it cuts (and those past it)
// moves element by element, loads clamped to that column.  NARROW: most groups
// are past it, and left out (100000 x 5 x 64: 16.6 -> 15.4 us; in the cut tiles
// of 1000 x 1500 x 700 the branch costs more than it saves, 14.9 -> 15.0).
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));

template <int TN, int RPW, int CPW, bool NARROW = false, class Acc>
FE2O3_DEVICE void general_epilogue(const Acc& acc, float* c_tile, uint32_t rows, uint32_t cols,
                                   uint32_t ldc, float alpha, float beta) {
#pragma clang fp contract(off)
  constexpr int RB = RPW / 16, CB = CPW / 16;
  const uint32_t row0 = gemm_pipe::acc16_row0<RPW>(), col0 = gemm_pipe::acc16_col0<CPW>();
  auto combined = [&](int i, int j, const f32x4_t& cv) {
    f32x4_t y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float product = alpha * acc.v[i][j][e];
      const float initial = beta * cv[e];
      y[e] = product + initial;
    }
    return y;
  };
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const uint32_t r = row0 + 16u * i;
    if (r >= rows) continue;
    float* out = c_tile + (uint64_t)r * ldc;
    f32x4_t cv[CB];
    if (cols == (uint32_t)TN) {
#pragma unroll
      for (int j = 0; j < CB; ++j)
        cv[j] = *reinterpret_cast<const f32x4_any_t*>(out + col0 + 16u * j);
#pragma unroll
      for (int j = 0; j < CB; ++j)
        *reinterpret_cast<f32x4_any_t*>(out + col0 + 16u * j) = combined(i, j, cv[j]);
    } else {
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const uint32_t col = col0 + 16u * j;
        if (col + 4u <= cols) {
          *reinterpret_cast<f32x4_any_t*>(out + col) =
              combined(i, j, *reinterpret_cast<const f32x4_any_t*>(out + col));
        } else if (!NARROW || col < cols) {
#pragma unroll
          for (int e = 0; e < 4; ++e) cv[j][e] = out[min(col + e, cols - 1u)];
          const f32x4_t y = combined(i, j, cv[j]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < cols) out[col + e] = y[e];
        }
      }
    }
  }
}

// k: A's k extent and the K loop's; kb: B's rows (its k extent), at most k
// and more than k - 64.  KT: k or kb is not a multiple of 64; A's chunks
// past k and B's rows past kb load zeros (gemm_pipe::Rows MASK), so each
// accumulator gets the register tiles' zero-padded 32-k blocks.
template <bool KT = false>
__global__ void __launch_bounds__(256, 1) gemm_general_pipe_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, float* __restrict__ c,
    uint32_t m, uint32_t n, uint32_t k, uint32_t kb, uint32_t lda, uint32_t ldb, uint32_t ldc,
    float alpha, float beta, uint32_t xcds) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const uint32_t tiles_m = (m + 255u) / 256u, tiles_n = (n + 255u) / 256u;
  uint32_t tm, tn;
  gemm_core::xcd_tile_order(blockIdx.x, tiles_m, tiles_n, xcds, &tm, &tn);
  const uint32_t rows = min(256u, m - tm * 256u), cols = min(256u, n - tn * 256u);
  const auto ar =
      gemm_pipe::dense_rows<kGpRowBytes, 256, KT>(a + (uint64_t)tm * 256u * lda, lda, rows, k);
  const auto br = gemm_pipe::kn_rows<KT>(b + (uint64_t)tn * 256u, ldb, cols, kb);
  gemm_pipe::Acc16 acc;
  gemm_pipe::mainloop<gemm_pipe::Bf16MmaKN, kGpRowBytes, kGpStages, KT>(ar, br, k, smem, acc);
  general_epilogue<256, 128, 128>(acc, c + (uint64_t)tm * 256u * ldc + (uint64_t)tn * 256u, rows,
                                  cols, ldc, alpha, beta);
}

// The same GEMM on 128 x 128 tiles (Bf16MmaKN64), for problems whose
// 256 x 256 tiles would not fill the CUs: two stages (64 KiB of LDS, two
// workgroups per CU) when there are more tiles than CUs, else three (96 KiB,
// one workgroup per CU, copies two stages ahead: +24% at 2048^3, -5% at
// 4096 x 2048 x 2048 where two workgroups per CU pay more).  The k order of
// every output's MFMAs is that of the 256 x 256 tile, so C is bit-identical
// to it.
template <int STAGES>
constexpr int kGp64Smem =
    STAGES * (128 * kGpRowBytes + gemm_pipe::Bf16MmaKN64::kBTileBytes);
// TAIL: the last, partial round of a 256 x 256 grid (tiles first_big .. end
// of gemm_core::xcd_tile_order's list), each as four 128 x 128 quarters
// (gemm_core::tail_quarter).
// k, kb, KT: as for gemm_general_pipe_kernel.
template <int STAGES, bool TAIL = false, bool KT = false>
__global__ void __launch_bounds__(256, STAGES == 2 ? 2 : 1) gemm_general_pipe128_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, float* __restrict__ c,
    uint32_t m, uint32_t n, uint32_t k, uint32_t kb, uint32_t lda, uint32_t ldb, uint32_t ldc,
    float alpha, float beta, uint32_t xcds, uint32_t first_big = 0) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  uint32_t tm, tn;
  if constexpr (TAIL) {
    if (!gemm_core::tail_quarter(blockIdx.x, first_big, m, n, xcds, &tm, &tn)) return;
  } else {
    gemm_core::xcd_tile_order(blockIdx.x, (m + 127u) / 128u, (n + 127u) / 128u, xcds, &tm, &tn);
  }
  const uint32_t rows = min(128u, m - tm * 128u), cols = min(128u, n - tn * 128u);
  const auto ar =
      gemm_pipe::dense_rows<kGpRowBytes, 128, KT>(a + (uint64_t)tm * 128u * lda, lda, rows, k);
  const auto br = gemm_pipe::kn_rows128<KT>(b + (uint64_t)tn * 128u, ldb, cols, kb);
  gemm_pipe::Bf16MmaKN64::Acc acc;
  gemm_pipe::mainloop<gemm_pipe::Bf16MmaKN64, kGpRowBytes, STAGES, KT>(ar, br, k, smem, acc);
  general_epilogue<128, 64, 64>(acc, c + (uint64_t)tm * 128u * ldc + (uint64_t)tn * 128u, rows,
                                cols, ldc, alpha, beta);
}

// ---- 64 x 64 tiles through registers: any alignment, any K ------------------------------
// For outputs too small for the pipelined tiles to fill the device, and for
// operands they would need repacked: 16-byte loads at the operand's own
// alignment into registers, kGsDepth steps of 64 k ahead, then through LDS
// (two buffers, one barrier per step).  Four waves, 2 x 2, own 32 x 32
// outputs each.  B's [k][n] rows are read back with the transposing LDS read,
// as in gemm_pipe::Bf16MmaKN.  Every accumulator gets the MFMAs of the
// pipelined tiles in the same k order over the same zero-padded 32-k blocks,
// so C is bit-identical to theirs.
//
// Bound by LDS, which moves three bytes per byte loaded at this tile (two
// steps of 64 k take 0.6 us alone on a CU); against the masked scalar loads
// it replaces 2000 x 100 x 2000 takes 18.6 us for 177.7, and against
// repacking for the pipelined tile 1000 x 1500 x 700 takes 15.1 for 30.1.
constexpr int kGsThreads = 256, kGsDepth = 4;
constexpr uint32_t kGsBuf = 64 * 128;  // bytes of one operand's step: 64 rows of 128

// 16-byte piece position of B's k row in LDS: the rows that one half wave of
// a transposing read touches (8g + q, g < 2, q < 4) fall on distinct banks
FE2O3_DEVICE uint32_t gs_swz_b(uint32_t krow) {
  return 2u * (((krow >> 1) & 1u) | (((krow >> 3) & 1u) << 1));
}

// How a tile reads B's columns: all 64 valid; cut by the last column; or a
// row of B shorter than a 16-byte piece.
enum class Cols { whole, cut, narrow };

template <Cols MODE>
FE2O3_DEVICE void general_tile(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
                               float* __restrict__ c, uint32_t n, uint32_t k, uint32_t lda,
                               uint32_t ldb, uint32_t ldc, float alpha, float beta, uint32_t tm,
                               uint32_t tn, uint32_t rows, uint32_t cols, uint8_t* smem) {
  using G = gemm_pipe::Geo<128>;
  using gemm_direct::load16;
  using gemm_direct::load_end;
  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = gemm_pipe::wave_id();
  // this thread's pieces of a step: place pc of rows pr and pr + 32 of A's
  // 64 (rows past m repeat the last) and of B's 64 k rows.  A piece that the
  // last column cuts is read 8 columns before it and shifted down; one past
  // it reads the same, and its columns are not stored.
  const uint32_t pr = t >> 3, pc = t & 7u;
  const uint32_t b_first = tn * 64u + 8u * pc;
  const uint32_t b_read = MODE == Cols::whole ? b_first
                          : MODE == Cols::cut ? min(b_first, n - 8u) : 0u;
  const uint32_t b_shift = 16u * (b_first - b_read);  // bits
  const uint8_t* row_a[2];
  const uint8_t* ap[2];
  const uint8_t* bp[2];
  uint32_t aw[2], bw[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t r = pr + 32u * h;
    row_a[h] = reinterpret_cast<const uint8_t*>(
        a + ((uint64_t)tm * 64u + min(r, rows - 1u)) * lda);
    ap[h] = row_a[h] + 16u * pc;
    bp[h] = reinterpret_cast<const uint8_t*>(b + (uint64_t)r * ldb + b_read);
    aw[h] = r * 128u + ((pc ^ G::swz(r)) << 4);
    bw[h] = 2u * kGsBuf + r * 128u + ((pc ^ gs_swz_b(r)) << 4);
  }
  const uint64_t b_step = (uint64_t)ldb * 128u;
  const uint32_t steps = k / 64u, k_rest = k % 64u;
  // the partial last step, fetched first, without a branch, and kept: A's
  // pieces that K cuts (or that lie past it) are read 16 bytes before the
  // row's end, B's rows past K repeat the last; end_a and end_b make of them
  // what the step needs, zeros past K
  u32x4_t last_a[2], last_b[2];
  const bool short_row = k < 8u || MODE == Cols::narrow;  // no whole piece in a row
  const uint64_t a_at = (uint64_t)steps * 128u + 16u * pc;
  const uint64_t a_last = min(a_at, (uint64_t)k * 2u - 16u);
  if (k_rest != 0u && !short_row) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t r = pr + 32u * h, rb = min(r, k_rest - 1u);
      last_a[h] = load16(row_a[h] + a_last);
      last_b[h] = load16(bp[h] + steps * b_step - (uint64_t)(r - rb) * ldb * 2u);
    }
  }
  auto end_a = [&](int h) {
    if (short_row) return load_end<2, uint64_t>(row_a[h], a_at, (uint64_t)k * 2u);
    const uint64_t past = a_at - a_last;
    return past < 16u ? gemm_direct::shift_down(last_a[h], 8u * (uint32_t)past) : u32x4_t{};
  };
  auto end_b = [&](int h) {
    const uint32_t r = pr + 32u * h;
    if (r >= k_rest) return u32x4_t{};
    if (short_row)
      return load_end<2, uint64_t>(
          reinterpret_cast<const uint8_t*>(b + ((uint64_t)steps * 64u + r) * ldb),
          (uint64_t)b_first * 2u, (uint64_t)n * 2u);
    return MODE == Cols::cut ? gemm_direct::shift_down(last_b[h], b_shift) : last_b[h];
  };

  gemm_pipe::Acc16T<2, 2> acc;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc.v[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  constexpr int D = MODE == Cols::narrow ? 2 : kGsDepth;
  u32x4_t ra[D][2], rb[D][2];
  // the next step to load; the last one is loaded again past it (unless the
  // loads of B's short rows cost more than the branch)
  uint32_t loaded = 0;
  auto load = [&](int s) {
    __builtin_amdgcn_sched_barrier(0);
    if (MODE == Cols::narrow && loaded >= steps) return;
    const bool more = loaded + 1u < steps;
    ++loaded;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[s][h] = load16(ap[h]);
      if constexpr (MODE == Cols::narrow)
        rb[s][h] = load_end<2, uint64_t>(bp[h], (uint64_t)b_first * 2u, (uint64_t)n * 2u);
      else
        rb[s][h] = load16(bp[h]);
      ap[h] += more ? 128u : 0u;
      bp[h] += more ? b_step : 0u;
    }
  };
  auto put = [&](uint32_t buf, int h, u32x4_t pa, u32x4_t pb) {
    *reinterpret_cast<u32x4_t*>(smem + buf * kGsBuf + aw[h]) = pa;
    *reinterpret_cast<u32x4_t*>(smem + buf * kGsBuf + bw[h]) = pb;
  };
  auto put_set = [&](uint32_t buf, int s) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      put(buf, h, ra[s][h],
          MODE == Cols::cut ? gemm_direct::shift_down(rb[s][h], b_shift) : rb[s][h]);
    __builtin_amdgcn_sched_barrier(0);
  };
  // fragments: wave rows wm * 32, columns wn * 32
  const uint32_t wm = wave >> 1, wn = wave & 1u, lr = lane & 15u, g = lane >> 4;
  auto compute = [&](uint32_t buf) {
    const uint8_t* la = smem + buf * kGsBuf;
    const uint8_t* lb = la + 2u * kGsBuf;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8_t fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t r = wm * 32u + 16u * i + lr;
        fa[i] =
            *reinterpret_cast<const bf16x8_t*>(la + r * 128u + (((4u * ks + g) ^ G::swz(r)) << 4));
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t kr = 32u * ks + 8u * g + (lr >> 2);
        const uint32_t piece = wn * 4u + 2u * j + ((lr & 3u) >> 1), off = (lr & 1u) * 8u;
        const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (lds_bf16x4_t*)(lb + kr * 128u + ((piece ^ gs_swz_b(kr)) << 4) + off));
        const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (lds_bf16x4_t*)(lb + (kr + 4u) * 128u + ((piece ^ gs_swz_b(kr + 4u)) << 4) + off));
        fb[j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc.v[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc.v[i][j], 0, 0, 0);
    }
  };
  // Step t is in buffer t % 2 when its turn comes.  It writes step t + 1 into
  // the other buffer, which every wave left at the barrier before, and loads
  // step t + D into the set that step t came from.
  if (steps != 0u) {
#pragma unroll
    for (int s = 0; s < D; ++s) load(s);
    put_set(0, 0);
    lds_barrier();
    for (uint32_t t0 = 0; t0 < steps; t0 += D) {
#pragma unroll
      for (int s = 0; s < D; ++s) {
        if (t0 + s >= steps) break;
        if (MODE != Cols::narrow || t0 + s + 1u < steps) put_set((s + 1) & 1, (s + 1) % D);
        load(s);
        compute(s & 1);
        lds_barrier();
      }
    }
  }
  if (k_rest != 0u) {
#pragma unroll
    for (int h = 0; h < 2; ++h) put(steps & 1u, h, end_a(h), end_b(h));
    lds_barrier();
    compute(steps & 1u);
  }
  general_epilogue<64, 32, 32, MODE == Cols::narrow>(
      acc, c + (uint64_t)tm * 64u * ldc + (uint64_t)tn * 64u, rows, cols, ldc, alpha, beta);
}

__global__ void __launch_bounds__(kGsThreads, 3) gemm_general_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, float* __restrict__ c,
    uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb, uint32_t ldc, float alpha,
    float beta, uint32_t xcds) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[4 * kGsBuf];  // A0 A1 B0 B1
  uint32_t tm, tn;
  const uint32_t tiles_m = (m - 1u) / 64u + 1u, tiles_n = (n - 1u) / 64u + 1u;
  if (gemm_direct::list_id() >= tiles_m * tiles_n) return;
  gemm_core::xcd_tile_order(gemm_direct::list_id(), tiles_m, tiles_n, xcds, &tm, &tn);
  const uint32_t rows = min(64u, m - tm * 64u), cols = min(64u, n - tn * 64u);
  if (n < 8u)
    general_tile<Cols::narrow>(a, b, c, n, k, lda, ldb, ldc, alpha, beta, tm, tn, rows, cols, smem);
  else if (cols < 64u)
    general_tile<Cols::cut>(a, b, c, n, k, lda, ldb, ldc, alpha, beta, tm, tn, rows, cols, smem);
  else
    general_tile<Cols::whole>(a, b, c, n, k, lda, ldb, ldc, alpha, beta, tm, tn, rows, cols, smem);
}

// ---- operands the pipelined tile cannot read directly ---------------------------
// Rows that are not 16-byte aligned (A or B two bytes past a boundary, a
// stride that is not a multiple of 8) or an A whose K is not a multiple of
// 8 are first copied into aligned scratch rows: A as [m][kp] with kp = K
// rounded up to 64 and zeros from K on, B as [K][np] with np = N rounded up
// to 8.  The pipelined tile then reads the copies; its products are the same
// MFMAs over the same zero-padded 32-k blocks.  8 elements (16 bytes) per
// thread per step, written as one 16-byte store.  A whole 8-element piece
// of a source row is read as one 16-byte load at its own (2-byte) alignment
// (gfx950 global loads take any alignment); the piece that holds a row's
// end is read element by element.
__global__ void __launch_bounds__(256) repack_rows_kernel(const uint16_t* __restrict__ src,
                                                          uint32_t rows, uint32_t cols,
                                                          uint32_t ld, uint16_t* __restrict__ dst,
                                                          uint32_t dst_cols) {
  const uint64_t per_row = dst_cols / 8u, groups = (uint64_t)rows * per_row;
  for (uint64_t g = (uint64_t)blockIdx.x * 256u + threadIdx.x; g < groups;
       g += (uint64_t)gridDim.x * 256u) {
    const uint64_t r = g / per_row;
    const uint32_t c0 = (uint32_t)(g % per_row) * 8u;
    const uint16_t* row = src + r * ld;
    u32x4_t p;
    if (c0 + 8u <= cols) {
      __builtin_memcpy(&p, row + c0, 16);
    } else {
      uint16_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = c0 + e < cols ? row[c0 + e] : (uint16_t)0;
#pragma unroll
      for (int q = 0; q < 4; ++q) p[q] = (uint32_t)v[2 * q] | ((uint32_t)v[2 * q + 1] << 16);
    }
    *reinterpret_cast<u32x4_t*>(dst + r * dst_cols + c0) = p;
  }
}

#define FE2O3_GENERAL_PIPE_KERNELS(entry)                                                        \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe_kernel", (const void*)gemm_general_pipe_kernel<false>, 256, kGpSmem}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe_kernel<k tail>", (const void*)gemm_general_pipe_kernel<true>, 256, kGpSmem}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<2>", (const void*)gemm_general_pipe128_kernel<2>, 256, kGp64Smem<2>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<3>", (const void*)gemm_general_pipe128_kernel<3>, 256, kGp64Smem<3>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<2, tail>", (const void*)gemm_general_pipe128_kernel<2, true>, 256, kGp64Smem<2>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<3, tail>", (const void*)gemm_general_pipe128_kernel<3, true>, 256, kGp64Smem<3>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<2, k tail>", (const void*)gemm_general_pipe128_kernel<2, false, true>, 256, kGp64Smem<2>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<3, k tail>", (const void*)gemm_general_pipe128_kernel<3, false, true>, 256, kGp64Smem<3>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<2, tail, k tail>", (const void*)gemm_general_pipe128_kernel<2, true, true>, 256, kGp64Smem<2>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_pipe128_kernel<3, tail, k tail>", (const void*)gemm_general_pipe128_kernel<3, true, true>, 256, kGp64Smem<3>}), \
  fe2o3_host::KernelRegistrar({entry, "gemm_general_kernel", (const void*)gemm_general_kernel, kGsThreads, 0}), \
  fe2o3_host::KernelRegistrar({entry, "repack_rows_kernel", (const void*)repack_rows_kernel, 256, 0})

const fe2o3_host::KernelRegistrar kRegisteredPipe[] = {
    FE2O3_GENERAL_PIPE_KERNELS("fe2o3_tiled_gemm_general_v1"),
    FE2O3_GENERAL_PIPE_KERNELS("fe2o3_tiled_gemm_general_vector_a_v1"),
    // fe2o3_gemm_bf16_nt repacks misaligned operand rows with it (gemm_bf16.hip)
    fe2o3_host::KernelRegistrar({"fe2o3_gemm_bf16_nt", "repack_rows_kernel", (const void*)repack_rows_kernel, 256, 0})};

// Raises every pipelined kernel's dynamic-LDS limit once per process.
int32_t set_general_lds() {
  static const int32_t rc = [] {
    int32_t r = fe2o3_host::set_dynamic_lds(
        {(const void*)gemm_general_pipe_kernel<false>, (const void*)gemm_general_pipe_kernel<true>},
        kGpSmem);
    if (r == FE2O3_OK)
      r = fe2o3_host::set_dynamic_lds({(const void*)gemm_general_pipe128_kernel<2>,
                                       (const void*)gemm_general_pipe128_kernel<2, true>,
                                       (const void*)gemm_general_pipe128_kernel<2, false, true>,
                                       (const void*)gemm_general_pipe128_kernel<2, true, true>},
                                      kGp64Smem<2>);
    if (r == FE2O3_OK)
      r = fe2o3_host::set_dynamic_lds({(const void*)gemm_general_pipe128_kernel<3>,
                                       (const void*)gemm_general_pipe128_kernel<3, true>,
                                       (const void*)gemm_general_pipe128_kernel<3, false, true>,
                                       (const void*)gemm_general_pipe128_kernel<3, true, true>},
                                      kGp64Smem<3>);
    return r;
  }();
  return rc;
}

// The launches of `plan` over A (lda, k) and B (ldb, kb rows); KT: k or kb
// is not a multiple of 64.
template <bool KT>
int32_t launch_general_pipe(const uint16_t* a, const uint16_t* b, float* c, uint32_t m,
                            uint32_t n, uint32_t k, uint32_t kb, uint32_t lda, uint32_t ldb,
                            uint32_t ldc, float alpha, float beta, const tile_plan::Plan& plan,
                            uint32_t xcds, hipStream_t s) {
  if (plan.small) {  // 256 x 256 tiles would leave most CUs idle
    if (plan.stages == 2)
      gemm_general_pipe128_kernel<2, false, KT><<<(unsigned)plan.grid, 256, kGp64Smem<2>, s>>>(
          a, b, c, m, n, k, kb, lda, ldb, ldc, alpha, beta, xcds);
    else
      gemm_general_pipe128_kernel<3, false, KT><<<(unsigned)plan.grid, 256, kGp64Smem<3>, s>>>(
          a, b, c, m, n, k, kb, lda, ldb, ldc, alpha, beta, xcds);
    return fe2o3_host::after_launch();
  }
  gemm_general_pipe_kernel<KT><<<(unsigned)plan.grid, 256, kGpSmem, s>>>(
      a, b, c, m, n, k, kb, lda, ldb, ldc, alpha, beta, xcds);
  const int32_t big_rc = fe2o3_host::after_launch();
  if (big_rc != FE2O3_OK || !plan.tail) return big_rc;
  // the last round of at most half the CUs' tiles as 128 x 128 quarters
  if (plan.tail_stages == 2)  // more quarters than CUs: two per CU
    gemm_general_pipe128_kernel<2, true, KT><<<(unsigned)plan.tail_grid, 256, kGp64Smem<2>, s>>>(
        a, b, c, m, n, k, kb, lda, ldb, ldc, alpha, beta, xcds, plan.first_big);
  else
    gemm_general_pipe128_kernel<3, true, KT><<<(unsigned)plan.tail_grid, 256, kGp64Smem<3>, s>>>(
        a, b, c, m, n, k, kb, lda, ldb, ldc, alpha, beta, xcds, plan.first_big);
  return fe2o3_host::after_launch();
}

// Whether the pipelined tile reads an operand in place: 16-byte aligned
// rows, and its 256-row (A) or K-row (B) panel within a buffer resource's
// 32-bit range.  A also needs K a multiple of 8 (chunks past K are masked
// whole).
bool a_direct(const uint16_t* a, uint32_t k, uint32_t lda) {
  return k % 8 == 0 && lda % 8 == 0 && ((uintptr_t)a & 15u) == 0 &&
         (255ull * lda + k) * 2 < (1ull << 31);
}
bool b_direct(const uint16_t* b, uint32_t k, uint32_t ldb) {
  return ldb % 8 == 0 && ((uintptr_t)b & 15u) == 0 &&
         ((uint64_t)(k - 1) * ldb + 256) * 2 < (1ull << 31);
}

// Operands the tile cannot read in place are repacked (repack_rows_kernel)
// when M and N are at least one 128 x 128 tile; smaller problems, and those
// below register_tiles' line, stay on the register tiles.
constexpr uint32_t kRepackMin = 128;

// Whether the 64 x 64 register tiles take a GEMM that the pipelined tiles
// could run, in place (`in_place`) or on repacked operands.  Both sides in us
// (pipelined, register); `rounds` is what the busiest CU walks, in steps.
//   in place       1024 x 1024 x 1024  11.2, 10.2    1024 x 512 x 2048   15.7, 15.9
//                  1200 x 1200 x 256    9.3,  7.7    1024 x 2048 x 512    9.4,  9.8
//                  512^3                7.6,  5.4    1024 x 1024 x 4096  26.3, 28.9
//   repacked       1000 x 1500 x 700   30.3, 15.1    1500^3              31.9, 32.9
//                  2048 x 2048 x 512   27.6, 21.7    2000 x 2000 x 1000  30.1, 32.2
//                  1024 x 1024 x 4096  40.9, 35.3    512 x 512 x 8192    62.2, 63.9
bool register_tiles(uint32_t m, uint32_t n, uint32_t k, bool in_place, uint32_t cus) {
  const uint64_t tiles = (((uint64_t)m + 63u) / 64u) * (((uint64_t)n + 63u) / 64u);
  const uint64_t rounds = (tiles + cus - 1u) / cus * (((uint64_t)k + 63u) / 64u);
  if (in_place) return 2u * tiles <= 3ull * cus && rounds <= 32u;
  return rounds <= 48u || (tiles <= cus && rounds <= 96u);
}

int32_t general_gemm(const uint16_t* a, uint64_t a_len, const uint16_t* b, uint64_t b_len,
                     float* c, uint64_t c_len, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                     uint32_t ldb, uint32_t ldc, float alpha, float beta, void* stream) {
  // examples/tiled_gemm_general_v1/src/kernel.rs:80-89
  if ((m != 0 && k != 0 && lda < k) || (k != 0 && n != 0 && ldb < n) ||
      (m != 0 && n != 0 && ldc < n))
    return FE2O3_ERR_STRIDE;
  uint64_t ea, eb, ec;
  fe2o3_host::extent_ok(m, k, lda, &ea);
  fe2o3_host::extent_ok(k, n, ldb, &eb);
  fe2o3_host::extent_ok(m, n, ldc, &ec);
  if (a_len < ea || b_len < eb || c_len < ec) return FE2O3_ERR_LENGTH;
  if (m == 0 || n == 0) return FE2O3_OK;  // empty output: no dispatch
  if ((ea && !a) || (eb && !b) || !c) return FE2O3_ERR_NULL;
  const bool ad = k != 0 && a_direct(a, k, lda), bd = k != 0 && b_direct(b, k, ldb);
  const bool repack = k != 0 && (!ad || !bd) && m >= kRepackMin && n >= kRepackMin;
  tile_plan::Topology topo;
  const int32_t topo_rc = fe2o3_host::device_topology(&topo);
  if (topo_rc != FE2O3_OK) return topo_rc;
  if (k != 0 && ((ad && bd) || repack) && !register_tiles(m, n, k, ad && bd, topo.cus)) {
    // every kernel's LDS limit is raised before anything is launched, so a
    // failure leaves C untouched
    const int32_t lds_rc = set_general_lds();
    if (lds_rc != FE2O3_OK) return lds_rc;
    const tile_plan::Plan plan = tile_plan::plan(m, n, topo);
    if (plan.grid > 0x7fffffffu || plan.tail_grid > 0x7fffffffu) return FE2O3_ERR_SHAPE;
    hipStream_t s = (hipStream_t)stream;
    if (!repack) {
      if (k % 64 != 0)
        return launch_general_pipe<true>(a, b, c, m, n, k, k, lda, ldb, ldc, alpha, beta, plan,
                                         topo.xcds, s);
      return launch_general_pipe<false>(a, b, c, m, n, k, k, lda, ldb, ldc, alpha, beta, plan,
                                        topo.xcds, s);
    }
    // repack what cannot be read in place into one stream-ordered scratch
    // block: A as [m][kp] (zeros from K on), B as [K][np]
    const uint32_t kp = (k + 63u) & ~63u, np = (n + 7u) & ~7u;
    const uint64_t a_elems = ad ? 0 : (uint64_t)m * kp, b_elems = bd ? 0 : (uint64_t)k * np;
    if ((!ad && 256ull * kp * 2 >= (1ull << 31)) ||
        (!bd && ((uint64_t)(k - 1) * np + 256) * 2 >= (1ull << 31)))
      return FE2O3_ERR_SHAPE;
    void* scratch = nullptr;
    int32_t rc = fe2o3_host::scratch_alloc(&scratch, (a_elems + b_elems) * 2, s);
    if (rc != FE2O3_OK) {
      // no stream-ordered scratch on this device or process: the register
      // kernel reads the operands as they are
      (void)hipGetLastError();
      goto in_registers;
    }
    uint16_t* ap = static_cast<uint16_t*>(scratch);
    uint16_t* bp = ap + a_elems;
    auto grid = [](uint64_t groups) {
      const uint64_t g = (groups + 255) / 256;
      return (unsigned)(g < 16384 ? g : 16384);
    };
    if (!ad) repack_rows_kernel<<<grid((uint64_t)m * (kp / 8)), 256, 0, s>>>(a, m, k, lda, ap, kp);
    if (!bd) repack_rows_kernel<<<grid((uint64_t)k * (np / 8)), 256, 0, s>>>(b, k, n, ldb, bp, np);
    rc = fe2o3_host::after_launch();
    if (rc == FE2O3_OK) {
      const uint16_t* ra = ad ? a : ap;
      const uint16_t* rb = bd ? b : bp;
      const uint32_t rlda = ad ? lda : kp, rldb = bd ? ldb : np;
      // a repacked A holds zeros up to kp: the K loop runs whole stages over
      // it; an A read in place masks its chunks past K.  B's rows past K
      // are masked either way.
      const uint32_t kloop = ad ? k : kp;
      rc = k % 64 != 0
               ? launch_general_pipe<true>(ra, rb, c, m, n, kloop, k, rlda, rldb, ldc, alpha,
                                           beta, plan, topo.xcds, s)
               : launch_general_pipe<false>(ra, rb, c, m, n, kloop, k, rlda, rldb, ldc, alpha,
                                            beta, plan, topo.xcds, s);
    }
    const int32_t free_rc = fe2o3_host::scratch_free(scratch, s);
    return rc != FE2O3_OK ? rc : free_rc;
  }
in_registers:
  const uint64_t tiles = (((uint64_t)m + 63u) / 64u) * (((uint64_t)n + 63u) / 64u);
  if (((uint64_t)m + 63u) / 64u > 65535u || tiles > 0x7fffffffu) return FE2O3_ERR_SHAPE;
  gemm_general_kernel<<<gemm_direct::list_grid(tiles), kGsThreads, 0, (hipStream_t)stream>>>(
      a, b, c, m, n, k, lda, ldb, ldc, alpha, beta, topo.xcds);
  return fe2o3_host::after_launch();
}

}  // namespace

namespace fe2o3_host {

int32_t repack_bf16_rows(const uint16_t* src, uint32_t rows, uint32_t cols, uint32_t ld,
                         uint16_t* dst, uint32_t dst_cols, hipStream_t s) {
  const uint64_t g = ((uint64_t)rows * (dst_cols / 8u) + 255u) / 256u;
  repack_rows_kernel<<<(unsigned)(g < 16384u ? g : 16384u), 256, 0, s>>>(src, rows, cols, ld, dst,
                                                                         dst_cols);
  return after_launch();
}

}  // namespace fe2o3_host

extern "C" {

int32_t fe2o3_tiled_gemm_general_v1(const uint16_t* a, uint64_t a_len, const uint16_t* b,
                                    uint64_t b_len, float* c, uint64_t c_len, uint32_t m,
                                    uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb,
                                    uint32_t ldc, float alpha, float beta, void* stream) {
  FE2O3_ENTRY("fe2o3_tiled_gemm_general_v1");
  return general_gemm(a, a_len, b, b_len, c, c_len, m, n, k, lda, ldb, ldc, alpha, beta,
                             stream);
}

int32_t fe2o3_tiled_gemm_general_vector_a_v1(const uint16_t* a, uint64_t a_len,
                                             const uint16_t* b, uint64_t b_len, float* c,
                                             uint64_t c_len, uint32_t m, uint32_t n, uint32_t k,
                                             uint32_t lda, uint32_t ldb, uint32_t ldc,
                                             float alpha, float beta, void* stream) {
  FE2O3_ENTRY("fe2o3_tiled_gemm_general_vector_a_v1");
  return general_gemm(a, a_len, b, b_len, c, c_len, m, n, k, lda, ldb, ldc, alpha, beta,
                            stream);
}

int32_t fe2o3_scalar_gemm_v1(const float* a, uint64_t a_len, const float* b, uint64_t b_len,
                             float* c, uint64_t c_len, uint32_t m, uint32_t n, uint32_t k,
                             void* stream) {
  FE2O3_ENTRY("fe2o3_scalar_gemm_v1");
  const uint64_t ea = (uint64_t)m * k, eb = (uint64_t)k * n, ec = (uint64_t)m * n;
  if (a_len < ea || b_len < eb || c_len < ec) return FE2O3_ERR_LENGTH;
  if (ec == 0) return FE2O3_OK;
  if ((ea && !a) || (eb && !b) || !c) return FE2O3_ERR_NULL;
  const uint64_t tiles = (((uint64_t)m + S_BM - 1) / S_BM) * (((uint64_t)n + S_BN - 1) / S_BN);
  if (tiles > 0x7fffffffu) return FE2O3_ERR_SHAPE;
  scalar_gemm_kernel<<<(unsigned)tiles, 256, 0, (hipStream_t)stream>>>(a, b, c, m, n, k);
  return fe2o3_host::after_launch();
}

}  // extern "C"
