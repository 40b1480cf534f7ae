// Row-wise scaled FP8 (e4m3fn) GEMM for MI355X (gfx950, CDNA4): kernels and C ABI.
//
//   C[M,N] bf16 = bf16( (sum_k A[m,k] * B[n,k]) * a_scale[m] * b_scale[n] + bias[n] )
//
// A is [M,K] and B is [N,K], both K-contiguous, one byte per element. The contraction runs
// on the gfx950 f8f6f4 MFMA instructions (full FP8 rate) with fp32 accumulation; scales and
// bias are applied in fp32 to the accumulator and the result is rounded to bf16 once.
//
// Kernels:
//   gemm_tiled_kernel        persistent workgroups walk (split, tile) work items; BM x BN x 128
//                            steps staged global->LDS with direct-to-LDS loads into swizzled
//                            rings (2 or 3 stages of A, one more of B), 32x32x64 MFMA, epilogue
//                            turned through LDS into 16-byte row stores. Tiles of 256x256,
//                            128x128 (two ring depths), 256x128, 64x256, 128x256 and 192x256; grouped
//                            and block-scaled forms.
//   gemm_block_kernel        block-scaled form for shapes that fill the chip with 256x256 tiles: two groups of
//                            four waves take turns between memory and matrix work.
//   splitk_finalize_kernel   adds the fp32 partial sums of a split-K launch, applies scales/bias
//                            (splitk_finalize_rows_kernel: four rows a thread, for large results).
//   gemm_skinny_kernel       M <= 64: every workgroup owns 16 rows of B and all of K, its waves
//                            split K between them and reduce through LDS; B is streamed once.
//   gemm_skinny_persistent_kernel  M <= 16 (M <= 32 at K = 4096): one 16-wave workgroup per CU keeps
//                            its share of A in registers and walks 16-row tiles of B.
//   gemm_skinny_pair_kernel  M <= 16, N <= 8192, K <= 8192: one or two 16-row tiles of B per CU, A parked
//                            in LDS, a tile's rows requested in one burst.
//   gemm_narrow_kernel       M <= 64 (M <= 256 in row blocks), K in 512-byte steps, at most one tile of
//                            up to 64 columns per CU: a workgroup owns all of K (no split, no second
//                            launch); separate waves fetch A and B.
//   gemm_any_kernel          any K, leading dimension and alignment (more than 64 rows; up to 64 the skinny
//                            kernel has a form for them): unaligned loads, binary16 MFMA on the widened codes.
//   quantize_rows_*_kernel   row-wise e4m3fn quantiser (amax, scale, convert), a row per workgroup or per wave.
//   quantize_blocks_kernel   128 x 128 block-wise e4m3fn quantiser, one block per workgroup.
//   fused_rowwise_quant_kernel  RMSNorm or SiLU-mul of bf16 rows followed by the same quantiser, one pass.
//
// Operand roles inside the MFMA are swapped on purpose (rows of B feed the instruction's
// "A" port, rows of A its "B" port) so each lane ends up holding 4 consecutive columns n of
// one output row m (8 bytes of 16-bit results for the epilogue's LDS turn and for the skinny
// kernels' direct stores).

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "../../include/mi355x_fp8_rowwise.h"

// ------------------------------------------------------------------------------------
// Building in parts. This file compiles on its own (`hipcc -shared` on it gives the library), and
// it compiles faster as several translation units in parallel, which is what the package's build
// script does: with -DMI355X_TILED_PART=<k> a unit holds only the instantiations of tile
// configuration k of the plain tiled kernel (where nearly all of the compile time goes), with
// -DMI355X_SPLIT_MAIN it holds everything else and calls those through the functions below.
// What the units share lives in this namespace (hidden from the library's users): the parameter
// block, the error text, the table of kernels that need a raised LDS limit, the device set-up.
// ------------------------------------------------------------------------------------
#if defined(MI355X_TILED_PART) && defined(MI355X_SPLIT_MAIN)
#error "a translation unit is either a part or the main unit"
#endif
namespace mi355x_shared __attribute__((visibility("hidden"))) {
struct GemmParams {
  const uint8_t* a;
  const uint8_t* b;
  const float* a_scale;
  const float* b_scale;
  const uint16_t* bias;  // bf16 bits or nullptr
  uint16_t* c;           // bf16 bits
  int M, N, K;
  long lda, ldb, ldc;
  int tiles_m, tiles_n;
  // grouped form: rows of C past the last group's are set to zero (else they are left alone). Here, because the others lie so
  // that the kernels' argument fetch is a few wide loads: between `groups` and `out_f16` this field took it apart, with a
  // wait between the pieces (1000x3000x4112, one round of workgroups: 22.67 -> 22.87 us)
  int clear_rest;
  // split-K: every tile is cut into `splits` work items of `steps_per_split` 128-byte K steps
  // (the last one takes what is left); with splits > 1 the items write fp32 partial sums to
  // partial[split][M][N] and a second kernel adds them up and applies the epilogue
  int splits, steps_per_split;
  float* partial;
  // grouped form: `groups` consecutive row blocks of A and C, block g of m_sizes[g] rows
  // (device memory) multiplied with rows [g*N, (g+1)*N) of B and scaled by b_scale[g*N + n]
  const int32_t* m_sizes;
  int groups;
  int out_f16;  // C holds IEEE binary16 instead of bf16 (same size, same stores)
  // tiled kernel, plain form: reciprocals of the two run-time divisors of the tile walk (the number
  // of tiles, and the tiles of a full group of tile rows), prepared on the host: see fast_div()
  uint32_t div_tiles_mul, div_tiles_shift, div_group_mul, div_group_shift;
  // tiled kernel: where every workgroup leaves its start and end readings of the shader clock and of
  // the constant 100 MHz clock (4 values per workgroup), or nullptr
  unsigned long long* stamps;
  int store;  // tiles: how their pieces of C are stored (kStoreStream ...)
};

extern thread_local char err[512];
struct LdsKernel {
  const void* kernel;
  size_t lds_bytes;
};
constexpr int kMaxLdsKernels = 512;
extern LdsKernel lds_kernels[kMaxLdsKernels];
extern int num_lds_kernels;
extern bool lds_table_overflow;
int ready_device(int* dev_out);
// tile configuration k of the plain tiled kernel: picks the instantiation for the plan in `p` and launches it
constexpr int kNumTiledParts = 7;
int tiled_config_0(const GemmParams& p, hipStream_t stream);
int tiled_config_1(const GemmParams& p, hipStream_t stream);
int tiled_config_2(const GemmParams& p, hipStream_t stream);
int tiled_config_3(const GemmParams& p, hipStream_t stream);
int tiled_config_4(const GemmParams& p, hipStream_t stream);
int tiled_config_5(const GemmParams& p, hipStream_t stream);
int tiled_config_6(const GemmParams& p, hipStream_t stream);
}  // namespace mi355x_shared

namespace {

typedef int   v4i  __attribute__((ext_vector_type(4)));
typedef int   v8i  __attribute__((ext_vector_type(8)));
typedef float v4f  __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned short us4 __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
// the same in memory at any address (one instruction each on this chip)
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
typedef int v4i_by4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t v2u_any __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef float v4f_by4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kNumXcd = 8;       // accelerator complex dies; workgroup ids round-robin over them
constexpr int kNumCu = 256;
constexpr int kChunk = 16;       // bytes moved per lane per load

using mi355x_shared::GemmParams;

// Where a tile sits: rows [m0, m_end) of A and C it may touch, first column, group.
struct TileLoc {
  int m0, m_end, n0, group;
  int tiles_m;  // (grouped form: tile rows of the group)
};

// Cursor over the groups for the grouped form. Tiles are numbered group by group; inside a
// group column-major (consecutive tiles share a B panel). A walker only moves forward.
struct GroupWalk {
  int group, tile_begin, tile_end, row_begin, tiles_m;
};

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x0040u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float(((uint32_t)h) << 16);
}

// Two f32 -> two bf16 (round to nearest even, NaN kept) in one gfx950 instruction;
// `lo` lands in bits 0..15.
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(lo), "v"(hi));
  return r;
}

// Two f32 -> two IEEE binary16 (round to nearest even; beyond 65504 rounds to infinity as the
// conversion instruction does); `lo` lands in bits 0..15.
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
  const _Float16 l = (_Float16)lo, h = (_Float16)hi;
  return (uint32_t)__builtin_bit_cast(uint16_t, l) | ((uint32_t)__builtin_bit_cast(uint16_t, h) << 16);
}

// Output element type is a launch parameter (uniform branch, outside the hot loop).
__device__ __forceinline__ uint32_t pack_out_x2(float lo, float hi, bool f16) {
  return f16 ? pack_f16x2(lo, hi) : pack_bf16x2(lo, hi);
}

// Kernel arguments live in memory and reach a wave through scalar loads that the compiler issues
// where it first needs each value: several dependent round trips of a few hundred nanoseconds each at
// the start of a kernel (the argument block is cold in the scalar cache at every launch). The decode
// kernels are a few microseconds long, so they ask for everything they will use in one batch, first
// thing (measured on the pair kernel at M=16, N=K=8192: 13.2 -> 12.6 us; whether the compiler's own
// placement is the fast or the slow one changes with unrelated edits).
__device__ __forceinline__ void fetch_arguments_now(const GemmParams& p) {
  asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.a_scale), "s"(p.b_scale), "s"(p.bias), "s"(p.c), "s"(p.M), "s"(p.N), "s"(p.K),
               "s"(p.lda), "s"(p.ldb), "s"(p.ldc), "s"(p.tiles_m), "s"(p.tiles_n), "s"(p.out_f16));
}

// Grouped form: zeros into rows first .. M-1 of C, shared out over `of` workgroups of this launch (this one is number `who`).
// As a fill of all of C in front of the launch it took a launch of its own and a write of everything that the product
// then writes again (8192 x 4096: 10 us of 115).
__device__ __forceinline__ void clear_rows(const GemmParams& p, int first, int who, int of) {
  const int threads = (int)blockDim.x, tid = (int)threadIdx.x;
  if (p.ldc == p.N && p.N % 8 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0) {
    v4i* c = (v4i*)(p.c + (size_t)first * p.N);
    const size_t count = (size_t)(p.M - first) * p.N / 8;
    for (size_t i = (size_t)who * threads + tid; i < count; i += (size_t)of * threads) c[i] = (v4i){0, 0, 0, 0};
  } else {
    for (long r = (long)first + who; r < p.M; r += of)
      for (long n = tid; n < p.N; n += threads) p.c[(size_t)r * p.ldc + n] = 0;
  }
}

// the same for what only the tiled kernel and its second pass read
__device__ __forceinline__ void fetch_tiled_arguments_now(const GemmParams& p) {
  asm volatile("" ::"s"(p.splits), "s"(p.steps_per_split), "s"(p.partial), "s"(p.m_sizes), "s"(p.groups), "s"(p.div_tiles_mul),
               "s"(p.div_tiles_shift), "s"(p.div_group_mul), "s"(p.div_group_shift), "s"(p.stamps), "s"(p.store));
}

// ------------------------------------------------------------------------------------
// Tile scheduler: static, no atomics (safe under graph capture).
//
// Hardware hands consecutive workgroup ids to consecutive XCDs, each with a private L2.
// Workgroup b therefore belongs to XCD b % 8 and is that XCD's slot b / 8. The tile list is
// cut into 8 contiguous chunks, one per XCD, and walked in "grouped" order (kGroupM tile
// rows at a time, column-major inside a group) so the tiles an XCD has in flight at any
// moment form a compact rectangle sharing A row panels and B column panels in its L2.
// ------------------------------------------------------------------------------------
struct TileWalk {
  int chunk_begin, chunk_len, slot, slots;
};

__device__ __forceinline__ TileWalk make_walk(int total_tiles) {
  const int xcd = blockIdx.x % kNumXcd;
  const int q = total_tiles / kNumXcd, rem = total_tiles % kNumXcd;
  TileWalk w;
  w.chunk_begin = xcd * q + (xcd < rem ? xcd : rem);
  w.chunk_len = q + (xcd < rem ? 1 : 0);
  w.slot = blockIdx.x / kNumXcd;
  w.slots = gridDim.x / kNumXcd;
  return w;
}

// Division of a wave-uniform n < 2^31 by a run-time divisor d whose reciprocal the host prepared:
// mul = ceil(2^shift / d), shift = 31 + ceil(log2 d), and then floor(n / d) = (n * mul) >> shift
// exactly (mul * d lies within 2^(shift-31) of 2^shift). Three scalar instructions where the
// compiler's expansion of a division is a few dozen, on the path that moves a load cursor from one
// tile to the next in the middle of the K pipeline.
__device__ __forceinline__ int fast_div(int n, uint32_t mul, uint32_t shift) {
  return (int)(uint32_t)(((uint64_t)(uint32_t)n * mul) >> shift);
}
inline void make_fast_div(uint32_t d, uint32_t& mul, uint32_t& shift) {
  int l = 0;
  while ((1ull << l) < d) ++l;
  shift = 31u + (uint32_t)l;
  mul = (uint32_t)(((1ull << shift) + d - 1) / d);
}

constexpr int kGroupM = 4;  // tile rows walked together (a group); the last group may hold fewer

// tile number -> tile row and column in grouped order (kGroupM tile rows at a time, column-major inside a group)
__device__ __forceinline__ void tile_coords(int t, int tiles_m, int tiles_n, uint32_t group_mul, uint32_t group_shift,
                                            int& tm, int& tn) {
  const int per_group = kGroupM * tiles_n;
  const int g = fast_div(t, group_mul, group_shift);
  const int first_m = g * kGroupM;
  const int gsz = min(tiles_m - first_m, kGroupM);
  const int in_g = t - g * per_group;
  // in_g / gsz for gsz in 1..4
  tn = gsz == 4 ? in_g >> 2 : gsz == 3 ? fast_div(in_g, 0xAAAAAAABu, 33) : gsz == 2 ? in_g >> 1 : in_g;
  tm = first_m + in_g - tn * gsz;
}

// ------------------------------------------------------------------------------------
// LDS layout of the tiled kernel. A "stage" of an operand holds a 128-byte K slab of the
// tile's rows: 128 bytes per row = 8 chunks of 16 bytes, fetched from global memory as whole
// 128-byte lines. Chunk c of row r sits at chunk position c ^ ((r >> 1) & 7): the MFMA
// operand reads (consecutive lanes = consecutive rows, same logical chunk) then spread over
// all banks. With a load distance of 2 steps A has two stages,
// B three (2*32 KB + 3*32 KB = all 160 KB of a 256x256 tile's LDS); the 256x128 tile runs at a
// distance of 3 (3*32 KB + 4*16 KB). (Distances of 3 and 4 were measured on the 128x128 tile with one
// workgroup per CU and bought under 10 %: that tile is bound by what the L2->L1->LDS path delivers
// per CU, about 48 bytes per clock against the 64 its two workgroups ask for at the full MFMA
// rate, not by the latency of a load.)
// ------------------------------------------------------------------------------------
constexpr int kStepK = 128;
constexpr int kDefaultDist = 2;  // steps a load runs ahead of its use; A ring = DIST stages, B ring = DIST + 1

__device__ __forceinline__ int swz128(int row) { return (row >> 1) & 7; }

// One wave-wide load of 16 bytes per lane from a buffer straight into LDS: lane i's bytes land at
// lds_wave_base + 16*i. The address is the descriptor's base + lane_off + wave_off, range-checked
// against the descriptor's extent (bytes past it arrive as zeros). STREAM marks the lines as used
// once (the instruction's `nt` bit): they leave the L2 early instead of pushing out lines other
// workgroups will ask for again.
template <bool STREAM>
__device__ __forceinline__ void load_chunk_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint8_t* lds_wave_base,
                                                  uint32_t lane_off, uint32_t wave_off) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not know the builtin)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds_wave_base, 16,
                                           (int)lane_off, (int)wave_off, 0, STREAM ? 2 : 0);
#endif
}

// Range-checked register loads through a buffer descriptor: 4 floats / 4 bf16 / one bf16 per lane;
// elements past the descriptor's extent read as zero bits.
__device__ __forceinline__ v4f load_f32x4_checked(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)lane_off, 0, 0));
#else
  return (v4f){0.f, 0.f, 0.f, 0.f};
#endif
}
__device__ __forceinline__ us4 load_u16x4_checked(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(us4, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)lane_off, 0, 0));
#else
  return (us4){0, 0, 0, 0};
#endif
}
__device__ __forceinline__ uint16_t load_u16_checked(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_raw_buffer_load_b16(rsrc, (int)lane_off, 0, 0);
#else
  return 0;
#endif
}

// Range-checked store of 4 floats per lane through a buffer descriptor (dropped past the extent).
__device__ __forceinline__ void store_f32x4_checked(v4f data, __amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off, uint32_t wave_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, data), rsrc, (int)lane_off, (int)wave_off, 0);
#endif
}

// How tiles store their 16-byte pieces of C (the host decides, store_policy()).
//   kStoreStream  aligned, with the streaming policy: C is written once and read by a later kernel at best, and what ordinary
//                 stores leave in the L2s is written back when the kernel ends (2048x4096x4096: 30.9 us, 34.3 with those)
//   kStoreKeep    aligned, without it (gemm_block_kernel)
//   kStoreAny     at any 2 bytes, without it
constexpr int kStoreStream = 0, kStoreKeep = 1, kStoreAny = 2;

// One wave-wide store of 16 bytes per lane through a buffer descriptor (address = base + lane_off + wave_off).
template <bool STREAM>
__device__ __forceinline__ void store_chunk(v4i data, __amdgpu_buffer_rsrc_t rsrc, uint32_t lane_off, uint32_t wave_off) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_buffer_store_b128(data, rsrc, (int)lane_off, (int)wave_off, STREAM ? 2 : 0);
#endif
}

// The first `valid` of 8 consecutive 16-bit results (none below 1, all from 8 on) to a row of C that starts at any 2 bytes: one
// unaligned store, pieces of 4, 2 and 1 where the row ends.
// (`valid` is opaque: the comparisons stay here, where as common values of many stores they would live in scalar registers)
__device__ __forceinline__ void store_columns(uint8_t* dst, v4i out, int valid) {
  asm volatile("" : "+v"(valid));
  if (valid >= 8) {
    *(v4i_any*)dst = out;
  } else if (valid > 0) {
    uint32_t first = (uint32_t)out[0], second = (uint32_t)out[1];
    if (valid & 4) {
      *(v2u_any*)dst = (v2u){first, second};
      first = (uint32_t)out[2];
      second = (uint32_t)out[3];
      dst += 8;
    }
    if (valid & 2) {
      *(u32_any*)dst = first;
      first = second;
      dst += 4;
    }
    if (valid & 1) *(uint16_t*)dst = (uint16_t)first;
  }
}

// A factor f of a block-scaled product in two parts: f = factor_mantissa(f) * 2^(e - 127), e being the biased exponent that the
// matrix instruction takes as the scale of an operand. Exact; between 2^-23 and 2 in magnitude but for an infinity or NaN, which
// stays one, and for zero, which counts as one with both operands scaled by 2^-126 (a product of codes is below 2^25: nothing is left).
__device__ __forceinline__ int factor_exponent(float f) { return min(max((__float_as_int(f) >> 23) & 0xff, 1), 254); }
__device__ __forceinline__ float factor_mantissa(float f) { return f == 0.0f ? 1.0f : ldexpf(f, 127 - factor_exponent(f)); }
// the scales of the two operands, a byte each
__device__ __forceinline__ int factor_scales(float f) { return factor_exponent(f) | (f == 0.0f ? 1 : 127) << 8; }

// Waits until at most VM of this wave's global loads and none of its LDS operations are
// outstanding, then joins the workgroup barrier. Written with the s_waitcnt builtin (not
// inline asm) so the compiler's own wait-count bookkeeping knows the LDS queue is empty
// afterwards and does not add full waits in front of the MFMAs that follow.
template <int VM>
__device__ __forceinline__ void wait_loads_and_barrier() {
  // gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] at [15:14]
  constexpr int imm = (VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (0 << 8);
  __builtin_amdgcn_s_waitcnt(imm);
  __builtin_amdgcn_s_barrier();
}

// what the block-scaled kernels read their factors through: constant memory, wave-uniform addresses, scalar loads
typedef const __attribute__((address_space(4))) float* scalar_floats;

// waits until at most VM of this wave's global loads are outstanding (LDS operations are not waited for)
template <int VM>
__device__ __forceinline__ void wait_loads() {
  constexpr int imm = (VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8);
  __builtin_amdgcn_s_waitcnt(imm);
}

// Cursor over the (tile, K step) sequence a workgroup walks; one for the A loads, one for
// the B loads (which run a step further ahead).
struct StepCursor {
  int item, kt, kt_begin, kt_end, left, issued;  // kt walks [kt_begin, kt_end) cyclically, `left` steps to go
};

// The kernel is one software pipeline over "steps" (a 128-byte K slab of one tile) that runs
// through all tiles a workgroup owns without draining at tile boundaries. For step g, with
// loads running DIST (= 2) steps ahead:
//
//   [A] MFMAs of (g, first K half), interleaved with the LDS reads of (g, second half) and
//       the loads of B(g+DIST) (its stage was released at the previous barrier)
//       wait for own loads of A(g+1) and B(g+1); workgroup barrier
//   [B] MFMAs of (g, second half), interleaved with the LDS reads of (g+1, first half) and
//       the loads of A(g+DIST) into the A stage step g just released
//   after a tile's last step: epilogue (loads of the next tile are already in flight)
//
// Two register sets of operand fragments alternate between the halves; one barrier per step.
//
// EPI selects what happens to a finished accumulator tile: scaled bf16 store (kEpiPlain),
// the same with the bias added (kEpiBias), or a raw fp32 partial-sum store for split-K
// (kEpiPartial). Tiles small enough for two workgroups per CU are compiled for two waves per
// SIMD (256 registers each).
constexpr int kEpiPlain = 0, kEpiBias = 1, kEpiPartial = 2;

constexpr size_t tiled_lds_bytes(int BM, int BN, int dist = kDefaultDist) {
  return (size_t)(dist * BM + (dist + 1) * BN) * kStepK;
}
constexpr int tiled_wgs_per_cu(int BM, int BN, int dist = kDefaultDist) { return tiled_lds_bytes(BM, BN, dist) <= 80 * 1024 ? 2 : 1; }
// waves per SIMD the registers are budgeted for. The block-scaled form is always held to 256 registers: with more
// the compiler puts the accumulators where the vector ALU cannot reach them and copies them back and
// forth in every step (512x4096x4096, deep ring: 28.5 us that way).
constexpr int tiled_waves_per_simd(int BM, int BN, int waves, bool blockscale, int dist) {
  const int n = tiled_wgs_per_cu(BM, BN, dist) * waves / 4;
  return blockscale && n < 2 ? 2 : n;
}

//
// GROUPED walks the tiles of a stack of row blocks whose sizes are read from device memory.
//
// BLOCKSCALE turns the kernel into the 128x128x128 block-scaled GEMM: a_scale is then
// [ceil(M/128)][ceil(K/128)], b_scale [ceil(N/128)][ceil(K/128)], and every K step's product
// is multiplied by a_scale[mb][kb] * b_scale[nb][kb] before it is added up. With wave tiles
// inside one scale block and 128-byte steps that factor is one number per wave and step:
// the accumulators are kept in units of the current step's factor (multiplied by the ratio of
// consecutive factors in front of each step's MFMAs) and by the last factor in the epilogue.
//
// STREAM_B: the rows of B are fetched with the streaming cache policy. For launches with one or
// two tile rows, where a panel of B is read by one or two workgroups and never again
// (measured: M=128, N=K=8192 27.6 -> 24.2 us, M=64 22.5 -> 19.6 us; with more tile rows the
// panels are shared through the L2 and the same policy costs 5-8 %). The grouped form has it for groups of
// about one tile row (grouped_form).
// CLEAR: the grouped form that sets the rows of C past the last group's to zero. Instances of their own: with the test
// and the loop in the others, which a call with a result of its own runs, those were 1-3 % slower (1704x1280x768 in 12 groups
// 11.46 -> 11.76 us, 450x1024x576 6.47 -> 6.61).
// OFF_LINES: a STREAM_B launch whose rows of B are off the 128-byte lines keeps the rotated walk but not the policy, with which the
// line that two steps of a row share would come from memory twice: 119x55346x4112 73.9 -> 62.8 us, 32x57344x4112 68.5 -> 50.2,
// 128x28672x8256 68.9 -> 63.7, 256x28672x8256 82.0 -> 78.9 (without the rotation 63.6, 51.0, 70.6 and 108).
// LINES: rows off the 128-byte lines (their base or pitch no multiple of 128) are fetched in whole lines all the same. A row's windows start
// at the line that its first byte lies in, so its chunks sit up to seven places further back than its neighbour's: chunk c of step g is
// chunk c + shift of window g, or of window g + 1, whatever of the next row or of the one before lies in a window is never read, and an item
// has one window more than steps. Eight rows on, the shift is the same (pitches are multiples of 16), so it is one number a lane for
// the loads and one for the operand reads. For launches of at most one item a workgroup (a second one would start in another place of the
// ring). From L2 a CU takes in 123 bytes/ns in whole lines and 83 in 128-byte pieces 16 bytes off them.
template <int BM, int BN, int WAVES_M, int WAVES_N, bool KTAIL, int EPI, bool GROUPED = false, bool BLOCKSCALE = false,
          int DIST = kDefaultDist, bool STREAM_B = false, bool CLEAR = false, bool OFF_LINES = false, bool LINES = false>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64)
__attribute__((amdgpu_waves_per_eu(tiled_waves_per_simd(BM, BN, WAVES_M * WAVES_N, BLOCKSCALE, DIST),
                                   tiled_waves_per_simd(BM, BN, WAVES_M * WAVES_N, BLOCKSCALE, DIST))))
void gemm_tiled_kernel(GemmParams p) {
  constexpr int kStagesA = DIST, kStagesB = DIST + 1;
  static_assert(DIST >= 2 && tiled_lds_bytes(BM, BN, DIST) <= 160 * 1024, "the stage rings must fit the LDS");
  static_assert(!GROUPED || EPI == kEpiPlain, "the grouped form has neither bias nor split-K");
  static_assert(!OFF_LINES || (STREAM_B && !GROUPED), "a variant of the streaming launches");
  static_assert(!CLEAR || GROUPED, "only the grouped form has rows past its groups'");
  static_assert(!LINES || (KTAIL && DIST >= 3 && !GROUPED && !BLOCKSCALE && !STREAM_B), "a window more has to have landed; the walk over K starts at its beginning");
  static_assert(!BLOCKSCALE || (128 % (BM / WAVES_M) == 0 && 128 % (BN / WAVES_N) == 0 && EPI != kEpiBias && !GROUPED),
                "a wave's tile must lie inside one 128x128 scale block: one factor per wave and step");
  constexpr bool HAS_BIAS = EPI == kEpiBias;
  constexpr int NW = WAVES_M * WAVES_N;
  constexpr int WTM = BM / WAVES_M;    // wave tile rows (m)
  constexpr int WTN = BN / WAVES_N;    // wave tile cols (n)
  constexpr int MT = WTM / 32, NT = WTN / 32;
  constexpr int STAGE_A = BM * kStepK, STAGE_B = BN * kStepK;
  constexpr int LDS_B0 = kStagesA * STAGE_A;  // B stages follow the A stages
  constexpr int A_GROUPS = BM / 8 / NW;       // 8-row groups (1 KB of LDS) each wave fetches per step
  constexpr int B_GROUPS = BN / 8 / NW;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "tile rows must split over waves");
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of 32x32");
  static_assert(DIST * (A_GROUPS + B_GROUPS) < 64, "outstanding-load count must fit the vmcnt field");

  fetch_arguments_now(p);
  fetch_tiled_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  // (diagnostic launches only: the shader clock and the constant 100 MHz clock at this workgroup's start)
  unsigned long long stamp_cycles = 0, stamp_ticks = 0;
  if (p.stamps) {
    stamp_cycles = __builtin_readcyclecounter();
    stamp_ticks = __builtin_amdgcn_s_memrealtime();
  }

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int l32 = lane & 31, half = lane >> 5;

  // ---- per-lane constants of the global->LDS copy: a wave-wide load fills 8 rows
  const int ld_row = lane >> 3;
  const int ld_pc = lane & 7;  // physical chunk this lane's 16 bytes land in
  // 8*group + ld_row: the swizzle key depends on ld_row and the parity of the group only
  auto ld_chunk_off = [&](int group) { return (ld_pc ^ swz128(group * 8 + ld_row)) * kChunk; };

  // ---- per-lane constants of the LDS->register operand reads. For K half s (64 bytes) and
  // j in {0,1}, lane (l32, half) takes logical chunk 4*half + 2*s + j of its row. Any
  // assignment is valid as long as A and B use the same one; this one keeps the two halves
  // of the wave in different 64-byte halves of a row.
  int rd_off[2][2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      rd_off[s][j] = l32 * kStepK + (((4 * half + 2 * s + j) ^ swz128(l32)) * kChunk);
  // LINES: a row's shift in chunks, by its number modulo 8; the reads of either operand, and whether they are the next window's
  auto row_shift = [](const uint8_t* base, long ld, int row) { return (int)(((uint32_t)reinterpret_cast<uintptr_t>(base) + (uint32_t)row * (uint32_t)ld) & 127u) / kChunk; };
  int rd_off_a[2][2], rd_off_b[2][2];
  bool rd_next_a[2][2], rd_next_b[2][2];
  if constexpr (LINES) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int ca = 4 * half + 2 * s + j + row_shift(p.a, p.lda, l32 & 7), cb = 4 * half + 2 * s + j + row_shift(p.b, p.ldb, l32 & 7);
        rd_off_a[s][j] = l32 * kStepK + (((ca & 7) ^ swz128(l32)) * kChunk);
        rd_off_b[s][j] = l32 * kStepK + (((cb & 7) ^ swz128(l32)) * kChunk);
        rd_next_a[s][j] = ca >= 8;
        rd_next_b[s][j] = cb >= 8;
      }
  }
  const int a_rd_base = (wm * WTM) * kStepK;
  const int b_rd_base = LDS_B0 + (wn * WTN) * kStepK;

  // Work items are (split, tile) pairs, split-major: consecutive items are neighbouring
  // tiles of the same K range, so an XCD's chunk of the list still shares operand panels.
  int total_tiles = p.tiles_m * p.tiles_n;
  // rows of group g, given the rows before it: never negative, never past row M
  auto group_rows = [&](int g, int row_begin) { return min(max(p.m_sizes[g], 0), p.M - row_begin); };
  if (GROUPED) {
    total_tiles = 0;
    int rows = 0;
    for (int g = 0; g < p.groups; ++g) {
      const int mg = group_rows(g, rows);
      total_tiles += ((mg + BM - 1) / BM) * p.tiles_n;
      rows += mg;
    }
    if (CLEAR && rows < p.M) clear_rows(p, rows, (int)blockIdx.x, (int)gridDim.x);
  }
  const TileWalk walk = make_walk(total_tiles * p.splits);
  if (walk.slot >= walk.chunk_len) return;  // uniform over the workgroup
  const int k_full = p.K / kStepK;             // whole 128-byte steps
  const int k_tail = p.K - k_full * kStepK;    // 0 or a multiple of 16
  const int k_steps = k_full + (k_tail ? 1 : 0);
  // (the grouped form counts its tiles on the device and divides the ordinary way; an unsplit launch has
  // nothing to divide)
  auto item_split = [&](int li) {
    const int t = walk.chunk_begin + li;
    return GROUPED ? t / total_tiles : p.splits == 1 ? 0 : fast_div(t, p.div_tiles_mul, p.div_tiles_shift);
  };
  auto item_tile = [&](int li) {
    const int t = walk.chunk_begin + li;
    return GROUPED ? t % total_tiles : p.splits == 1 ? t : t - fast_div(t, p.div_tiles_mul, p.div_tiles_shift) * total_tiles;
  };
  auto split_begin = [&](int sp) { return sp * p.steps_per_split; };
  auto split_end = [&](int sp) { return min((sp + 1) * p.steps_per_split, k_steps); };
  int total_steps = 0;
  for (int li = walk.slot; li < walk.chunk_len; li += walk.slots)
    total_steps += split_end(item_split(li)) - split_begin(item_split(li)) + (LINES ? 1 : 0);

  // item -> tile location. Plain form: grouped walk order over the tile grid. Grouped form:
  // the walker steps through m_sizes until it reaches the group that holds the tile.
  auto locate = [&](GroupWalk& w, int li) -> TileLoc {
    const int tile = item_tile(li);
    if (!GROUPED) {
      int tm, tn;
      tile_coords(tile, p.tiles_m, p.tiles_n, p.div_group_mul, p.div_group_shift, tm, tn);
      return TileLoc{tm * BM, p.M, tn * BN, 0, 0};
    }
    while (tile >= w.tile_end && w.group + 1 < p.groups) {
      w.row_begin += group_rows(w.group, w.row_begin);
      ++w.group;
      w.tiles_m = (group_rows(w.group, w.row_begin) + BM - 1) / BM;
      w.tile_begin = w.tile_end;
      w.tile_end += w.tiles_m * p.tiles_n;
    }
    const int t = tile - w.tile_begin;
    const int tm = t % max(w.tiles_m, 1), tn = t / max(w.tiles_m, 1);
    return TileLoc{w.row_begin + tm * BM, w.row_begin + group_rows(w.group, w.row_begin), tn * BN, w.group, STREAM_B ? w.tiles_m : 0};
  };
  auto first_group = [&]() -> GroupWalk {
    GroupWalk w = {0, 0, 0, 0, 0};
    if (GROUPED) {
      w.tiles_m = (group_rows(0, 0) + BM - 1) / BM;
      w.tile_end = w.tiles_m * p.tiles_n;
    }
    return w;
  };
  GroupWalk walk_a = first_group(), walk_b = first_group(), walk_c = first_group();

  // ---- load side of the pipeline
  StepCursor ca = {walk.slot, 0, 0, 0, 0, 0}, cb = {walk.slot, 0, 0, 0, 0, 0};
  // STREAM_B launches start every tile column at a different K step and wrap around. Their
  // workgroups stream disjoint rows of B in lockstep; with a power-of-two row pitch all the
  // addresses in flight at one moment would agree in their low bits and crowd a few memory
  // channels (M=32, N=57344, K=8192 with an 8192-byte pitch: 100 us; the same data at a pitch
  // of 8320 bytes: 71 us). The sum over K does not care where it starts. Launches whose tiles
  // share panels of B through the L2 keep the common order: there the sharing needs it. So do
  // plans with more than two splits, whose items are already spread over K (M=128, N=K=8192 with
  // four splits lost 5 % to the rotation; two splits gain 5 %, unsplit plans 11-28 %).
  // The streaming grouped form decides by group, as its tiles are taken up: those of a group of several tile rows share panels of
  // B like any others (half of all rows at one of 8 experts, 256x14336x4096 105 -> 84 us, one of 32, 1800x4096x4096 123 -> 112; all
  // of them 51 -> 38). From two tile rows on with 128 columns a tile, from three on with 256 (1000x14336x4096 in 8 groups, most
  // of one or two tile rows of those: 105, without streaming those of two 109). Rows off the 128-byte lines are not streamed.
  constexpr bool STREAM_BY_GROUP = GROUPED && STREAM_B;
  const int stream_rows = p.ldb % kStepK == 0 ? (BN == 256 ? 2 : 1) : 0;  // tile rows of a group up to which its tiles stream B
  auto group_streams = [&](const TileLoc& loc) { return loc.tiles_m <= stream_rows; };
  auto first_step = [&](const TileLoc& loc, int begin, int count) {
    const bool rotated = STREAM_B && p.splits <= 2 && (!STREAM_BY_GROUP || group_streams(loc));
    return begin + (rotated ? (loc.n0 / BN) % count : 0);
  };
  auto start_cursor = [&](StepCursor& c, int li, const TileLoc& loc) {
    c.kt_begin = split_begin(item_split(li));
    c.kt_end = split_end(item_split(li)) + (LINES ? 1 : 0);
    c.left = c.kt_end - c.kt_begin;
    c.kt = first_step(loc, c.kt_begin, c.left);
  };
  // Source of the loads: one buffer descriptor per operand and tile, base = the tile's first row,
  // extent = its valid rows (the hardware returns zeros for anything past the extent, so rows past
  // the matrix edge need neither clamping nor predication: they read as zeros and are never
  // stored). A lane's 16 bytes in the i-th 8-row group a wave fetches (grp = wave + NW*i) lie at
  //   lane part (vector register, the same for every group, step and tile: ld_row*ld + chunk,
  //              the chunk swizzle depends on the group's parity only, which a wave's groups share)
  // + scalar part (K offset + 8*grp*ld, one scalar add per load).
  // The range check adds the two before it compares, so the sum must stay below 2^32: the host
  // admits leading dimensions up to 2^31 / 256.
  static_assert(NW % 2 == 0, "all groups of a wave must share their parity");
  struct OperandSrc {
    const uint8_t* base;
    uint32_t extent;                  // bytes from base that may be read
    uint32_t wave_off, group_stride;  // 8*wave*ld and 8*NW*ld
  };
  constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format: plain byte addressing with range check
  constexpr uint32_t kLead = LINES ? 7 * kChunk : 0;  // (the most that a window starts in front of its row: offsets stay positive)
  auto make_src = [&](const uint8_t* base, int rows_valid, int rows_tile, long ld) -> OperandSrc {
    // (a tile always starts on a valid row, so rows_valid >= 1; clamping at zero as well would turn
    // the pair into a three-operand median, which exists as a vector instruction only and would
    // pull the descriptor out of the scalar registers)
    const uint32_t extent = (uint32_t)min(rows_valid, rows_tile) * (uint32_t)ld + kLead;
    // Base and extent are the same for every lane; they are pinned to scalar registers because a
    // descriptor that the compiler takes for lane-dependent (the grouped form derives these from
    // sizes it loads, through a clamp that only exists as a vector instruction) makes every load a
    // loop over the distinct descriptors of the wave.
    OperandSrc o;
    const uintptr_t b = reinterpret_cast<uintptr_t>(base) - kLead;
    o.base = reinterpret_cast<const uint8_t*>(
        ((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
        (uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
    o.extent = (uint32_t)__builtin_amdgcn_readfirstlane((int)extent);
    o.wave_off = 8u * (uint32_t)wave * (uint32_t)ld;
    o.group_stride = 8u * NW * (uint32_t)ld;
    return o;
  };
  // 24-bit multiplies (row < 8, leading dimension < 2^24 by the host's check)
  const uint32_t lane_chunk = (uint32_t)ld_chunk_off(wave);
  const int a_shift = LINES ? row_shift(p.a, p.lda, ld_row) : 0, b_shift = LINES ? row_shift(p.b, p.ldb, ld_row) : 0;
  const uint32_t a_lane = __umul24((uint32_t)ld_row, (uint32_t)p.lda) + lane_chunk + kLead - (uint32_t)(a_shift * kChunk);
  const uint32_t b_lane = __umul24((uint32_t)ld_row, (uint32_t)p.ldb) + lane_chunk + kLead - (uint32_t)(b_shift * kChunk);
  // K tail (KTAIL kernels only): in the partial last step, lanes whose chunk lies at or past K
  // must fetch zeros (whatever follows a row in memory could decode to NaN): their lane part is
  // pushed past every extent for that step. A lane's logical chunk is the same for all its
  // groups.
  const bool tail_chunk_ok = ((ld_pc ^ swz128(wave * 8 + ld_row)) * kChunk) < k_tail;
  constexpr uint32_t kPastExtent = 0x80000000u;  // extents and scalar parts stay below 2^31
  // LINES: the lane's chunk of window w is chunk 8w + c - shift of its row, which a window at either end need not have
  const int chunk_c = (int)lane_chunk / kChunk, chunks_left = k_tail / kChunk;  // of the row, past its whole steps
  const uint32_t a_lane_tail = (LINES ? chunk_c - a_shift < chunks_left : tail_chunk_ok) ? a_lane : kPastExtent;
  const uint32_t b_lane_tail = (LINES ? chunk_c - b_shift < chunks_left : tail_chunk_ok) ? b_lane : kPastExtent;
  const uint32_t a_lane_end = 8 + chunk_c - a_shift < chunks_left ? a_lane : kPastExtent;
  const uint32_t b_lane_end = 8 + chunk_c - b_shift < chunks_left ? b_lane : kPastExtent;
  const uint32_t a_lane_head = chunk_c >= a_shift ? a_lane : kPastExtent, b_lane_head = chunk_c >= b_shift ? b_lane : kPastExtent;
  OperandSrc a_src = {nullptr, 0, 0, 0}, b_src = {nullptr, 0, 0, 0};
  auto setup_a = [&](int li) {
    const TileLoc loc = locate(walk_a, li);
    start_cursor(ca, li, loc);
    a_src = make_src(p.a + (size_t)loc.m0 * p.lda, loc.m_end - loc.m0, BM, p.lda);
  };
  int b_streams = 0;  // whether the loads of B take the streaming policy (STREAM_BY_GROUP: in the tile being loaded)
  auto setup_b = [&](int li) {
    const TileLoc loc = locate(walk_b, li);
    start_cursor(cb, li, loc);
    if (STREAM_BY_GROUP) b_streams = __builtin_amdgcn_readfirstlane(group_streams(loc));
    b_src = make_src(p.b + ((size_t)loc.group * p.N + loc.n0) * p.ldb, p.N - loc.n0, BN, p.ldb);
  };
  // i-th group of one operand's step kt into the stage at sbase
  // (step_off: K offset of the step + the wave's first group, prepared once per step)
  auto load_group = [&](auto stream_tag, const OperandSrc& src, uint32_t lane_off, uint32_t step_off, int i, uint8_t* sbase) {
    // (the descriptor is put together from its scalar parts here: one scalar instruction)
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(src.base), 0, (int)src.extent, kRsrcFlags);
    load_chunk_to_lds<decltype(stream_tag)::value>(rsrc, sbase + (wave + NW * i) * 1024, lane_off,
                                                   step_off + (uint32_t)i * src.group_stride);
  };
  auto lane_part = [&](uint32_t whole, uint32_t tail, uint32_t end, int kt) -> uint32_t {
    if (LINES && kt > k_full) return end;
    return KTAIL && kt >= k_full ? tail : whole;
  };
  // (the first windows of an item; a row of one step has both its ends in window 0)
  auto first_lane_part = [&](uint32_t whole, uint32_t tail, uint32_t end, uint32_t head, int kt) -> uint32_t {
    const uint32_t part = lane_part(whole, tail, end, kt);
    return LINES && kt == 0 ? max(part, head) : part;
  };
  // Ring positions the next loads of A and of B go to (= issued % stages, kept as counters that wrap).
  int fill_a = 0, fill_b = 0;
  auto next_fill_a = [&]() { fill_a = (fill_a + 1 == kStagesA) ? 0 : fill_a + 1; };
  auto next_fill_b = [&]() { fill_b = (fill_b + 1 == kStagesB) ? 0 : fill_b + 1; };
  // Issues one operand's loads for its cursor's step into the next stage of its ring. Past the
  // last step it re-issues the last one into a stage nobody reads again, which keeps the
  // path free of branches.
  auto issue_a = [&]() {
    const uint32_t lo = first_lane_part(a_lane, a_lane_tail, a_lane_end, a_lane_head, ca.kt);
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i)
      load_group(std::false_type{}, a_src, lo, (uint32_t)ca.kt * kStepK + a_src.wave_off, i, lds + fill_a * STAGE_A);
    next_fill_a();
    ++ca.issued;
  };
  auto issue_b = [&]() {
    const uint32_t lo = first_lane_part(b_lane, b_lane_tail, b_lane_end, b_lane_head, cb.kt);
#pragma unroll
    for (int i = 0; i < B_GROUPS; ++i)
      load_group(std::integral_constant<bool, STREAM_B && !OFF_LINES>{}, b_src, lo, (uint32_t)cb.kt * kStepK + b_src.wave_off, i,
                 lds + LDS_B0 + fill_b * STAGE_B);
    next_fill_b();
    ++cb.issued;
  };
  // Moves a load cursor to its next step. PLAIN: the caller knows that the next step belongs to the
  // same work item (true for all but the last DIST + 1 steps of an item): no branch, no tile set-up.
  auto advance_a = [&](auto plain_tag) {
    if (!decltype(plain_tag)::value) {
      if (ca.issued >= total_steps) return;  // stay on the last step
      if (--ca.left == 0) {
        ca.item += walk.slots;
        setup_a(ca.item);
        return;
      }
    } else {
      --ca.left;
    }
    ca.kt = (ca.kt + 1 == ca.kt_end) ? ca.kt_begin : ca.kt + 1;
  };
  auto advance_b = [&](auto plain_tag) {
    if (!decltype(plain_tag)::value) {
      if (cb.issued >= total_steps) return;
      if (--cb.left == 0) {
        cb.item += walk.slots;
        setup_b(cb.item);
        return;
      }
    } else {
      --cb.left;
    }
    cb.kt = (cb.kt + 1 == cb.kt_end) ? cb.kt_begin : cb.kt + 1;
  };

  // ---- operand fragments: two register sets; each fragment is two 16-byte LDS reads
  struct Frag {
    v4i lo, hi;
  };
  Frag xa[MT], xb[NT], ya[MT], yb[NT];
  // (next: where the same rows' next window lies, LINES only)
  auto read_a = [&](const uint8_t* rows, const uint8_t* next, int s, int j, int i) -> v4i {
    if constexpr (LINES) return *(const v4i*)((rd_next_a[s][j] ? next : rows) + rd_off_a[s][j] + i * 32 * kStepK);
    else return *(const v4i*)(rows + i * 32 * kStepK + rd_off[s][j]);
  };
  auto read_b = [&](const uint8_t* rows, const uint8_t* next, int s, int j, int i) -> v4i {
    if constexpr (LINES) return *(const v4i*)((rd_next_b[s][j] ? next : rows) + rd_off_b[s][j] + i * 32 * kStepK);
    else return *(const v4i*)(rows + i * 32 * kStepK + rd_off[s][j]);
  };
  auto as_v8 = [](const Frag& f) -> v8i {
    return (v8i){f.lo[0], f.lo[1], f.lo[2], f.lo[3], f.hi[0], f.hi[1], f.hi[2], f.hi[3]};
  };

  v16f acc[MT][NT];  // defined by the first step of every work item
  // BLOCKSCALE only. The sum over K blocks of s_k * P_k (P_k the unscaled product of block k) is
  // kept in units of the current block's factor: before step k adds P_k the accumulators are
  // multiplied by s_(k-1) / s_k, and the epilogue multiplies by the last factor. One multiply per
  // accumulator and step on the vector ALU, under the MFMAs' cover, and no second accumulator
  // set: the kernel keeps the register budget of the plain 128x128 tile (two workgroups per CU).
  // A factor of exactly zero is replaced by 2^-60 (its block then contributes P_k * 2^-60, nothing
  // at the output's precision); factors are expected to span less than 2^60 within a row of blocks.
  // ANY_FACTORS: the parts of a split launch, which runs shapes whose form without a workspace adds every block's products with the
  // factor as it is, and so takes any. There the accumulators are in units of the factor's mantissa, and the matrix
  // instructions take its exponent as a scale: the same products and ratios times powers of two, hence the same bits where
  // the other units do not overflow (and 1.6e-3 of the result's norm off float64 either way, nearly all of it the rounding to bf16; the
  // f32 sums 1.5e-5, what the matrix instruction itself leaves). It costs nothing: a part's steps are half of all at most, and
  // with two registers to look them up in instead of four 1047x1566x12800 in two parts takes 39.6 us, in units of the factors 41.9,
  // 32x1024x28672 18.5 and 19.2.
  // Blocks 0 .. n-2 are rescaled in phase [B] of the step before (each under the cover of the next
  // block's MFMA), the last one under the first MFMA of the step itself.
  // s_pend / s_cur: the ratios to the next step / to this one; kt_c: the K step the compute side is
  // at; the lane's share of the item's factors and ratios (sc[r], rt[r] belong to step 64*r + lane).
  float s_pend = 1.0f, s_cur = 1.0f, s_last = 1.0f, n_pend = 1.0f, n_last = 1.0f;
  int kt_c = 0;
  constexpr bool ANY_FACTORS = BLOCKSCALE && EPI == kEpiPartial;
  int scales = 0, n_scales = 0;  // ANY_FACTORS: of this step's operands, and of the next one's
  auto unit = [](float f) { return ANY_FACTORS ? factor_mantissa(f) : f; };  // what the accumulators are in units of
  constexpr int SC_REGS = ANY_FACTORS ? 2 : 4;  // 256 steps = K up to 32768; a part has half of them at most, and its first one is lane 0's
  float sc[SC_REGS] = {}, rt[SC_REGS] = {};
  auto load_block_scales = [&](const TileLoc& loc, int first) {
    // the scale block of this wave's tile (clamped for waves that lie past the matrix edge)
    const int mb = min(loc.m0 + wm * WTM, p.M - 1) / 128, nb = min(loc.n0 + wn * WTN, p.N - 1) / 128;
    const float* sa = p.a_scale + (size_t)mb * k_steps;
    const float* sb = p.b_scale + (size_t)nb * k_steps;
    auto factor = [&](int kb) -> float {
      const float f = sa[kb] * sb[kb];
      return f == 0.0f && !ANY_FACTORS ? 0x1p-60f : f;
    };
    float before[SC_REGS];  // ANY_FACTORS: the factor of the step before
#pragma unroll
    for (int r = 0; r < SC_REGS; ++r) {
      const int kb = min(first + r * 64 + lane, k_steps - 1);
      sc[r] = factor(kb);
      if (STREAM_B) rt[r] = factor(kb > 0 ? kb - 1 : k_steps - 1) / sc[r];  // (a rotated walk passes from the last step to the first)
      else if (ANY_FACTORS) before[r] = factor(max(kb - 1, 0));
      else rt[r] = kb > 0 ? factor(kb - 1) / sc[r] : 1.0f;
    }
    if constexpr (ANY_FACTORS) {
      bool normal = true;
#pragma unroll
      for (int r = 0; r < SC_REGS; ++r) {
        auto bits = [](float f) { return __int_as_float((__float_as_int(f) & 0x807fffff) | 0x3f800000); };
        rt[r] = bits(before[r]) / bits(sc[r]);
        normal = normal && __builtin_isnormal(before[r]) && __builtin_isnormal(sc[r]);
      }
      if (!__all(normal)) {  // (zeros, subnormal products, infinities, NaN)
#pragma unroll
        for (int r = 0; r < SC_REGS; ++r) rt[r] = unit(before[r]) / unit(sc[r]);
      }
    }
  };
  // (kt at most k_steps past the end. A walk that wraps around finds the first steps there; what lies past the end of one that
  // does not is never used, and keeping to the last step costs less scalar work in every step: 721x528x1152 9.85 -> 9.54 us,
  // 404x3104x464 7.44 -> 7.20.)
  auto lane_value = [&](const float (&regs)[SC_REGS], int kt) -> float {
    if (STREAM_B) kt = kt >= k_steps ? kt - k_steps : kt;
    else kt = min(kt, ANY_FACTORS ? 64 * SC_REGS - 1 : k_steps - 1);
    const int r = kt >> 6;
    const float v = r == 0 ? regs[0] : r == 1 || SC_REGS == 2 ? regs[1] : r == 2 ? regs[SC_REGS - 2] : regs[SC_REGS - 1];
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), kt & 63));
  };
  // brings block t of the accumulators from one step's factor to the next one's
  auto fold_block = [&](int t, float ratio) {
    const int i = t / NT, j = t % NT;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][j][v] *= ratio;
  };

  // t-th MFMA of a half step (t = i*NT + j) on fragment set (fa, fb)
  // (fresh: the block's first MFMA of a tile starts from zero instead of the old contents)
  auto mfma_one = [&](const Frag (&fa)[MT], const Frag (&fb)[NT], int t, bool fresh) {
    const int i = t / NT, j = t % NT;
    const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if constexpr (ANY_FACTORS)
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(as_v8(fb[j]), as_v8(fa[i]), fresh ? zero : acc[i][j], 0, 0, 0, scales, 1, scales);
    else
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(as_v8(fb[j]), as_v8(fa[i]), fresh ? zero : acc[i][j], 0, 0, 0, 0, 0, 0);
  };
  // u-th of the 2*(MT+NT) LDS reads that fill fragment set (fa, fb) with K half s
  auto read_one = [&](Frag (&fa)[MT], Frag (&fb)[NT], const uint8_t* rows_a, const uint8_t* next_a, const uint8_t* rows_b,
                      const uint8_t* next_b, int s, int u) {
    const int f = u >> 1;
    if (f < MT) {
      if (u & 1) fa[f].hi = read_a(rows_a, next_a, s, 1, f);
      else fa[f].lo = read_a(rows_a, next_a, s, 0, f);
    } else {
      if (u & 1) fb[f - MT].hi = read_b(rows_b, next_b, s, 1, f - MT);
      else fb[f - MT].lo = read_b(rows_b, next_b, s, 0, f - MT);
    }
  };
  constexpr int AHEAD = LINES ? 1 : 0;  // windows behind a step's own that have to have landed for it
  // Per half step: NMFMA MFMAs, NREAD LDS reads, A_GROUPS or B_GROUPS global->LDS loads, the
  // memory instructions placed behind the MFMAs: load l in slot l*NMFMA/GROUPS, the reads RPS
  // per slot in the first half of the slots. The reads have then returned while the last
  // MFMAs still execute, so the wait at the end of the half step (for the barrier, or for
  // the fragments of the next half) costs the matrix pipe nothing.
  constexpr int NMFMA = MT * NT, NREAD = 2 * (MT + NT);
  constexpr int RPS = (NREAD + NMFMA / 2 - 1) / (NMFMA / 2);

  // ---- prologue: A(0) B(0) .. A(DIST-1) B(DIST-1) in flight, first fragments in registers
  setup_a(ca.item);
  setup_b(cb.item);
#pragma unroll
  for (int d = 0; d < DIST; ++d) {
    issue_a(); advance_a(std::false_type{});
    issue_b(); advance_b(std::false_type{});
  }
  wait_loads_and_barrier<(DIST - 1 - AHEAD) * (A_GROUPS + B_GROUPS)>();
#pragma unroll
  for (int u = 0; u < NREAD; ++u) read_one(xa, xb, lds + a_rd_base, lds + a_rd_base + STAGE_A, lds + b_rd_base, lds + b_rd_base + STAGE_B, 0, u);

  // ---- epilogue. The MFMA leaves lane (l32, half) with row l32 of every 32x32 block and the
  // columns 8*q + 4*half + e (register 4*q + e): storing from there would touch 32 rows per
  // instruction. Instead a lane finishes its own elements first - a_scale[m], b_scale[n], bias[n]
  // in fp32, one rounding to the 16-bit output type, two results per register - and each 32-row
  // block of the wave's tile is then turned through LDS, PASS_J 32-column blocks at a time, as
  // 16-bit values: read back, a lane holds 8 consecutive columns of one row and stores its 16
  // bytes, so a wave-wide store covers whole rows of the pass.
  //
  // The turn-table is the wave's own share (the 1 KB groups it fills itself) of the B stage
  // that held this tile's last step: every wave finished reading that stage before the
  // step's barrier, and only this wave will load into these groups again. A pass fills half of
  // it, so the passes alternate between two halves: while one pass is read back and stored, the
  // next is converted and written (LDS runs a wave's operations in order, so neither half needs
  // a wait before it is written again). A pass row is CPR 16-byte chunks; chunk c of row r sits
  // at chunk position c ^ key(r): the 16-byte reads of 8 lanes spread over all banks, the 8-byte
  // writes of 16 consecutive rows meet in pairs (a two-way conflict on 64 of the epilogue's
  // instructions, which are bound by their arithmetic; undoing it costs the readers register moves).
  constexpr int PASS_J = B_GROUPS / 4;          // 32-column blocks per pass (2 KB of 16-bit values each)
  constexpr int NJP = NT / PASS_J;              // passes per 32-row block
  constexpr int CPR = PASS_J * 4;               // 16-byte chunks per pass row
  constexpr int ROW_BYTES = CPR * 16;
  constexpr int ROWS_PER_GROUP = 1024 / ROW_BYTES;
  constexpr int GROUPS_PER_PASS = 32 / ROWS_PER_GROUP;  // = B_GROUPS / 2
  constexpr int LPR = CPR;                      // lanes per row when reading back (one chunk each)
  constexpr int ROWS_PER_READ = 64 / LPR;
  constexpr int ITERS = 32 / ROWS_PER_READ;
  static_assert(B_GROUPS % 4 == 0 && NT % PASS_J == 0 && (CPR == 4 || CPR == 8) && 2 * GROUPS_PER_PASS == B_GROUPS,
                "turn-table geometry");
  auto epilogue = [&](const TileLoc& loc, auto store_tag, auto f16_tag, uint8_t* free_b_stage) {
    const int m0 = loc.m0, n0 = loc.n0;
    // Aligned stores: no lane's 8 columns straddle the edge. Edge tiles take them too: rows past the edge fall outside the output
    // descriptor's extent and lanes past column N are sent there.
    constexpr int STORE = decltype(store_tag)::value;
    constexpr bool OUT_F16 = decltype(f16_tag)::value;      // IEEE binary16 instead of bf16
    // row r of the pass kept in half h of the table
    auto row_addr = [&](int h, int r) -> uint8_t* {
      return free_b_stage + (wave + NW * (h * GROUPS_PER_PASS + r / ROWS_PER_GROUP)) * 1024 + (r % ROWS_PER_GROUP) * ROW_BYTES;
    };
    auto key = [](int r) { return (r * ROW_BYTES / 128) % CPR; };
    // The lane-dependent addresses below are the same for every tile; derived from an opaque
    // copy of the lane id they are recomputed here (a few integer operations) instead of
    // being hoisted out of the tile loop, where they would occupy registers through the K loop.
    // (the lane id itself comes from the hardware's lane count, inside the opaque statement: as a
    // loop invariant it would be moved in front of the K loop and, with no register to spare there,
    // spilled; its reload at this point waits for every load in flight)
    int lane_e;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_e));
    const int l32 = lane_e & 31, half = lane_e >> 5;
    const int wr_key = key(l32);
    const int wr_half = half * 8;  // where this lane's 8 bytes sit inside a chunk
    const int rd_row = lane_e / LPR, rd_chunk = lane_e % LPR;  // 8 columns of the pass row this lane stores
    const int rd_col = rd_chunk * 8;

    // scales and bias of the lane's own elements: row l32 of every 32-row block, columns
    // 32*j + 8*q + 4*half + e, fetched through descriptors that end at column N (whatever lies
    // past it reads as zero and belongs to columns that are never stored), four at a time
    // whatever the alignment; only a bias that starts on an odd element is fetched one by one.
    // (the bias stays as loaded, two bf16 per register, and is widened where it is used)
    float sam[MT], sbv[NT][4][4];
    us4 bv[HAS_BIAS ? NT : 1][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
      sam[i] = BLOCKSCALE ? s_last : p.a_scale[min(m0 + wm * WTM + i * 32 + l32, loc.m_end - 1)];
    if (!BLOCKSCALE) {
      const int n_wave = n0 + wn * WTN;               // first column of the wave's tile
      const int n_left = __builtin_amdgcn_readfirstlane(max(p.N - n_wave, 0));  // columns from there to the edge
      const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(p.b_scale) + ((GROUPED ? (size_t)loc.group * p.N : 0) + n_wave), 0, n_left * 4, 0x00020000);
      const __amdgpu_buffer_rsrc_t bias_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t*>(HAS_BIAS ? p.bias + n_wave : nullptr), 0, HAS_BIAS ? n_left * 2 : 0, 0x00020000);
      // (the check works on whole 4-byte words: with an odd N the last word of the bias is half inside.
      // Fetched four at a time from a 4-byte aligned base that word is read whole: it cannot cross a
      // page, and its upper half belongs to a column that is never stored.)
      const __amdgpu_buffer_rsrc_t bias4_rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint16_t*>(HAS_BIAS ? p.bias + n_wave : nullptr), 0, HAS_BIAS ? ((n_left + 1) & ~1) * 2 : 0, 0x00020000);
      const bool bias_by_four = (reinterpret_cast<uintptr_t>(p.bias) & 3) == 0;  // (n_wave is a multiple of 32)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t col = (uint32_t)(j * 32 + 8 * q + 4 * half);
          const v4f s4 = load_f32x4_checked(s_rsrc, col * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) sbv[j][q][e] = s4[e];
          if (HAS_BIAS) {
            if (bias_by_four) {
              bv[HAS_BIAS ? j : 0][q] = load_u16x4_checked(bias4_rsrc, col * 2);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) bv[HAS_BIAS ? j : 0][q][e] = load_u16_checked(bias_rsrc, (col + e) * 2);
            }
          }
        }
      }
    } else {  // the factors were applied step by step
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) sbv[j][q][e] = 1.0f;
    }
    // pass pp = (32-row block i, column blocks jp*PASS_J ..): finished 16-bit values into half pp & 1.
    // One 32x32 block at a time in three sweeps over its 16 values (row scale, column scale and
    // bias, rounding): neighbouring instructions then do not wait for each other's results.
    auto convert_and_write = [&](int pp) {
      const int i = pp / NJP, jp = pp % NJP;
      uint8_t* const wr_row = row_addr(pp & 1, l32);
#pragma unroll
      for (int jj = 0; jj < PASS_J; ++jj) {
        const int j = jp * PASS_J + jj;
        float t[16], x[16];
        uint32_t packed[8];
#pragma unroll
        for (int v = 0; v < 16; ++v) t[v] = acc[i][j][v] * sam[i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 16; ++v)
          x[v] = HAS_BIAS ? __builtin_fmaf(t[v], sbv[j][v / 4][v % 4], bf16_to_f32(bv[HAS_BIAS ? j : 0][v / 4][v % 4]))
                          : t[v] * sbv[j][v / 4][v % 4];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int v = 0; v < 8; ++v) packed[v] = pack_out_x2(x[2 * v], x[2 * v + 1], OUT_F16);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(v2u*)(wr_row + (((jj * 4 + q) ^ wr_key) * 16) + wr_half) = (v2u){packed[2 * q], packed[2 * q + 1]};
      }
    };
    // The wave's part of the tile as a buffer: origin at its first element, extent = its valid rows
    // (none for a wave that lies past the edge); offsets stay below 2^31 by the host's check of ldc.
    // (opaque: its multiples are worked out here, not in front of the item loop where the epilogues' common ones would be kept)
    uint32_t c_row_bytes = (uint32_t)p.ldc * 2u;
    asm volatile("" : "+s"(c_row_bytes));
    // (pinned to a scalar register: the double clamp exists as a vector instruction only, and a
    // descriptor held in vector registers makes every store a loop)
    const int c_rows = __builtin_amdgcn_readfirstlane(min(max(loc.m_end - (m0 + wm * WTM), 0), WTM));
    uint16_t* const c_wave = p.c + ((size_t)(m0 + wm * WTM) * p.ldc + n0 + wn * WTN);
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(c_wave, 0, (int)((uint32_t)c_rows * c_row_bytes), 0x00020000);
    const uint32_t c_lane = (uint32_t)rd_row * c_row_bytes + (uint32_t)rd_col * 2u;
    constexpr int NP = MT * NJP;
    __builtin_amdgcn_sched_barrier(0);
    convert_and_write(0);
#pragma unroll
    for (int pp = 0; pp < NP; ++pp) {
      const int i = pp / NJP, jp = pp % NJP;
      __builtin_amdgcn_sched_barrier(0);
      v4i rows16[ITERS];
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int r = it * ROWS_PER_READ + rd_row;
        rows16[it] = *(const v4i*)(row_addr(pp & 1, r) + ((rd_chunk ^ key(r)) * 16));
      }
      __builtin_amdgcn_sched_barrier(0);
      if (pp + 1 < NP) convert_and_write(pp + 1);  // under the latency of the reads above
      __builtin_amdgcn_sched_barrier(0);
      const int n = n0 + wn * WTN + jp * PASS_J * 32 + rd_col;
      // (a lane whose columns lie past N is sent past the extent: its stores are dropped)
      const uint32_t c_lane_pass = n < p.N ? c_lane : 0x80000000u;
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int r = it * ROWS_PER_READ + rd_row;
        const v4i out = rows16[it];
        if (STORE != kStoreAny) {
          // lane part (rd_row, rd_col) + scalar part (block row, read round, pass column)
          store_chunk<STORE == kStoreStream>(out, c_rsrc, c_lane_pass,
                                             (uint32_t)(i * 32 + it * ROWS_PER_READ) * c_row_bytes + (uint32_t)(jp * PASS_J * 32 * 2));
        } else {
          store_columns((uint8_t*)c_wave + c_lane + ((uint32_t)(i * 32 + it * ROWS_PER_READ) * c_row_bytes + (uint32_t)(jp * PASS_J * 32 * 2)),
                        out, i * 32 + r < c_rows ? p.N - n : 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- split-K: raw fp32 partial sums of this item to partial[split][m][n]: the lane layout the
  // MFMA leaves (4 consecutive n per lane), one 16-byte buffer store per 4 values (rows of partials start on 4 bytes, which
  // is all it asks for): rows past M fall outside the descriptor's extent, lanes whose 4 columns are not all below N are sent
  // there, and the values go from the accumulators to memory without passing through other registers. Where N is no
  // multiple of 4 the quad at the edge follows value by value. (All of them one by one, as such rows went before, and read one by one by
  // the second pass: 1042x719x10624 30.5 us, now 21.2; 512x2049x8192 34.8, now 25.3; 128x8194x8192 37.2, now 27.0.)
  auto store_partial = [&](int m0, int n0, int split) {
    int lane_e;  // (inside the opaque statement for the reason given in the epilogue)
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_e));
    const int l32 = lane_e & 31, half = lane_e >> 5;
    float* base = p.partial + (size_t)split * p.M * p.N;
    const float last_unit = unit(s_last);
    const uint32_t row_bytes = (uint32_t)p.N * 4u;  // (N*4*128 < 2^31 by the host's check of the workspace plan)
    const int rows = __builtin_amdgcn_readfirstlane(min(max(p.M - (m0 + wm * WTM), 0), WTM));  // (scalar: see the epilogue)
    float* const tile = base + ((size_t)(m0 + wm * WTM) * p.N + n0 + wn * WTN);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(tile, 0, (int)((uint32_t)rows * row_bytes), 0x00020000);
    const uint32_t lane_off = (uint32_t)l32 * row_bytes + (uint32_t)(4 * half) * 4u;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn * WTN + j * 32 + 8 * q + 4 * half;
        const uint32_t lo = n + 3 < p.N ? lane_off : 0x80000000u;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          v4f v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          if (BLOCKSCALE) v = v * last_unit;  // (back from the units of the last step's factor)
          store_f32x4_checked(v, rsrc, lo, (uint32_t)(i * 32) * row_bytes + (uint32_t)(j * 32 + 8 * q) * 4u);
        }
      }
    }
    const int n_left = p.N - (n0 + wn * WTN);  // columns of the wave's tile, or more
    if ((p.N & 3) != 0 && n_left > 0 && n_left < WTN) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = j * 32 + 8 * q + 4 * half;
          if (n < n_left && n + 3 >= n_left) {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              if (i * 32 + l32 < rows) {
                float* dst = tile + ((size_t)(i * 32 + l32) * p.N + n);
#pragma unroll
                for (int e = 0; e < 3; ++e)
                  if (n + e < n_left) dst[e] = BLOCKSCALE ? acc[i][j][4 * q + e] * last_unit : acc[i][j][4 * q + e];
              }
            }
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  int sa = 0, sb = 0;  // stages holding the step being computed
  const uint8_t* cur_a = lds + a_rd_base;  // where this wave reads the step being computed ...
  const uint8_t* cur_b = lds + b_rd_base;
  const uint8_t* nxt_a = LINES ? cur_a + STAGE_A : cur_a;  // ... and the step after it
  const uint8_t* nxt_b = LINES ? cur_b + STAGE_B : cur_b;
  const uint8_t *then_a = nxt_a, *then_b = nxt_b;  // (LINES: and the window after that)
  // What a phase's loads need, put together while the previous phase's last MFMAs run: between
  // the last MFMA of one phase and the first of the next a wave, which issues its instructions in
  // order, should find as little as possible (every scalar instruction there is time the matrix
  // pipe waits once its 64 cycles of cover are used up).
  struct LoadPhase {
    uint32_t lane_off, step_off;
    uint8_t* stage;
  };
  LoadPhase ph_a = {0, 0, lds}, ph_b = {0, 0, lds};  // loads of A (issued in phase [B]) / of B (issued in phase [A])
  auto prepare_b_loads = [&]() {
    ph_b.lane_off = lane_part(b_lane, b_lane_tail, b_lane_end, cb.kt);
    ph_b.step_off = (uint32_t)cb.kt * kStepK + b_src.wave_off;
    ph_b.stage = lds + LDS_B0 + fill_b * STAGE_B;
    next_fill_b();
    ++cb.issued;
  };
  auto prepare_a_loads = [&]() {
    ph_a.lane_off = lane_part(a_lane, a_lane_tail, a_lane_end, ca.kt);
    ph_a.step_off = (uint32_t)ca.kt * kStepK + a_src.wave_off;
    ph_a.stage = lds + fill_a * STAGE_A;
    next_fill_a();
    ++ca.issued;
  };
  constexpr int B_LAST = (B_GROUPS - 1) * NMFMA / B_GROUPS;  // slots of a phase's last load
  constexpr int A_LAST = (A_GROUPS - 1) * NMFMA / A_GROUPS;
  // One K step. READ_NEXT: fetch the first-half fragments of the following step behind the
  // second-half MFMAs (left out on a tile's last step, so that the epilogue has those
  // registers; the fragments are then read after it).
  // PLAIN: neither load cursor leaves its work item in this step.
  // slots behind which the next phase is prepared (two, so that neither holds more scalar work than
  // an MFMA covers)
  constexpr int PREP_T = NMFMA / 2, PREP_T2 = NMFMA >= 8 ? NMFMA / 2 + 1 : NMFMA / 2;
  auto step = [&](auto first_tag, auto read_next_tag, auto plain_tag, auto stream_tag) {
    constexpr bool FIRST = decltype(first_tag)::value;
    constexpr bool READ_NEXT = decltype(read_next_tag)::value;
    if (BLOCKSCALE) {  // (fetched from the lanes that hold them during the previous step, or at the item's start)
      s_cur = s_pend;    // ratio that brought the accumulators to this step
      s_pend = n_pend;   // ratio to the next step (applied in phase [B])
      s_last = n_last;   // this step's factor: what the epilogue multiplies by after the last step
      if (ANY_FACTORS) scales = n_scales;
    }

    // [A] MFMAs on x* (first K half of this step). Behind them, one per MFMA: the LDS reads
    //     of the second half (-> y*), and behind every other one a global->LDS load of
    //     B(g+DIST) into the B stage released at the previous barrier. The fences pin this
    //     interleaving: every wave-level memory instruction hides behind an MFMA, and the
    //     load queue never holds more than the matrix pipe can cover. Half way through, phase [B]
    //     is prepared; behind the last loads the B cursor moves on. Behind the phase's last MFMA
    //     there is nothing but the wait and the barrier, which its 64 cycles cover.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NMFMA; ++t) {
      mfma_one(xa, xb, t, FIRST);
      __builtin_amdgcn_sched_barrier(0);  // the MFMA goes first: what follows is issued under its cover
      // (the last block of the previous step is brought to this step's units here, under the first MFMA's cover)
      if (BLOCKSCALE && !FIRST && t == 0) fold_block(NMFMA - 1, s_cur);
#pragma unroll
      for (int l = 0; l < B_GROUPS; ++l)
        if (l * NMFMA / B_GROUPS == t)
          load_group(stream_tag, b_src, ph_b.lane_off, ph_b.step_off, l, ph_b.stage);
#pragma unroll
      for (int u = t * RPS; u < (t + 1) * RPS; ++u)
        if (u < NREAD) read_one(ya, yb, cur_a, nxt_a, cur_b, nxt_b, 1, u);
      if (t == B_LAST) advance_b(plain_tag);
      if (t == PREP_T) prepare_a_loads();
      if (BLOCKSCALE && t == PREP_T) {
        n_pend = lane_value(rt, STREAM_B && k_steps == 1 ? 0 : kt_c + 2);
        n_last = lane_value(sc, kt_c + 1);
        if (ANY_FACTORS) n_scales = factor_scales(n_last);
      }
      if (t == PREP_T2) {
        sa = (sa + 1 == kStagesA) ? 0 : sa + 1;
        sb = (sb + 1 == kStagesB) ? 0 : sb + 1;
        if constexpr (LINES) {  // (this phase's reads, which end in front of this slot or behind it, have the next window's place in nxt_*)
          then_a = lds + a_rd_base + (sa + 1 == kStagesA ? 0 : sa + 1) * STAGE_A;
          then_b = lds + b_rd_base + (sb + 1 == kStagesB ? 0 : sb + 1) * STAGE_B;
        } else {
          nxt_a = lds + a_rd_base + sa * STAGE_A;
          nxt_b = lds + b_rd_base + sb * STAGE_B;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }

    // own loads of A(g+1) and B(g+1) have landed (the younger B(g+2) .. B(g+DIST) and
    // A(g+2) .. A(g+DIST-1) may still be in flight); past the barrier everyone's have, and
    // every wave is done reading this step's stages
    wait_loads_and_barrier<(DIST - 1 - AHEAD) * B_GROUPS + (DIST - 2 - AHEAD) * A_GROUPS>();

    // [B] MFMAs on y* (second K half); behind them the loads of A(g+DIST) into the A stage just
    //     released and the LDS reads of step g+1's first half (-> x*; at the end of a tile
    //     these already belong to the next tile)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NMFMA; ++t) {
      mfma_one(ya, yb, t, false);
      __builtin_amdgcn_sched_barrier(0);
      // block t-1 has had its last MFMA of this step: into the next step's units, under this MFMA's cover
      if (BLOCKSCALE && READ_NEXT && t >= 1) fold_block(t - 1, s_pend);
#pragma unroll
      for (int l = 0; l < A_GROUPS; ++l)
        if (l * NMFMA / A_GROUPS == t) load_group(std::false_type{}, a_src, ph_a.lane_off, ph_a.step_off, l, ph_a.stage);
#pragma unroll
      for (int u = t * RPS; u < (t + 1) * RPS; ++u)
        if (READ_NEXT && u < NREAD) read_one(xa, xb, nxt_a, then_a, nxt_b, then_b, 0, u);
      if (t == A_LAST) advance_a(plain_tag);
      if (t == PREP_T) {
        prepare_b_loads();
        cur_a = nxt_a;
        cur_b = nxt_b;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LINES) {
      nxt_a = then_a;
      nxt_b = then_b;
    }
    if (BLOCKSCALE) kt_c = STREAM_B && kt_c + 1 == k_steps ? 0 : kt_c + 1;
  };
  auto read_first_half = [&]() {
#pragma unroll
    for (int u = 0; u < NREAD; ++u) read_one(xa, xb, cur_a, nxt_a, cur_b, nxt_b, 0, u);
  };

  // Item loop around the K loop. The first step of an item is its own copy of the step code
  // whose first-half MFMAs start from zero: the accumulators then have one live range per
  // item (defined there, dead after the epilogue) and need no clearing or copying between
  // items.
  prepare_b_loads();  // of the first step's phase [A]
  for (int c_item = walk.slot; c_item < walk.chunk_len; c_item += walk.slots) {
    const int c_split = item_split(c_item);
    const int n_steps = split_end(c_split) - split_begin(c_split);
    if (BLOCKSCALE) {
      const TileLoc loc = locate(walk_c, c_item);
      load_block_scales(loc, ANY_FACTORS ? split_begin(c_split) : 0);
      kt_c = ANY_FACTORS ? 0 : first_step(loc, split_begin(c_split), n_steps);
      n_pend = lane_value(rt, kt_c + 1);
      n_last = lane_value(sc, kt_c);
      if (ANY_FACTORS) n_scales = factor_scales(n_last);
    }
    // step k loads for step k + DIST and then moves the cursors to step k + DIST + 1, which is still this item's for
    // k < n_steps - DIST - 1. (Text and not a function: as a lambda around `step` it cost every grouped launch 1-2 %, 282x1536x1024
    // in 30 groups 26.7 -> 27.1 us.)
#define MI355X_ALL_STEPS(stream_tag)                                                                                           \
  if (n_steps == 1) {                                                                                                          \
    step(std::true_type{}, std::false_type{}, std::false_type{}, stream_tag);                                                  \
  } else {                                                                                                                     \
    step(std::true_type{}, std::true_type{}, std::false_type{}, stream_tag);                                                   \
    int k = 1;                                                                                                                 \
    for (; k < n_steps - DIST - 1; ++k) step(std::false_type{}, std::true_type{}, std::true_type{}, stream_tag);               \
    for (; k < n_steps - 1; ++k) step(std::false_type{}, std::true_type{}, std::false_type{}, stream_tag);                     \
    step(std::false_type{}, std::false_type{}, std::false_type{}, stream_tag);                                                 \
  }
    if constexpr (STREAM_BY_GROUP) {  // (the cursor of B is a few steps ahead, as a rule in this item; the policy is a hint either way)
      if (b_streams) {
        MI355X_ALL_STEPS(std::true_type{})
      } else {
        MI355X_ALL_STEPS(std::false_type{})
      }
    } else {
      MI355X_ALL_STEPS((std::integral_constant<bool, STREAM_B && !OFF_LINES>{}))
    }
#undef MI355X_ALL_STEPS
    {
      const TileLoc loc = locate(walk_c, c_item);
      if (EPI == kEpiPartial) {
        store_partial(loc.m0, loc.n0, c_split);
      } else {
        // sb already names the next step's stage; the one before it held this tile's last step
        uint8_t* free_b = lds + LDS_B0 + ((sb + kStagesB - 1) % kStagesB) * STAGE_B;
        // (kind of store and output type are compile-time properties of the epilogue code: one uniform branch per tile)
        auto finish = [&](auto store_tag) {
          // (Grouped and block-scaled calls have one output type. With code for the other beside it grouped launches of few steps took 1.6 %
          // longer on average, 1953x896x768 in 55 groups 36.9 us, without 35.7. With a K tail it stays: without it the compiler keeps the lane
          // parts of the loads in scratch memory, 2881x5632x3904 in 5 groups 92.7 -> 96.3.)
          if constexpr ((GROUPED && !KTAIL) || BLOCKSCALE) epilogue(loc, store_tag, std::false_type{}, free_b);
          else if (p.out_f16) epilogue(loc, store_tag, std::true_type{}, free_b);
          else epilogue(loc, store_tag, std::false_type{}, free_b);
        };
        // (no kStoreKeep here: its code costs all other launches 1-2 %, up to 5 where a tile has few steps)
        // (Without the hint 256x256 tiles with a K tail kept values of the other form in registers and the lane parts of the loads in scratch
        // memory, where a read waits for every load in flight: 8192x4608x2064 in 4 groups 84.2 -> 88.4 us, 4096x8192x4112 114.2 -> 116.6.)
        if (__builtin_expect(p.store == kStoreStream, true)) finish(std::integral_constant<int, kStoreStream>{});
        else finish(std::integral_constant<int, kStoreAny>{});
      }
    }
    read_first_half();  // of the next item's first step (landed before this item's last barrier)
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // the trailing dummy loads must land before LDS is released
  if (p.stamps && threadIdx.x == 0) {
    unsigned long long* out = p.stamps + 4 * (size_t)blockIdx.x;
    out[0] = stamp_cycles;
    out[1] = __builtin_readcyclecounter();
    out[2] = stamp_ticks;
    out[3] = __builtin_amdgcn_s_memrealtime();
  }
}

// ------------------------------------------------------------------------------------
// Block-scaled kernel for shapes that fill the chip with 256x256 tiles: two groups of four waves take turns.
//
// The accumulators are kept in units of the current K block's factor (see the tiled kernel's BLOCKSCALE
// form): one multiply per accumulator and step on the vector ALU, which reaches accumulators in
// ordinary registers only. A 256x256 tile therefore needs eight waves (128x64 each: 128 accumulators), two per
// SIMD. Each wave alternates between a memory phase (all of a step's operand fragments from LDS, the
// rescaling) and a matrix phase (the step's 16 MFMAs); waves 4..7 run one phase behind waves 0..3, and
// a SIMD hosts one wave of either group, so one of its waves feeds the matrix pipe while the other one
// reads and rescales. A barrier ends every phase.
//
//   phase 2k      waves 0..3: memory(k)    waves 4..7: matrix(k-1)     everyone loads A(k+1)
//   phase 2k + 1  waves 0..3: matrix(k)    waves 4..7: memory(k)       everyone loads B(k+2), then waits for
//                                                                       its own loads of A(k+1) and B(k+1)
//
// LDS: two stages of A, three of B (32 KB each), as in the plain 256x256 tile. B(k+2) goes where B(k-1) was,
// last read in phase 2k-1; A(k+1) where A(k-1) was, last read in the same phase.
//
// What bounds it: 8192^3 416 us (2.64 PFLOP/s), with the rescaling taken out 366, which is what the plain 256x256 tile
// takes; the 128x128 form 542. The eight waves read 192 KB of fragments from LDS per step (four waves of
// 128x128 would read 128, but have no registers the multiplies can reach), beside the 64 KB that arrive there.
// Measured on the way: the same waves in step with each other (the tiled kernel's schedule) 464-470 us; this one with
// the cursors' scalar work in the memory phase 430; all 128 multiplies in the memory phase 426, all behind the
// MFMAs 447; the loads in front of the fragment reads instead of behind them 427.
// ------------------------------------------------------------------------------------
constexpr int kBlockTile = 256, kBlockWaves = 8;
constexpr size_t kBlockLdsBytes = tiled_lds_bytes(kBlockTile, kBlockTile);

template <bool KTAIL>
__global__ __launch_bounds__(kBlockWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_block_kernel(GemmParams p) {
  constexpr int BT = kBlockTile, NW = kBlockWaves, MT = 4, NT = 2;  // wave tile: 4 x 2 blocks of 32x32
  constexpr int STAGE = BT * kStepK;
  constexpr int LDS_B0 = 2 * STAGE;
  constexpr int GROUPS = BT / 8 / NW;  // 8-row groups of A, and of B, a wave fetches per step
  fetch_arguments_now(p);
  fetch_tiled_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool lead = wave < NW / 2;         // waves 0..3
  const int wm = (wave >> 1) & 1, wn = (wave & 1) * 2 + (wave >> 2);
  const int l32 = lane & 31, half = lane >> 5;

  const TileWalk walk = make_walk(p.tiles_m * p.tiles_n);
  if (walk.slot >= walk.chunk_len) return;  // uniform over the workgroup
  const int k_full = p.K / kStepK, k_tail = p.K - k_full * kStepK;
  const int k_steps = k_full + (k_tail ? 1 : 0);
  const int total_steps = ((walk.chunk_len - walk.slot + walk.slots - 1) / walk.slots) * k_steps;
  auto tile_of = [&](int li, int& m0, int& n0) {
    int tm, tn;
    tile_coords(walk.chunk_begin + li, p.tiles_m, p.tiles_n, p.div_group_mul, p.div_group_shift, tm, tn);
    m0 = tm * BT;
    n0 = tn * BT;
  };

  // ---- load side: one cursor per operand. `mem` is the operand a wave loads in its memory phases, `mat` the one
  // it loads in its matrix phases: A and B for waves 0..3, the other way round for waves 4..7.
  struct Cursor {
    bool is_a;
    int item, kt, issued, stage;
    const uint8_t* base;
    uint32_t extent, wave_off, group_stride, lane_off, lane_off_tail;
  };
  const int ld_row = lane >> 3, ld_pc = lane & 7;
  const uint32_t chunk = (uint32_t)((ld_pc ^ swz128(wave * 8 + ld_row)) * kChunk);  // (a wave's groups share their parity)
  auto enter_item = [&](Cursor& c) {
    int m0, n0;
    tile_of(c.item, m0, n0);
    const int row0 = c.is_a ? m0 : n0, rows = min((c.is_a ? p.M : p.N) - row0, BT);
    const long ld = c.is_a ? p.lda : p.ldb;
    const uintptr_t b = reinterpret_cast<uintptr_t>(c.is_a ? p.a : p.b) + (size_t)row0 * ld;
    c.base = reinterpret_cast<const uint8_t*>(
        ((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
        (uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b));
    c.extent = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)rows * (uint32_t)ld));
    c.kt = 0;
  };
  auto make_cursor = [&](bool is_a) {
    Cursor c;
    c.is_a = is_a;
    c.item = walk.slot;
    c.issued = 0;
    c.stage = 0;
    const uint32_t ld = (uint32_t)(is_a ? p.lda : p.ldb);
    c.wave_off = 8u * (uint32_t)wave * ld;
    c.group_stride = 8u * NW * ld;
    c.lane_off = __umul24((uint32_t)ld_row, ld) + chunk;
    c.lane_off_tail = (int)chunk < k_tail ? c.lane_off : 0x80000000u;  // past K: outside every extent, zeros arrive
    enter_item(c);
    return c;
  };
  auto load_one = [&](const Cursor& c, int i) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(c.base), 0, (int)c.extent, 0x00020000);
    uint8_t* const stage = lds + (c.is_a ? 0 : LDS_B0) + c.stage * STAGE;
    load_chunk_to_lds<false>(rsrc, stage + (wave + NW * i) * 1024, KTAIL && c.kt >= k_full ? c.lane_off_tail : c.lane_off,
                             (uint32_t)c.kt * kStepK + c.wave_off + (uint32_t)i * c.group_stride);
  };
  // past the last step the last one is fetched again, into a stage nobody reads any more
  auto advance = [&](Cursor& c) {
    c.stage = c.stage + 1 == (c.is_a ? 2 : 3) ? 0 : c.stage + 1;
    if (++c.issued >= total_steps) return;
    if (++c.kt == k_steps) {
      c.item += walk.slots;
      enter_item(c);
    }
  };
  Cursor c_mem = make_cursor(lead), c_mat = make_cursor(!lead);
  auto load_step = [&](Cursor& c) {
#pragma unroll
    for (int i = 0; i < GROUPS; ++i) load_one(c, i);
    advance(c);
  };

  // ---- factors: one per wave and step; a factor of zero (a block of zeros) counts as 2^-60
  scalar_floats sa_row = nullptr, sb_row = nullptr;
  auto factor = [&](float a, float b) {
    const float f = a * b;
    return f == 0.0f ? 0x1p-60f : f;
  };

  v16f acc[MT][NT];
  v4i fa[MT][4], fb[NT][4];
  int rd[4];  // logical chunks 4*half + 0..3 of row l32
#pragma unroll
  for (int c = 0; c < 4; ++c) rd[c] = l32 * kStepK + (((4 * half + c) ^ swz128(l32)) * kChunk);
  const int a_rows = wm * 128 * kStepK, b_rows = LDS_B0 + wn * 64 * kStepK;
  int sa = 0, sb = 0;  // stages of the step being computed
  // factor of the step whose products the accumulators are in units of, of the step after it, and their ratio
  float s_now = 1.0f, s_next = 1.0f, ratio = 1.0f;

  // A wave issues an instruction every four cycles at best, so a phase of 1024 cycles (its 16 MFMAs, or the other
  // group's) has room for 256 instructions: the memory phase is kept to the loads, the fragment reads and as much
  // of the rescaling as fits beside them; the last FOLD_LATE blocks are rescaled and everything scalar is done
  // behind the MFMAs of the matrix phase.
  constexpr int FOLD_LATE = 3, READS_PER_BLOCK = 8;
  auto rescale = [&](int t, int v0, int v1) {
    v16f& block = acc[t / NT][t % NT];
#pragma unroll
    for (int v = v0; v < v1; ++v) block[v] *= ratio;
    asm volatile("" : "+v"(block));  // here: the compiler would sink the multiplies to the MFMAs
  };
  auto memory_phase = [&](auto first_tag) {
    constexpr bool FIRST = decltype(first_tag)::value;
    __builtin_amdgcn_sched_barrier(0);
    const uint8_t* rows_a = lds + sa * STAGE + a_rows;
    const uint8_t* rows_b = lds + sb * STAGE + b_rows;
#pragma unroll
    for (int t = 0; t < MT * NT; ++t) {
#pragma unroll
      for (int u = READS_PER_BLOCK * t; u < READS_PER_BLOCK * (t + 1); ++u) {
        const int c = u / (MT + NT), f = u % (MT + NT);
        if (u >= 4 * (MT + NT)) continue;
        if (f < NT) fb[f < NT ? f : 0][c] = *(const v4i*)(rows_b + f * 32 * kStepK + rd[c]);
        else fa[f < NT ? 0 : f - NT][c] = *(const v4i*)(rows_a + (f - NT) * 32 * kStepK + rd[c]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (!FIRST && t < MT * NT - FOLD_LATE) rescale(t, 0, 16);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < GROUPS; ++i) load_one(c_mem, i);
    if (!lead) wait_loads<GROUPS>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments are in registers, the stage may be written
    __builtin_amdgcn_s_barrier();
  };
  auto matrix_phase = [&](auto first_tag, int kt) {
    constexpr bool FIRST = decltype(first_tag)::value;
    const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto join = [](const v4i& lo, const v4i& hi) { return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}; };
    float next_a = 0.f, next_b = 0.f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2 * MT * NT; ++t) {
      const int h = t / (MT * NT), i = t / NT % MT, j = t % NT;
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(join(fb[j][2 * h], fb[j][2 * h + 1]), join(fa[i][2 * h], fa[i][2 * h + 1]),
                                                                  FIRST && h == 0 ? zero : acc[i][j], 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (t == 0) {
        const int kn = min(kt + 1, k_steps - 1);
        next_a = sa_row[kn];
        next_b = sb_row[kn];
        sa = sa ^ 1;
        sb = sb == 2 ? 0 : sb + 1;
      }
      if (!FIRST && FOLD_LATE && t < 2 * FOLD_LATE) rescale(MT * NT - FOLD_LATE + t / 2, 8 * (t & 1), 8 * (t & 1) + 8);
      if (t >= 5 && t < 5 + GROUPS) load_one(c_mat, t - 5);
      if (t == 5 + GROUPS) advance(c_mat);
      if (t == 6 + GROUPS) advance(c_mem);
      if (t == 13) {
        s_now = FIRST ? s_now : s_next;
        s_next = factor(next_a, next_b);
        ratio = s_now / s_next;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (lead) wait_loads<GROUPS>();
    __builtin_amdgcn_s_barrier();
  };

  // ---- epilogue: each 32-row block of the wave's tile is turned through LDS as 16-bit values, in the four
  // 1 KB groups this wave fetches itself of the B stage the tile's last step was read from
  auto epilogue = [&](int m0, int n0, uint8_t* table, auto store_tag) {
    constexpr int STORE = decltype(store_tag)::value;
    int lane_e;  // (an opaque copy: see the tiled kernel's epilogue)
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_e));
    const int row = lane_e & 31, hi = lane_e >> 5, rd_row = lane_e >> 3, rd_c = lane_e & 7;
    auto at = [&](int r, int c) { return table + (wave + NW * (r >> 3)) * 1024 + (r & 7) * 128 + ((c ^ (r & 7)) * 16); };
    const int m_wave = m0 + wm * 128, n_wave = n0 + wn * 64;
    uint32_t c_row_bytes = (uint32_t)p.ldc * 2u;
    asm volatile("" : "+s"(c_row_bytes));
    const int c_rows = __builtin_amdgcn_readfirstlane(min(max(p.M - m_wave, 0), 128));
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.c + ((size_t)m_wave * p.ldc + n_wave), 0,
                                                                            (int)((uint32_t)c_rows * c_row_bytes), 0x00020000);
    const int n = n_wave + rd_c * 8;
    const uint32_t c_lane = n < p.N ? (uint32_t)rd_row * c_row_bytes + (uint32_t)rd_c * 16u : 0x80000000u;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(v2u*)(at(row, j * 4 + q) + hi * 8) = (v2u){pack_bf16x2(acc[i][j][4 * q] * s_now, acc[i][j][4 * q + 1] * s_now),
                                                       pack_bf16x2(acc[i][j][4 * q + 2] * s_now, acc[i][j][4 * q + 3] * s_now)};
      __builtin_amdgcn_sched_barrier(0);
      v4i out[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) out[it] = *(const v4i*)at(it * 8 + rd_row, rd_c);
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        if (STORE != kStoreAny) {
          store_chunk<STORE == kStoreStream>(out[it], c_rsrc, c_lane, (uint32_t)(i * 32 + it * 8) * c_row_bytes);
        } else {
          const int r = i * 32 + it * 8 + rd_row;
          store_columns((uint8_t*)(p.c + ((size_t)(m_wave + r) * p.ldc + n)), out[it], r < c_rows ? p.N - n : 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- A(0) B(0) B(1) in flight; step 0 landed at the first barrier
  if (lead) {
    load_step(c_mem);
    load_step(c_mat);
    load_step(c_mat);
  } else {
    load_step(c_mat);
    load_step(c_mem);
    load_step(c_mem);
  }
  wait_loads<GROUPS>();
  __builtin_amdgcn_s_barrier();
  if (!lead) {  // the phase the second group runs behind: it loads its share of A(1) (its matrix phases' operand)
    load_step(c_mat);
    __builtin_amdgcn_s_barrier();
  }
  for (int item = walk.slot; item < walk.chunk_len; item += walk.slots) {
    int m0, n0;
    tile_of(item, m0, n0);
    // the scale block of this wave's tile (clamped for waves that lie past the matrix edge)
    sa_row = (scalar_floats)(p.a_scale + (size_t)(min(m0 + wm * 128, p.M - 1) / 128) * k_steps);
    sb_row = (scalar_floats)(p.b_scale + (size_t)(min(n0 + wn * 64, p.N - 1) / 128) * k_steps);
    s_now = factor(sa_row[0], sb_row[0]);
    memory_phase(std::true_type{});
    matrix_phase(std::true_type{}, 0);
    for (int kt = 1; kt < k_steps; ++kt) {
      memory_phase(std::false_type{});
      matrix_phase(std::false_type{}, kt);
    }
    uint8_t* table = lds + LDS_B0 + (sb == 0 ? 2 : sb - 1) * STAGE;
    if (p.store == kStoreStream) epilogue(m0, n0, table, std::integral_constant<int, kStoreStream>{});
    else if (p.store == kStoreKeep) epilogue(m0, n0, table, std::integral_constant<int, kStoreKeep>{});
    else epilogue(m0, n0, table, std::integral_constant<int, kStoreAny>{});
  }
  if (lead) __builtin_amdgcn_s_barrier();  // the second group's last phase
  wait_loads<0>();  // (loads into LDS land before it is released)
}

constexpr int kFinalizeRows = 4;

// Second pass of a split-K launch: sums the splits' partials in a fixed order (results do not
// depend on scheduling), applies the scales and the bias and rounds to bf16. One thread per
// 4 consecutive columns of ROWS consecutive rows.
// Bound by the partial planes' bytes where it is more than a round of workgroups, which needs loads in flight: every
// row's loads of two splits (one row: four) are issued before the first is used. (One row a thread, a 64-bit division for its place and
// two splits' loads one behind the other: 1024x8192, two splits, 22.6 us = 3.7 TB/s; with four
// rows 15.6 = 5.4 TB/s.)
template <int ROWS>
__device__ __forceinline__ void splitk_finalize(const GemmParams& p) {
  const long quads_per_row = (p.N + 3) / 4;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= quads_per_row * ((p.M + ROWS - 1) / ROWS)) return;
  // (the division's factors belong to a quad index below 2^31; larger results divide in 64 bits)
  const long row_group = p.div_group_mul ? (long)fast_div((int)idx, p.div_group_mul, p.div_group_shift) : idx / quads_per_row;
  const int m0 = (int)row_group * ROWS;
  const int n = (int)(idx - row_group * quads_per_row) * 4;
  const size_t plane = (size_t)p.M * p.N;
  // (the quad at the edge reads the row's last four values and moves its own down: read one by one, split after split, they took
  // longer than all the others together, 2x707x25888 in sixteen parts 18.9 -> 20.0 us in all)
  const int first = p.N >= 4 ? min(n, p.N - 4) : n, shift = n - first;
  const float* src[ROWS];
  float sa[ROWS], sb[4];
  uint16_t bias[4] = {0, 0, 0, 0};
  v4f sum[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int m = min(m0 + i, p.M - 1);  // (rows past the last one read it again)
    src[i] = p.partial + (size_t)m * p.N + first;
    sa[i] = p.a_scale ? p.a_scale[m] : 1.0f;  // fetched beside the partial sums, not after them
    sum[i] = (v4f){0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) sb[e] = p.b_scale ? p.b_scale[min(n + e, p.N - 1)] : 1.0f;
  if (p.bias)
#pragma unroll
    for (int e = 0; e < 4; ++e) bias[e] = p.bias[min(n + e, p.N - 1)];
  if (p.N >= 4) {  // (a row of partials starts on any 4 bytes)
    // added in split order, as the scalar form does
    auto add = [&](int s, auto count) {
      constexpr int COUNT = decltype(count)::value;
      v4f part[COUNT][ROWS];
#pragma unroll
      for (int u = 0; u < COUNT; ++u)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) part[u][i] = __builtin_nontemporal_load((const v4f_by4*)(src[i] + (s + u) * plane));
#pragma unroll
      for (int u = 0; u < COUNT; ++u)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) sum[i] += part[u][i];
    };
    int s = 0;
    constexpr int BATCH = ROWS > 1 ? 2 : 4;
    for (; s + BATCH <= p.splits; s += BATCH) add(s, std::integral_constant<int, BATCH>{});
    const int rest = p.splits - s;
    if (BATCH > 3 && rest == 3) add(s, std::integral_constant<int, 3>{});
    else if (BATCH > 2 && rest == 2) add(s, std::integral_constant<int, 2>{});
    else if (rest == 1) add(s, std::integral_constant<int, 1>{});
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      if (shift & 1) sum[i] = (v4f){sum[i][1], sum[i][2], sum[i][3], 0.f};
      if (shift & 2) sum[i] = (v4f){sum[i][2], sum[i][3], 0.f, 0.f};
    }
  } else {
    for (int s = 0; s < p.splits; ++s) {
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int e = 0; e < 3; ++e)
          if (n + e < p.N) sum[i][e] += src[i][s * plane + e];
    }
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (m0 + i >= p.M) break;
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = sum[i][e] * sa[i];
      r[e] = p.bias ? __builtin_fmaf(t, sb[e], bf16_to_f32(bias[e])) : t * sb[e];
    }
    const uint32_t lo = pack_out_x2(r[0], r[1], p.out_f16), hi = pack_out_x2(r[2], r[3], p.out_f16);
    uint16_t* dst = p.c + (size_t)(m0 + i) * p.ldc + n;
    if (n + 3 < p.N) {
      *(v2u_any*)dst = (v2u){lo, hi};
    } else {
      dst[0] = (uint16_t)lo;
      if (n + 1 < p.N) dst[1] = (uint16_t)(lo >> 16);
      if (n + 2 < p.N) dst[2] = (uint16_t)hi;
    }
  }
}
__global__ __launch_bounds__(256) void splitk_finalize_kernel(GemmParams p) {
  fetch_arguments_now(p);
  fetch_tiled_arguments_now(p);
  splitk_finalize<1>(p);
}
__global__ __launch_bounds__(256) void splitk_finalize_rows_kernel(GemmParams p) {
  fetch_arguments_now(p);
  fetch_tiled_arguments_now(p);
  splitk_finalize<kFinalizeRows>(p);
}

// ------------------------------------------------------------------------------------
// Generic kernels: operands the other families cannot take (K, lda or ldb not a multiple of 16,
// A or B not 16-byte aligned, leading dimensions beyond a buffer descriptor's range). Rows start at
// any byte. The streaming form loads a lane's 16 bytes where they lie (one instruction on this chip; the pieces of a
// row lie across two cache lines more often than not), the tiles in whole dwords, and the last chunk of a row is put
// together from its last 16 bytes: nothing outside the dwords that a row's K bytes lie in is ever read.
//
// The products run on the 16-bit matrix instructions with the codes widened to binary16, which is
// exact (e4m3fn reaches from 2^-9 to 448), and f32 accumulation that is as accurate as a chain of f32
// multiply-adds (measured over K = 1024 standard normal codes: 4e-8 of the result's norm for both,
// 1.5e-5 for the fp8 matrix instructions, which align a group of products before they add). One
// conversion instruction of 8 cycles widens two codes, and over many rounds of tiles the conversions are what bounds them (4096x8192x2047:
// 810 TFLOP/s, 0.32 of the 16-bit matrix rate). Against byte loads and f32 multiply-adds on the
// vector ALU, which this family was at first, 517x3000x1041 took 212 us.
// ------------------------------------------------------------------------------------
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef uint16_t u16_any __attribute__((aligned(1)));

// bytes [k, k + 16) of a row of K bytes; those at or past K count as zero
__device__ __forceinline__ v4i load16_any(const uint8_t* row, int k, int K) {
  if (k + kChunk <= K) return *(const v4i_any*)(row + k);
  uint64_t lo = 0, hi = 0;
  if (K >= kChunk) {  // the row's last 16 bytes, moved down to where the chunk wants them
    if (k < K) {
      const v4i x = *(const v4i_any*)(row + K - kChunk);
      lo = (uint32_t)x[0] | ((uint64_t)(uint32_t)x[1] << 32);
      hi = (uint32_t)x[2] | ((uint64_t)(uint32_t)x[3] << 32);
      const int n = 8 * (k + kChunk - K);  // 8 .. 120
      lo = n < 64 ? (lo >> n) | (hi << (64 - n)) : hi >> (n & 63);
      hi = n < 64 ? hi >> n : 0;
    }
  } else if (k == 0) {  // the whole row, in pieces of 8, 4, 2 and 1 bytes
    int at = K & 8, bits = 0;
    uint64_t rest = 0;
    if (K & 4) {
      rest = *(const u32_any*)(row + at);
      at += 4;
      bits = 32;
    }
    if (K & 2) {
      rest |= (uint64_t)*(const u16_any*)(row + at) << bits;
      at += 2;
      bits += 16;
    }
    if (K & 1) rest |= (uint64_t)row[at] << bits;
    lo = rest;
    if (K & 8) {
      const v2u_any first = *(const v2u_any*)row;
      lo = first[0] | ((uint64_t)first[1] << 32);
      hi = rest;
    }
  }
  return (v4i){(int)(uint32_t)lo, (int)(uint32_t)(lo >> 32), (int)(uint32_t)hi, (int)(uint32_t)(hi >> 32)};
}

// eight e4m3fn codes in two registers -> binary16 (exact; NaN codes become NaN)
__device__ __forceinline__ v8h e4m3fn_to_f16x8(int lo, int hi) {
#if defined(__HIP_DEVICE_COMPILE__)
  const v2h a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false), b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true);
  const v2h c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false), d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true);
  return (v8h){a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
#else
  return (v8h){};
#endif
}

// Generic form for more than 64 rows: BM x BN tile per workgroup of WAVES_M x WAVES_N x WAVES_K waves, K in 128-byte steps.
// Global memory -> registers (DEPTH steps ahead) -> LDS in the tiled kernel's swizzled layout, two stages,
// one barrier per step; a fragment's codes are widened as they are read from LDS. The partial step
// at the end of K is multiplied first, so that the loop over whole steps has no conditional loads (its wait
// counts are then exact and DEPTH steps stay in flight).
//
// What bounds it over many rounds of tiles is the vector ALU, which widens every fragment in each wave that multiplies it (an instruction of 8 cycles
// for two codes), beside MFMAs that it hardly overlaps with: of the 340000 cycles of 4096x8192x2047 on 128x128 tiles a SIMD converts for 133000, has
// 57000 of other vector instructions and 131000 of MFMAs. One round on short rows waits instead, for its first data and at its few barriers: waves of
// 517x3000x1041 are in s_waitcnt for half of their time. With 2x2 waves of 32x32 on a 64x64 tile it is 64 conversions a step and wave beside 8 MFMAs of
// 32 cycles. Waves that share out a step's K
// instead (WAVES_K) widen nothing twice and have wave tiles of twice the size, for one exchange of the sums at the end: 517x3000x1041 with
// its bias 16.7 -> 14.3 us, 517x3000x4113 36.6 -> 28.4, 1000x3000x4111 52.9 -> 39.4. Where tiles of 64x64 a wave are several rounds
// of the chip the exchange costs more than it saves and the waves share out the tile (4096x8192x2047 171 us, with WAVES_K 191).
//
// The bytes are fetched in whole dwords and moved into place on their way into LDS (load rates a CU from L2, 128-byte pieces of 256 rows: rows on
// 16 or 4 bytes 83 bytes/ns, on 2 bytes 64, on odd ones 49). The last dword of the chunk in front, which a row that starts
// off the dwords needs too, is in the lane beside it or was in the step before (a load of its own for it cost more than it gained:
// 128x8192x8191 33.4 -> 43.0 us). Without that 1000x3000x4111 takes 47.9 us, 517x3000x1041 15.6.
// DWORDS: rows that all start on a dword lie in place already: their chunks go into LDS as they are (64x64 tiles 0.89 of the time on average with waves that
// share out K and 0.95 with waves that share out the tile, 128x64 0.97 and 0.90, 128x128 0.98 and 0.96; 423 shapes. Moved like the others, 152x24457x820 took
// 26.4 us where 22.4 are had).
constexpr size_t any_stage_bytes(int BM, int BN, int WAVES_K, int WAVES_MN) {
  const size_t stages = (size_t)2 * (BM + BN) * kStepK, sums = (size_t)WAVES_MN * WAVES_K * (WAVES_K - 1) * 32 * 32 * 4;
  return stages > sums ? stages : sums;
}
constexpr size_t any_lds_bytes(int BM, int BN, int WAVES_K, int WAVES_MN) { return any_stage_bytes(BM, BN, WAVES_K, WAVES_MN) + (size_t)(BM + 2 * BN) * 4; }

// PARTIAL: K in p.splits parts of p.steps_per_split steps, each an item of its own that leaves its sums in its plane of p.partial
// for the second pass. The last part has the partial step.
template <int BM, int BN, int WAVES_M, int WAVES_N, int WAVES_K, int DEPTH, bool PARTIAL, bool DWORDS>
__global__ __launch_bounds__(WAVES_M* WAVES_N* WAVES_K * 64) void gemm_any_kernel(GemmParams p) {
  constexpr int THREADS = WAVES_M * WAVES_N * WAVES_K * 64;
  constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N, MT = WTM / 32, NT = WTN / 32;
  constexpr int STAGE = (BM + BN) * kStepK;  // A's rows, then B's
  constexpr int ROWS = THREADS / 8;          // rows a round of the workgroup's lanes fetches, eight lanes each
  constexpr int LA = BM / ROWS, LOADS = (BM + BN) / ROWS;  // chunks of A, and of both, a lane fetches per step
  constexpr int PAIRS = 4 / WAVES_K;         // pairs of chunks of a row's eight that a wave multiplies, one for each half of its lanes
  constexpr int OWN = MT * NT / WAVES_K;     // 32x32 blocks that a wave finishes
  static_assert(BM % ROWS == 0 && BN % ROWS == 0 && ROWS % 16 == 0, "whole rounds of rows of one operand, which share their swizzle");
  static_assert(WAVES_K == 1 || (WAVES_K == 4 && WAVES_K % NT == 0 && OWN * WAVES_K == MT * NT), "each wave finishes blocks of one column");
  fetch_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % WAVES_K, wmn = wave / WAVES_K, wm = wmn / WAVES_N, wn = wmn % WAVES_N, l32 = lane & 31, half = lane >> 5;

  // each XCD takes a contiguous run of the tile list (kGroupM tile rows at a time, column-major inside)
  const int tiles = p.tiles_m * p.tiles_n;
  const TileWalk walk = make_walk(PARTIAL ? tiles * p.splits : tiles);
  if (walk.slot >= walk.chunk_len) return;
  const int item = walk.chunk_begin + walk.slot;
  const int part = PARTIAL ? fast_div(item, p.div_tiles_mul, p.div_tiles_shift) : 0;
  int tm, tn;
  tile_coords(item - part * tiles, p.tiles_m, p.tiles_n, p.div_group_mul, p.div_group_shift, tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BN;

  // Steps of this item from step `first` on but for the row's last one, which has 1 to 128 bytes and is its last part's.
  const int whole = (p.K - 1) / kStepK;
  const int first = PARTIAL ? part * p.steps_per_split : 0;
  const int full = PARTIAL ? min(p.steps_per_split, whole - first) : whole;
  const bool has_tail = !PARTIAL || part == p.splits - 1;

  // Lane's chunk ld_c of rows ld_row, ld_row + ROWS, ... (rows past an edge repeat the last one).
  // The bytes of a step are fetched as the whole dwords behind the one that its first byte lies in (DWORDS: from that one on), and moved into place when
  // they are parked: a chunk begins in the last dword of the chunk in front of it, the lane's beside it, or the step's before.
  // (Every dword that is fetched holds bytes of its row: the first one byte 0, the last one byte 128 * whole.)
  const int ld_row = tid >> 3, ld_c = tid & 7;
  const uint8_t* at[LOADS];  // what is fetched next
  uint32_t shift[LOADS];
  int before[LOADS];  // the last dword of the step that was parked last
  v4i land[DEPTH][LOADS];
  const uint8_t* row[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = ld_row + ROWS * (i < LA ? i : i - LA);
    row[i] = i < LA ? p.a + (size_t)min(m0 + r, (long)p.M - 1) * p.lda : p.b + (size_t)min(n0 + r, (long)p.N - 1) * p.ldb;
    shift[i] = DWORDS ? 0 : (uint32_t)(reinterpret_cast<uintptr_t>(row[i]) & 3);
    at[i] = row[i] - shift[i] + (long)first * kStepK + ld_c * kChunk + (DWORDS ? 0 : 4);
    before[i] = !DWORDS && full > 0 ? *(const int*)(row[i] - shift[i] + (long)first * kStepK) : 0;
  }
  // the factors and the bias of the tile's rows and columns, which wait in LDS behind the stages for the end
  uint8_t* const ends = lds + any_stage_bytes(BM, BN, WAVES_K, WAVES_M * WAVES_N);
  float end_a = 0.0f, end_b = 0.0f, end_bias = 0.0f;
  if constexpr (!PARTIAL) {
    if (tid < BM) end_a = p.a_scale[min(m0 + tid, (long)p.M - 1)];
    if (tid < BN) {
      const long n = min(n0 + tid, (long)p.N - 1);
      end_b = p.b_scale[n];
      if (p.bias) end_bias = bf16_to_f32(p.bias[n]);
    }
  }
  auto park_ends = [&]() {  // (after the first steps have been asked for)
    if constexpr (!PARTIAL) {
      if (tid < BM) *(float*)(ends + tid * 4) = end_a;
      if (tid < BN) {
        *(float*)(ends + (BM + tid) * 4) = end_b;
        *(float*)(ends + (BM + BN + tid) * 4) = end_bias;
      }
    }
  };
  int to_fetch = full;  // whole steps that have not been asked for
  auto fetch = [&](v4i (&to)[LOADS]) {
    const long on = --to_fetch > 0 ? kStepK : 0;  // past the last whole step: that one again, for nobody
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      to[i] = *(const v4i_by4*)at[i];
      at[i] += on;
    }
  };
  const int park_pos = ld_row * kStepK + ((ld_c ^ swz128(ld_row)) * kChunk);  // (ROWS rows on: the same swizzle)
  auto park_one = [&](const v4i& chunk, int i, int stage) { *(v4i*)(lds + park_pos + stage * STAGE + i * ROWS * kStepK) = chunk; };
  auto park = [&](const v4i (&from)[LOADS], int stage) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const v4i x = from[i];
      if constexpr (DWORDS) {
        park_one(x, i, stage);
        continue;
      }
      // the lane beside it; for the first of a row's eight lanes the last one's of the step before
      const int left = __builtin_amdgcn_update_dpp(0, x[3], 0x111, 0xf, 0xf, true);       // row_shr:1
      const int back = __builtin_amdgcn_update_dpp(0, before[i], 0x141, 0xf, 0xf, true);  // row_half_mirror
      before[i] = x[3];
      const int front = ld_c == 0 ? back : left;
      park_one((v4i){(int)__builtin_amdgcn_alignbyte(x[0], front, shift[i]), (int)__builtin_amdgcn_alignbyte(x[1], x[0], shift[i]),
                     (int)__builtin_amdgcn_alignbyte(x[2], x[1], shift[i]), (int)__builtin_amdgcn_alignbyte(x[3], x[2], shift[i])}, i, stage);
    }
  };
  auto join = [&]() {  // this wave's LDS accesses are done, then everyone's; global loads stay in flight
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
  };

  v16f acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (v16f){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int frag_pos[PAIRS];
#pragma unroll
  for (int c = 0; c < PAIRS; ++c) frag_pos[c] = l32 * kStepK + (((2 * (wk * PAIRS + c) + half) ^ swz128(l32)) * kChunk);
  const int rows_a = wm * WTM * kStepK, rows_b = (BM + wn * WTN) * kStepK;
  auto multiply = [&](int stage) {
    v4i ra[PAIRS][MT], rb[PAIRS][NT];
#pragma unroll
    for (int c = 0; c < PAIRS; ++c) {
#pragma unroll
      for (int i = 0; i < MT; ++i) ra[c][i] = *(const v4i*)(lds + frag_pos[c] + rows_a + stage * STAGE + i * 32 * kStepK);
#pragma unroll
      for (int j = 0; j < NT; ++j) rb[c][j] = *(const v4i*)(lds + frag_pos[c] + rows_b + stage * STAGE + j * 32 * kStepK);
    }
    if (PAIRS > 1) __builtin_amdgcn_sched_barrier(0);  // (left alone, the reads of a pair wait for the products of the one before)
#pragma unroll
    for (int c = 0; c < PAIRS; ++c) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {  // 8 codes of a lane per instruction
        v8h fa[MT], fb[NT];
#pragma unroll
        for (int i = 0; i < MT; ++i) fa[i] = e4m3fn_to_f16x8(ra[c][i][2 * u], ra[c][i][2 * u + 1]);
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[j] = e4m3fn_to_f16x8(rb[c][j][2 * u], rb[c][j][2 * u + 1]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
    }
  };

  if (full > 0)
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(land[d]);
  park_ends();
  if (has_tail) {
    v4i tail[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) tail[i] = load16_any(row[i], whole * kStepK + ld_c * kChunk, p.K);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) park_one(tail[i], i, 1);
    join();
    multiply(1);
    if (full <= 0) join();
  }
  if (full > 0) {
    // a step on the stage it was parked in; its registers take the step DEPTH on, the other stage the next one
    auto step = [&](int d, int stage) {
      fetch(land[d]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(stage);
      park(land[(d + 1) % DEPTH], stage ^ 1);
      join();
    };
    park(land[0], 0);
    join();
    constexpr int TURN = DEPTH % 2 ? 2 * DEPTH : DEPTH;  // steps after which registers and stages are the same again
    int s = 0;
    for (; s + TURN <= full; s += TURN)
#pragma unroll
      for (int d = 0; d < TURN; ++d) step(d % DEPTH, d & 1);
#pragma unroll
    for (int d = 0; d < TURN - 1; ++d)
      if (s + d < full) step(d % DEPTH, d & 1);
  }

  // Lane (l32, half) holds row l32 of a block, columns 8q + 4*half + 0..3: each four as one piece wherever it lies
  // (1795x84399x13, rows of C that start at any 2 bytes: 553 us with a store per element).
  auto finish = [&](const v16f& sum, int i, int j) {
    const int m_tile = wm * WTM + i * 32 + l32, n_tile = wn * WTN + j * 32 + 4 * half;
    const long m = m0 + m_tile;
    const float sa_m = PARTIAL ? 0.0f : *(const float*)(ends + m_tile * 4);
    v4f sb[4], bias[4];
    if constexpr (!PARTIAL) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sb[q] = *(const v4f*)(ends + (BM + n_tile + 8 * q) * 4);
        bias[q] = *(const v4f*)(ends + (BM + BN + n_tile + 8 * q) * 4);
      }
    }
    if (m < p.M) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const long n = n0 + n_tile + 8 * q;
        if constexpr (PARTIAL) {
          float* dst = p.partial + ((size_t)part * p.M + m) * p.N + n;
          if (n + 3 < p.N) {
            *(v4f_by4*)dst = (v4f){sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
          } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (n + e < p.N) dst[e] = sum[4 * q + e];
          }
        } else {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float t = sum[4 * q + e] * sa_m;
            v[e] = p.bias ? __builtin_fmaf(t, sb[q][e], bias[q][e]) : t * sb[q][e];
          }
          const uint32_t lo = pack_out_x2(v[0], v[1], p.out_f16), hi = pack_out_x2(v[2], v[3], p.out_f16);
          uint16_t* dst = p.c + (size_t)m * p.ldc + n;
          if (n + 3 < p.N) {
            *(v2u_any*)dst = (v2u){lo, hi};
          } else {
            if (n < p.N) dst[0] = (uint16_t)lo;
            if (n + 1 < p.N) dst[1] = (uint16_t)(lo >> 16);
            if (n + 2 < p.N) dst[2] = (uint16_t)hi;
          }
        }
      }
    }
  };
  if constexpr (WAVES_K == 1) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) finish(acc[i][j], i, j);
  } else {
    // The sums of the waves that shared out K meet in LDS, where the stages were, a block for each of them at a time: the wave that
    // finishes it adds what the others left to its own, in their order.
    constexpr int kBlockBytes = 32 * 32 * 4;
    uint8_t* const slots = lds + wmn * (WAVES_K * (WAVES_K - 1) * kBlockBytes) + lane * 16;
    auto slot = [&](int writer, int owner) { return slots + (owner * (WAVES_K - 1) + (writer < owner ? writer : writer - 1)) * kBlockBytes; };
#pragma unroll
    for (int r = 0; r < OWN; ++r) {
      v16f mine;
#pragma unroll
      for (int o = 0; o < WAVES_K; ++o) {
        const v16f& block = acc[o / NT * OWN + r][o % NT];
        if (wk == o) {
          mine = block;
        } else {
          uint8_t* const to = slot(wk, o);
#pragma unroll
          for (int q = 0; q < 4; ++q) *(v4f*)(to + q * 1024) = (v4f){block[4 * q], block[4 * q + 1], block[4 * q + 2], block[4 * q + 3]};
        }
      }
      join();
#pragma unroll
      for (int o = 0; o < WAVES_K - 1; ++o) {
        const uint8_t* const from = slot(o < wk ? o : o + 1, wk);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const v4f x = *(const v4f*)(from + q * 1024);
#pragma unroll
          for (int e = 0; e < 4; ++e) mine[4 * q + e] += x[e];
        }
      }
      if (r + 1 < OWN) join();
      finish(mine, wk / NT * OWN + r, wk % NT);
    }
  }
}

// Grouped form: the group that row block `item` belongs to when every group's rows are cut into blocks of BM, and what
// precedes it. Each lane takes one size of 64, and two scans across the wave give the rows and the blocks in front of
// every group: one trip to memory however many groups there are (up to 64), where a walk over the sizes makes one each.
// Sizes are clamped as in the tiled kernel (negative -> 0, the running sum cut at M): additions that saturate at M, which
// a scan may regroup. group < 0: there is no such block, and row_end and blocks_before are the totals.
struct RowBlock {
  int group, row_begin, row_end, blocks, blocks_before;
};
template <int BM>
__device__ __forceinline__ RowBlock find_row_block(const GemmParams& p, int item) {
  const int lane = threadIdx.x & 63;
  int rows_before = 0, blocks_before = 0;
  for (int g0 = 0; g0 < p.groups; g0 += 64) {
    const int size = g0 + lane < p.groups ? min(max(p.m_sizes[g0 + lane], 0), p.M) : 0;
    uint32_t row_end = (uint32_t)size + (lane == 0 ? (uint32_t)rows_before : 0u);
    row_end = min(row_end, (uint32_t)p.M);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t below = __shfl_up(row_end, o);
      if (lane >= o) row_end = min(row_end + below, (uint32_t)p.M);
    }
    const uint32_t prev = __shfl_up(row_end, 1);
    const int row_begin = lane == 0 ? rows_before : (int)prev;
    const int blocks = ((int)row_end - row_begin + BM - 1) / BM;
    int blocks_end = blocks + (lane == 0 ? blocks_before : 0);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int below = __shfl_up(blocks_end, o);
      if (lane >= o) blocks_end += below;
    }
    const uint64_t past = __ballot(item < blocks_end);
    if (past) {
      const int at = __builtin_ctzll(past);
      RowBlock r;
      r.group = g0 + at;
      r.row_begin = __builtin_amdgcn_readlane(row_begin, at);
      r.row_end = __builtin_amdgcn_readlane((int)row_end, at);
      r.blocks = __builtin_amdgcn_readlane(blocks, at);
      r.blocks_before = __builtin_amdgcn_readlane(blocks_end, at) - r.blocks;
      return r;
    }
    rows_before = __builtin_amdgcn_readlane((int)row_end, 63);
    blocks_before = __builtin_amdgcn_readlane(blocks_end, 63);
  }
  return RowBlock{-1, rows_before, rows_before, 0, blocks_before};
}

// ------------------------------------------------------------------------------------
// Skinny kernel (M <= 16*MT, HBM-bound): B is streamed exactly once and nothing is reused, so
// what matters is whole-line coalesced loads and as many bytes in flight as a plain copy has.
//
// A workgroup owns 16*NTW rows of B and all of K; its KW waves split K between them in
// interleaved 128-byte steps (wave w takes steps w, w+KW, ...: the workgroup reads KW*128-byte runs
// of every row). Registers are the landing zone: a wave keeps DEPTH steps of loads in flight
// (16 bytes per lane, 8 lanes per row, so every wave-wide load moves 8 whole 128-byte lines;
// letting each MFMA lane fetch its own row instead costs the memory pipeline four times the
// tag look-ups). A landed step is transposed into the MFMA lane layout through a small
// wave-private LDS buffer (swizzled like the tiled kernel's stages); LDS executes a wave's
// operations in order, so the loop needs no barrier. A [16*MT rows] takes the same route.
// Partial 16x16 results are summed across the waves through LDS at the end.
// ------------------------------------------------------------------------------------
// ANY: the generic family's form for up to 64 rows: unaligned loads, 16-bit matrix instructions on the
// widened codes, any K (see the generic kernels above).
// BLOCK: the block-scaled form (a step is one K block, all rows of A are in one row block and a tile of B in one
// column block): a step's products are scaled by its factor as they are added up.
// GROUPED: the grouped form for few rows a group. A workgroup is 16*NTW columns of one block of up to 16*MT rows of
// a group; the row blocks of one group's columns are neighbours on one XCD (workgroup ids go round the XCDs), so that
// the group's rows of B come from HBM once. The grid covers the most row blocks that any sizes with these M and G can
// give; the surplus comes last and returns at once.
// OFF_LINES: for rows of B that do not start on 128-byte lines: no streaming policy.
template <int MT, int NTW, int DEPTH, int KW, bool ANY = false, bool BLOCK = false, bool GROUPED = false, bool OFF_LINES = false>
__global__ __launch_bounds__(KW * 64) void gemm_skinny_kernel(GemmParams p) {
  static_assert((int)ANY + (int)BLOCK + (int)GROUPED <= 1, "at most one of them");
  using Chunk = std::conditional_t<ANY, v4i_any, v4i>;
  constexpr int TILE = 16 * kStepK;                 // one 16-row operand tile of one step: 2 KB
  constexpr int NTILE = NTW + MT;                   // tiles per step: B tiles then A tiles
  constexpr int BUF = NTILE * TILE;                 // wave-private transpose buffer
  static_assert(NTW * MT * 1024 <= BUF, "the reduction reuses a wave's buffer for its partials");
  fetch_arguments_now(p);

  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* buf = lds + wave * BUF;
  int n0 = blockIdx.x * (16 * NTW), m0 = 0, m_end = p.M;
  const uint8_t* b_rows = p.b;
  const float* b_scales = p.b_scale;
  if constexpr (GROUPED) {
    const int tiles = (p.tiles_n + kNumXcd - 1) / kNumXcd * kNumXcd;
    const RowBlock at = find_row_block<16 * MT>(p, (int)blockIdx.x / tiles);
    if (at.group < 0) {  // surplus
      if (p.clear_rest && at.row_end < p.M) {
        const int used = at.blocks_before * tiles;
        clear_rows(p, at.row_end, (int)blockIdx.x - used, (int)gridDim.x - used);
      }
      return;
    }
    // t runs over the group's tiles and row blocks: the XCD's place, then the row block, then the round of tiles
    const int t = (int)blockIdx.x - at.blocks_before * tiles;
    const int slot = t / kNumXcd;
    const int tile = slot / at.blocks * kNumXcd + t % kNumXcd;
    if (tile >= p.tiles_n) return;
    n0 = tile * (16 * NTW);
    m0 = at.row_begin + slot % at.blocks * (16 * MT);
    m_end = at.row_end;
    b_rows += (size_t)at.group * p.N * p.ldb;
    b_scales += (size_t)at.group * p.N;
  }

  // global load: lane (ld_row, ld_c) of a wave-wide load fetches chunk ld_c (16 bytes) of row
  // ld_row of an 8-row half tile and parks it in LDS at the swizzled chunk position
  const int ld_row = lane >> 3, ld_c = lane & 7;
  const uint8_t* src[NTILE][2];
  int wr_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = h * 8 + ld_row;
    wr_off[h] = r * kStepK + ((ld_c ^ swz128(r)) * kChunk);
#pragma unroll
    for (int t = 0; t < NTW; ++t)
      src[t][h] = b_rows + (size_t)min(n0 + t * 16 + r, p.N - 1) * p.ldb + ld_c * kChunk;
#pragma unroll
    for (int t = 0; t < MT; ++t)
      src[NTW + t][h] = p.a + (size_t)min(m0 + t * 16 + r, m_end - 1) * p.lda + ld_c * kChunk;
  }
  // LDS->register: lane (r, g) of the 16x16x128 MFMA takes logical chunks 2g, 2g+1 of row r
  const int r16 = lane & 15, g4 = lane >> 4;
  const int rd0 = r16 * kStepK + (((2 * g4) ^ swz128(r16)) * kChunk);
  const int rd1 = r16 * kStepK + (((2 * g4 + 1) ^ swz128(r16)) * kChunk);

  const int k_full = p.K / kStepK;
  const int k_tail = p.K - k_full * kStepK;
  const int my_steps = (k_full > wave) ? (k_full - wave + KW - 1) / KW : 0;  // whole steps this wave owns

  v4f acc[NTW][MT];
#pragma unroll
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) acc[t][u] = (v4f){0.f, 0.f, 0.f, 0.f};

  // The lanes that will finish an output quad (one per lane of each 16x16 result) fetch its
  // scales and bias now, so that their latency is not left over at the end of the kernel.
  // Lane layout of a 16x16 result: m = u*16 + lane%16, n = n0 + t*16 + 4*(lane/16) + e.
  static_assert(NTW * MT * 64 <= KW * 64, "one finishing lane per output quad");
  const bool finisher = threadIdx.x < NTW * MT * 64;
  const int fin_tu = threadIdx.x >> 6;
  const int fin_m = m0 + (fin_tu % MT) * 16 + (lane & 15);
  const int fin_n = n0 + (fin_tu / MT) * 16 + 4 * (lane >> 4);
  float fin_sa = 0.f, fin_sb[4] = {0.f, 0.f, 0.f, 0.f}, fin_bias[4] = {0.f, 0.f, 0.f, 0.f};
  if (finisher && !BLOCK) {
    fin_sa = p.a_scale[min(fin_m, m_end - 1)];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ne = min(fin_n + e, p.N - 1);
      fin_sb[e] = b_scales[ne];
      if (p.bias) fin_bias[e] = bf16_to_f32(p.bias[ne]);
    }
  }

  // the factors of K block kb: a_scale's and, per 16 rows of B, b_scale's
  const int k_blocks = k_full + (k_tail ? 1 : 0);
  scalar_floats block_a = (scalar_floats)p.a_scale, block_b[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) block_b[t] = (scalar_floats)(p.b_scale + (size_t)(min(n0 + t * 16, p.N - 1) / 128) * k_blocks);
  struct Factors {
    float a, b[NTW];
  };
  auto fetch_factors = [&](int kb, Factors& f) {
    if constexpr (BLOCK) {
      f.a = block_a[kb];
#pragma unroll
      for (int t = 0; t < NTW; ++t) f.b[t] = block_b[t][kb];
    }
  };

  // DEPTH register sets, one per step in flight
  v4i land[DEPTH][NTILE][2];
  Factors land_f[DEPTH];
  auto fetch = [&](int i, v4i (&dst)[NTILE][2], Factors& f) {
    fetch_factors(wave + KW * i, f);
    const size_t kb = (size_t)(wave + KW * i) * kStepK;
#pragma unroll
    for (int t = 0; t < NTILE; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // B is read once and never again: stream it past the caches; A is shared by everyone. (ANY: an
        // unaligned piece shares its lines with the neighbouring steps, which the streaming policy would
        // fetch again: 1x8192x8191 19.6 -> 14.4 us without it, 16x8192x8191 25.6 -> 19.1. The same for rows that start
        // off a line: 128 rows in 16 groups of 4096x4112 75 -> 60, 64 in 8 of 14336x4112 128 -> 101, 1x12544x5968 17.4 -> 16.2,
        // 54x3584x4288 9.0 -> 6.9.)
        if (t < NTW && !ANY && !OFF_LINES) dst[t][h] = __builtin_nontemporal_load((const Chunk*)(src[t][h] + kb));
        else dst[t][h] = *(const Chunk*)(src[t][h] + kb);
      }
  };
  // one step's products; ANY: a lane's 32 codes of a row are four 16-bit instructions of 8 codes per lane
  auto multiply = [&](const v8i (&bf)[NTW], const v8i (&af)[MT], const Factors& f) {
    if constexpr (BLOCK) {
      const v4f zero = {0.f, 0.f, 0.f, 0.f};
      v4f part[NTW][MT];
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int u = 0; u < MT; ++u)
          part[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[t], af[u], zero, 0, 0, 0, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NTW; ++t) {
        const float s = f.a * f.b[t];
#pragma unroll
        for (int u = 0; u < MT; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][u][e] = __builtin_fmaf(part[t][u][e], s, acc[t][u][e]);
      }
    } else if constexpr (ANY) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v8h hb[NTW], ha[MT];
#pragma unroll
        for (int t = 0; t < NTW; ++t) hb[t] = e4m3fn_to_f16x8(bf[t][2 * q], bf[t][2 * q + 1]);
#pragma unroll
        for (int u = 0; u < MT; ++u) ha[u] = e4m3fn_to_f16x8(af[u][2 * q], af[u][2 * q + 1]);
#pragma unroll
        for (int t = 0; t < NTW; ++t)
#pragma unroll
          for (int u = 0; u < MT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hb[t], ha[u], acc[t][u], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int u = 0; u < MT; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[t], af[u], acc[t][u], 0, 0, 0, 0, 0, 0);
    }
  };
  auto consume = [&](const v4i (&got)[NTILE][2], const Factors& factors) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) *(v4i*)(buf + t * TILE + wr_off[h]) = got[t][h];
    v8i bf[NTW], af[MT];
#pragma unroll
    for (int t = 0; t < NTILE; ++t) {
      const v4i lo = *(const v4i*)(buf + t * TILE + rd0);
      const v4i hi = *(const v4i*)(buf + t * TILE + rd1);
      const v8i f = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if (t < NTW) bf[t] = f;
      else af[t - NTW] = f;
    }
    multiply(bf, af, factors);
  };

  // K tail (K % 128 != 0): one partial step, taken by the wave whose turn it would be; the
  // lanes fetch their own 16-byte chunks and chunks (ANY: bytes) at or past K count as zero. Behind the first steps' loads and in front of
  // their products: at the end its trip to memory is on its own (2x6400x3008 7.46 -> 7.03 us, 12x1916x752 3.37 -> 3.16). ANY: at the end after all, where
  // the one wave that has it holds the others' lines up less (42x33317x2297 57.4 us so, 52.2 at the end).
  auto multiply_tail = [&]() {
    if (!k_tail || (k_full % KW) != wave) return;
    const int kb = k_full * kStepK;
    auto chunk_of = [&](const uint8_t* row, int c) -> v4i {
      if constexpr (ANY) return load16_any(row, kb + c * kChunk, p.K);
      return c * kChunk < k_tail ? *(const v4i*)(row + kb + c * kChunk) : (v4i){0, 0, 0, 0};
    };
    v8i bf[NTW], af[MT];
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      const uint8_t* row = b_rows + (size_t)min(n0 + t * 16 + r16, p.N - 1) * p.ldb;
      const v4i lo = chunk_of(row, 2 * g4), hi = chunk_of(row, 2 * g4 + 1);
      bf[t] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      const uint8_t* row = p.a + (size_t)min(m0 + u * 16 + r16, m_end - 1) * p.lda;
      const v4i lo = chunk_of(row, 2 * g4), hi = chunk_of(row, 2 * g4 + 1);
      af[u] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    Factors f;
    fetch_factors(k_full, f);
    multiply(bf, af, f);
  };

  // (Block scaling: at the end where its wave has one or two whole steps and less than half of the waves one more. 198 shapes of 40 to 260 chunks: in front
  // such calls took 1.01 to 1.06 of the time at the end, 4x128x1200 3.07 us and 2.95, the others 0.95 to 1.03. Row-wise in front is ahead or level in all of them.)
  const int tail_steps = k_full / KW;
  const bool tail_first = !ANY && !(BLOCK && tail_steps >= 1 && tail_steps <= 2 && k_full % KW < KW / 2);

  // The loop is unrolled DEPTH times so every register set has a fixed name; the compiler's
  // own wait counts then make each consume() wait for exactly its set's loads (they return
  // in issue order, so the younger sets stay in flight). That only works on paths without
  // conditional fetches: where paths with different numbers of younger loads meet, the
  // compiler has to assume the fewest and ends up draining the whole queue once per round.
  // So the rounds in which every consume is followed by a fetch form their own loop, the
  // last full round (consumes only) is straight-line code, and only ragged step counts take
  // the conditional form. (Measured: worth 2 % with four steps in flight; with two steps in
  // flight the drained form is 8-11 % faster, so those configurations keep it.)
  constexpr bool kSteadyLoop = DEPTH >= 4;
  int i = 0;
  if (kSteadyLoop && my_steps >= DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(d, land[d], land_f[d]);
    if (tail_first) multiply_tail();
    for (; i + 2 * DEPTH <= my_steps; i += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        consume(land[d], land_f[d]);
        fetch(i + d + DEPTH, land[d], land_f[d]);
      }
    }
    if (i + DEPTH == my_steps) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) consume(land[d], land_f[d]);
      i += DEPTH;
    }
  } else {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (d < my_steps) fetch(d, land[d], land_f[d]);
    if (tail_first) multiply_tail();
  }
  for (; i < my_steps; i += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (i + d < my_steps) {
        consume(land[d], land_f[d]);
        if (i + d + DEPTH < my_steps) fetch(i + d + DEPTH, land[d], land_f[d]);
      }
    }
  }
  if (!tail_first) multiply_tail();

  // ---- cross-wave reduction through each wave's own (now idle) buffer
  v4f* mine = (v4f*)buf;
#pragma unroll
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) mine[(t * MT + u) * 64 + lane] = acc[t][u];
  __syncthreads();

  if (finisher && fin_m < m_end && fin_n < p.N) {
    v4f sum = ((const v4f*)lds)[fin_tu * 64 + lane];
#pragma unroll
    for (int w = 1; w < KW; ++w) sum += ((const v4f*)(lds + w * BUF))[fin_tu * 64 + lane];
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] = BLOCK ? sum[e] : sum[e] * fin_sa * fin_sb[e];
      if (!BLOCK && p.bias) r[e] += fin_bias[e];
    }
    const uint32_t lo = pack_out_x2(r[0], r[1], p.out_f16), hi = pack_out_x2(r[2], r[3], p.out_f16);
    uint16_t* dst = p.c + (size_t)fin_m * p.ldc + fin_n;
    if (fin_n + 3 < p.N && ((p.ldc & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.c) & 7) == 0)) {
      *(v2u*)dst = (v2u){lo, hi};
    } else {
      dst[0] = (uint16_t)lo;
      if (fin_n + 1 < p.N) dst[1] = (uint16_t)(lo >> 16);
      if (fin_n + 2 < p.N) dst[2] = (uint16_t)hi;
      if (fin_n + 3 < p.N) dst[3] = (uint16_t)(hi >> 16);
    }
  }
}

// ------------------------------------------------------------------------------------
// Persistent skinny kernel for M <= 16*MT (MT = 1, 2) and K = 16*SPW 128-byte steps (K = 2048 ..
// 8192): one workgroup of 16 waves per CU walks a contiguous run of 16-row tiles of B. Wave w
// owns the K steps w, w+16, ... of every tile and keeps its share of A (MT*SPW fragments, 8
// registers each) in registers for the whole launch: A crosses the L2->L1 path once per CU
// instead of once per tile, which is where the one-tile-per-workgroup kernel above loses a
// tenth of its time at M = 16 and a quarter at M = 32. The loads of B run LAG steps ahead of
// their use (a whole tile with one block of A; two steps with two, whose fragments take the
// registers); per tile the waves' partial 16x16 results meet in LDS (two alternating areas, one
// barrier per tile) and one wave per 16x16 result, a different one every time, adds them in
// wave order and stores.
// Workgroup g starts its K walk at step 2*(g/8) (workgroups g, g+8, ... share an XCD): the
// workgroups of an XCD then ask its L2 for different lines of A at any one time, and the
// addresses of B in flight do not all agree in their low bits (measured at N=K=8192, M=16:
// 13.2 -> 12.7 us).
// ------------------------------------------------------------------------------------
constexpr int kPersistWaves = 16;

constexpr size_t persistent_lds_bytes(int MT) { return (size_t)kPersistWaves * 2048 + (size_t)2 * kPersistWaves * MT * 1024; }

// VEC: b_scale, bias and C are aligned for 16-, 8- and 8-byte accesses (else element by element).
template <int SPW, int MT, int LAG, bool VEC>
__global__ __launch_bounds__(kPersistWaves * 64) void gemm_skinny_persistent_kernel(GemmParams p) {
  constexpr int WAVES = kPersistWaves;
  constexpr int STEPS = WAVES * SPW;
  static_assert(LAG >= 1 && LAG <= SPW && SPW % LAG == 0, "the landing registers are a ring of LAG steps");
  fetch_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* buf = lds + wave * 2048;             // this wave's transpose buffer (one 16 x 128 B step)
  v4f* red = (v4f*)(lds + WAVES * 2048);        // [2][MT][WAVES][64] partial results

  // this workgroup's run of tiles: the first `rem` workgroups take one tile more (quotient and
  // remainder of tiles by workgroups come from the host: the division would sit in front of the
  // first load)
  const int g = blockIdx.x;
  const int q = p.tiles_m, rem = p.tiles_n;
  const int tile0 = g * q + min(g, rem);
  const int count = q + (g < rem ? 1 : 0);
  if (count <= 0) return;

  // byte offset of this wave's i-th K step inside a row; wave-uniform, pinned to scalar registers
  const int base_step = (wave + 2 * (g >> 3)) % STEPS;
  uint32_t kofs[SPW];
#pragma unroll
  for (int i = 0; i < SPW; ++i) {
    int s = base_step + WAVES * i;
    if (s >= STEPS) s -= STEPS;
    kofs[i] = (uint32_t)__builtin_amdgcn_readfirstlane(s * kStepK);
  }
  // a wave-uniform 64-bit offset pinned to scalar registers: loads then take the scalar-base +
  // 32-bit lane-offset form instead of a 64-bit address pair per lane and load
  auto uniform = [](size_t v) -> size_t {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((size_t)hi << 32) | lo;
  };
  const int r16 = lane & 15, g4 = lane >> 4;
  const int ld_row = lane >> 3, ld_c = lane & 7;
  uint32_t b_lane[2];
  int wr_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = h * 8 + ld_row;
    wr_off[h] = r * kStepK + ((ld_c ^ swz128(r)) * kChunk);
    b_lane[h] = (uint32_t)r * (uint32_t)p.ldb + ld_c * kChunk;
  }
  const int rd0 = r16 * kStepK + (((2 * g4) ^ swz128(r16)) * kChunk);
  const int rd1 = r16 * kStepK + (((2 * g4 + 1) ^ swz128(r16)) * kChunk);

  v4i land[LAG][2];
  const size_t tile_pitch = (size_t)16 * p.ldb;
  size_t cur_tile = uniform((size_t)tile0 * tile_pitch);  // byte offset of the tile being multiplied
  auto fetch = [&](int slot, size_t tile_off, int i) {
    const uint8_t* sbase = p.b + (tile_off + kofs[i]);
#pragma unroll
    for (int h = 0; h < 2; ++h) land[slot][h] = __builtin_nontemporal_load((const v4i*)(sbase + b_lane[h]));
  };
  // The first rows of B are asked for before anything else: they come from HBM.
#pragma unroll
  for (int i = 0; i < LAG; ++i) fetch(i, cur_tile, i);
  __builtin_amdgcn_sched_barrier(0);
  // A: whole-line loads (8 lanes per row, rows past M repeat the last one), turned into the
  // MFMA lane layout through the transpose buffer, once, one 16-row block at a time
  v8i fa[MT][SPW];
#pragma unroll
  for (int u = 0; u < MT; ++u) {
    v4i la[SPW][2];
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
      const uint8_t* sbase = p.a + kofs[i];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        la[i][h] = *(const v4i*)(sbase + ((uint32_t)min(u * 16 + h * 8 + ld_row, p.M - 1) * (uint32_t)p.lda + ld_c * kChunk));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
      *(v4i*)(buf + wr_off[0]) = la[i][0];
      *(v4i*)(buf + wr_off[1]) = la[i][1];
      const v4i lo = *(const v4i*)(buf + rd0);
      const v4i hi = *(const v4i*)(buf + rd1);
      fa[u][i] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // The 16x16 results are numbered q = MT*j + u (tile j of the run, block u of A); wave w finishes
  // the results q = w, w + 16, ...: lane (m = 16u + lane % 16, quad lane / 16) owns
  // C[m, 16*tile + 4*(lane/16) .. +3]. The column scales and bias of a wave's next result are
  // fetched long before they are used (here, and after each finished result) and kept as loaded;
  // a run without a result for this wave reads the run's last tile instead.
  // Without a bias the same loads read the head of b_scale instead and the bits are masked off:
  // the loads stay unconditional and in the global address space either way.
  const uint16_t* const bias_src = p.bias ? p.bias : reinterpret_cast<const uint16_t*>(p.b_scale);
  const int bias_stride = p.bias ? 1 : 0;
  const uint16_t bias_mask = p.bias ? 0xffffu : 0u;
  float sb_raw[4], fin_sa;
  uint16_t bias_raw[4];
  auto load_epi = [&](int qi) {
    const int qc = min(qi, count * MT - 1);
    const int n = (tile0 + qc / MT) * 16 + 4 * g4;
    fin_sa = p.a_scale[min((qc % MT) * 16 + r16, p.M - 1)];
    if (VEC) {
      const v4f s4 = *(const v4f*)(p.b_scale + n);
      const us4 b4 = *(const us4*)(bias_src + n * bias_stride);
#pragma unroll
      for (int x = 0; x < 4; ++x) sb_raw[x] = s4[x], bias_raw[x] = b4[x];
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) sb_raw[x] = p.b_scale[n + x], bias_raw[x] = bias_src[(n + x) * bias_stride];
    }
  };
  load_epi(wave);

  auto consume = [&](int slot, int i, v4f (&acc)[MT]) {
    *(v4i*)(buf + wr_off[0]) = land[slot][0];
    *(v4i*)(buf + wr_off[1]) = land[slot][1];
    const v4i lo = *(const v4i*)(buf + rd0);
    const v4i hi = *(const v4i*)(buf + rd1);
    const v8i fb = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
    for (int u = 0; u < MT; ++u)
      acc[u] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa[u][i], acc[u], 0, 0, 0, 0, 0, 0);
  };
  auto finish = [&](int j, const v4f (&acc)[MT]) {
    v4f* area = red + (j & 1) * (MT * WAVES * 64);
#pragma unroll
    for (int u = 0; u < MT; ++u) area[(u * WAVES + wave) * 64 + lane] = acc[u];
    __syncthreads();
    // (the area is written again two tiles later, behind the next barrier, which the finishing
    // waves reach only after these reads)
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      if (wave == ((j * MT + u) & (WAVES - 1))) {
        const v4f* part = area + u * WAVES * 64 + lane;
        v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int w0 = 0; w0 < WAVES; w0 += 8) {  // eight partials in flight at a time: all sixteen cost 64 registers
#pragma unroll
          for (int w = 0; w < 8; ++w) sum += part[(w0 + w) * 64];
        }
        const int m = u * 16 + r16;
        if (m < p.M) {
          float r[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) r[x] = __builtin_fmaf(sum[x] * fin_sa, sb_raw[x], bf16_to_f32(bias_raw[x] & bias_mask));
          const uint32_t lo = pack_out_x2(r[0], r[1], p.out_f16), hi = pack_out_x2(r[2], r[3], p.out_f16);
          uint16_t* dst = p.c + (size_t)m * p.ldc + (tile0 + j) * 16 + 4 * g4;
          if (VEC) {
            *(v2u*)dst = (v2u){lo, hi};
          } else {
            dst[0] = (uint16_t)lo; dst[1] = (uint16_t)(lo >> 16);
            dst[2] = (uint16_t)hi; dst[3] = (uint16_t)(hi >> 16);
          }
        }
        load_epi(j * MT + u + WAVES);
      }
    }
  };

  int j = 0;
  for (; j + 1 < count; ++j) {
    const size_t next_tile = uniform(cur_tile + tile_pitch);
    v4f acc[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) acc[u] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
      consume(i % LAG, i, acc);
      if (i + LAG < SPW) fetch(i % LAG, cur_tile, i + LAG);
      else fetch(i % LAG, next_tile, i + LAG - SPW);
    }
    finish(j, acc);
    cur_tile = next_tile;
  }
  {
    v4f acc[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) acc[u] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
      consume(i % LAG, i, acc);
      if (i + LAG < SPW) fetch(i % LAG, cur_tile, i + LAG);
    }
    finish(j, acc);
  }
}

// ------------------------------------------------------------------------------------
// Narrow-tile kernel: one workgroup per tile of 32*MB rows and 32*NB columns of C (MB, NB = 1, 2)
// owns all of K, so there are no partial sums and no second launch. It is the form for shapes
// that give every CU at most one such tile when A has more rows than the persistent kernel
// above keeps in registers: up to 64 rows on any panel, up to 256 in row blocks.
//
// Eight waves. A K step is 512 bytes: wave w of the first four fetches and multiplies the
// step's w-th 128-byte slab of A (rows of A are L2 hits: a short queue, DA steps ahead), wave
// 4+w fetches the same slab of the tile's rows of B (from HBM, DB steps ahead).
// Loads return to a wave in order: with A and B in one queue every A line would wait behind
// the B lines in front of it and see HBM's latency. Both go straight into LDS stages laid out
// as [slab][row][128 bytes] with the tiled kernel's chunk swizzle; one barrier per step. The
// four partial 32x32 (x MB x NB) results meet in LDS at the end; wave w finishes columns 8w..8w+7
// of every 32-row block.
// What bounds it (measured with the loads taken out of the K loop: M=128, N=K=8192 13.5 instead of
// 21.7 us; M=64, N=4096 8.2 instead of 13.0): the bytes the CUs pull from L2 together, about 17 TB/s
// chip-wide in every form (32 KB per step and CU with 32x32 tiles, 64 KB with 64x64), not the depth of
// either ring and not the order of LDS reads and MFMAs.
// Workgroup g starts its walk over K at step 5g mod steps and wraps around: with a power-of-two
// row pitch the rows in flight at one moment would otherwise agree in their low address bits
// and crowd a few memory channels (measured, M=32, N=K=8192, K loop only: 19.8 -> 13.4 us).
// ------------------------------------------------------------------------------------
constexpr int kNarrowKS = 512;
// NB: 32-column blocks per tile (2: 64-column tiles, for panels of one to two 32-column tiles per CU).
// Steps the loads run ahead of their use: what the 160 KB of LDS allow.
constexpr int narrow_b_dist(int MB, int NB) { return NB == 1 ? 5 : MB == 1 ? 3 : 2; }
// A's stages: a compute wave is the only reader of the slab it fetches, so it refills a stage as soon as
// its own fragment reads of it have returned, in the same step: as many steps ahead as there are stages.
constexpr int narrow_a_dist(int MB, int NB) { return MB == 1 && NB == 1 ? 3 : 2; }
constexpr size_t narrow_lds_bytes(int MB, int NB) {
  return (size_t)narrow_a_dist(MB, NB) * MB * 32 * kNarrowKS + (size_t)(narrow_b_dist(MB, NB) + 1) * NB * 32 * kNarrowKS;
}
static_assert(narrow_lds_bytes(2, 1) <= 160 * 1024 && narrow_lds_bytes(1, 2) <= 160 * 1024 && narrow_lds_bytes(2, 2) <= 160 * 1024,
              "stage rings must fit the LDS");

__constant__ float kZeroFactor = 0.0f;

// BLOCK: the block-scaled form. A wave's slab of a step is one K block; the slab's products are scaled by that
// block's factor as they are added up. A tile's columns may straddle two column blocks of B: every group of 4
// columns takes the factor of its own.
// OFF_LINES: rows of B off the 128-byte lines, without the streaming policy.
template <int MB, int NB, bool BLOCK = false, bool OFF_LINES = false>
__global__ __launch_bounds__(512) void gemm_narrow_kernel(GemmParams p) {
  constexpr int BM = 32 * MB, BN = 32 * NB, KS = kNarrowKS;
  constexpr int DA = narrow_a_dist(MB, NB), DB = narrow_b_dist(MB, NB);
  constexpr int RA = DA, RB = DB + 1;
  constexpr int STA = BM * KS, STB = BN * KS;  // bytes per stage
  constexpr int LA = BM / 8, LB = BN / 8;      // wave-wide loads per wave and step (8 rows x 128 bytes each)
  static_assert((DA - 1) * LA < 64 && (DB - 1) * LB < 64, "outstanding-load counts must fit the wait instruction");
  fetch_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // More than BM rows of A: a workgroup per tile and row block. The workgroups of one tile sit next to
  // each other on one XCD (workgroup ids go round the XCDs), so the tile's rows of B come from HBM once
  // and from that XCD's L2 for the others.
  const int row_blocks = (p.M + BM - 1) / BM;
  // Columns of C a tile owns: BN, or fewer where that deals the columns out evenly over the CUs (the host's
  // choice, a multiple of 4). Rows of B past them lie outside the tile's descriptor and read as zeros without
  // a memory access; their products are computed and not stored.
  const int tile_cols = p.tiles_n;
  int tile = blockIdx.x, row_block = 0;
  if (row_blocks > 1) {
    const int slot = blockIdx.x / kNumXcd;
    row_block = slot % row_blocks;
    tile = (slot / row_blocks) * kNumXcd + (blockIdx.x % kNumXcd);
    if (tile * tile_cols >= p.N) return;  // (the grid is rounded up to whole rounds of the XCDs)
  }
  const int n0 = tile * tile_cols, m0 = row_block * BM;
  const int n_end = min(n0 + tile_cols, p.N);
  const int ksteps = (p.K + KS - 1) / KS;  // the last step may be partial (K is a multiple of 16)
  const int rot = (int)(((unsigned)tile * 5u) % (unsigned)ksteps);
  // a lane's 16 bytes of an 8-row group: row lane/8; LDS position lane%8 holds logical chunk
  // position ^ key(row), key = (row >> 1) & 7: for the even groups of a slab that is ld_row >> 1, for
  // the odd ones 4 more, which flips bit 6 of the byte offset
  const int ld_row = lane >> 3, ld_pc = lane & 7;
  const uint32_t chunk_even = (uint32_t)((ld_pc ^ (ld_row >> 1)) * kChunk);
  auto step_of = [&](int s) { const int t = s + rot; return t >= ksteps ? t - ksteps : t; };
  // A lane whose 16 bytes lie at or past K (only in the last step of a K that is not a multiple of 512)
  // asks for an offset outside every descriptor instead: zeros arrive, and the load still counts.
  constexpr uint32_t kOutside = 0x80000000u;
  auto lane_part = [&](uint32_t inside, uint32_t chunk, uint32_t k_slab) { return k_slab + chunk < (uint32_t)p.K ? inside : kOutside; };

  if (wave < 4) {
    // ---- compute wave: slab `wave` of every step
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.a) + (size_t)m0 * p.lda, 0, (int)((uint32_t)min(p.M - m0, BM) * (uint32_t)p.lda), 0x00020000);
    const uint32_t a_even = (uint32_t)ld_row * (uint32_t)p.lda + chunk_even;
    const uint32_t a_odd = (uint32_t)ld_row * (uint32_t)p.lda + (chunk_even ^ 64u);
    auto issue_a = [&](int s) {
      if (s >= ksteps) return;
      uint8_t* dst = lds + (s % RA) * STA + wave * (BM * kStepK);
      const uint32_t koff = (uint32_t)step_of(s) * KS + (uint32_t)wave * kStepK;
      const uint32_t even = lane_part(a_even, chunk_even, koff), odd = lane_part(a_odd, chunk_even ^ 64u, koff);
#pragma unroll
      for (int g = 0; g < LA; ++g)
        load_chunk_to_lds<false>(ra, dst + g * 1024, (g & 1) ? odd : even, (uint32_t)(g * 8) * (uint32_t)p.lda + koff);
    };
    // this lane's scales and bias, asked for before the loop: row l32 of every 32-row block, columns
    // n0 + 32*jb + 8*wave + 4*half .. +3 of every 32-column block (indices clamped; what lies past an
    // edge is never stored)
    const int l32 = lane & 31, half = lane >> 5;
    const int nq = n0 + 8 * wave + 4 * half;
    float sa[MB], sb[NB][4], bias_f[NB][4];
    if (!BLOCK) {
#pragma unroll
      for (int i = 0; i < MB; ++i) sa[i] = p.a_scale[min(m0 + i * 32 + l32, p.M - 1)];
#pragma unroll
      for (int jb = 0; jb < NB; ++jb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int ne = min(nq + 32 * jb + e, p.N - 1);
          sb[jb][e] = p.b_scale[ne];
          bias_f[jb][e] = p.bias ? bf16_to_f32(p.bias[ne]) : 0.0f;
        }
    }
    // BLOCK: rows of factors of this row block and of the (at most two) column blocks 32 columns lie in
    const int k_blocks = (p.K + kStepK - 1) / kStepK;
    scalar_floats block_a = nullptr, block_lo[NB], block_hi[NB];
    bool in_lo[NB][4];
    if (BLOCK) {
      const int last_nb = (p.N - 1) / 128;
      block_a = (scalar_floats)(p.a_scale + (size_t)(m0 / 128) * k_blocks);
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) {
        const int nb = min((n0 + 32 * jb) / 128, last_nb);
        block_lo[jb] = (scalar_floats)(p.b_scale + (size_t)nb * k_blocks);
        block_hi[jb] = (scalar_floats)(p.b_scale + (size_t)min(nb + 1, last_nb) * k_blocks);
#pragma unroll
        for (int q = 0; q < 4; ++q) in_lo[jb][q] = n0 + 32 * jb + 8 * q + 4 * half < (nb + 1) * 128;
      }
    }
#pragma unroll
    for (int s = 0; s < DA; ++s) issue_a(s);
    if (ksteps > DA) wait_loads<(DA - 1) * LA>(); else wait_loads<0>();
    __builtin_amdgcn_s_barrier();

    v16f acc[MB][NB];
    const v16f zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) acc[i][jb] = zero;
    // fragment of K half sh (64 bytes) of this wave's slab: logical chunks 4*half + 2*sh + {0, 1} of row l32
    int rd[2][2];
#pragma unroll
    for (int sh = 0; sh < 2; ++sh)
#pragma unroll
      for (int j = 0; j < 2; ++j) rd[sh][j] = l32 * kStepK + (((4 * half + 2 * sh + j) ^ swz128(l32)) * kChunk);

    // The two K halves of a step are read and multiplied out of phase: while the MFMAs of one half
    // run, the fragment reads of the next are under way (the second half of the same step, or, past
    // the step's barrier, the first half of the next step), so neither the LDS reads nor the MFMAs
    // of the one wave a SIMD has here wait for the other.
    auto read_half = [&](int s, int sh, v4i (&fbh)[NB][2], v4i (&fah)[MB][2]) {
      const uint8_t* sa_rows = lds + (s % RA) * STA + wave * (BM * kStepK);
      const uint8_t* sb_rows = lds + RA * STA + (s % RB) * STB + wave * (BN * kStepK);
#pragma unroll
      for (int jb = 0; jb < NB; ++jb)
#pragma unroll
        for (int j = 0; j < 2; ++j) fbh[jb][j] = *(const v4i*)(sb_rows + jb * 32 * kStepK + rd[sh][j]);
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) fah[i][j] = *(const v4i*)(sa_rows + i * 32 * kStepK + rd[sh][j]);
    };
    v16f part[BLOCK ? MB : 1][BLOCK ? NB : 1];  // BLOCK: the step's products
    auto mfma_half = [&](const v4i (&fbh)[NB][2], const v4i (&fah)[MB][2], bool first) {
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) {
        const v8i vb = (v8i){fbh[jb][0][0], fbh[jb][0][1], fbh[jb][0][2], fbh[jb][0][3],
                             fbh[jb][1][0], fbh[jb][1][1], fbh[jb][1][2], fbh[jb][1][3]};
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const v8i va = (v8i){fah[i][0][0], fah[i][0][1], fah[i][0][2], fah[i][0][3],
                               fah[i][1][0], fah[i][1][1], fah[i][1][2], fah[i][1][3]};
          if constexpr (BLOCK) {
            part[i][jb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vb, va, first ? zero : part[i][jb], 0, 0, 0, 0, 0, 0);
          } else {
            acc[i][jb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vb, va, acc[i][jb], 0, 0, 0, 0, 0, 0);
          }
        }
      }
    };
    auto add_scaled = [&](float fa, const float (&flo)[NB], const float (&fhi)[NB]) {
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) {
        const float lo = fa * flo[jb], hi = fa * fhi[jb];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float f = in_lo[jb][q] ? lo : hi;
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[i][jb][4 * q + e] = __builtin_fmaf(part[BLOCK ? i : 0][BLOCK ? jb : 0][4 * q + e], f, acc[i][jb][4 * q + e]);
        }
      }
    };
    v4i fb0[NB][2], fa0[MB][2], fb1[NB][2], fa1[MB][2];
    read_half(0, 0, fb0, fa0);
    for (int s = 0; s < ksteps; ++s) {
      float f_a = 0.f, f_lo[NB] = {}, f_hi[NB] = {};
      if (BLOCK) {
        // A slab past K adds nothing, but an infinite factor of the last block would turn its zeros into NaN: it takes factors of
        // zero. (By address: zeros chosen behind the loads, or a branch around the additions, are 247x768x1328 5.15 -> 5.4 us.)
        const int kb = step_of(s) * 4 + wave;
        const bool inside = kb < k_blocks;
        const scalar_floats zero = (scalar_floats)&kZeroFactor;
        f_a = *(inside ? block_a + kb : zero);
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) {
          f_lo[jb] = *(inside ? block_lo[jb] + kb : zero);
          f_hi[jb] = *(inside ? block_hi[jb] + kb : zero);
        }
      }
      read_half(s, 1, fb1, fa1);
      __builtin_amdgcn_sched_barrier(0);
      mfma_half(fb0, fa0, true);
      // every fragment of the step is in registers: this wave's slab of the A stage is free again, and
      // the loads of step s + DA go into it (nobody else reads or writes that slab)
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the LDS reads above have returned
      issue_a(s + DA);
      // own loads of A(s+1) have landed (the younger A(s+2) .. A(s+DA) may be in flight); past the barrier
      // everyone's have, B's included, and every wave is done reading this step's stages
      if (s + DA < ksteps) wait_loads<(DA - 1) * LA>(); else wait_loads<0>();
      __builtin_amdgcn_s_barrier();
      if (s + 1 < ksteps) read_half(s + 1, 0, fb0, fa0);
      __builtin_amdgcn_sched_barrier(0);
      mfma_half(fb1, fa1, false);
      if (BLOCK) add_scaled(f_a, f_lo, f_hi);
      __builtin_amdgcn_sched_barrier(0);
    }

    // ---- the four waves' partial results meet in LDS (the stages are free: last barrier passed)
    v4f* area = (v4f*)lds;  // [wave][32x32 block][q][lane]
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int jb = 0; jb < NB; ++jb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          area[(((wave * MB + i) * NB + jb) * 4 + q) * 64 + lane] =
              (v4f){acc[i][jb][4 * q], acc[i][jb][4 * q + 1], acc[i][jb][4 * q + 2], acc[i][jb][4 * q + 3]};
    __syncthreads();
    const bool vec = ((p.ldc & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.c) & 7) == 0);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) {
        v4f sum = area[(((0 * MB + i) * NB + jb) * 4 + wave) * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) sum += area[(((w * MB + i) * NB + jb) * 4 + wave) * 64 + lane];
        const int m = m0 + i * 32 + l32, n = nq + 32 * jb;
        if (m < p.M && n < n_end) {
          float r[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float t = BLOCK ? sum[e] : sum[e] * sa[i];
            r[e] = BLOCK ? t : p.bias ? __builtin_fmaf(t, sb[jb][e], bias_f[jb][e]) : t * sb[jb][e];
          }
          const uint32_t lo = pack_out_x2(r[0], r[1], p.out_f16), hi = pack_out_x2(r[2], r[3], p.out_f16);
          uint16_t* dst = p.c + (size_t)m * p.ldc + n;
          if (vec && n + 3 < n_end) {
            *(v2u*)dst = (v2u){lo, hi};
          } else {
            dst[0] = (uint16_t)lo;
            if (n + 1 < n_end) dst[1] = (uint16_t)(lo >> 16);
            if (n + 2 < n_end) dst[2] = (uint16_t)hi;
            if (n + 3 < n_end) dst[3] = (uint16_t)(hi >> 16);
          }
        }
      }
    }
  } else {
    // ---- loader wave for B: slab `wave - 4` of every step, 8 rows per load
    const int w = wave - 4;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.b) + (size_t)n0 * p.ldb, 0, (int)((uint32_t)(n_end - n0) * (uint32_t)p.ldb), 0x00020000);
    const uint32_t b_even = (uint32_t)ld_row * (uint32_t)p.ldb + chunk_even;
    const uint32_t b_odd = (uint32_t)ld_row * (uint32_t)p.ldb + (chunk_even ^ 64u);
    auto issue_b = [&](int s) {
      if (s >= ksteps) return;
      uint8_t* dst = lds + RA * STA + (s % RB) * STB + w * (BN * kStepK);
      const uint32_t koff = (uint32_t)step_of(s) * KS + (uint32_t)w * kStepK;
      const uint32_t even = lane_part(b_even, chunk_even, koff), odd = lane_part(b_odd, chunk_even ^ 64u, koff);
#pragma unroll
      for (int g = 0; g < LB; ++g)
        load_chunk_to_lds<!OFF_LINES>(rb, dst + g * 1024, (g & 1) ? odd : even, (uint32_t)(g * 8) * (uint32_t)p.ldb + koff);
    };
#pragma unroll
    for (int s = 0; s < DB; ++s) issue_b(s);
    if (ksteps > DB) wait_loads<(DB - 1) * LB>(); else wait_loads<0>();
    __builtin_amdgcn_s_barrier();
    for (int s = 0; s < ksteps; ++s) {
      issue_b(s + DB);
      if (s + DB < ksteps) wait_loads<(DB - 1) * LB>(); else wait_loads<0>();
      __builtin_amdgcn_s_barrier();
    }
    __syncthreads();  // the compute waves' hand-over of their partial results
  }
}

// ------------------------------------------------------------------------------------
// Pair kernel: M <= 16, N a multiple of 16 up to 8192 (at most two 16-row tiles of B per CU),
// K up to 8192 (any multiple of 16). The decode shapes proper: the whole launch is one or two
// tiles per workgroup, so there is no steady state to reach and what counts is the order in
// which the requests leave the CU.
//
// One workgroup of 16 waves per CU; wave w owns the K steps w, w+16, ... (SPW of them, those past
// K read as zeros) as in the persistent kernel above. Differences:
//  * A is not kept in registers: each wave copies its SPW-1 first steps of A straight from memory
//    into LDS, already in the order the MFMA lanes read them, and reads a step's fragment from there
//    when it multiplies; only its last step goes through the transpose buffer into registers (LDS:
//    3 x 32 KB of A at SPW = 4, 32 KB of transpose buffers, 32 KB of partial results).
//  * A tile's loads of B leave in one burst: step 0 of the first tile first, then A, then the rest
//    of the first tile together with step 0 of the second; the rest of the second tile follows the
//    first tile's reduction. A tile is 16 rows x K contiguous bytes, so a burst asks for one
//    contiguous region, and at no time is more than one tile per CU in flight: measured cold at
//    M=16, N=K=8192, this order 12.9 us against 13.4 us for the persistent kernel's rolling
//    prefetch (four steps per wave in flight all the time) and 13.9 us for the same rolling
//    prefetch with A in LDS; K = 4096 8.0 against 8.6 us, K = 2048 5.3 against 5.9, N = 4096 9.0
//    against 9.5, M = 1 12.2 against 12.6. Everything requested at once (both tiles) takes 14.9 us.
// All loads of B are range-checked buffer loads: a lane whose 16 bytes lie past K, and every lane of
// a tile that does not exist, asks for an offset outside the descriptor and gets zeros without a
// memory access, so the instruction stream is the same for every wave and the wait counts are exact.
// ------------------------------------------------------------------------------------
constexpr size_t pair_lds_bytes(int SPW) {
  return (size_t)kPersistWaves * 2048 * SPW + (size_t)2 * kPersistWaves * 1024;
}

// KTAIL: K is no multiple of 2048, so some waves own steps that lie (partly) past K and their lanes need a
// predicate per load; HAS_BIAS: a bias vector is added. Both are compile-time properties: this kernel's
// time hangs on how fast a wave gets its burst of loads out, and the few vector instructions either adds
// in front of the loads measured 0.3 and 0.1 us at M=16, N=K=8192.
// OFF_LINES: rows of B off the 128-byte lines, without the streaming policy (16x8192x4112 12.2 -> 11.0 us, 16x4096x4112 7.1 -> 5.8).
// BLOCK: the block-scaled product. A step's product is multiplied by its a_scale[0][kb] * b_scale[nb][kb] before it is added up; a wave's
// factors, one for each of its steps of either tile, lie in its first lanes (16x8192x8192 15.4 us with narrow tiles, 14.1 here, 16x8192x8176 18.9 and
// 16.7, 16x8192x4096 10.9 and 9.2, with one tile a workgroup 9.6).
template <int SPW, bool VEC, bool KTAIL, bool HAS_BIAS, bool OFF_LINES = false, bool BLOCK = false>
__global__ __launch_bounds__(kPersistWaves * 64) void gemm_skinny_pair_kernel(GemmParams p) {
  static_assert(!BLOCK || !HAS_BIAS, "the block-scaled product has no bias");
  constexpr int WAVES = kPersistWaves;
  constexpr int STEPS = WAVES * SPW;
  constexpr int A_LDS = SPW - 1;  // steps of A per wave that live in LDS
  fetch_arguments_now(p);
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* a_mine = lds + wave * (A_LDS * 2048);             // this wave's steps of A
  uint8_t* buf = lds + WAVES * A_LDS * 2048 + wave * 2048;   // this wave's transpose buffer (one 16 x 128 B step)
  v4f* red = (v4f*)(lds + WAVES * SPW * 2048);               // [2][WAVES][64] partial results

  // this workgroup's one or two tiles (quotient and remainder of tiles by workgroups come from the host)
  const int g = blockIdx.x;
  const int tile0 = g * p.tiles_m + min(g, p.tiles_n);
  const int count = p.tiles_m + (g < p.tiles_n ? 1 : 0);
  if (count <= 0) return;

  // byte offset of this wave's i-th K step inside a row; workgroups of one XCD start at different steps
  const int base_step = (wave + 2 * (g >> 3)) % STEPS;
  uint32_t kofs[SPW];
#pragma unroll
  for (int i = 0; i < SPW; ++i) {
    int s = base_step + WAVES * i;
    if (s >= STEPS) s -= STEPS;
    kofs[i] = (uint32_t)__builtin_amdgcn_readfirstlane(s * kStepK);
  }
  const int r16 = lane & 15, g4 = lane >> 4;
  const int ld_row = lane >> 3, ld_c = lane & 7;
  constexpr uint32_t kOutside = 0x80000000u;  // past every extent (the host keeps extents below 2^31)
  uint32_t b_lane[2], a_lane[2];
  int wr_off[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = h * 8 + ld_row;
    wr_off[h] = r * kStepK + ((ld_c ^ swz128(r)) * kChunk);
    b_lane[h] = (uint32_t)r * (uint32_t)p.ldb + ld_c * kChunk;
    // the direct-to-LDS copy puts lane l at position l of a 1 KB half step (8 rows x 128 bytes): the lane
    // asks for the chunk whose swizzled place that is; rows past M repeat the last one
    a_lane[h] = (uint32_t)min(r, p.M - 1) * (uint32_t)p.lda + (uint32_t)((ld_c ^ swz128(r)) * kChunk);
  }
  // the lane's chunk of a step lies inside K? (only the last step of a K that is no multiple of 128 cuts lanes off)
  auto in_k = [&](uint32_t step_off, int chunk) { return !KTAIL || step_off + (uint32_t)(chunk * kChunk) < (uint32_t)p.K; };
  const int rd0 = r16 * kStepK + (((2 * g4) ^ swz128(r16)) * kChunk);
  const int rd1 = r16 * kStepK + (((2 * g4 + 1) ^ swz128(r16)) * kChunk);

  const uint32_t tile_pitch = 16u * (uint32_t)p.ldb;
  const uintptr_t bb = reinterpret_cast<uintptr_t>(p.b) + (size_t)tile0 * tile_pitch;
  const uint8_t* b_base = reinterpret_cast<const uint8_t*>(
      ((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(bb >> 32)) << 32) |
      (uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bb));
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(b_base), 0, (int)((uint32_t)count * tile_pitch), 0x00020000);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(p.a), 0, (int)((uint32_t)p.M * (uint32_t)p.lda), 0x00020000);

  v4i land[2][SPW][2];
  auto fetch = [&](int t, int i) {
    const uint32_t so = (uint32_t)t * tile_pitch + kofs[i];
    const bool ok = t < count && in_k(kofs[i], ld_c);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#if defined(__HIP_DEVICE_COMPILE__)
      land[t][i][h] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)(ok ? b_lane[h] : kOutside), (int)so, OFF_LINES ? 0 : 2));
#else
      land[t][i][h] = (v4i){0, 0, 0, 0};
#endif
    }
  };
  fetch(0, 0);  // the first rows of B are asked for before anything else: they come from HBM
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < SPW; ++i) {
    uint8_t* dst = i < A_LDS ? a_mine + i * 2048 : buf;
    // (the chunk a lane fetches for LDS position ld_c of row r is ld_c ^ swz128(r))
#pragma unroll
    for (int h = 0; h < 2; ++h)
      load_chunk_to_lds<false>(ra, dst + h * 1024, in_k(kofs[i], ld_c ^ swz128(h * 8 + ld_row)) ? a_lane[h] : kOutside, kofs[i]);
  }
  __builtin_amdgcn_sched_barrier(0);
  // Wave j finishes tile j: lane (m = lane % 16, quad lane / 16) owns C[m, 16*tile + 4*(lane/16) .. +3] (waves
  // without a result read the run's last tile and drop it). Its scales and bias come from memory nobody has
  // touched yet, so they are asked for here, while the wave waits for A anyway - but the wait below must not
  // include them (it holds the burst back: 0.3 us at M=16, N=K=8192), so it has to know how many load
  // instructions they are. With aligned vectors that is exact: one buffer load each through descriptors of
  // their own (nothing the compiler could merge or split). The unaligned form asks behind the burst instead.
  const int fin_n = (tile0 + min(wave, count - 1)) * 16 + 4 * g4;
  float fin_sa = 0.f, sb_raw[4] = {0.f, 0.f, 0.f, 0.f};
  uint16_t bias_raw[4] = {0, 0, 0, 0};
  if constexpr (BLOCK) {
    // lane t * SPW + i: step i of tile t (a step past K has no block: its factors are outside both vectors and read as zeros)
    const uint32_t blocks = (uint32_t)(p.K + kStepK - 1) / kStepK;
    uint32_t kb = (uint32_t)(base_step + WAVES * (lane % SPW));
    if (kb >= STEPS) kb -= STEPS;
    const uint32_t nb = (uint32_t)(tile0 + min(lane / SPW, 1)) / (kStepK / 16);
    const bool inside = kb < blocks && nb < ((uint32_t)p.N + kStepK - 1) / kStepK;
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.a_scale), 0, (int)(blocks * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.b_scale), 0, (int)(((uint32_t)p.N + kStepK - 1) / kStepK * blocks * 4u), 0x00020000);
    fin_sa = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, (int)(inside ? kb * 4u : kOutside), 0, 0));
    sb_raw[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsb, (int)(inside ? (nb * blocks + kb) * 4u : kOutside), 0, 0));
#endif
    __builtin_amdgcn_sched_barrier(0);
    wait_loads<2>();
  } else if constexpr (VEC) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.a_scale), 0, p.M * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.b_scale), 0, p.N * 4, 0x00020000);
    fin_sa = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, min(r16, p.M - 1) * 4, 0, 0));
    const v4f s4 = load_f32x4_checked(rsb, (uint32_t)fin_n * 4u);
#pragma unroll
    for (int x = 0; x < 4; ++x) sb_raw[x] = s4[x];
    if (HAS_BIAS) {
      const __amdgpu_buffer_rsrc_t rbias = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.bias), 0, p.N * 2, 0x00020000);
      const us4 b4 = load_u16x4_checked(rbias, (uint32_t)fin_n * 2u);
#pragma unroll
      for (int x = 0; x < 4; ++x) bias_raw[x] = b4[x];
    }
#endif
    __builtin_amdgcn_sched_barrier(0);
    // A has landed once everything in front of those two or three loads has (loads return in order)
    wait_loads<2 + (HAS_BIAS ? 1 : 0)>();
  } else {
    wait_loads<0>();
  }
  v8i fa_last;
  {
    const v4i lo = *(const v4i*)(buf + rd0);
    const v4i hi = *(const v4i*)(buf + rd1);
    fa_last = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): in registers before the buffer is written again
  }
  __builtin_amdgcn_sched_barrier(0);

  auto consume = [&](int t, int i, v4f& acc) {
    *(v4i*)(buf + wr_off[0]) = land[t][i][0];
    *(v4i*)(buf + wr_off[1]) = land[t][i][1];
    const v4i lo = *(const v4i*)(buf + rd0);
    const v4i hi = *(const v4i*)(buf + rd1);
    const v8i fb = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    v8i fa = fa_last;
    if (i < A_LDS) {
      const v4i alo = *(const v4i*)(a_mine + i * 2048 + rd0);
      const v4i ahi = *(const v4i*)(a_mine + i * 2048 + rd1);
      fa = (v8i){alo[0], alo[1], alo[2], alo[3], ahi[0], ahi[1], ahi[2], ahi[3]};
    }
    if constexpr (BLOCK) {
      const v4f product = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
      const float factor = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fin_sa * sb_raw[0]), t * SPW + i));
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[x] = __builtin_fmaf(product[x], factor, acc[x]);
    } else {
      acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, acc, 0, 0, 0, 0, 0, 0);
    }
  };
  // tile 0: the rest of its loads in one burst, the first step of tile 1 behind them
#pragma unroll
  for (int i = 1; i < SPW; ++i) fetch(0, i);
  fetch(1, 0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!VEC && !BLOCK) {  // (element by element: a count the compiler may change, so behind the burst)
    fin_sa = p.a_scale[min(r16, p.M - 1)];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      sb_raw[x] = p.b_scale[fin_n + x];
      if (HAS_BIAS) bias_raw[x] = p.bias[fin_n + x];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // the 16 partial results of tile j meet in LDS (one area per tile); wave j adds them in wave order and stores
  auto finish = [&](int j, const v4f& acc) {
    v4f* area = red + j * (WAVES * 64);
    area[wave * 64 + lane] = acc;
    __syncthreads();
    if (wave == j) {
      const v4f* part = area + lane;
      v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int w0 = 0; w0 < WAVES; w0 += 8) {  // eight partials in flight at a time
#pragma unroll
        for (int w = 0; w < 8; ++w) sum += part[(w0 + w) * 64];
      }
      if (r16 < p.M) {
        float r[4];
#pragma unroll
        for (int x = 0; x < 4; ++x)
          r[x] = BLOCK      ? sum[x]
                 : HAS_BIAS ? __builtin_fmaf(sum[x] * fin_sa, sb_raw[x], bf16_to_f32(bias_raw[x]))
                            : sum[x] * fin_sa * sb_raw[x];
        const uint32_t lo = pack_out_x2(r[0], r[1], p.out_f16), hi = pack_out_x2(r[2], r[3], p.out_f16);
        uint16_t* dst = p.c + (size_t)r16 * p.ldc + (tile0 + j) * 16 + 4 * g4;
        if (VEC) {
          *(v2u*)dst = (v2u){lo, hi};
        } else {
          dst[0] = (uint16_t)lo; dst[1] = (uint16_t)(lo >> 16);
          dst[2] = (uint16_t)hi; dst[3] = (uint16_t)(hi >> 16);
        }
      }
    }
  };

  v4f acc0 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < SPW; ++i) consume(0, i, acc0);
  __builtin_amdgcn_sched_barrier(0);
  finish(0, acc0);
  __builtin_amdgcn_sched_barrier(0);
  // tile 1 (loads that ask for nothing when there is none: the instruction stream stays the same)
#pragma unroll
  for (int i = 1; i < SPW; ++i) fetch(1, i);
  __builtin_amdgcn_sched_barrier(0);
  if (count > 1) {
    v4f acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SPW; ++i) consume(1, i, acc1);
    finish(1, acc1);
  }
}

// ------------------------------------------------------------------------------------
// Row-wise quantiser: one workgroup per row, two passes over the row (amax, then scale
// and convert). e4m3fn encoding is done with integer arithmetic so the rounding
// (nearest, ties to even, subnormals below 2^-6) does not depend on conversion hardware.
// ------------------------------------------------------------------------------------
__device__ __forceinline__ uint8_t f32_to_e4m3fn_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  const uint32_t sign = (u >> 24) & 0x80u;
  const uint32_t mag = u & 0x7fffffffu;
  if (mag > 0x7f800000u) return (uint8_t)(sign | 0x7fu);  // NaN
  if (mag >= 0x43e80000u) {                                // |f| >= 464: beyond the last finite code
    return (uint8_t)(sign | (mag == 0x43e80000u ? 0x7eu : 0x7fu));
  }
  if (mag < 0x3c800000u) {  // |f| < 2^-6: subnormal target, spacing 2^-9
    const float scaled = __uint_as_float(mag) * 512.0f;  // exact
    const float rounded = __builtin_rintf(scaled);       // ties to even
    return (uint8_t)(sign | (uint32_t)rounded);          // 8 -> 0x08 = 2^-6, the first normal
  }
  // normal: keep 3 mantissa bits, round to nearest even on the 20 dropped bits
  uint32_t v = mag + 0x7ffffu + ((mag >> 20) & 1u);
  v >>= 20;                                // exponent(8) | mantissa(3)
  v -= (uint32_t)(127 - 7) << 3;           // rebias
  return (uint8_t)(sign | v);
}

// A reduction over the wave, in every lane: each lane's value with that of the lane whose number differs in one bit, from bit 5 down to bit 0. In the
// register file: __shfl_xor goes through LDS, six round trips in a row (0.1 to 0.3 us of a call of few rows: RMSNorm 32x8192, which has two
// reductions, 4.95 -> 4.64 us in four rounds of 256 lanes, SiLU-mul 32x8192 3.76 -> 3.63).
template <typename Op>
__device__ __forceinline__ float row_reduce(float v, Op op) {  // bits 3 to 0: within each row of 16 lanes
#if defined(__HIP_DEVICE_COMPILE__)
  auto dpp = [](float from, float old, auto ctrl, auto banks) -> float {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(from), decltype(ctrl)::value, 0xf, decltype(banks)::value, false));
  };
  using std::integral_constant;
  v = op(v, dpp(v, v, integral_constant<int, 0x128>{}, integral_constant<int, 0xf>{}));  // row_ror:8
  const float up = dpp(v, v, integral_constant<int, 0x104>{}, integral_constant<int, 0x5>{});  // row_shl:4 into the even fours
  v = op(v, dpp(v, up, integral_constant<int, 0x114>{}, integral_constant<int, 0xa>{}));       // row_shr:4 into the odd ones
  v = op(v, dpp(v, v, integral_constant<int, 0x4E>{}, integral_constant<int, 0xf>{}));         // quad_perm [2, 3, 0, 1]
  v = op(v, dpp(v, v, integral_constant<int, 0xB1>{}, integral_constant<int, 0xf>{}));         // quad_perm [1, 0, 3, 2]
#endif
  return v;
}
// Either half of a wave, and either row of two, in both: {lower, lower} and {upper, upper}.
struct Halves {
  float lower, upper;
};
__device__ __forceinline__ Halves halves_of_wave(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto both = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
  return {__int_as_float(both[0]), __int_as_float(both[1])};
#else
  return {v, v};
#endif
}
__device__ __forceinline__ Halves rows_of_pair(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto both = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
  return {__int_as_float(both[0]), __int_as_float(both[1])};
#else
  return {v, v};
#endif
}
template <typename Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
  const Halves halves = halves_of_wave(v);
  v = op(halves.lower, halves.upper);
  const Halves rows = rows_of_pair(v);
  return row_reduce(op(rows.lower, rows.upper), op);
}

template <typename SrcT>
struct SrcTraits;
// fp32 source: every step rounds to fp32 once, as the eager PyTorch program does.
template <>
struct SrcTraits<float> {
  static __device__ __forceinline__ float load(const float* p) { return *p; }
  static __device__ __forceinline__ float round(float v) { return v; }
};
// bf16 source: PyTorch evaluates each elementwise op in fp32 and rounds its result back to
// bf16, so amax, the scale, the scaled value and the inverse scale each pass through bf16.
template <>
struct SrcTraits<uint16_t> {
  static __device__ __forceinline__ float load(const uint16_t* p) { return bf16_to_f32(*p); }
  static __device__ __forceinline__ float round(float v) { return bf16_to_f32(f32_to_bf16_rne(v)); }
};

// max(a, b) that returns NaN when either operand is NaN (torch.max does; fmaxf drops the NaN).
// One gfx950 instruction (v_maximum3_f32).
__device__ __forceinline__ float max_keep_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// The row's quantisation scale from its absolute maximum, as eager PyTorch computes it:
// `448.0 / clamp(amax, 1e-12)` evaluates as reciprocal * 448, and clamp keeps a NaN (so a row
// holding a NaN gets a NaN scale, a row holding an infinity the scale 0).
template <typename SrcT>
__device__ __forceinline__ float row_scale(float amax) {
  using T = SrcTraits<SrcT>;
  const float floor_ = T::round(1e-12f);
  const float clamped = amax < floor_ ? floor_ : amax;  // false for NaN: it stays
  const float recip = T::round(1.0f / clamped);
  return T::round(recip * 448.0f);
}

// One element the way the PyTorch program treats it, NaN included: scale, clamp to +-448 (a NaN
// passes the clamp), round to e4m3fn with the integer encoder (NaN -> 0x7f with the sign kept).
template <typename SrcT>
__device__ __forceinline__ uint8_t quantize_one(float x, float scale) {
  using T = SrcTraits<SrcT>;
  float v = T::round(x * scale);
  v = v < -448.0f ? -448.0f : v;
  v = v > 448.0f ? 448.0f : v;
  return f32_to_e4m3fn_rne(v);
}

template <typename SrcT>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const SrcT* x, uint8_t* xq,
                                                            float* inv_scale, int K, long ldx,
                                                            long ldq) {
  using T = SrcTraits<SrcT>;
  __shared__ float wave_max[4];
  const long row = blockIdx.x;
  const SrcT* xr = x + row * ldx;
  uint8_t* qr = xq + row * ldq;

  float amax = 0.0f;
  for (int k = threadIdx.x; k < K; k += 256) amax = max_keep_nan(amax, fabsf(T::load(xr + k)));
  amax = wave_reduce(amax, [](float a, float b) { return max_keep_nan(a, b); });
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = max_keep_nan(max_keep_nan(wave_max[0], wave_max[1]), max_keep_nan(wave_max[2], wave_max[3]));

  const float scale = row_scale<SrcT>(amax);
  if (threadIdx.x == 0) inv_scale[row] = T::round(1.0f / scale);
  for (int k = threadIdx.x; k < K; k += 256) qr[k] = quantize_one<SrcT>(T::load(xr + k), scale);
}

// Vector form of the quantiser for 16-byte aligned rows: one workgroup per row, every lane
// moves 16 source bytes per load (a wave-wide load covers whole lines). The first CACHE
// chunks a lane reads stay in registers between the amax pass and the convert pass, so rows
// of up to THREADS*CACHE chunks are read from memory once; the rest of a longer row is read
// again (from cache). The e4m3fn rounding is done by the gfx950 pack-convert instruction
// (OCP format, round to nearest even) on values already clamped to +-448.
template <typename SrcT>
struct VecTraits;
template <>
struct VecTraits<float> {
  static constexpr int EPV = 4;  // elements per 16-byte chunk
  static __device__ __forceinline__ void unpack(const v4i& c, float (&f)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = __int_as_float(c[e]);
  }
};
template <>
struct VecTraits<uint16_t> {
  static constexpr int EPV = 8;
  static __device__ __forceinline__ void unpack(const v4i& c, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = __uint_as_float((uint32_t)c[e] << 16);
      f[2 * e + 1] = __uint_as_float((uint32_t)c[e] & 0xffff0000u);
    }
  }
};

// THREADS lanes per row, ROWS rows per workgroup. Rows short enough for one wave's registers take
// THREADS = 64 with several rows per workgroup: no LDS, no barrier, and a fraction of the workgroups
// (short rows are bound by the rate at which workgroups start, about one per 1.2-2 ns).
// ANY: rows that start at any element and end anywhere (K >= one chunk): the same passes on unaligned accesses, which cost
// a wave-wide load one line more. The last chunk is the row's last 16 bytes, which may repeat part of the chunk before it:
// harmless for the maximum, and the codes come out and are stored the same twice. Its loads do without the streaming
// policy (neighbouring waves share the lines at their borders).
template <typename SrcT, int CACHE, int THREADS, int ROWS = 1, bool ANY = false>
__global__ __launch_bounds__(THREADS* ROWS) void quantize_rows_vec_kernel(const SrcT* x, uint8_t* xq,
                                                                        float* inv_scale, int K, long ldx,
                                                                        long ldq, long rows) {
  static_assert(ROWS == 1 || THREADS == 64, "several rows per workgroup: one wave each");
  using T = SrcTraits<SrcT>;
  using V = VecTraits<SrcT>;
  constexpr int EPV = V::EPV;
  __shared__ float wave_max[THREADS / 64];
  const long row = (long)blockIdx.x * ROWS + (ROWS > 1 ? (long)(threadIdx.x >> 6) : 0);
  if (ROWS > 1 && row >= rows) return;  // (whole waves; this form has no barrier)
  using Chunk = std::conditional_t<ANY, v4i_any, v4i>;
  using Codes = std::conditional_t<ANY, v4i_any, v4i>;
  using Codes8 = std::conditional_t<ANY, v2u_any, v2u>;
  using Codes4 = std::conditional_t<ANY, u32_any, uint32_t>;
  const SrcT* xr = x + row * ldx;
  uint8_t* qr = xq + row * ldq;
  const int nchunks = ANY ? (K + EPV - 1) / EPV : K / EPV;
  // first element of chunk c
  auto start = [&](int c) { return ANY ? min(c * EPV, K - EPV) : c * EPV; };
  auto load = [&](int c) -> v4i { return *(const Chunk*)(xr + start(c)); };
  const int tid = ROWS > 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;

  v4i cache[CACHE];
  float amax = 0.0f;
  auto fold = [&](const v4i& c) {
    float f[EPV];
    V::unpack(c, f);
#pragma unroll
    for (int e = 0; e < EPV; ++e) amax = max_keep_nan(amax, fabsf(f[e]));
  };
#pragma unroll
  for (int i = 0; i < CACHE; ++i) {
    // past the row's end a lane re-reads the last chunk: harmless for the maximum, never
    // stored, and it keeps the loads free of branches
    const int c = min(tid + THREADS * i, nchunks - 1);
    if constexpr (ANY) cache[i] = load(c);
    else cache[i] = __builtin_nontemporal_load((const v4i*)xr + c);
  }
#pragma unroll
  for (int i = 0; i < CACHE; ++i) fold(cache[i]);
  for (int c = tid + THREADS * CACHE; c < nchunks; c += THREADS) fold(load(c));
  amax = wave_reduce(amax, [](float a, float b) { return max_keep_nan(a, b); });
  if (THREADS > 64) {
    if ((tid & 63) == 0) wave_max[tid >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) amax = max_keep_nan(amax, wave_max[w]);
  }

  const float scale = row_scale<SrcT>(amax);
  if (tid == 0) inv_scale[row] = T::round(1.0f / scale);
  // A row that holds a NaN or an infinity (the whole workgroup sees the same amax) takes the
  // element-by-element route, whose clamp and encoder carry NaN through as PyTorch does; the
  // pack-convert route below is for finite rows.
  if (!(amax < __builtin_inff())) {
    const SrcT* xs = x + row * ldx;
    for (int k = tid; k < K; k += THREADS) qr[k] = quantize_one<SrcT>(T::load(xs + k), scale);
    return;
  }

  auto convert = [&](const v4i& src, uint32_t (&out)[EPV / 4]) {
    float f[EPV];
    V::unpack(src, f);
#pragma unroll
    for (int e = 0; e < EPV; ++e) f[e] = fminf(fmaxf(T::round(f[e] * scale), -448.0f), 448.0f);
#pragma unroll
    for (int w = 0; w < EPV / 4; ++w) {
      int packed = __builtin_amdgcn_cvt_pk_fp8_f32(f[4 * w], f[4 * w + 1], 0, false);
      packed = __builtin_amdgcn_cvt_pk_fp8_f32(f[4 * w + 2], f[4 * w + 3], packed, true);
      out[w] = (uint32_t)packed;
    }
  };
  auto convert_store = [&](const v4i& src, int c) {
    uint32_t out[EPV / 4];
    convert(src, out);
    if (EPV == 4) *(Codes4*)(qr + start(c)) = out[0];
    else *(Codes8*)(qr + start(c)) = (v2u){out[0], out[EPV / 4 - 1]};
  };
  // A chunk turns into EPV output bytes per lane (4 or 8): too little per store instruction.
  // BATCH = 16 / EPV consecutive rounds of the cached chunks are therefore gathered through
  // a wave-private LDS strip (LDS executes a wave's operations in order: no barrier) and
  // leave as one 16-byte store per lane, BATCH runs of 1024 / BATCH contiguous bytes each.
  constexpr int BATCH = 16 / EPV;
  __shared__ __attribute__((aligned(16))) uint8_t strip[THREADS * ROWS / 64][1024];
  uint8_t* mine = strip[threadIdx.x >> 6];
  const int lane = tid & 63;
  constexpr int LPR = 64 / BATCH;  // lanes that store one round's bytes of this wave
#pragma unroll
  for (int i0 = 0; i0 < CACHE; i0 += BATCH) {
    if (i0 + BATCH <= CACHE && THREADS * (i0 + BATCH) <= K / EPV) {  // uniform: every lane of every wave has all BATCH rounds
#pragma unroll
      for (int b = 0; b < BATCH; ++b) {
        uint32_t out[EPV / 4];
        convert(cache[min(i0 + b, CACHE - 1)], out);
        if (EPV == 4) *(uint32_t*)(mine + b * 256 + lane * 4) = out[0];
        else *(v2u*)(mine + b * 512 + lane * 8) = (v2u){out[0], out[EPV / 4 - 1]};
      }
      const int b = lane / LPR, piece = lane % LPR;
      const v4i bytes = *(const v4i*)(mine + lane * 16);
      // round i0+b, this wave's 64 chunks start at chunk THREADS*(i0+b) + 64*wave
      *(Codes*)(qr + ((size_t)THREADS * (i0 + b) + (tid & ~63)) * EPV + piece * 16) = bytes;
    } else {
#pragma unroll
      for (int b = 0; b < BATCH && i0 + b < CACHE; ++b) {
        const int c = tid + THREADS * (i0 + b);
        if (c < nchunks) convert_store(cache[i0 + b], c);
      }
    }
  }
  for (int c = tid + THREADS * CACHE; c < nchunks; c += THREADS) convert_store(load(c), c);
}


// ------------------------------------------------------------------------------------
// Block-wise quantiser: one scale per 128 x 128 block of the source, the input step of the
// block-scaled GEMM. One workgroup per block keeps the block in registers between the
// maximum and the conversion, so the source is read once. Follows the eager PyTorch program of
// tritonbench/operators/fp8_gemm_blockwise/operator.py:86-118:
//   amax  = max |x| over the block (elements past M or K count as zero), clamped from below
//           with 1e-12 in the source type, then widened to f32
//   scale = fl(fl(1 / amax) * 448) in f32 (how PyTorch evaluates 448 / tensor); +inf -> 1
//   xq    = e4m3fn(fl(x * scale)), the product in f32 whatever the source type, no clamp
//           (|x * scale| cannot reach 464, the first value the cast turns into NaN)
//   inv   = fl(1 / scale)
// A block that holds a NaN comes out as NaN codes with a NaN inverse scale; a block that holds an
// infinity gets scale 0 and inverse scale +inf, its finite elements become zero, the infinities NaN.
// ------------------------------------------------------------------------------------
constexpr int kQuantBlock = 128;

template <typename SrcT>
__device__ __forceinline__ float block_scale(float amax) {
  const float floor_ = SrcTraits<SrcT>::round(1e-12f);
  const float clamped = amax < floor_ ? floor_ : amax;  // false for NaN: it stays
  const float scale = (1.0f / clamped) * 448.0f;
  return scale == __builtin_inff() ? 1.0f : scale;
}

// VEC: 16-byte source chunks (rows 16-byte aligned, K a whole number of chunks), 4- or 8-byte stores.
// Otherwise element by element, the block read twice (the second time from cache).
template <typename SrcT, bool VEC>
__global__ __launch_bounds__(256) void quantize_blocks_kernel(const SrcT* x, uint8_t* xq, float* inv_scale, int M,
                                                              int K, long ldx, long ldq, int grid_k) {
  using T = SrcTraits<SrcT>;
  using V = VecTraits<SrcT>;
  constexpr int EPV = V::EPV;
  constexpr int CPR = kQuantBlock / EPV;   // chunks per block row
  constexpr int RPP = 256 / CPR;           // block rows per pass of the workgroup
  constexpr int PASSES = kQuantBlock / RPP;
  __shared__ float wave_max[4];
  const int bk = blockIdx.x, bm = blockIdx.y;
  const int m0 = bm * kQuantBlock, k0 = bk * kQuantBlock;
  const int tid = threadIdx.x;
  const int chunk = tid % CPR, row0 = tid / CPR;

  v4i cache[VEC ? PASSES : 1];
  float amax = 0.0f;
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int r = m0 + row0 + i * RPP, c = k0 + chunk * EPV;
      const bool inside = r < M && c < K;
      // (outside the matrix a lane reads the block's first chunk, which exists, and drops it)
      const v4i got = __builtin_nontemporal_load((const v4i*)(x + (inside ? (long)r * ldx + c : (long)m0 * ldx + k0)));
      cache[i] = inside ? got : (v4i){0, 0, 0, 0};
      float f[EPV];
      V::unpack(cache[i], f);
#pragma unroll
      for (int e = 0; e < EPV; ++e) amax = max_keep_nan(amax, fabsf(f[e]));
    }
  } else {
    for (int idx = tid; idx < kQuantBlock * kQuantBlock; idx += 256) {
      const int r = m0 + idx / kQuantBlock, c = k0 + idx % kQuantBlock;
      if (r < M && c < K) amax = max_keep_nan(amax, fabsf(T::load(x + (long)r * ldx + c)));
    }
  }
  amax = wave_reduce(amax, [](float a, float b) { return max_keep_nan(a, b); });
  if ((tid & 63) == 0) wave_max[tid >> 6] = amax;
  __syncthreads();
  amax = max_keep_nan(max_keep_nan(wave_max[0], wave_max[1]), max_keep_nan(wave_max[2], wave_max[3]));

  const float scale = block_scale<SrcT>(amax);
  if (tid == 0) inv_scale[(long)bm * grid_k + bk] = 1.0f / scale;
  const bool finite = amax < __builtin_inff();  // false for NaN and infinity: the integer encoder carries them

  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int r = m0 + row0 + i * RPP, c = k0 + chunk * EPV;
      if (r >= M || c >= K) continue;
      float f[EPV];
      V::unpack(cache[i], f);
      uint32_t out[EPV / 4];
      if (finite) {
#pragma unroll
        for (int w = 0; w < EPV / 4; ++w) {
          // (the clamp changes nothing for a finite block; it keeps the pack-convert inside its range)
          float g[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) g[e] = fminf(fmaxf(f[4 * w + e] * scale, -448.0f), 448.0f);
          int packed = __builtin_amdgcn_cvt_pk_fp8_f32(g[0], g[1], 0, false);
          packed = __builtin_amdgcn_cvt_pk_fp8_f32(g[2], g[3], packed, true);
          out[w] = (uint32_t)packed;
        }
      } else {
#pragma unroll
        for (int w = 0; w < EPV / 4; ++w) {
          out[w] = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) out[w] |= (uint32_t)f32_to_e4m3fn_rne(f[4 * w + e] * scale) << (8 * e);
        }
      }
      uint8_t* dst = xq + (long)r * ldq + c;
      if (EPV == 4) *(uint32_t*)dst = out[0];
      else *(v2u*)dst = (v2u){out[0], out[EPV / 4 - 1]};
    }
  } else {
    for (int idx = tid; idx < kQuantBlock * kQuantBlock; idx += 256) {
      const int r = m0 + idx / kQuantBlock, c = k0 + idx % kQuantBlock;
      if (r < M && c < K) xq[(long)r * ldq + c] = f32_to_e4m3fn_rne(T::load(x + (long)r * ldx + c) * scale);
    }
  }
}

// ------------------------------------------------------------------------------------
// Fused front ends of the row-wise GEMM: the activation is normalised (RMSNorm with a weight
// vector) or gated (SiLU(x1) * x2) and quantised row-wise in one pass, so the bf16 row is read
// from memory once and nothing but the e4m3fn codes and one scale per row is written.
// One workgroup per row; a lane keeps the fp32 values of up to CACHE 16-byte chunks (8 bf16
// each) in registers across the passes: [sum of squares ->] value and row maximum -> convert.
// Rows longer than THREADS*CACHE chunks re-read and recompute the rest. All arithmetic is fp32:
//   RMSNorm   y = (x * rstd) * w,  rstd = 1 / sqrt(mean(x^2) + eps)
//   SiLU-mul  y = (x1 / (1 + exp(-x1))) * x2
// then the quantiser's arithmetic on y as on an fp32 tensor (row_scale<float>, clamp, RNE).
// ------------------------------------------------------------------------------------
constexpr int kFusedRmsNorm = 0, kFusedSiluMul = 1;

// A row's sum of squares is added up in an order that hangs on the row's length alone (in another order rstd can move by a unit in its last
// place, which sends exact ties between two codes the other way), so a row has the same codes however many rows the call has:
// as by this many lanes, of which lane o adds up chunks o, o + S, o + 2 S, ... element by element in one chain, then the lanes of each
// 64 pairwise from bit 5 of their numbers down to bit 0, then the 64s one after another.
constexpr int rms_sum_lanes(int64_t chunks) { return chunks <= 256 ? 64 : chunks <= 1024 ? 256 : chunks <= 4096 ? 512 : 1024; }
// Whether a form of the RMSNorm kernel asks for the weights beside x. (With 512 lanes and 8 chunks each the weights' registers cost more than
// the second trip, 8192 x 28672 245 us with them, 167 without, and 1024 lanes have 128 registers each and none to spare.)
constexpr bool rms_early_weights(int lanes, int chunks) { return lanes <= 256 || (lanes == 512 && chunks <= 4); }

template <int OP, int CACHE, int THREADS, int ROWS = 1>
__global__ __launch_bounds__(THREADS* ROWS) void fused_rowwise_quant_kernel(const uint16_t* x1, const uint16_t* x2,
                                                                             float eps, uint8_t* xq, float* inv_scale,
                                                                             int K, long ld1, long ld2, long ldq, long rows) {
  static_assert(ROWS == 1 || THREADS == 64, "several rows per workgroup: one wave each (as in the quantiser)");
  using V = VecTraits<uint16_t>;
  constexpr int EPV = 8;
  // Rows of up to 256 chunks on 256 lanes, with one chunk each: the order's 64 lanes are 64 chains that four lanes of a wave hand on, one in each
  // row of 16, where that is one instruction. (All of them add at each turn. 32x2048 2.71 us, on 64 lanes with four chunks 3.26.)
  constexpr int SUM_LANES = OP == kFusedRmsNorm ? rms_sum_lanes((int64_t)THREADS * CACHE) : THREADS;
  constexpr bool HANDED_ON = SUM_LANES != THREADS;
  static_assert(!HANDED_ON || (SUM_LANES == 64 && THREADS == 256 && CACHE == 1), "the other forms have the lanes of the order");
  __shared__ float wave_part[THREADS / 64];
  __shared__ __attribute__((aligned(16))) float sum_part[HANDED_ON ? SUM_LANES : THREADS / 64];  // (of its own: no wait for the other's readers)
  const long row = (long)blockIdx.x * ROWS + (ROWS > 1 ? (long)(threadIdx.x >> 6) : 0);
  if (ROWS > 1 && row >= rows) return;  // (whole waves; this form has no barrier)
  const v4i* r1 = (const v4i*)(x1 + row * ld1);
  // RMSNorm: the weight vector, shared by all rows; SiLU-mul: the row of the second operand
  const v4i* r2 = (const v4i*)(OP == kFusedRmsNorm ? x2 : x2 + row * ld2);
  uint8_t* qr = xq + row * ldq;
  const int nchunks = K / EPV;
  const int tid = ROWS > 1 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  const int lane = tid & 63;
  // Round i of lane t is chunk first_chunk(t) + THREADS * i. (Handed on: the rows of a wave have turns 0, 1, 3, 2, so that each finds what it goes
  // on with in the other row of its pair or in the other half.)
  auto turn_of = [](int t) { return (t & 63) / 16 ^ (t & 63) / 32; };
  auto first_chunk = [&](int t) { return HANDED_ON ? (t >> 6) * 16 + t % 16 + SUM_LANES * turn_of(t) : t; };
  const int at = first_chunk(tid);
  const int rest = HANDED_ON ? nchunks : tid + THREADS * CACHE;  // what the registers do not hold (0.1 us of a call of 2 where there never is any)
  // (hardware exponential and reciprocal, about one ulp each: the result is rounded to 4 significant
  // bits next; the library exponential costs six times the instructions and a correctly rounded
  // quotient ten, which together made the kernel compute-bound)
  auto silu_mul = [](float a, float b) -> float { return (a * __builtin_amdgcn_rcpf(1.0f + __expf(-a))) * b; };

  float vals[CACHE][EPV];
  constexpr bool EARLY_WEIGHTS = OP == kFusedRmsNorm && rms_early_weights(THREADS, CACHE);
  v4i wts[EARLY_WEIGHTS ? CACHE : 1];
  float rstd = 0.0f;
  if (OP == kFusedRmsNorm) {
    // pass 1: x to registers, sum of squares (lanes past the row's end re-read the last chunk and
    // leave it out of the sum). The weights of the cached chunks are asked for here as well: fetched
    // after the reduction they would put a second trip to the L2 on every row's critical path.
    if (EARLY_WEIGHTS) {
#pragma unroll
      for (int i = 0; i < CACHE; ++i) wts[EARLY_WEIGHTS ? i : 0] = r2[min(at + THREADS * i, nchunks - 1)];
    }
#pragma unroll
    for (int i = 0; i < CACHE; ++i) V::unpack(__builtin_nontemporal_load(r1 + min(at + THREADS * i, nchunks - 1)), vals[i]);
    auto add_squares = [](const float (&f)[EPV], float s) -> float {
#pragma unroll
      for (int e = 0; e < EPV; ++e) s = __builtin_fmaf(f[e], f[e], s);
      return s;
    };
    float ss = 0.0f;
    auto add = [](float a, float b) { return a + b; };
    if constexpr (HANDED_ON) {
#pragma unroll
      for (int turn = 0; turn < 4; ++turn) {
        if (turn > 0) ss = turn == 1 ? rows_of_pair(ss).lower : turn == 2 ? halves_of_wave(ss).lower : rows_of_pair(ss).upper;
        const float with = add_squares(vals[0], ss);
        ss = at < nchunks ? with : ss;
      }
      // the chains' sums, those of the lanes that are added first beside one another
      if (turn_of(tid) == 3) sum_part[lane % 16 * 4 + (tid >> 6)] = ss;
      __syncthreads();
      const v4f four = *(const v4f*)(sum_part + lane % 16 * 4);
      ss = row_reduce((four[0] + four[2]) + (four[1] + four[3]), add);
    } else {
#pragma unroll
      for (int i = 0; i < CACHE; ++i) {
        const float with = add_squares(vals[i], ss);
        ss = at + THREADS * i < nchunks ? with : ss;
      }
      for (int c = rest; c < nchunks; c += THREADS) {
        float f[EPV];
        V::unpack(r1[c], f);
        ss = add_squares(f, ss);
      }
      ss = wave_reduce(ss, add);
      if (THREADS > 64) {
        if (lane == 0) sum_part[tid >> 6] = ss;
        __syncthreads();
        ss = sum_part[0];
#pragma unroll
        for (int w = 1; w < THREADS / 64; ++w) ss += sum_part[w];
      }
    }
    rstd = 1.0f / sqrtf(ss / (float)K + eps);
  }
  // value of chunk c from its raw operands
  auto value = [&](const float (&a)[EPV], const float (&b)[EPV], float (&y)[EPV]) {
#pragma unroll
    for (int e = 0; e < EPV; ++e) y[e] = OP == kFusedRmsNorm ? (a[e] * rstd) * b[e] : silu_mul(a[e], b[e]);
  };
  // pass 2: values (kept for the cached chunks) and the row's absolute maximum
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < CACHE; ++i) {
    const int c = min(at + THREADS * i, nchunks - 1);
    float a[EPV], b[EPV];
    if (OP == kFusedRmsNorm) {
#pragma unroll
      for (int e = 0; e < EPV; ++e) a[e] = vals[i][e];
    } else {
      V::unpack(__builtin_nontemporal_load(r1 + c), a);
    }
    V::unpack(EARLY_WEIGHTS ? wts[EARLY_WEIGHTS ? i : 0] : OP == kFusedRmsNorm ? r2[c] : __builtin_nontemporal_load(r2 + c), b);
    value(a, b, vals[i]);
#pragma unroll
    for (int e = 0; e < EPV; ++e) amax = max_keep_nan(amax, fabsf(vals[i][e]));
  }
  for (int c = rest; c < nchunks; c += THREADS) {
    float a[EPV], b[EPV], y[EPV];
    V::unpack(r1[c], a);
    V::unpack(r2[c], b);
    value(a, b, y);
#pragma unroll
    for (int e = 0; e < EPV; ++e) amax = max_keep_nan(amax, fabsf(y[e]));
  }
  amax = wave_reduce(amax, [](float a, float b) { return max_keep_nan(a, b); });
  if (THREADS > 64) {
    if (lane == 0) wave_part[tid >> 6] = amax;
    __syncthreads();
    amax = wave_part[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) amax = max_keep_nan(amax, wave_part[w]);
  }

  const float scale = row_scale<float>(amax);
  if (tid == 0) inv_scale[row] = 1.0f / scale;
  const bool finite_row = amax < __builtin_inff();  // a NaN or an infinity takes the integer encoder, which carries NaN through
  auto convert_store = [&](const float (&y)[EPV], int c) {
    if (finite_row) {
      float f[EPV];
#pragma unroll
      for (int e = 0; e < EPV; ++e) f[e] = fminf(fmaxf(y[e] * scale, -448.0f), 448.0f);
      int lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
      lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
      int hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
      hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
      *(v2u*)(qr + (size_t)c * 8) = (v2u){(uint32_t)lo, (uint32_t)hi};
    } else {
#pragma unroll
      for (int e = 0; e < EPV; ++e) qr[(size_t)c * 8 + e] = quantize_one<float>(y[e], scale);
    }
  };
  // pass 3: convert. Two consecutive rounds of cached chunks meet in a wave-private LDS strip and
  // leave as one 16-byte store per lane (LDS executes a wave's operations in order: no barrier).
  __shared__ __attribute__((aligned(16))) uint8_t strip[THREADS * ROWS / 64][1024];
  uint8_t* mine = strip[threadIdx.x >> 6];
#pragma unroll
  for (int i0 = 0; i0 < CACHE; i0 += 2) {
    if (i0 + 2 <= CACHE && finite_row && THREADS * (i0 + 2) <= nchunks) {  // uniform: every lane of every wave has both rounds
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        float f[EPV];
#pragma unroll
        for (int e = 0; e < EPV; ++e) f[e] = fminf(fmaxf(vals[min(i0 + b, CACHE - 1)][e] * scale, -448.0f), 448.0f);
        int lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], lo, true);
        int hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], hi, true);
        *(v2u*)(mine + b * 512 + lane * 8) = (v2u){(uint32_t)lo, (uint32_t)hi};
      }
      const int b = lane / 32, piece = lane % 32;
      const v4i bytes = *(const v4i*)(mine + lane * 16);
      *(v4i*)(qr + (size_t)(THREADS * (i0 + b) + first_chunk((tid & ~63) + 2 * piece)) * EPV) = bytes;
    } else {
#pragma unroll
      for (int b = 0; b < 2 && i0 + b < CACHE; ++b) {
        const int c = at + THREADS * (i0 + b);
        if (c < nchunks) convert_store(vals[i0 + b], c);
      }
    }
  }
  for (int c = rest; c < nchunks; c += THREADS) {
    float a[EPV], b[EPV], y[EPV];
    V::unpack(r1[c], a);
    V::unpack(r2[c], b);
    value(a, b, y);
    convert_store(y, c);
  }
}

// ------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------
int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(mi355x_shared::err, sizeof(mi355x_shared::err), fmt, ap);
  va_end(ap);
  return code;
}

constexpr int kSkinnyMaxM = 64;

// A launch holds fewer than 2^32 lanes. Kernels whose grid grows with an operand (rather than with the chip) are taken
// only where theirs does; beyond, the form with the next larger tiles runs.
constexpr bool grid_fits(int64_t workgroups, int64_t lanes) { return workgroups * lanes <= (int64_t)UINT32_MAX; }

int check_shape(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 1) return fail(MI355X_FP8_EINVAL, "M, N, K must be >= 1 (got %lld, %lld, %lld)",
                                           (long long)M, (long long)N, (long long)K);
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
    return fail(MI355X_FP8_ENOTSUP, "dimension exceeds 2^31-1");
  return MI355X_FP8_OK;
}
// What the MFMA families ask of the operands beyond check_shape (the generic family asks nothing).
int check_fast_shape(int64_t K) {
  if (K % 16 != 0) return fail(MI355X_FP8_ENOTSUP, "K must be a multiple of 16 (got %lld)", (long long)K);
  return MI355X_FP8_OK;
}

// ---- tiled-kernel plans: tile configuration x split-K factor
struct TileConfig {
  int bm, bn, wgs_per_cu;
  float us_per_step;        // one 128-byte K step of a work item, every workgroup slot busy
  float us_per_step_alone;  // the same with at most one workgroup per CU
  float us_per_item;        // pipeline refill + epilogue of one work item
  float stream_bytes_per_us;  // operand bytes per microsecond the configuration can stream from HBM
  float wg_stream_share;      // what one workgroup can stream, in units of 1/256 of that rate
};
constexpr int kNumTileConfigs = 7;
static_assert(kNumTileConfigs == mi355x_shared::kNumTiledParts, "one part function per tile configuration");
constexpr int kDeepSmallConfig = 6;  // 128x128 tiles with three steps in flight, one workgroup per CU
constexpr int kNumGroupedTileConfigs = 3;  // the grouped form uses the first three
// Measured on MI355X with normally distributed operands (clock under sustained MFMA load).
constexpr TileConfig kTileConfigs[kNumTileConfigs] = {
    {256, 256, tiled_wgs_per_cu(256, 256), 1.30f, 1.30f, 6.0f, 3.6e6f, 1.8f},
    {128, 128, tiled_wgs_per_cu(128, 128), 1.00f, 0.60f, 5.0f, 4.4e6f, 1.18f},
    {256, 128, tiled_wgs_per_cu(256, 128), 0.87f, 0.87f, 5.0f, 4.0e6f, 1.1f},
    {64, 256, tiled_wgs_per_cu(64, 256), 0.75f, 0.75f, 9.0f, 5.7e6f, 1.42f},
    // (one tile row against a wide panel: 128 x 57344 x 8192 75.2 us with 224 tiles, bound by the stream rate;
    // several tile rows: 512 x 16384 x 16384 125 us with 256 tiles, 4096 x 5120 x 13824 269 us with 640)
    // (a step and a tile's refill and epilogue, from launches that are not bound by the stream rate: 4096 x 2048 x 2048
    // 18.1 us with 256 tiles of 16 steps, 636 x 12288 x 6144 50.3 with 240 of 48, 512 x 16384 x 16384 125 with 256 of 128)
    {128, 256, tiled_wgs_per_cu(128, 256), 0.97f, 0.97f, 2.6f, 5.8e6f, 1.42f},
    // (panels whose 256-column tiles come to more than half a round with 256 rows each but fit one with 192:
    // 1024 x 10240 x 8192 73.3 us with 240 tiles, 2048 x 10240 x 8192 135.4 us with 440)
    // (one tile row against a wide panel: 192 x 57344 x 8192 89.2 us)
    // (one round of tiles costs 7 us beside its steps, not 9: plan_cost_us has it)
    {192, 256, tiled_wgs_per_cu(192, 256), 1.00f, 1.00f, 9.0f, 4.9e6f, 1.42f},
    // 128x128 tiles with loads three steps ahead (112 KB of LDS: one workgroup per CU), for launches of at most
    // one workgroup per CU, where a CU has one wave per SIMD and nothing but the depth of the ring to cover
    // the memory latency with. Operands from HBM, against the two-step form: 1024 x 2048 x 4096 25.4 -> 20.4 us
    // with 128 tiles, 512 x 4096 x 4096 25.6 -> 21.1, 1536 x 1536 x 4096 25.4 -> 20.6, 2048 x 2048 x 4096 27.2 ->
    // 23.0 with 256, 2048^3 15.9 -> 14.4; split (work items still at most one per CU): 1024 x 2048 x 8192 36.1 ->
    // 31.3 in two, 1024 x 2048 x 16384 67.3 -> 48.9 in two, 1024 x 1024 x 8192 36.3 -> 26.5 in two -> 23.0 in four.
    // Operands from the memory-side cache: 0.31 us per step instead of 0.49 (1024 x 2048 x 8192 29.1 -> 24.6).
    // A ring one step deeper measured the same. The step time is the one with operands from HBM and half the
    // CUs at work; plan_cost_us adds what a fuller chip costs.
    {128, 128, 1, 0.49f, 0.49f, 4.8f, 4.4e6f, 1.18f},
};

// The skinny kernel's run time for comparison with the tiled plans at M <= 64: a fixed part
// plus B streamed at a rate that falls with the number of 16-row blocks of A every workgroup
// has to pull through L1 beside its rows of B (measured, MB per microsecond). With three or
// four blocks the register budget leaves one workgroup per CU, and a last round of workgroups
// that fills only part of the CUs streams at that fraction of the rate.
inline bool persistent_skinny_fits(int64_t M, int64_t N, int64_t K);
// The pair kernel: up to 16 rows of A, at most two 16-row tiles of B per CU, K that fits the LDS.
inline bool pair_skinny_fits(int64_t M, int64_t N, int64_t K) {
  return M <= 16 && N % 16 == 0 && N <= 2 * 16 * kNumCu && K <= 4 * kPersistWaves * kStepK;
}
// The narrow-tile kernel. With all rows in one workgroup (M <= 64) its cost is one round of workgroups per
// 256 tiles (measured at N = 8192, cold: 9.8 / 14.3 / 43.0 us for K = 4096 / 8192 / 28672 with up to
// 32 rows of A, 17.1-17.9 / 49.9 us for K = 8192 / 28672 with up to 64).
// Up to 256 rows of A it runs in row blocks where that is one round of workgroups, one per CU
// (measured, K = 8192 unless given: 64x64 tiles 13.7 / 21.5 / 67.6 us for K = 4096 / 8192 / 28672 at
// M = 128, N = 8192; 64x32 tiles 10.7 / 16.0 / 24.2 us for K = 4096 / 8192 / 14336 at M = 128, N = 4096,
// 14.0 us at 192 x 1536; 32x32 tiles 12.6 us at 64 x 4096, 11.3 us at 128 x 2048, 11.0 us at 64 x 1024,
// 8.3 us at 64 x 4096 x 4096, 37.1 us at 64 x 4096 x 28672).
constexpr int kNarrowMaxM = 256;
inline bool narrow_fits(int64_t M, int64_t N, int64_t K) {
  (void)K;
  if (M <= kSkinnyMaxM) return true;
  const long tiles = ((N + 63) / 64 + kNumXcd - 1) / kNumXcd * kNumXcd, row_blocks = (M + 63) / 64;
  return M <= kNarrowMaxM && tiles * row_blocks <= kNumCu;
}
// The form for a shape: 32-row blocks of A per workgroup (the rows beyond them go to further row
// blocks) and 32-column blocks per tile. Up to 32 rows, and up to 64 on panels too wide for row
// blocks: all rows in one workgroup, tiles of narrow_tile_cols() columns (two blocks from 33 columns up).
// Otherwise the smallest tile whose row blocks are one round of workgroups: more CUs at work, and
// less to deliver into each one's LDS.
struct NarrowForm {
  int mb, nb;
};
inline long narrow_workgroups(int64_t M, int64_t N, NarrowForm f) {
  const long tiles = (N + 32 * f.nb - 1) / (32 * f.nb), row_blocks = (M + 32 * f.mb - 1) / (32 * f.mb);
  return row_blocks == 1 ? tiles : (tiles + kNumXcd - 1) / kNumXcd * kNumXcd * row_blocks;
}
// Columns per tile where all rows sit in one workgroup: the columns dealt out evenly over the CUs, in multiples
// of 4 (8-byte stores), up to the 64 a workgroup can take; beyond 64 x 256 columns the launch needs several
// rounds of workgroups anyway and the tiles stay 32 wide.
inline int narrow_tile_cols(int64_t N) {
  if (N > 64 * (int64_t)kNumCu) return 32;
  const int64_t per_cu = (N + kNumCu - 1) / kNumCu;
  const int w = (int)((per_cu + 3) / 4 * 4);
  return w < 4 ? 4 : w;
}
inline NarrowForm narrow_form(int64_t M, int64_t N) {
  if (M <= 32) return {1, narrow_tile_cols(N) > 32 ? 2 : 1};
  static const NarrowForm by_size[3] = {{1, 1}, {2, 1}, {2, 2}};
  for (const NarrowForm f : by_size)
    if (narrow_workgroups(M, N, f) <= kNumCu) return f;
  return {2, narrow_tile_cols(N) > 32 ? 2 : 1};  // (M <= 64: all rows in one workgroup)
}
inline float narrow_cost_us(int64_t M, int64_t N, int64_t K) {
  const NarrowForm f = narrow_form(M, N);
  if (M > 32 * f.mb) {  // row blocks, one round
    const float k1024 = (float)K / 1024.0f;
    const float share = (float)narrow_workgroups(M, N, f) / (float)kNumCu;  // of the CUs at work
    // (64x64 tiles: 1.9 us per 1024 bytes of K with every CU at work, 1.7 with 160 of them, 256 x 2304 x 6656 17.0 us)
    if (f.nb == 2) return 6.0f + k1024 * (K > 16384 ? 2.15f : 1.34f + 0.56f * share);
    if (f.mb == 2) return 5.4f + k1024 * (0.75f + 0.575f * share);
    return 3.5f + k1024 * (0.9f + 0.25f * share);
  }
  // All rows in one workgroup, one round of workgroups: the columns are dealt out evenly (narrow_tile_cols), and
  // what a workgroup waits for is its operands against the fetches a CU can have outstanding (about 64 KB): its
  // rows of B at HBM's latency (2 us), its rows of A at the L2's (0.6 us), plus start and launch. Measured cold at
  // M = 32, K = 8192: N = 1024 8.5 us, 2048 8.9, 4096 11.9, 5120 11.7, 8192 14.5, 10240 17.2, 16384 23.5 (N = 12288:
  // 21.1, three more than this says: with 48-column tiles the chip as a whole delivers less); K = 4096: N = 4096 7.3,
  // 14336 12.9; M = 64: 8192 x 8192 17.9, 10240 x 8192 20.6; M = 16: 13312 x 13312 29.3.
  // (Fewer than 16 rows of A cost what 16 do: 1 x 5120 x 8192 10.1 us, 16 x 5120 x 8192 10.2.)
  if (N <= 64 * (int64_t)kNumCu) {
    const float w = (float)narrow_tile_cols(N);
    // (Narrow panels: with 4 to 16 columns a workgroup there is little to fetch, and what a step of K costs is its
    // trip to memory against the depth of the ring, 0.07 to 0.1 us per 128 bytes. Up to 16 rows, N = 2048: 5.8 / 8.3 /
    // 11.8 / 21.8 us at K = 4096 / 8192 / 13312 / 28672; N = 1024 5.7 / 8.2 / - / 20.6, 3072 6.1 / 8.9 / 12.6 / 23.7;
    // 32 rows, K = 28672: N = 1024 21.7, 2048 23.4, 3072 26.0, 3584 28.8.)
    const float rows = (float)(M < 16 ? 16 : M);
    return fmaxf(4.4f + w * (float)K / 32768.0f + rows * (float)K * (0.6f / 65536.0f),
                 3.2f + (float)K * (5.0e-4f + 0.135e-4f * w + 0.035e-4f * rows));
  }
  const long tiles = (N + 31) / 32;
  const long rounds = (tiles + kNumCu - 1) / kNumCu;
  // per 1024 bytes of K: what the CUs at work can pull from L2, or, with most of them at work and up to 32
  // rows, what HBM delivers of B (measured at M <= 32: 8.6 us at 5120 x 5120, 8.3 at 4096 x 4096, 14.3 at 8192 x 8192)
  const float share = fminf(1.0f, (float)tiles / (float)kNumCu);
  const float k1024 = (float)K / 1024.0f;
  // (with fewer than half the CUs at work the fixed part is larger than this form has it: the old rate stays)
  if (M <= 32) return (float)rounds * (3.5f + k1024 * (tiles >= kNumCu / 2 ? fmaxf(1.08f, 1.38f * share) : 1.38f));
  return (float)rounds * (4.5f + k1024 * (1.1f + 0.52f * share));
}
// The pair kernel. Its time follows the CU with the most tiles, and the K steps are dealt to its 16 waves in whole
// rounds (K = 2304 is 18 steps in 32 slots): half the columns count as dealt evenly, half as the busiest CU's, and K
// as rounded up to 2048. Measured cold: 16 x 8192 x 8192 12.75 us, K = 4096 7.9, K = 2048 5.4; M = 1: 8192 x 8192
// 12.4, 4096 x 8192 8.0, 4096 x 4096 5.6, 8192 x 2048 5.1, 4096 x 2304 5.0; M = 16: 5120 x 8192 11.2, 6144 x 8192 11.5.
// With one tile a CU there is little of B to hide the fetch of A behind (N = 2048, K = 8192: 6.8 us with one row of A,
// 7.8 with 16; K = 4096: 5.1 / 5.5; N = 8192, K = 8192: 12.4 / 12.75).
inline float pair_cost_us(int64_t M, int64_t N, int64_t K) {
  const float cols_busiest = (float)(16 * ((N / 16 + kNumCu - 1) / kNumCu) * kNumCu);
  const float k_slots = (float)((K + 16 * kStepK - 1) / (16 * kStepK) * (16 * kStepK));
  const float a_rows = N <= 16 * kNumCu ? (float)M * (float)K * (1.1e-4f / 16.0f) : 0.0f;
  // (a quarter of the CUs at work: 1 x 1024 x 4096 4.95 us, 1 x 1024 x 8192 6.5)
  const float fixed = N <= 1536 ? 3.35f : N <= 16 * kNumCu ? 3.1f : 2.75f;
  return fixed + 0.5f * ((float)N + cols_busiest) * k_slots / 6.7e6f + a_rows;
}
// The general kernel, one 16- or 32-row tile of B per workgroup.
inline float one_tile_cost_us(int64_t M, int64_t N, int64_t K) {
  static const float rate[4] = {6.0e6f, 4.5e6f, 3.44e6f, 3.6e6f};
  const int blocks = (int)((M + 15) / 16);
  const int b = blocks < 1 ? 0 : blocks > 4 ? 3 : blocks - 1;
  float r = M <= 8 ? 7.2e6f : rate[b];  // (a few rows of A: its loads hit in L1 almost always)
  // two blocks, one round of workgroups (two per CU) and a short K: everything is in flight at once
  if (b == 1 && N <= 16 * 2 * kNumCu && K <= 8192) r = 4.9e6f;
  // The kernel takes as long as its busiest CU: workgroups are dealt out in rounds of one per CU, and a last
  // round that reaches only some CUs costs a whole one (16 x 5120 x 13824: 20.8 us with 320 workgroups, where
  // 4096 x 14336 with 256 takes 12.9).
  // (With one or two blocks of A a single round that leaves CUs idle is left as it was: those shapes are a few
  // microseconds long and bound by the launch, 32 x 2048 x 2048 4.5 us.)
  const long wgs = (N + (b == 3 ? 31 : 15)) / (b == 3 ? 32 : 16);
  const long rounds = (wgs + kNumCu - 1) / kNumCu;
  if (b >= 2 || rounds > 1) r *= (float)wgs / (float)(rounds * kNumCu);
  // (up to 16 rows, measured cold: 1 x 8192 x 8192 12.1 us, 1 x 4096 x 8192 7.5, 1 x 2304 x 2048 3.7,
  // 16 x 8192 x 8192 13.8, 16 x 4096 x 4096 5.6)
  // (two blocks: 32 x 2048 x 2048 4.5 us)
  float t = (b == 0 ? 3.0f : b == 1 ? 3.7f : 5.0f) + (float)N * (float)K / r;
  // (Wide panels with short rows: every workgroup has a start and an end that no other hides, 1.7 ns apiece beyond the
  // first 512, which shows where a workgroup's share of K is short: 3 x 45376 x 1024 14.7 us for 46 MB, 1 x 103104 x
  // 1664 38.1 for 172 MB, 3 x 97728 x 2304 44.6; at K = 8192 half of it is left, 1 x 57344 x 8192 71.5.)
  if (b == 0 && wgs > 2 * kNumCu) t += (float)(wgs - 2 * kNumCu) * 1.66e-3f * fminf(1.0f, 4096.0f / (float)K);
  // Part of the chip at work, up to 32 rows: a workgroup has its CU to itself, and a byte of K costs it what its 16
  // rows of B (from HBM) and its rows of A (from L2) take against the fetches a CU can have outstanding, whatever
  // the number of workgroups. Measured with 128 workgroups (N = 2048) at K = 4096 / 8192 / 16384 / 28672: one row of
  // A 4.5 / 6.2 / 9.7 / 14.9 us, 8 rows 4.7 / 6.6 / 10.6 / 17.0, 16 rows 5.1 / 7.6 / 12.2 / 20.5, 32 rows 6.2 / 9.8 /
  // - / -; with 64 (N = 1024): one row 4.2 / 6.0 / 8.8 / 13.8, 16 rows 4.9 / 7.1 / 11.6 / 19.3; 144 workgroups,
  // K = 16384: 10.8 / 12.5 / 16.4 us with 8 / 16 / 32 rows.
  // (Rows that do not start on a 128-byte boundary: every 128-byte piece of a row lies across two cache lines, and a
  // workgroup alone on its CU, which asks for its rows 128 bytes at a time, takes 1.4-1.5 times as long per byte of K:
  // 17 x 2816 x 18832 23.6 us where aligned rows would take 15.5, 14 x 1536 x 9760 11.4 against 8.4; the narrow-tile
  // kernel, 512 bytes of a row at a time, loses 0-12 % on the same shapes. With several rounds of workgroups every
  // kernel loses about the same, 1.25-1.4, and the order of the estimates holds. K stands in for the row pitch.)
  const float pitch = K % kStepK != 0 ? 1.45f : 1.0f;
  if (b <= 1 && wgs < kNumCu) t = fmaxf(t, 2.6f + pitch * (float)K * (4.1e-4f + 0.13e-4f * (float)M));
  // (three blocks of A, the same way: 48 x 2048 x 4096 7.5-8.0 us, 48 x 2048 x 8192 12.1-12.6, 34 x 2048 x 1024 3.4,
  // 48 x 3584 x 28672 36.8; the rate above, scaled by the share of the CUs at work, has these shapes a quarter slower)
  if (b == 2 && wgs < kNumCu) t = fminf(t, 3.0f + 1.08f * pitch * (float)K * (4.1e-4f + 0.13e-4f * (float)M));
  return t;
}
// The streaming members of the family and which of them runs a shape: the pair kernel where it fits, unless the
// one-tile kernel is expected ahead (at M <= 8 by a few per cent on most shapes, by 15-20 % where K fills the pair
// kernel's step slots badly: 1 x 4096 x 2304 4.3 us against 5.0); the persistent kernel beyond the pair kernel's N.
enum SkinnyStreaming { kStreamPair, kStreamPersistent, kStreamOneTile };
inline SkinnyStreaming skinny_streaming_choice(int64_t M, int64_t N, int64_t K) {
  if (pair_skinny_fits(M, N, K)) return one_tile_cost_us(M, N, K) < pair_cost_us(M, N, K) ? kStreamOneTile : kStreamPair;
  return persistent_skinny_fits(M, N, K) ? kStreamPersistent : kStreamOneTile;
}
inline float skinny_streaming_cost_us(int64_t M, int64_t N, int64_t K) {
  switch (skinny_streaming_choice(M, N, K)) {
    case kStreamPair: return pair_cost_us(M, N, K);
    // the persistent form (measured: 71 us at 16 x 57344 x 8192; two blocks of A, K = 4096: 9.9 us at N = 8192, 8.9 at
    // 24 x 6144 x 4096; one step per wave, K = 2048: a tile is over before the next one's rows have arrived, 4 x 13312 x 2048 8.2 us)
    // (K = 2048, one step per wave: 1 x 128256 x 2048 50.6 us, 4 x 13312 x 2048 8.2)
    case kStreamPersistent:
      if (K <= 2048 && M <= 16) return 3.4f + (float)N * (float)K / 5.7e6f;
      return (K <= 2048 ? 4.2f : 3.0f) + (float)N * (float)K / (M <= 16 ? 6.9e6f : 4.4e6f);
    default: return one_tile_cost_us(M, N, K);
  }
}
// the cheapest member of the M <= 64 family: streaming (persistent or one tile per workgroup) or narrow tiles
inline bool narrow_preferred(int64_t M, int64_t N, int64_t K) {
  if (M > kSkinnyMaxM) return narrow_fits(M, N, K);  // (the streaming kernels stop at 64 rows)
  return narrow_fits(M, N, K) && narrow_cost_us(M, N, K) < skinny_streaming_cost_us(M, N, K);
}
inline float skinny_cost_us(int64_t M, int64_t N, int64_t K) {
  if (M > kSkinnyMaxM && !narrow_fits(M, N, K)) return 1e30f;
  return narrow_preferred(M, N, K) ? narrow_cost_us(M, N, K) : skinny_streaming_cost_us(M, N, K);
}
constexpr int kMaxSplits = 16;
// Tile rows up to which a launch fetches B with the streaming policy (see gemm_tiled_kernel).
constexpr int kStreamTileRows = 2;
// (256x256 tiles: one tile row only. M=256, N=57344, K=8192 120.3 -> 109.7 us; with two tile rows, M=512, the
// policy costs 2-3 %.)
constexpr int stream_tile_rows(int bm, int bn) { return bm == 256 && bn == 256 ? 1 : kStreamTileRows; }

struct TiledPlan {
  int config, splits, steps_per_split;
  float cost_us;
};

inline int k_steps_of(int64_t K) { return (int)((K + kStepK - 1) / kStepK); }

// Splits actually used when `want` are asked for: every split gets the same whole number of
// steps and none is empty.
inline void normalise_splits(int k_steps, int want, int& splits, int& sps) {
  want = want < 1 ? 1 : (want > k_steps ? k_steps : want);
  sps = (k_steps + want - 1) / want;
  splits = (k_steps + sps - 1) / sps;
}

// What a step takes on rows off the 128-byte lines against rows on them, by configuration: the deep 128x128 form fetches them in whole lines from
// kWindowSteps steps an item on, the others' pieces lie across two. Fitted to what the choice then costs: 1260 shapes of more than 256 rows,
// 16 to 30000 columns, every configuration in one to sixteen parts. (Medians of the launches alone 1.21, 1.14,
// 1.34, 1.37, 1.38, 1.29 and, deep, 1.06: what a factor also makes up for is where a configuration's estimate on the lines is off.)
// Up to 640 rows 256x128 and 128x256 tiles have their own: 450x9481x6368 53 us on the former, 66 on 256x256 in three parts; 3471x1640x13728 132 us on
// them, 99 on 192x256. 3846x1656x2384 27.2 us with these or none, 31.1 with one factor of 1.2; 411x4682x10848 51.6 with the one or none, 46.3.
// Not on rows of fewer steps than kOffLinesMinSteps, where parts of few steps look like a gain that they are not: 563x64x752 in six 1.34 times
// as long as in one. On longer rows parts have kOffLinesMinPart steps at least: 3836x19x3920 15.2 us in sixteen, 11.7 in eight.
constexpr int kWindowSteps = 12, kOffLinesMinSteps = 16, kOffLinesMinPart = 3;
inline bool priced_off_lines(int64_t M, int64_t K, bool off_lines) { return off_lines && M > kNarrowMaxM && k_steps_of(K) >= kOffLinesMinSteps; }
inline float off_lines_step(int config, int64_t M, int splits, int sps) {
  static const float step[kNumTileConfigs] = {1.06f, 1.17f, 1.5f, 1.04f, 1.08f, 1.11f, 1.17f};
  if (config == kDeepSmallConfig && sps >= kWindowSteps) return 0.95f;
  if (config == 0 && splits > 1) return 1.14f;
  if (M <= 640 && (config == 2 || config == 4)) return config == 2 ? 1.11f : 1.14f;
  return step[config];
}

// Estimated run time of a plan. Work items are dealt to 256 * wgs_per_cu workgroup slots in
// rounds; a last round that fills at most one slot per CU runs at the faster stand-alone
// rate. The operands cannot arrive faster than the configuration streams from HBM. Split
// plans add a launch and the partial sums' trip through memory (written once, read once).
inline float plan_cost_us(int64_t M, int64_t N, int64_t K, bool off_lines, int config, int splits, int sps) {
  const TileConfig& c = kTileConfigs[config];
  const long tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
  const long items = tiles * splits;
  const long slots = (long)kNumCu * c.wgs_per_cu;
  const long full_rounds = items / slots, rest = items % slots;
  // (256x128 tiles are bound by the delivery of their operands, and rows of a tile past M are not fetched: with a last
  // tile row that is half empty a step takes less, 384 x 16384 x 16384 106.5 us = 0.79 us per step instead of 0.87,
  // 384 x 13312 x 13312 85.7, 640 x 8192 x 8192 53.5, 448 x 10240 x 8192 51.4 where three splits of 256x256 tiles take
  // 62.8. Unsplit plans only: with the same allowance split plans were taken where they measure behind, 448 x 2304 x
  // 13312 in seven 33.0 us against 28.5 for the deep 128x128 form in three.)
  const float rows_fetched = (float)M / (float)((M + c.bm - 1) / c.bm);
  const float step_scale = config == 2 && splits == 1 ? 0.5f + 0.5f * (rows_fetched + (float)c.bn) / (float)(c.bm + c.bn) : 1.0f;
  // (192x256 tiles in a single round: 4712 x 2048 x 1024 14.0-14.8 us with 200 tiles of 8 steps, 416 x 21312 x 1024 15.0
  // with 252, 2560 x 8192 x 1024 26.6 with 448 where 128x256 tiles take 30.3; over several rounds the table's 9 us per
  // tile stands: it leaves the estimate as far above the measurement as that of the 256x256 tiles, 3-4 %, and the order
  // of the two right: 896 x 57344 x 8192 343 us with 256x256 tiles, 354 with these)
  // (64x256 tiles, unsplit, over very short rows, K up to 1664: the table's constants are those of long weight panels;
  // here a step takes 0.54 us and a tile 5 beside its steps: 400 x 8704 x 1536 10.8 us with 238 tiles, 3 x 45376 x 1024
  // 11.6 with 178, 192 x 21312 x 1024 8.9 with 252. Only where 128x128 tiles are more than one round: up to that the
  // deep 128x128 form measures ahead, 400 x 8192 x 1024 7.7 us against 8.5, and its own estimate is a cautious one.)
  const bool short_c3 = config == 3 && splits == 1 && K <= 13 * kStepK && ((M + 127) / 128) * ((N + 127) / 128) > kNumCu;
  // (128x256 tiles over fewer than 8 steps: what a launch costs before its first step is not in the table's 2.6 us a
  // tile, 2129 x 32 x 512 7.2 us with 17 tiles where 128x128 tiles take 5.2: such launches are left to those)
  const float us_per_item = config == 5 && items <= 2 * slots ? 7.0f : short_c3 ? 5.0f : config == 4 && sps < 8 ? 10.0f : c.us_per_item;
  // (Rows off the lines: see off_lines_step. Above the rows of the narrow tiles, whose own estimate has K stand in for the pitch.)
  const float off = priced_off_lines(M, K, off_lines) ? off_lines_step(config, M, splits, sps) : 1.0f;
  const float us_step = off * (short_c3 ? 0.54f : c.us_per_step), us_step_alone = off * (short_c3 ? 0.54f : c.us_per_step_alone);
  float t = full_rounds * (sps * us_step * step_scale + us_per_item);
  if (rest) t += sps * (rest <= kNumCu ? us_step_alone : us_step) * step_scale + us_per_item;
  // (the deep 128x128 form is for one round only; beyond 128 workgroups its steps slow down with the chip's
  // clock and the shared L2: 0.49 us with 128, 0.58 with 256)
  if (config == kDeepSmallConfig) {
    if (items > kNumCu) return 1e30f;
    if (items > kNumCu / 2) t += sps * 0.09f * (float)(items - kNumCu / 2) / (float)(kNumCu / 2);
  }
  // (one or two tile rows, one for 256x256 tiles: B is fetched with the streaming policy, which is worth 8 % or more)
  const bool streams_b = (M + c.bm - 1) / c.bm <= stream_tile_rows(c.bm, c.bn);
  // (fewer work items than CUs: the busy CUs cannot make up for the idle ones beyond their share)
  const float busy = items >= kNumCu ? 1.0f : fminf(1.0f, c.wg_stream_share * (float)items / (float)kNumCu);
  // (64x256 tiles, unsplit: the rotated K order lifts the rate further; with two splits the plan measured at the
  // plain rate, 48 x 28672 x 8192 47.5 us)
  // (256x256 tiles gain the most: their rate without the policy is the lowest)
  const float policy = !streams_b || config == kDeepSmallConfig ? 1.0f
                       : (config == 3 && splits == 1) ? 1.08f * 1.1f : config == 0 ? 1.2f : 1.08f;
  // (128x128 tiles: the rate was measured with full tiles; rows of a tile past M are not fetched, and what a CU
  // has to take in beside its rows of B shrinks with them: 64 x 28672 x 8192 unsplit 42.4 us = 6.3 MB/us)
  const float rows_a = (float)M / (float)((M + c.bm - 1) / c.bm);
  // (not below 33 rows: there the estimate would undercut the streaming kernels, which measure 25 % ahead)
  // (with short rows, K up to 4096, the allowance holds for any M: there the streaming kernels pay for every workgroup's
  // start and do not measure ahead, 1 x 128256 x 2048 44.7 us with 128x128 tiles against 50.6)
  const float fill = (config == 1 || config == kDeepSmallConfig) && (M > 32 || K <= 4096) ? fmaxf(0.75f, (rows_a + (float)c.bn) / (float)(c.bm + c.bn)) : 1.0f;
  // (the 256-column tiles of one tile row stream less with short rows, where a tile is over after a few steps: of
  // their rate at K >= 4096 they reach 0.8 up to K = 2048 and 0.87 at 2560; 1 x 128256 x 2048 46.8 us with 64x256
  // tiles and 49.6 with 128x256, 2 x 115072 x 2560 50.6 and 53.2, 1 x 128256 x 4096 79.5 and 81.7)
  const float short_rows = (config == 3 || config == 4) && K < 4096 ? fmaxf(0.8f, 0.8f + 0.2f * (float)(K - 2048) / 2048.0f) : 1.0f;
  const float stream = ((float)M * (float)K + (float)N * (float)K) * fill / (c.stream_bytes_per_us * policy * busy * short_rows);
  if (t < stream) t = stream;
  if (splits > 1) t += 3.0f + 2.0f * (float)splits * (float)M * (float)N * 4.0f / 5.0e6f;
  return t;
}

// Cheapest plan by the model above; `max_splits` = 1 restricts it to plans without workspace.
inline TiledPlan plan_tiled(int64_t M, int64_t N, int64_t K, bool off_lines, int force_config, int force_splits,
                            int max_splits) {
  const int k_steps = k_steps_of(K);
  TiledPlan best = {0, 1, k_steps, 0.0f};
  float best_cost = -1.0f;
  for (int c = 0; c < kNumTileConfigs; ++c) {
    if (force_config >= 0 && c != force_config) continue;
    for (int want = 1; want <= max_splits; ++want) {
      if (force_splits > 0 && want != force_splits) continue;
      int splits, sps;
      normalise_splits(k_steps, want, splits, sps);
      if (force_splits <= 0 && splits != want) continue;  // duplicate of a smaller request
      // (128x256 tiles are the plan for whole rows of K against wide panels; split, they measured behind what
      // their estimate says: 128 x 8192 x 28672 66.3 us against 56.5 with 128x128 tiles)
      // (192x256 tiles were not measured split either)
      if ((c == 4 || c == 5) && force_splits <= 0 && splits > 1) continue;
      // (the deep ring takes three steps to fill: short rows of K stay with the two-step form, 2048 x 2048 x 512
      // 6.5 us against 6.9)
      if (c == kDeepSmallConfig && force_config < 0 && sps < 8) continue;
      if (splits > 1 && sps < kOffLinesMinPart && force_splits <= 0 && priced_off_lines(M, K, off_lines)) continue;
      // (With one or two tile rows the other configurations fetch B with the streaming policy; the deep form with
      // that policy measured 37.7 us on 256 x 4096 x 8192 against 20.1 for the 64x256 tiles, so it does not have it.
      // Without it B's lines stay in the caches: on weights small enough to be found there again it is the fastest
      // plan of all at 96 to 256 rows (operands from the memory-side cache: 256 x 6144 x 4096 14.6 us against 23.8,
      // 128 x 13312 x 2048 10.0 against 13.9; from HBM level with the 128x128 form), on large ones the policy wins
      // (64 x 28672 x 8192 from HBM: 51.7 us against 42.7).)
      if (c == kDeepSmallConfig && force_config < 0 && M <= 2 * 128 && N * K > (int64_t)48 << 20) continue;
      const float cost = plan_cost_us(M, N, K, off_lines, c, splits, sps);
      if (best_cost < 0.0f || cost < best_cost) {
        best_cost = cost;
        best = {c, splits, sps, cost};
      }
    }
  }
  return best;
}

// variant word: bits 0..7 kernel family, bits 8..15 tile configuration + 1 (0 = automatic),
// bits 16..23 split-K factor (0 = automatic)
inline TiledPlan plan_from_variant(int64_t M, int64_t N, int64_t K, bool off_lines, int variant, int max_splits) {
  const int cfg = ((variant >> 8) & 0xff) - 1;
  const int spl = (variant >> 16) & 0xff;
  return plan_tiled(M, N, K, off_lines, cfg, spl, spl > 0 ? spl : max_splits);
}

constexpr int kMaxDevices = 64;
// The tile walk, the grid sizes and the cost tables are written for the whole part: 256 CUs in 8
// XCDs. A device that reports another CU count (a partitioned mode, another product) would be
// scheduled wrongly without any error, so it is turned away, once per device, when the device is
// set up.
int check_device_shape(int dev) {
  int cus = 0;
  const hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "hipDeviceGetAttribute: %s", hipGetErrorString(e));
  if (cus != kNumCu)
    return fail(MI355X_FP8_ENOTSUP, "device %d does not report the %d compute units these kernels are scheduled for "
                "(a partitioned mode or another part)", dev, kNumCu);
  return MI355X_FP8_OK;
}

// Every kernel instantiation that needs more dynamic LDS than the default limit enters itself in
// this table while the library is loaded (static initialisation, before any call can arrive).
// Setting a device up walks the table once and raises each kernel's limit there, so that no
// launch path has anything but the launch itself to do: a caller whose first use of some
// instantiation happens under graph capture meets no attribute call.
// (The table is shared by the translation units of a build in parts; it is zero-initialised storage,
// so registrations from any unit's static initialisers find it ready.)
bool register_lds_kernel(const void* kernel, size_t lds_bytes) {
  using namespace mi355x_shared;
  if (num_lds_kernels < mi355x_shared::kMaxLdsKernels) lds_kernels[num_lds_kernels++] = {kernel, lds_bytes};
  else lds_table_overflow = true;
  return true;
}
template <auto Kernel, size_t LdsBytes>
struct LdsLimit {
  static inline const bool registered = register_lds_kernel(reinterpret_cast<const void*>(Kernel), LdsBytes);
};

// 0 = not set up, 1 = ready, -1 = refused (wrong device shape). Setting a device up twice from two
// threads is harmless: every step is idempotent.
#if !defined(MI355X_TILED_PART)
std::atomic<int> g_device_state[kMaxDevices];
std::atomic<void*> g_scratch_ptr[kMaxDevices];
int setup_device(int dev);
#endif
inline int ready_device(int* dev_out = nullptr) { return mi355x_shared::ready_device(dev_out); }
}  // namespace

#if !defined(MI355X_TILED_PART)
thread_local char mi355x_shared::err[512] = "";
mi355x_shared::LdsKernel mi355x_shared::lds_kernels[mi355x_shared::kMaxLdsKernels];
int mi355x_shared::num_lds_kernels = 0;
bool mi355x_shared::lds_table_overflow = false;

// The current device, set up. The only HIP call on the ready path is hipGetDevice.
int mi355x_shared::ready_device(int* dev_out) {
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(MI355X_FP8_ENOTSUP, "device index %d beyond %d", dev, kMaxDevices - 1);
  if (dev_out) *dev_out = dev;
  if (g_device_state[dev].load(std::memory_order_acquire) == 1) return MI355X_FP8_OK;
  return setup_device(dev);
}
#endif

namespace {
// How a launch of tiles stores C. The streaming policy is for rows on 64 bytes, or a C that is not much more than the
// L2s hold (32 MB): with others two pieces share 64 bytes, which then go to memory twice in parts. us streaming / ordinary,
// rows 16 to 32 bytes off the lines: 4924x9808x1024 (97 MB) 80 / 66, 3000x9736x2304 (58) 77 / 63, 6935x5200x1200 (72) 75 / 68,
// block-scaled 4096x8208x1024 (67) 65 / 57, 16384x1040x1024 (34) 32 / 33, 2048x4112x4096 (17) 35.5 / 38.9; on the lines
// 3122x9728x2304 59 / 63; on 64 bytes 5000x9760x1024 68.6 / 70.4, block-scaled 1129x24928x1504 50 / 58.
// Pieces that start at any 2 bytes, as one store each where they were eight of 2 bytes: 4924x9807x1024 127 -> 68, 5203x3266x1152
// 56 -> 31, 1024x5203x1200 23.4 -> 15.4, 16 groups of 8192x4111x1024 112 -> 63 (streaming ones of that kind 97, 38, 17, 73).
constexpr int64_t kLargeResult = (int64_t)48 << 20;
inline int store_policy(const GemmParams& p) {
  const uintptr_t base = reinterpret_cast<uintptr_t>(p.c), pitch = (uintptr_t)(p.ldc * 2);
  if ((base | pitch | (uintptr_t)p.N * 2) & 15) return kStoreAny;
  return ((base | pitch) & 63) != 0 && (int64_t)p.M * p.N * 2 > kLargeResult ? kStoreKeep : kStoreStream;
}

// The second pass of a launch whose items left partial sums.
int launch_finalize(GemmParams p, hipStream_t stream) {
  // Four rows a thread where one row each would be more workgroups than the chip holds at once (8 of 256 lanes on a
  // CU): fewer of them to start, more loads in flight each. Below that they would leave CUs idle.
  const long quads_per_row = ((long)p.N + 3) / 4;
  const bool many = (quads_per_row * p.M + 255) / 256 > 8L * kNumCu;
  const long quads = quads_per_row * (many ? ((long)p.M + kFinalizeRows - 1) / kFinalizeRows : p.M);
  p.div_group_mul = p.div_group_shift = 0;
  if (quads <= (long)INT32_MAX - 255) make_fast_div((uint32_t)quads_per_row, p.div_group_mul, p.div_group_shift);
  hipLaunchKernelGGL(many ? splitk_finalize_rows_kernel : splitk_finalize_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0,
                     stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "split-K finalize launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, bool KTAIL, int EPI, bool GROUPED = false, bool BLOCKSCALE = false,
          int DIST = kDefaultDist, bool STREAM_B = false, bool CLEAR = false, bool OFF_LINES = false, bool LINES = false>
int launch_tiled(GemmParams p, hipStream_t stream) {
  p.store = store_policy(p);
  constexpr int threads = WAVES_M * WAVES_N * 64;
  constexpr size_t lds_bytes = tiled_lds_bytes(BM, BN, DIST);
  // grouped: the group sizes live on the device; every group adds at most one partial tile row
  p.tiles_m = GROUPED ? p.M / BM + p.groups : (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  make_fast_div((uint32_t)p.tiles_m * (uint32_t)p.tiles_n, p.div_tiles_mul, p.div_tiles_shift);
  make_fast_div((uint32_t)kGroupM * (uint32_t)p.tiles_n, p.div_group_mul, p.div_group_shift);
  const long total = (long)p.tiles_m * p.tiles_n * p.splits;
  if (total > (long)INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "more than 2^31-1 work items");
  const long slots = (long)kNumCu * tiled_wgs_per_cu(BM, BN, DIST);
  long grid = total < slots ? ((total + kNumXcd - 1) / kNumXcd) * kNumXcd : slots;
  constexpr auto kern = gemm_tiled_kernel<BM, BN, WAVES_M, WAVES_N, KTAIL, EPI, GROUPED, BLOCKSCALE, DIST, STREAM_B, CLEAR, OFF_LINES, LINES>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  if (const int st = ready_device()) return st;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), lds_bytes, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "tiled kernel launch: %s", hipGetErrorString(e));
  if (EPI == kEpiPartial) {
    if (BLOCKSCALE) p.a_scale = p.b_scale = nullptr;  // (the factors were applied block by block)
    return launch_finalize(p, stream);
  }
  return MI355X_FP8_OK;
}

// whether rows of B start off the 128-byte lines, or off their halves
inline bool off_lines(const GemmParams& p, int bytes = kStepK) { return ((reinterpret_cast<uintptr_t>(p.b) | (uintptr_t)p.ldb) & (bytes - 1)) != 0; }

template <int BM, int BN, int WAVES_M, int WAVES_N, bool STREAM_B, bool DEEP = false>
int launch_tiled_epilogue(const GemmParams& p, hipStream_t s) {
  // 256x128 tiles have the LDS for loads three steps ahead (3 A + 4 B stages = 160 KB): worth 6-10 % where
  // the operands come from HBM rather than the memory-side cache (M=1024, N=K=8192 cold: 65.9 -> 60.5 us;
  // K=28672: 220 -> 199 us). The 64x256 tile measured 1-3 % slower that way and stays at two.
  constexpr int D = DEEP || (BM == 256 && BN == 128) ? 3 : kDefaultDist;
  const bool ktail = p.K % kStepK;
  // The deep form, rows off the lines: in whole lines where the steps of an item pay for the window more that has to land before the first.
  // us so and as they lie, by items and steps of each: 1000x3000x4112 (192, 33) 24.5 and 28.9, 512x4096x4112 (128, 33) 24.4 and 31.4, 539x4260x6480
  // (170, 51) 30.8 and 39.6, 252x2688x13840 (in six) 26.3 and 31.7, 2048x2048x2064 (256, 17) 16.2 and 18.8, 1693x663x1488 (84, 12)
  // 12.2 and 13.1; with 10 steps 699x3051x1216 (144) 12.8 and 12.6, with 9 535x2440x1056 (100) 10.2 and 9.6.
  if constexpr (DEEP) {
    const long items = (long)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN) * p.splits;
    const uintptr_t off = reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | (uintptr_t)p.lda | (uintptr_t)p.ldb;
    if (off % kStepK != 0 && items <= kNumCu && p.steps_per_split >= kWindowSteps) {
      if (p.splits > 1) return launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPartial, false, false, D + 1, false, false, false, true>(p, s);
      return p.bias ? launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiBias, false, false, D + 1, false, false, false, true>(p, s)
                    : launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPlain, false, false, D + 1, false, false, false, true>(p, s);
    }
  }
  if constexpr (STREAM_B) {
    // (mostly because K is no multiple of a step: the kernels for that take the others too. 120 shapes of 33 to 256 rows: 1.035 times as
    // fast on average without the policy, 220x12704x17520 100 -> 88 us; at worst 210x8143x24896 78 -> 84)
    if (off_lines(p)) {
      if (p.splits > 1) return launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPartial, false, false, D, true, false, true>(p, s);
      return p.bias ? launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiBias, false, false, D, true, false, true>(p, s)
                    : launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPlain, false, false, D, true, false, true>(p, s);
    }
  }
  if (p.splits > 1)
    return ktail ? launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPartial, false, false, D, STREAM_B>(p, s)
                 : launch_tiled<BM, BN, WAVES_M, WAVES_N, false, kEpiPartial, false, false, D, STREAM_B>(p, s);
  if (p.bias)
    return ktail ? launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiBias, false, false, D, STREAM_B>(p, s)
                 : launch_tiled<BM, BN, WAVES_M, WAVES_N, false, kEpiBias, false, false, D, STREAM_B>(p, s);
  return ktail ? launch_tiled<BM, BN, WAVES_M, WAVES_N, true, kEpiPlain, false, false, D, STREAM_B>(p, s)
               : launch_tiled<BM, BN, WAVES_M, WAVES_N, false, kEpiPlain, false, false, D, STREAM_B>(p, s);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, bool MAY_STREAM, bool DEEP = false>
int launch_tiled_config(const GemmParams& p, hipStream_t s) {
  if constexpr (MAY_STREAM) {
    if ((p.M + BM - 1) / BM <= stream_tile_rows(BM, BN))
      return launch_tiled_epilogue<BM, BN, WAVES_M, WAVES_N, true, DEEP>(p, s);
  }
  return launch_tiled_epilogue<BM, BN, WAVES_M, WAVES_N, false, DEEP>(p, s);
}
}  // namespace

// The seven tile configurations of the plain tiled kernel, each behind a function of its own: a unit
// of a build in parts defines one of them, the main unit of such a build none, a single-unit build all.
#if !defined(MI355X_SPLIT_MAIN)
#define MI355X_DEFINE_TILED_PART(k, ...)                                                             \
  int mi355x_shared::tiled_config_##k(const GemmParams& p, hipStream_t stream) { return launch_tiled_config<__VA_ARGS__>(p, stream); }
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 0
MI355X_DEFINE_TILED_PART(0, 256, 256, 2, 2, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 1
MI355X_DEFINE_TILED_PART(1, 128, 128, 2, 2, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 2
MI355X_DEFINE_TILED_PART(2, 256, 128, 2, 2, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 3
MI355X_DEFINE_TILED_PART(3, 64, 256, 1, 4, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 4
MI355X_DEFINE_TILED_PART(4, 128, 256, 2, 2, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 5
MI355X_DEFINE_TILED_PART(5, 192, 256, 2, 2, true)
#endif
#if !defined(MI355X_TILED_PART) || MI355X_TILED_PART == 6
MI355X_DEFINE_TILED_PART(6, 128, 128, 2, 2, false, true)  // (never with the streaming policy)
#endif
#undef MI355X_DEFINE_TILED_PART
#endif

#if !defined(MI355X_TILED_PART)  // (everything from here on belongs to the main unit)
namespace {
// Whether the kernels of few rows ask for all of B, or of a row of it, at once: one step a wave, or a panel of at most 1.5 MB. Then both steps
// that share a line off the 128 bytes have asked for it before it comes, nothing comes twice, and the streaming policy stays:
// one tile a workgroup 8x714x800 2.96 us, without the policy 3.24, 47x26x3936 7.2 and 8.5, the pair kernel 0.2 to 0.3 us up to
// 1024 columns; with more columns and K up to 1024 within 4 % either way.
// (Rows that start on 64 bytes: memory is read by halves of lines, so no half is fetched twice with the policy, and the pair kernel and the narrow
// tiles keep it, 1.5 % ahead on 20 and 2 % on 34 shapes: 1x1600x3776 5.01 us, without 5.22, 2x4608x6848 9.36 and 9.69. One tile a workgroup
// is level, 1 % ahead without.)
constexpr int kHalfLine = 64;
inline bool asked_for_at_once(const GemmParams& p) { return k_steps_of(p.K) <= 8 || (int64_t)p.N * p.K <= (int64_t)3 << 19; }

template <int MT, int NTW, int DEPTH, int KW, bool ANY = false, bool BLOCK = false, bool OFF_LINES = false>
int launch_skinny(const GemmParams& p, hipStream_t stream) {
  if constexpr (!ANY && !OFF_LINES) {
    // (2x17533x10800 44.6 us with the streaming policy, 38.7 without, 1x6723x8272 14.9 and 13.9, 2x1021x3952 5.83 and 5.24, 3x945x20144
    // block-scaled 16.1 and 15.0)
    if (off_lines(p) && !asked_for_at_once(p)) return launch_skinny<MT, NTW, DEPTH, KW, false, BLOCK, true>(p, stream);
  }
  constexpr size_t lds_bytes = (size_t)KW * (NTW + MT) * 16 * kStepK;
  static_assert(lds_bytes <= 160 * 1024, "transpose buffers must fit the 160 KB LDS");
  constexpr auto kern = gemm_skinny_kernel<MT, NTW, DEPTH, KW, ANY, BLOCK, false, OFF_LINES>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  if (const int st = ready_device()) return st;
  const unsigned grid = (unsigned)((p.N + 16 * NTW - 1) / (16 * NTW));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(KW * 64), lds_bytes, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "skinny kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

// The grouped form for few rows a group. The most row blocks any sizes can give: every group that has rows at all
// wastes at most all but one row of a block.
constexpr int64_t grouped_row_blocks(int64_t G, int64_t M, int bm, bool clear_rest) {
  // (one more where rows past the groups' are to be cleared, so that there is a surplus to do it)
  return (M + (int64_t)(bm - 1) * (G < M ? G : M)) / bm + (clear_rest ? 1 : 0);
}
constexpr int64_t grouped_column_tiles(int64_t N, int bn) { return ((N + bn - 1) / bn + kNumXcd - 1) / kNumXcd * kNumXcd; }

template <int MT, int NTW, int DEPTH, int KW, bool OFF_LINES>
int launch_grouped_rows(const GemmParams& p, hipStream_t stream) {
  constexpr int BM = 16 * MT, BN = 16 * NTW;
  constexpr size_t lds_bytes = (size_t)KW * (NTW + MT) * 16 * kStepK;
  static_assert(lds_bytes <= 160 * 1024, "transpose buffers must fit the 160 KB LDS");
  constexpr auto kern = gemm_skinny_kernel<MT, NTW, DEPTH, KW, false, false, true, OFF_LINES>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  GemmParams q = p;
  q.tiles_n = (p.N + BN - 1) / BN;
  const int64_t tiles = grouped_column_tiles(p.N, BN), row_blocks = grouped_row_blocks(p.groups, p.M, BM, p.clear_rest != 0);
  if (!grid_fits(tiles * row_blocks, KW * 64)) return fail(MI355X_FP8_ENOTSUP, "more lanes than a launch holds");
  if (const int st = ready_device()) return st;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles * row_blocks)), dim3(KW * 64), lds_bytes, stream, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "grouped skinny kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

template <int MT, int NTW, int DEPTH, int KW>
int launch_grouped_skinny(const GemmParams& p, hipStream_t s) {
  return p.ldb % kStepK ? launch_grouped_rows<MT, NTW, DEPTH, KW, true>(p, s) : launch_grouped_rows<MT, NTW, DEPTH, KW, false>(p, s);
}

// The grouped form of the tiled kernel.
template <int BM, int BN, int DIST, bool STREAM_B>
int launch_grouped_tiles(const GemmParams& p, hipStream_t s) {
  if (p.clear_rest)
    return p.K % kStepK ? launch_tiled<BM, BN, 2, 2, true, kEpiPlain, true, false, DIST, STREAM_B, true>(p, s)
                        : launch_tiled<BM, BN, 2, 2, false, kEpiPlain, true, false, DIST, STREAM_B, true>(p, s);
  return p.K % kStepK ? launch_tiled<BM, BN, 2, 2, true, kEpiPlain, true, false, DIST, STREAM_B>(p, s)
                      : launch_tiled<BM, BN, 2, 2, false, kEpiPlain, true, false, DIST, STREAM_B>(p, s);
}

// Which form runs a grouped launch whose groups are up to a tile high on average: such a launch is bound by the
// stream of B, and the sizes themselves are on the device. Measured over G = 2 ... 64 with rows sent to groups at random
// and B read from memory, us, 128x128 tiles with B through the caches -> the form:
// * up to 8 rows a group on average, the 16-row streaming form (a group with more takes several blocks): 16 groups of
//   4096x4096 67 -> 47, 8 of 2048x7168 37 -> 21, 8 of 14336x4096 99 -> 77, 64 of 1536x1024 46 -> 21. Its tiles are 32
//   columns wide so that A passes the L1 half as often (16 columns: 57 on the first, 97 on the third). Four waves rather than
//   eight, so that twice as many workgroups are on a CU at different places of their short lives: eight waves 49, 21, 82
//   and 31, sixteen 60, 24, 101 and 50.
// * launches of at most 128 tiles leave half of the chip idle; on long rows the streaming forms with 32 and 64 rows are
//   ahead of them up to 16 and 32 rows a group: 8 groups of 2048x7168 38 -> 25 and 38 -> 31, 2 of 4096x4096 20 -> 13
//   with 32 rows. (64 rows a group: 39 -> 48.)
// * else tiles of one tile row with the streaming policy and the rotated walk: 16 groups of 4096x4096 with 16 to 64
//   rows 68 -> 51-53, 8 of 14336x4096 with 32 101 -> 88. (Fewer than 128 tiles: 18 -> 22. K = 1024: 14.4 -> 15.7.)
// * groups of 65 to 128 rows often are two tile rows high; 128x256 tiles then make fewer rounds: 16 groups of 4096x4096
//   with 128 rows 88 -> 73 (128x128 tiles with the streaming policy 99), 8 of 14336x4096 145 -> 109, 16 of 7168x2048
//   72 -> 63. (Fewer than 128 of them: 8 groups of 2048x7168 42 -> 57.)
// * Rows of B off the 128-byte lines: tiles take them without the streaming policy, and so without a reason to be other tiles
//   (400x4096x2064 in 16 groups 40, streaming 50; 700x4096x4112 in 8 39, 128x256 tiles 60, the same without the policy 55), but for
//   128x256 tiles that come to one full round (480x11584x9536 in 4 groups 131, now 110).
// The choice goes by the average. Where one group holds a large share of the rows the forms are still ahead of or level with
// the plain tiles up to about half of all rows (13 groups, 1076x4608x5120: 82 -> 88, the worst seen), and behind where it holds
// all of them: 64 groups, 512x4096x4096 34 -> 50, 51 of 346x11584x384 21 -> 43, against 203 -> 174 and 83 -> 74 with rows spread at random.
enum GroupedForm {
  kGroupedTiles = MI355X_FP8_GROUPED_TILES,
  kGroupedRows16 = MI355X_FP8_GROUPED_ROWS_16,
  kGroupedRows32 = MI355X_FP8_GROUPED_ROWS_32,
  kGroupedRows64 = MI355X_FP8_GROUPED_ROWS_64,
  kGroupedStream128 = MI355X_FP8_GROUPED_STREAM_128,
  kGroupedStream256 = MI355X_FP8_GROUPED_STREAM_256
};
constexpr bool grouped_rows16_fits(int64_t G, int64_t M, int64_t N) {
  return grid_fits(grouped_column_tiles(N, 32) * grouped_row_blocks(G, M, 16, true), 256);
}
static_assert(!grouped_rows16_fits(256, 256, 2200000) && grouped_rows16_fits(256, 2048, 57344), "a column tile and row block are 256 lanes");
inline GroupedForm grouped_form(int64_t G, int64_t M, int64_t N, int64_t K, int64_t ldb) {
  const bool rows_forms = G <= 256;  // (a workgroup's look-up goes over 64 groups at a time, the tiled kernel's once a launch)
  if (M <= 8 * G && rows_forms && grouped_rows16_fits(G, M, N)) return kGroupedRows16;
  const int64_t tiles_128 = G * ((N + 127) / 128), tiles_256 = G * ((N + 255) / 256);
  if (rows_forms && K >= 4096 && tiles_128 <= 128 && M <= 32 * G) return M <= 16 * G ? kGroupedRows32 : kGroupedRows64;
  if (K < 2048 || M > 128 * G) return kGroupedTiles;
  if (ldb % kStepK != 0) return M > 64 * G && tiles_256 >= 176 && tiles_256 <= kNumCu ? kGroupedStream256 : kGroupedTiles;
  if (M > 64 * G) return tiles_256 >= 128 ? kGroupedStream256 : kGroupedTiles;
  return tiles_128 >= 128 ? kGroupedStream128 : kGroupedTiles;
}

// Estimated times of the block-scaled forms over MFMA-bound shapes, from launches with 4 to 104 steps (us a 128-byte
// step of a round of tiles, and what a round costs beside its steps). 128x128 tiles, two workgroups per CU: 8192^3
// 545 us (8 rounds of 64 steps), 4096x10240x8192 350; alone on their CUs 1024x2048x4096 20 (128 tiles of 32
// steps), 2048x2048x4096 22.6 (256).
// One tile row against a wide panel is bound by the stream of B and fetches it with the streaming policy: K = 8192,
// N = 57344 78 / 83 / 98 us with 16 / 64 / 128 rows (96 / 109 / 117 without the policy), N = 28672 48 with 64 rows (63);
// with fewer workgroups it costs: 24x20480x5120 30.9 -> 31.9, 128x2304x6656 28 -> 34.
// It also costs where rows do not start on 128-byte lines, which pieces of two neighbouring steps then share (K = 3952, 9 rows,
// N = 64149 56 -> 68 us, K = 2640, 23 rows, N = 58574 43 -> 49), and on short rows (N = 65536, 64 rows: K = 128 6.7 -> 8.2, 512
// 11.2 -> 12.9; 128 rows, K = 1024: 21.4 -> 22.1) against all but the largest panels (one row, K = 768: N = 65536 15.0 -> 13.3,
// N = 40064 11.35 -> 11.8; 128 rows, N = 100096, K = 768 31.7 -> 29.2). From K = 2048 on it is never behind.
inline bool block_streams(int64_t M, int64_t N, int64_t K, bool off_lines) {
  const int64_t large = (int64_t)(M <= 48 ? 36 : M <= 64 ? 48 : 72) << 20;
  return M <= 128 && N >= 192 * 128 && !off_lines && (K >= 2048 || N * K >= large);
}
inline float block_small_cost_us(int64_t M, int64_t N, int64_t K, bool off_lines) {
  const float steps = (float)k_steps_of(K);
  if (block_streams(M, N, K, off_lines)) return fmaxf(5.0f + (float)N * (float)K * (1.0f + (float)M / 400.0f) / 6.4e6f, 6.0f + 0.62f * steps);
  const long tiles = ((M + 127) / 128) * ((N + 127) / 128), full = tiles / (2 * kNumCu), rest = tiles % (2 * kNumCu);
  // (one tile row: its steps wait for HBM, 16x8192x8192 40 us, 16x13312x13312 67)
  const float alone = M <= 128 ? 0.58f : 0.45f + 0.1f * (float)rest / (float)kNumCu;
  float t = (float)full * (steps + 5.0f);
  if (rest) t += steps * (rest <= kNumCu ? alone : 1.0f) + 5.0f;
  return t;
}
// 256x256 tiles: 8192^3 416-425 us (4 rounds of 64 steps), 2048x8192x2048 33.7 (one of 16), 4096x2304x13312 129 (144
// tiles of 104 steps), 1024x8192x8192 76.5 (128 of 64), 512x4096x4096 38.6 (64 of 32): a step slows down with the
// share of the chip at work beyond one half.
inline float block_large_cost_us(int64_t M, int64_t N, int64_t K) {
  const long tiles = ((M + kBlockTile - 1) / kBlockTile) * ((N + kBlockTile - 1) / kBlockTile), full = tiles / kNumCu, rest = tiles % kNumCu;
  const float steps = (float)k_steps_of(K), share = (float)rest / (float)kNumCu;
  float t = (float)full * (steps * 1.55f + 8.0f);
  if (rest) t += steps * (share <= 0.5f ? 1.1f : 1.1f + 0.9f * (share - 0.5f)) + 6.0f;
  // (one tile row against a wide panel: 128x57344x8192 122 us, 200x57344x4096 62)
  return M <= kBlockTile ? fmaxf(t, 4.0f + (float)N * (float)K / 4.0e6f) : t;
}

// Up to 64 rows (256 where row blocks of it are one round) the streaming forms of the row-wise product take over, whose waves
// share out the K blocks of a tile: measured against 128x128 tiles 1x2304x2048 12.1 -> 3.4 us, 16x8192x8192 40.0 -> 13.6,
// 16x2048x16384 76.8 -> 13.2, 32x8192x28672 142 -> 46, 64x4096x2048 12.2 -> 6.4, 128x8192x8192 42.9 -> 21.9,
// 256x4096x4096 19.9 -> 12.2. Their times are those of the row-wise forms within 3 %, and so are the estimates.
enum BlockForm {
  kBlockOneTile = MI355X_FP8_BLOCK_ONE_TILE,
  kBlockNarrow = MI355X_FP8_BLOCK_NARROW,
  kBlockSmall = MI355X_FP8_BLOCK_TILES_128,
  kBlockSmallStream = MI355X_FP8_BLOCK_TILES_128_STREAM,
  kBlockLarge = MI355X_FP8_BLOCK_TILES_256,
  kBlockResident = MI355X_FP8_BLOCK_RESIDENT  // the pair kernel
};
// (One 16-row tile a workgroup, many of them on short rows: what bounds it is the rate at which they come and go, which the
// row-wise estimate has too high there. us a workgroup beyond the first 256: 16x24576x256 2.9e-3, 16x24576x384 3.3e-3,
// 24x31841x16 2.6e-3, 28x66614x208 3.7e-3, 44x87564x32 4.2e-3, 49x18200x64 (32 columns each) 13e-3, 64x65536x128 8.7e-3.)
inline float block_one_tile_cost_us(int64_t M, int64_t N, int64_t K, float off_lines) {
  const long wgs = (N + (M > 48 ? 31 : 15)) / (M > 48 ? 32 : 16);
  const float steps = fminf((float)k_steps_of(K), 8.0f);
  const float per_wg = (M <= 16 ? 2.4e-3f : M <= 32 ? 2.8e-3f : M <= 48 ? 4.1e-3f : 10.0e-3f) + 0.2e-3f * steps;
  return fmaxf(off_lines * one_tile_cost_us(M, N, K), 3.0f + (wgs > kNumCu ? (float)(wgs - kNumCu) * per_wg : 0.0f));
}
// The form that keeps A on chip against its row-wise estimate, with one tile a workgroup as it is. One tile a CU: off the lines it is behind by more
// the more rows of A and the longer K, and with up to 4 rows its start shows. Two: it is behind off the lines, most on long rows (2x4368x7616
// 11.3 us, on narrow tiles 10.3), and where its second round of steps begins. (2420 shapes, weights from HBM: 0.998 of the time without this form on
// average, 1 % of them more than 2 % behind; by the row-wise estimate alone 1.000 and 5 %, 16x2528x3264 5.47 -> 6.08 us, 4x5376x3584 6.49 -> 7.08,
// 8x1088x4592 5.51 -> 6.07. What it is for: 16x8192x8192 14.1 -> 13.1, 16x8192x3600 9.88 -> 8.80, 16x512x5936 7.53 -> 7.14.)
inline float block_resident_factor(int64_t M, int64_t N, int64_t K, bool off_lines) {
  if (N <= 16 * kNumCu) return (off_lines ? 1.07f + 1.1e-6f * (float)M * (float)K : 1.01f) + (M <= 4 ? 0.08f : 0.0f);
  if (M > 8) return off_lines ? 1.2f : K > 4096 ? 1.0f : 1.09f;
  if (off_lines && K > 4096) return 1.17f;
  return (off_lines ? 1.07f : 1.01f) * (K > 2048 && K <= 4096 ? 1.08f : 1.0f);
}
inline BlockForm block_form(int64_t M, int64_t N, int64_t K, bool off_lines, float* cost_us = nullptr) {
  BlockForm best = block_streams(M, N, K, off_lines) ? kBlockSmallStream : kBlockSmall;
  float cost = block_small_cost_us(M, N, K, off_lines);
  auto weigh = [&](BlockForm form, float us) {
    if (us < cost) {
      best = form;
      cost = us;
    }
  };
  weigh(kBlockLarge, block_large_cost_us(M, N, K));
  // Rows off the 128-byte lines, K no multiple of a step (832 shapes of 1 to 256 rows, weights from HBM): times against the estimates, which are
  // of rows on the lines. Panels of several rounds of workgroups: 128x128 tiles 1.25 with 150 of them in the last round, 1.45 with 300, 1.6
  // with 450, less on short rows; one 16-row tile a workgroup 1.1 to 1.2 with up to four rows of A, 1.2 to 1.35 with 5 to 64; narrow tiles
  // 0.87 to 1.02 as they are. One round: narrow tiles 1.1 to 1.25 from K = 2048 on and up to 64 rows, 1.0 to 1.2 beyond; one tile a
  // workgroup 1.25 with 5 to 16 rows, 1.1 with fewer or more (below one a CU its estimate knows of rows off the lines). With the factors
  // below the form chosen is 0.7 % behind the quickest one on average and 38 of the shapes are more than 5 % behind; with those
  // of the kernels that fetched such rows with the streaming policy it was 2.4 % and 113: 48x35328x8432 109 us on 128x128 tiles, 88 on
  // narrow ones, 1x24904x1424 14.3 and 11.3 on one tile each, 5x570x11680 13.1 on narrow tiles and 9.9. (1000 other shapes: 1.016 times
  // as fast on average, 160 more than 2 % ahead, 23 behind, 32x43552x672 14.6 -> 16.7, 34x16528x8736 56 -> 63 and 59x3388x25840 39 -> 43.)
  float one_tile_off = 1.0f, narrow_off = 1.0f;
  if (off_lines && N > 64 * kNumCu) {
    if (M <= 128) {
      const long rest = (N + 127) / 128 % (2 * kNumCu);
      const float share = rest > kNumCu ? fminf(fmaxf((float)(K - 128) / 1400.0f, 0.0f), 1.0f) : K >= 1536 ? 1.0f : 0.3f;
      cost *= 1.0f + share * (0.25f + (float)rest / 1300.0f);
    }
    one_tile_off = 1.2f + 0.025f * (float)(M < 8 ? M : 8) * fminf((float)K / 8192.0f, 1.0f);
  } else if (off_lines && K >= 1536 && M <= kSkinnyMaxM) {
    narrow_off = 1.15f;
    if ((N + (M > 48 ? 31 : 15)) / (M > 48 ? 32 : 16) >= kNumCu) one_tile_off = M > 4 && M <= 16 ? 1.2f : 1.15f;
  }
  if (M <= kSkinnyMaxM) weigh(kBlockOneTile, block_one_tile_cost_us(M, N, K, one_tile_off));
  if (narrow_fits(M, N, K)) weigh(kBlockNarrow, narrow_off * narrow_cost_us(M, N, K));
  if (pair_skinny_fits(M, N, K)) weigh(kBlockResident, block_resident_factor(M, N, K, off_lines) * pair_cost_us(M, N, K));
  if (cost_us) *cost_us = cost;
  return best;
}

// K cut in parts where the tiles are few and K is long (with a workspace for the parts). us in the quickest form in one piece -> now:
// 1000x1000x28672 160 -> 47, 312x512x9088 37.3 -> 15.4, 1047x1566x12800 78 -> 40, 92x512x26368 29.5 -> 17.3, 32x1024x28672
// 27.1 -> 18.5, 500x5120x13824 80 -> 58, 96x16384x16384 96 -> 74. 265 shapes on the lines, 17 to 1500 rows and K from 2048: cut are 116, 0.60
// of the time on average, 3 of them behind by 2 to 5 %; the plan is 0.6 % behind the quickest one on average, most where it leaves
// 60 to 130 tiles with K = 4096 to 4700 in one piece (256x4098x4096 27.3, in two 21.7).
struct BlockPlan {
  BlockForm form;
  int splits, steps_per_split;
};
// 128x128 tiles with K cut into `splits` parts of `sps` steps: the times of block_small_cost_us over the work items, the second launch
// and the parts' trip through memory; bound by the stream of B where the tiles are one or two rows (64x28672x8192 in two
// 68 us, 128x57344x8192 142, where the streaming form takes 45 and 95 in one piece).
inline float block_split_cost_us(int64_t M, int64_t N, int64_t K, bool off_lines, int splits, int sps) {
  const long items = ((M + 127) / 128) * ((N + 127) / 128) * splits, full = items / (2 * kNumCu), rest = items % (2 * kNumCu);
  float t = (float)full * ((float)sps + 5.0f);
  if (rest) t += (float)sps * (rest <= kNumCu ? 0.45f + 0.1f * (float)rest / (float)kNumCu : 1.0f) + 5.0f;
  // (off the lines: 17x37568x10000 in two 103 us, in one piece 94)
  t = fmaxf(t, (off_lines ? 1.25f : 1.0f) * (float)(M + N) * (float)K / 4.4e6f);
  return t + 4.5f + 2.0f * (float)splits * (float)M * (float)N * 4.0f / 5.0e6f;
}
inline BlockPlan block_plan(int64_t M, int64_t N, int64_t K, bool off_lines, int max_splits) {
  const int k_steps = k_steps_of(K);
  float cost = 0.0f;
  BlockPlan best = {block_form(M, N, K, off_lines, &cost), 1, k_steps};
  for (int want = 2; want <= max_splits; ++want) {
    int splits, sps;
    normalise_splits(k_steps, want, splits, sps);
    if (splits != want || N * 512 > (int64_t)INT32_MAX) continue;
    // (Few rows: the estimate of the parts is low against those of the streaming forms. Off the lines, in parts and streaming: 6x1382x26000
    // 19.6 and 20.8 us, 6x780x20528 17.2 and 17.4, 4x1320x8048 11.9 and 8.1, 34x5029x16048 28.4 and 27.6, 33x894x24624 19.8 and 27.7.
    // From 65 rows on it is right, where 1.25 left 78x11956x10704 in one piece for 71 us, in two 47, and 110x8845x4592 for 36, in three 25.)
    const float few_rows = M <= 16 ? (off_lines ? 1.2f : 1.5f) : M <= kSkinnyMaxM && off_lines ? 1.1f : 1.0f;
    const float us = block_split_cost_us(M, N, K, off_lines, splits, sps) * few_rows;
    if (us < cost) {
      cost = us;
      best = {kBlockSmall, splits, sps};
    }
  }
  return best;
}

template <bool KTAIL>
int launch_block_form(GemmParams p, hipStream_t stream) {
  constexpr auto kern = gemm_block_kernel<KTAIL>;
  (void)LdsLimit<kern, kBlockLdsBytes>::registered;
  p.store = store_policy(p);
  p.tiles_m = (p.M + kBlockTile - 1) / kBlockTile;
  p.tiles_n = (p.N + kBlockTile - 1) / kBlockTile;
  make_fast_div((uint32_t)kGroupM * (uint32_t)p.tiles_n, p.div_group_mul, p.div_group_shift);
  const long total = (long)p.tiles_m * p.tiles_n;
  if (total > (long)INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "more than 2^31-1 tiles");
  const long grid = total < kNumCu ? (total + kNumXcd - 1) / kNumXcd * kNumXcd : kNumCu;
  if (const int st = ready_device()) return st;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kBlockWaves * 64), kBlockLdsBytes, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "block-scaled kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}
int launch_block(const GemmParams& p, hipStream_t s) { return p.K % kStepK ? launch_block_form<true>(p, s) : launch_block_form<false>(p, s); }

template <int BM, int BN, int WAVES_M, int WAVES_N, int WAVES_K, int DEPTH, bool PARTIAL, bool DWORDS>
int launch_any(GemmParams p, hipStream_t stream) {
  constexpr size_t lds_bytes = any_lds_bytes(BM, BN, WAVES_K, WAVES_M * WAVES_N);
  constexpr auto kern = gemm_any_kernel<BM, BN, WAVES_M, WAVES_N, WAVES_K, DEPTH, PARTIAL, DWORDS>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const long items = (long)p.tiles_m * p.tiles_n * p.splits;
  if (items > (long)INT32_MAX - kNumXcd || (long)kGroupM * p.tiles_n > (long)INT32_MAX)
    return fail(MI355X_FP8_ENOTSUP, "more than 2^31-1 tiles");
  make_fast_div((uint32_t)p.tiles_m * (uint32_t)p.tiles_n, p.div_tiles_mul, p.div_tiles_shift);
  make_fast_div((uint32_t)kGroupM * (uint32_t)p.tiles_n, p.div_group_mul, p.div_group_shift);
  if (const int st = ready_device()) return st;
  hipLaunchKernelGGL(kern, dim3((unsigned)((items + kNumXcd - 1) / kNumXcd * kNumXcd)), dim3(WAVES_M * WAVES_N * WAVES_K * 64), lds_bytes, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "generic kernel launch: %s", hipGetErrorString(e));
  return PARTIAL ? launch_finalize(p, stream) : MI355X_FP8_OK;
}

// Up to 64 rows: whether the streaming kernel's unaligned form runs. Its workgroups, one for 16 columns (32 from 33 rows on),
// share out the K steps among eight waves, so rows of one or two steps leave most of a workgroup idle, and on wide panels what
// it takes is the rate at which workgroups come and go: 1x30090x1 8.4 us against 4.9 for 64x64 tiles, 34x112402x13 54 against 11,
// 60x282266x3 156 against 29, 22x116414x94 42 against 19; the other way round 2x10559x202 4.8 against 5.7. (The grid: 512 lanes
// a workgroup, fewer than 2^32 in all.)
constexpr bool generic_streams(int64_t M, int64_t N, int64_t K) {
  if (M > kSkinnyMaxM || !grid_fits((N + 15) / 16, 512)) return false;
  return !(K <= (M <= 16 ? 128 : 256) && N > (M <= 32 ? 8192 : 4096));
}
static_assert(!generic_streams(1, 1 << 27, 1024) && generic_streams(1, (1 << 27) - 16, 1024), "2^27 columns are 2^32 lanes");
// Tiles of a launch above 64 rows, estimated from launches of 1 to 70 rounds of the CUs (1297 shapes, 65 to 8192 rows, K 100 to 16000): what
// starts and ends with the launch and with each tile, and the rounds of the CUs times a 128-byte step. Waves that share out K (64x64, 128x64 and 128x128
// tiles) are ahead while the tiles are few rounds, waves that share out the tile (128x128 and 64x64) on short rows and over many rounds: us in that
// order 463x1440x2101 14.2, 17.0, 23.9, 31.4 and 18.6; 362x5040x4907 39.8, 35.0, 45.6, 63.5 and 42.4; 243x15469x7535 105.6, 96.7, 76.8, 97.0 and 106.3;
// 707x19781x241 38.8, 51.8, 40.4, 33.1 and 35.8; 134x20332x519 19.9, 25.5, 26.0, 21.4 and 16.6. Rows on dwords have a sixth form, 128x64 tiles that
// the waves share out: 449x18784x3624 102.3, 107.4, 105.4, 105.2, 110.1 and 90.7; 152x24457x820 24.2, 28.2, 29.3, 23.9, 24.8 and 22.4. (Off the dwords it is
// never the quickest by more than noise.) The quickest is missed by 0.4 % on average off the dwords and by 0.5 % on them, and by more than 7 % on 4 of 674
// and 11 of 623. (With constants from 180 shapes for either 0.8 and 1.3 %: 210x193x356 8.04 us on 128x64, 6.60 on 64x64.)
enum GenericTiles { kGeneric64Shared, kGeneric128x64Shared, kGeneric128Shared, kGeneric128, kGeneric64, kGeneric128x64 };
static_assert(kGeneric64Shared + 1 == MI355X_FP8_GENERIC_TILES_64_K && kGeneric128x64Shared + 1 == MI355X_FP8_GENERIC_TILES_128X64_K &&
              kGeneric128Shared + 1 == MI355X_FP8_GENERIC_TILES_128_K && kGeneric128 + 1 == MI355X_FP8_GENERIC_TILES_128 &&
              kGeneric64 + 1 == MI355X_FP8_GENERIC_TILES_64 && kGeneric128x64 + 1 == MI355X_FP8_GENERIC_TILES_128X64, "the query's names, behind the streaming form's");
struct GenericChoice {
  GenericTiles tiles;
  float us;
};
struct GenericCost {
  int bm, bn, lanes, slots;  // slots: tiles of a round
  float start, tile, step, alone;  // us: of a launch, of each tile, of a step of a round, of a step at least
};
inline GenericChoice generic_tiles(int64_t M, int64_t N, int64_t K, bool dwords) {
  static const GenericCost any[] = {{64, 64, 256, kNumCu, 4.16f, 5.45e-3f, 0.433f, 0.0f},     {128, 64, 512, kNumCu, 3.64f, 9.56e-3f, 0.771f, 0.0f},
                                    {128, 128, 512, kNumCu, 3.86f, 21.1e-3f, 1.135f, 0.0f},    {128, 128, 256, 2 * kNumCu, 4.32f, 17.9e-3f, 1.682f, 0.0f},
                                    {64, 64, 256, kNumCu, 1.85f, 5.15e-3f, 0.385f, 1.371f}};
  static const GenericCost on_dwords[] = {{64, 64, 256, kNumCu, 3.86f, 3.28e-3f, 0.443f, 0.0f},  {128, 64, 512, kNumCu, 3.72f, 11.3e-3f, 0.629f, 0.0f},
                                          {128, 128, 512, kNumCu, 3.85f, 16.7e-3f, 1.086f, 0.0f}, {128, 128, 256, 2 * kNumCu, 5.06f, 12.1e-3f, 1.787f, 0.0f},
                                          {64, 64, 256, kNumCu, 1.81f, 4.46e-3f, 0.380f, 1.123f}, {128, 64, 256, kNumCu, 5.38f, 5.36e-3f, 0.568f, 0.769f}};
  const GenericCost* const forms = dwords ? on_dwords : any;
  const float steps = (float)k_steps_of(K);
  auto us = [&](int form) {
    const GenericCost& c = forms[form];
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    if (form != kGeneric128 && !grid_fits(tiles, c.lanes)) return 1e30f;  // (a launch takes fewer than 2^32 lanes)
    return c.start + c.tile * (float)tiles + steps * fmaxf(c.alone, c.step * (float)((tiles + c.slots - 1) / c.slots));
  };
  // (one step, or one row of tiles: nothing to gain from the larger tiles, 164x39275x3 21.6 us with 128x128, 14.0 with 64x64)
  if ((M <= kSkinnyMaxM || K <= kStepK) && us(kGeneric64) < 1e30f) return {kGeneric64, us(kGeneric64)};
  GenericChoice best = {kGeneric128, us(kGeneric128)};
  for (int f = kGeneric64Shared; f <= (dwords ? kGeneric128x64 : kGeneric64); ++f)
    if (us(f) < best.us) best = {(GenericTiles)f, us(f)};
  return best;
}

// Where the tiles are few and K is long, K is cut into parts (128x64 tiles, up to one item a CU): a launch is as quick as it has CUs at
// work. What the second pass adds is a launch and the planes' way through memory.
struct GenericPlan {
  int splits, steps_per_split;
};
inline GenericPlan generic_plan(int64_t M, int64_t N, int64_t K, int max_splits) {
  const int k_steps = k_steps_of(K);
  GenericPlan best = {1, k_steps};
  const int64_t tiles_64 = ((M + 63) / 64) * ((N + 63) / 64), tiles = ((M + 127) / 128) * ((N + 63) / 64);
  if (generic_streams(M, N, K) || tiles_64 >= kNumCu) return best;
  float cost = generic_tiles(M, N, K, K % 4 == 0).us;  // (by the sizes alone, like the query)
  for (int want = 2; want <= max_splits && tiles * want <= kNumCu; ++want) {
    int splits, sps;
    normalise_splits(k_steps, want, splits, sps);
    if (splits != want) continue;
    const float us = (float)sps * 0.62f + 7.5f + 2.0f * (float)splits * (float)M * (float)N * 4.0f / 5.0e6f;
    if (us < cost) {
      cost = us;
      best = {splits, sps};
    }
  }
  return best;
}

// The generic family: the streaming kernel's unaligned form up to 64 rows but for short rows on wide panels (measured cold: 1x8192x8191 14.4 us,
// 16x8192x8191 19.1, 64x8192x8191 29.7, where 64x64 tiles take 33), tiles beyond. Tiles whose waves share out K run two steps ahead
// (61.1 -> 41.8 us on 128x8192x8191), the others, of which a CU has several, one.
template <bool DWORDS>
int launch_generic_tiles(const GemmParams& p, hipStream_t s) {
  switch (generic_tiles(p.M, p.N, p.K, DWORDS).tiles) {
    case kGeneric64Shared: return launch_any<64, 64, 1, 1, 4, 2, false, DWORDS>(p, s);
    case kGeneric128x64Shared: return launch_any<128, 64, 2, 1, 4, 2, false, DWORDS>(p, s);
    case kGeneric128Shared: return launch_any<128, 128, 2, 1, 4, 2, false, DWORDS>(p, s);
    case kGeneric64: return launch_any<64, 64, 2, 2, 1, 1, false, DWORDS>(p, s);
    case kGeneric128x64:
      if constexpr (DWORDS) return launch_any<128, 64, 2, 2, 1, 1, false, true>(p, s);
      [[fallthrough]];
    default: return launch_any<128, 128, 2, 2, 1, 1, false, DWORDS>(p, s);
  }
}
int launch_generic(const GemmParams& p, hipStream_t s) {
  // (the documented range of the family, which the tests' sizes lie in)
  if (p.M > 65535 * 64) return fail(MI355X_FP8_ENOTSUP, "the generic family takes M <= %d", 65535 * 64);
  const bool dwords = ((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | (uintptr_t)p.lda | (uintptr_t)p.ldb) & 3) == 0;
  if (p.splits > 1) return dwords ? launch_any<128, 64, 2, 1, 4, 2, true, true>(p, s) : launch_any<128, 64, 2, 1, 4, 2, true, false>(p, s);
  if (generic_streams(p.M, p.N, p.K)) {
    if (p.M <= 16) return launch_skinny<1, 1, 4, 8, true>(p, s);
    if (p.M <= 32) return launch_skinny<2, 1, 2, 8, true>(p, s);
    return launch_skinny<4, 2, 2, 8, true>(p, s);
  }
  return dwords ? launch_generic_tiles<true>(p, s) : launch_generic_tiles<false>(p, s);
}

// ---- built-in scratch of the entry point that allocates nothing
// Split-K plans park their fp32 partial sums in device memory between the two launches. Callers
// that cannot bring a workspace (HIP graph capture, serving loops that may not allocate) get this
// array instead: every device the library is loaded on holds its own copy until the process
// ends. In host code the array's name is only a handle for the symbol look-up in setup_device();
// kernels, fills and copies take the per-device address that look-up returns.
constexpr size_t kScratchBytes = (size_t)MI355X_FP8_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Sets the current device `dev` up: checks its shape, raises the dynamic-LDS limit of every
// registered kernel on it and looks up the address of its copy of `scratch`. None of this is an
// enqueue, so it belongs in front of any graph capture: mi355x_fp8_rowwise_init() does it by name,
// and a first call on a device that was never initialised does it on the way.
int setup_device(int dev) {
  if (g_device_state[dev].load(std::memory_order_acquire) < 0)
    return fail(MI355X_FP8_ENOTSUP, "device %d does not report the %d compute units these kernels are scheduled for "
                "(a partitioned mode or another part)", dev, kNumCu);
  if (mi355x_shared::lds_table_overflow) return fail(MI355X_FP8_ELAUNCH, "kernel table overflow (more than %d instantiations)", mi355x_shared::kMaxLdsKernels);
  if (const int st = check_device_shape(dev)) {
    if (st == MI355X_FP8_ENOTSUP) g_device_state[dev].store(-1, std::memory_order_release);
    return st;
  }
  for (int i = 0; i < mi355x_shared::num_lds_kernels; ++i) {
    const hipError_t e = hipFuncSetAttribute(mi355x_shared::lds_kernels[i].kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)mi355x_shared::lds_kernels[i].lds_bytes);
    if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  }
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) return fail(MI355X_FP8_ELAUNCH, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
  g_scratch_ptr[dev].store(ptr, std::memory_order_release);  // every thread finds the same address
  g_device_state[dev].store(1, std::memory_order_release);
  return MI355X_FP8_OK;
}

// Address of the current device's copy of `scratch`.
int scratch_of_current_device(void** out) {
  int dev = 0;
  if (const int st = ready_device(&dev)) return st;
  *out = g_scratch_ptr[dev].load(std::memory_order_acquire);
  return MI355X_FP8_OK;
}

// The persistent skinny kernel takes N a multiple of 16 and K of 2048 up to 8192 with M <= 16,
// and K = 4096 with M <= 32. (Two blocks of A in registers leave room for two steps of B in
// flight per wave. At K = 4096 that is a whole tile ahead and the form wins: M=32, N=8192 9.9 us
// against 11.4 us for the one-tile kernel. At K = 8192 it is half a tile and loses, 20.6 against
// 17.9 us; four steps in flight do not fit the 128 registers of a 16-wave workgroup.)
inline bool persistent_skinny_fits(int64_t M, int64_t N, int64_t K) {
  if (N % 16 != 0 || K % (kPersistWaves * kStepK) != 0) return false;
  const int64_t spw = K / (kPersistWaves * kStepK);
  return (M <= 16 && spw <= 4) || (M <= 32 && spw == 2);
}

template <int SPW, int MT, int LAG, bool VEC>
int launch_skinny_persistent(const GemmParams& p, hipStream_t stream) {
  constexpr size_t lds_bytes = persistent_lds_bytes(MT);
  constexpr auto kern = gemm_skinny_persistent_kernel<SPW, MT, LAG, VEC>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  if (const int st = ready_device()) return st;
  const long ntiles = p.N / 16;
  const unsigned grid = (unsigned)(ntiles < kNumCu ? ntiles : kNumCu);
  GemmParams q = p;
  q.tiles_m = (int)(ntiles / grid);  // tiles per workgroup ...
  q.tiles_n = (int)(ntiles % grid);  // ... and how many workgroups take one more
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kPersistWaves * 64), lds_bytes, stream, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "persistent skinny kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

template <int SPW, bool VEC, bool KTAIL, bool HAS_BIAS, bool OFF_LINES = false, bool BLOCK = false>
int launch_skinny_pair(const GemmParams& p, hipStream_t stream) {
  if constexpr (KTAIL && !OFF_LINES) {  // (whole rounds of steps are off the lines with padded rows only)
    if (off_lines(p, kHalfLine) && !asked_for_at_once(p)) return launch_skinny_pair<SPW, VEC, KTAIL, HAS_BIAS, true, BLOCK>(p, stream);
  }
  constexpr size_t lds_bytes = pair_lds_bytes(SPW);
  static_assert(lds_bytes <= 160 * 1024, "A's steps, the transpose buffers and the partial results must fit the LDS");
  constexpr auto kern = gemm_skinny_pair_kernel<SPW, VEC, KTAIL, HAS_BIAS, OFF_LINES, BLOCK>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  if (const int st = ready_device()) return st;
  const long ntiles = p.N / 16;
  const unsigned grid = (unsigned)(ntiles < kNumCu ? ntiles : kNumCu);
  GemmParams q = p;
  q.tiles_m = (int)(ntiles / grid);  // tiles per workgroup ...
  q.tiles_n = (int)(ntiles % grid);  // ... and how many workgroups take one more
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kPersistWaves * 64), lds_bytes, stream, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "pair skinny kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

template <bool VEC, bool KTAIL, bool HAS_BIAS, bool BLOCK = false>
int launch_skinny_pair_steps(const GemmParams& p, hipStream_t s) {
  const int steps = (p.K + kStepK - 1) / kStepK;
  const int spw = (steps + kPersistWaves - 1) / kPersistWaves;
  switch (spw) {
    case 1: return launch_skinny_pair<1, VEC, KTAIL, HAS_BIAS, false, BLOCK>(p, s);
    case 2: return launch_skinny_pair<2, VEC, KTAIL, HAS_BIAS, false, BLOCK>(p, s);
    case 3: return launch_skinny_pair<3, VEC, KTAIL, HAS_BIAS, false, BLOCK>(p, s);
    default: return launch_skinny_pair<4, VEC, KTAIL, HAS_BIAS, false, BLOCK>(p, s);
  }
}
template <bool VEC>
int launch_skinny_pair_form(const GemmParams& p, hipStream_t s) {
  const bool ktail = p.K % (kPersistWaves * kStepK) != 0;
  if (p.bias) return ktail ? launch_skinny_pair_steps<VEC, true, true>(p, s) : launch_skinny_pair_steps<VEC, false, true>(p, s);
  return ktail ? launch_skinny_pair_steps<VEC, true, false>(p, s) : launch_skinny_pair_steps<VEC, false, false>(p, s);
}

int launch_skinny_pair_block(const GemmParams& p, hipStream_t s) {
  const bool vec = (reinterpret_cast<uintptr_t>(p.c) & 7) == 0 && (p.ldc & 3) == 0;  // (8-byte stores of C)
  const bool ktail = p.K % (kPersistWaves * kStepK) != 0;
  if (vec) return ktail ? launch_skinny_pair_steps<true, true, false, true>(p, s) : launch_skinny_pair_steps<true, false, false, true>(p, s);
  return ktail ? launch_skinny_pair_steps<false, true, false, true>(p, s) : launch_skinny_pair_steps<false, false, false, true>(p, s);
}

template <bool VEC>
int launch_skinny_persistent_steps(const GemmParams& p, hipStream_t s) {
  const int spw = p.K / (kPersistWaves * kStepK);
  if (p.M > 16) return launch_skinny_persistent<2, 2, 2, VEC>(p, s);
  switch (spw) {
    case 1: return launch_skinny_persistent<1, 1, 1, VEC>(p, s);
    case 2: return launch_skinny_persistent<2, 1, 2, VEC>(p, s);
    case 3: return launch_skinny_persistent<3, 1, 3, VEC>(p, s);
    default: return launch_skinny_persistent<4, 1, 4, VEC>(p, s);
  }
}

template <int MB, int NB, bool BLOCK, bool OFF_LINES = false>
int launch_narrow(const GemmParams& p, hipStream_t stream) {
  if constexpr (!OFF_LINES) {
    // Rows off the lines: without the streaming policy the wider tiles' launches are quicker (128x8192x4112 17.3 -> 15.8 us,
    // 256x4096x4112 16.0 -> 12.1, 1x19687x15024 67.4 -> 60.2, 8x5233x12976 18.3 -> 16.5, 24x10179x19168 block-scaled 44.0 -> 40.0). With all rows
    // in one block and few columns a tile there is so little to fetch that a step's trip is what it takes, and the next step finds the
    // shared line on its way: 8x714x800 3.52, without 3.78, 2x2177x27472 block-scaled 25.6 and 29.0, 9x2881x21200 21.2 and 24.4,
    // 7x3468x23088 23.5 and 27.0; row-wise it ends a little earlier, 16x3421x7824 10.9 and 10.3, 16x4274x8176 block-scaled 12.7 and 12.1.
    const int few_columns = p.M > 32 ? 0 : p.M <= (BLOCK ? 16 : 8) ? (BLOCK ? 20 : 16) : 8;
    // (row blocks find their neighbours' lines in the L2s: they are level at 0.5 MB, 0.95 with the policy at 1.5; 5 % ahead with it up to 0.4)
    const bool keep = p.M > 32 * MB ? (int64_t)p.N * p.K <= 400 << 10
                                    : !off_lines(p, kHalfLine) || asked_for_at_once(p) || narrow_tile_cols(p.N) <= few_columns;
    if (off_lines(p) && !keep) return launch_narrow<MB, NB, BLOCK, true>(p, stream);
  }
  constexpr size_t lds_bytes = narrow_lds_bytes(MB, NB);
  constexpr auto kern = gemm_narrow_kernel<MB, NB, BLOCK, OFF_LINES>;
  (void)LdsLimit<kern, lds_bytes>::registered;
  if (const int st = ready_device()) return st;
  const unsigned row_blocks = (unsigned)((p.M + 32 * MB - 1) / (32 * MB));
  GemmParams q = p;
  q.tiles_n = row_blocks == 1 ? narrow_tile_cols(p.N) : 32 * NB;  // columns per tile
  if (q.tiles_n > 32 * NB) return fail(MI355X_FP8_ELAUNCH, "narrow-tile form and tile width disagree");
  const unsigned tiles = (unsigned)((p.N + q.tiles_n - 1) / q.tiles_n);
  // (with row blocks the kernel deals tiles out per XCD: whole rounds of the XCDs)
  const unsigned grid = row_blocks == 1 ? tiles : (tiles + kNumXcd - 1) / kNumXcd * kNumXcd * row_blocks;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds_bytes, stream, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "narrow-tile kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

// the narrow-tile instantiation for a shape
template <bool BLOCK = false>
int launch_narrow_for(const GemmParams& p, hipStream_t s) {
  const NarrowForm f = narrow_form(p.M, p.N);
  if (f.mb == 1) return f.nb == 1 ? launch_narrow<1, 1, BLOCK>(p, s) : launch_narrow<1, 2, BLOCK>(p, s);
  return f.nb == 1 ? launch_narrow<2, 1, BLOCK>(p, s) : launch_narrow<2, 2, BLOCK>(p, s);
}

int run_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale, const void* bias, void* c,
             int out_type, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, void* workspace,
             size_t workspace_bytes, int variant, void* stream, unsigned long long* stamps);

}  // namespace

// What is chosen for a shape depends on its sizes alone and takes 0.7 to 1.5 us of the host to weigh up, two to four times a
// call, where the whole call is about 4 us and a launch of a few rows 3 us on the GPU: it is the host that such calls wait for. Every
// thread keeps the choices of the shapes it met last, one per entry of a table of fixed size: workspace_bytes + choice of
// 1x2304x2048 1.9 us -> 0.02.
template <typename Value>
struct Choices {
  static constexpr int kEntries = 128;
  struct Entry {
    int64_t m, n, k, how;  // (m = 0: empty)
    Value value;
  } entries[kEntries];
  template <typename Weigh>
  const Value& get(int64_t m, int64_t n, int64_t k, int64_t how, Weigh weigh) {
    const uint64_t h = ((uint64_t)m * 0x9E3779B97F4A7C15u ^ (uint64_t)n) * 0xC2B2AE3D27D4EB4Fu + (uint64_t)k * 0x165667B19E3779F9u + (uint64_t)how;
    Entry& e = entries[(h * 0x9E3779B97F4A7C15u) >> 57];
    if (e.m != m || e.n != n || e.k != k || e.how != how) e = {m, n, k, how, weigh()};
    return e.value;
  }
};
static_assert(kMaxSplits < 1 << 7, "the factor has seven bits of a plan's key");
static_assert(Choices<int>::kEntries == 1 << (64 - 57), "the hash's top bits index the table");
thread_local Choices<TiledPlan> known_plans;
thread_local Choices<int> known_families;
thread_local Choices<BlockPlan> known_block_plans;

// (`pitch`: lda | ldb)
inline TiledPlan known_plan(int64_t M, int64_t N, int64_t K, int64_t pitch, int variant, int max_splits) {
  variant &= ~0xff;  // (the plan does not depend on the family's number)
  const bool off_lines = pitch % kStepK != 0;
  return known_plans.get(M, N, K, (int64_t)variant << 8 | (int64_t)off_lines << 7 | max_splits,
                         [&] { return plan_from_variant(M, N, K, off_lines, variant, max_splits); });
}

// (the size query and the call behind it ask for the same entry: 0.2 us for both without it, 0.04 with it, on a call of 4)
inline BlockPlan known_block_plan(int64_t M, int64_t N, int64_t K, int64_t ldb, int max_splits) {
  const bool off_lines = ldb % kStepK != 0;  // (all that the plan depends on of ldb)
  return known_block_plans.get(M, N, K, (int64_t)off_lines << 8 | max_splits, [&] { return block_plan(M, N, K, off_lines, max_splits); });
}

extern "C" {

int mi355x_fp8_rowwise_abi_version(void) { return MI355X_FP8_ABI_VERSION; }

int mi355x_fp8_rowwise_init(void) { return ready_device(); }

const char* mi355x_fp8_rowwise_last_error(void) { return mi355x_shared::err; }

int mi355x_fp8_rowwise_select_variant(int64_t M, int64_t N, int64_t K) {
  const int st = check_shape(M, N, K);
  if (st != MI355X_FP8_OK) return st;
  if (K % 16 != 0) return MI355X_FP8_VARIANT_GENERIC;
  if (M > kSkinnyMaxM && !narrow_fits(M, N, K)) return MI355X_FP8_VARIANT_TILED;
  return known_families.get(M, N, K, 0, [&] {
    // M <= 64: the streaming kernel, unless a tiled plan (64- or 128-row tiles that stream B, split
    // K where the tiles are few) is expected to beat it: from two 16-row blocks of A up on most
    // shapes, with one block on the longest weight panels. Up to 8 rows the streaming kernel was
    // behind on one kind of shape only, few columns with very long rows, where a handful of workgroups
    // each stream a long tile and split tiles put the whole chip to work (8 x 1024 x 28672: 16.2 us
    // against 14.5); there a tiled plan has to be expected ahead by a tenth to be taken.
    // (above 64 rows the family's only member is the narrow-tile kernel in row blocks, where it fits)
    const float margin = M <= 8 ? 0.9f : 1.0f;
    return known_plan(M, N, K, K, MI355X_FP8_VARIANT_AUTO, kMaxSplits).cost_us < margin * skinny_cost_us(M, N, K) ? MI355X_FP8_VARIANT_TILED
                                                                                                              : MI355X_FP8_VARIANT_SKINNY;
  });
}

size_t mi355x_fp8_rowwise_workspace_bytes(int64_t M, int64_t N, int64_t K, int variant) {
  if (check_shape(M, N, K) != MI355X_FP8_OK) return 0;
  if ((variant & 0xff) == MI355X_FP8_VARIANT_AUTO)
    variant = (variant & ~0xff) | mi355x_fp8_rowwise_select_variant(M, N, K);
  if ((variant & 0xff) == MI355X_FP8_VARIANT_GENERIC) {
    const int splits = generic_plan(M, N, K, kMaxSplits).splits;
    return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
  }
  // (the skinny kernels reduce on chip)
  if ((variant & 0xff) != MI355X_FP8_VARIANT_TILED || K % 16 != 0) return 0;
  // (the pitch is not known here: enough for rows of K bytes and for rows padded onto the lines, whose plan can have more parts)
  int splits = known_plan(M, N, K, K, variant, kMaxSplits).splits;
  if (K % kStepK != 0) splits = std::max(splits, known_plan(M, N, K, 0, variant, kMaxSplits).splits);
  return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

int mi355x_fp8_rowwise_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale,
                            const void* bias, void* c, int64_t M, int64_t N, int64_t K, int64_t lda,
                            int64_t ldb, int64_t ldc, void* workspace, size_t workspace_bytes,
                            int variant, void* stream) {
  return mi355x_fp8_rowwise_gemm_ex(a, b, a_scale, b_scale, bias, c, MI355X_FP8_OUT_BF16, M, N, K, lda, ldb, ldc,
                                    workspace, workspace_bytes, variant, stream);
}

int mi355x_fp8_rowwise_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                               const void* bias, void* c, int out_type, int64_t M, int64_t N, int64_t K,
                               int64_t lda, int64_t ldb, int64_t ldc, void* workspace, size_t workspace_bytes,
                               int variant, void* stream) {
  return run_gemm(a, b, a_scale, b_scale, bias, c, out_type, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, variant,
                  stream, nullptr);
}

int mi355x_fp8_rowwise_gemm_stamped(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                    const void* bias, void* c, int64_t M, int64_t N, int64_t K, int64_t lda,
                                    int64_t ldb, int64_t ldc, void* workspace, size_t workspace_bytes, int variant,
                                    uint64_t* stamps, size_t stamp_entries, void* stream) {
  if (!stamps || stamp_entries < (size_t)MI355X_FP8_STAMP_ENTRIES)
    return fail(MI355X_FP8_EINVAL, "stamps must hold %d entries (got %zu)", MI355X_FP8_STAMP_ENTRIES, stamps ? stamp_entries : (size_t)0);
  if (reinterpret_cast<uintptr_t>(stamps) & 7) return fail(MI355X_FP8_EINVAL, "misaligned stamps pointer");
  return run_gemm(a, b, a_scale, b_scale, bias, c, MI355X_FP8_OUT_BF16, M, N, K, lda, ldb, ldc, workspace, workspace_bytes,
                  variant, stream, reinterpret_cast<unsigned long long*>(stamps));
}

}  // extern "C"

namespace {
int run_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale, const void* bias, void* c,
             int out_type, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, void* workspace,
             size_t workspace_bytes, int variant, void* stream, unsigned long long* stamps) {
  if (out_type != MI355X_FP8_OUT_BF16 && out_type != MI355X_FP8_OUT_F16)
    return fail(MI355X_FP8_EINVAL, "unknown output type %d", out_type);
  int st = check_shape(M, N, K);
  if (st != MI355X_FP8_OK) return st;
  if (!a || !b || !a_scale || !b_scale || !c) return fail(MI355X_FP8_EINVAL, "null operand pointer");
  if (lda < K || ldb < K || ldc < N) return fail(MI355X_FP8_EINVAL, "leading dimension smaller than the row length");
  if ((reinterpret_cast<uintptr_t>(a_scale) & 3) || (reinterpret_cast<uintptr_t>(b_scale) & 3) ||
      (reinterpret_cast<uintptr_t>(c) & 1) || (reinterpret_cast<uintptr_t>(bias) & 1))
    return fail(MI355X_FP8_EINVAL, "misaligned scale, bias or output pointer");
  if (variant < 0 || (variant >> 24) || ((variant >> 8) & 0xff) > kNumTileConfigs)
    return fail(MI355X_FP8_EINVAL, "unknown variant 0x%x", variant);
  const int plan_bits = variant & ~0xff;
  variant &= 0xff;
  // What the MFMA families ask of the operands; the generic family takes whatever is left, and AUTO
  // sends it there.
  const char* unfit = nullptr;
  if (K % 16 != 0) unfit = "K must be a multiple of 16";
  else if (lda % 16 || ldb % 16) unfit = "lda and ldb must be multiples of 16";
  else if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15)) unfit = "a and b must be 16-byte aligned";
  // (a tile's rows are addressed with 32-bit byte offsets that must stay below 2^31)
  else if (lda * 256 > (int64_t)INT32_MAX || ldb * 256 > (int64_t)INT32_MAX || ldc * 512 > (int64_t)INT32_MAX)
    unfit = "leading dimension too large";
  if (unfit && variant == MI355X_FP8_VARIANT_AUTO) variant = MI355X_FP8_VARIANT_GENERIC;
  if (unfit && variant != MI355X_FP8_VARIANT_GENERIC)
    return fail(MI355X_FP8_ENOTSUP, "%s for this kernel family (lda %lld, ldb %lld, ldc %lld, K %lld); the generic family or "
                "the automatic choice takes such operands", unfit, (long long)lda, (long long)ldb, (long long)ldc, (long long)K);
  if (variant == MI355X_FP8_VARIANT_GENERIC && stamps)
    return fail(MI355X_FP8_ENOTSUP, "the stamped entry point runs the tiled family only");
  if (variant == MI355X_FP8_VARIANT_AUTO) {
    variant = mi355x_fp8_rowwise_select_variant(M, N, K);
    if (variant == MI355X_FP8_VARIANT_TILED && (M <= kSkinnyMaxM || narrow_fits(M, N, K))) {
      // the choice assumed the plan's workspace; without it the plan changes and may lose
      const TiledPlan plan = known_plan(M, N, K, lda | ldb, plan_bits, kMaxSplits);
      const size_t need = plan.splits > 1 ? (size_t)plan.splits * M * N * sizeof(float) : 0;
      if (need && (!workspace || workspace_bytes < need) &&
          known_plan(M, N, K, lda | ldb, plan_bits, 1).cost_us >= skinny_cost_us(M, N, K))
        variant = MI355X_FP8_VARIANT_SKINNY;
    }
  }
  if (variant == MI355X_FP8_VARIANT_SKINNY && M > kSkinnyMaxM && !narrow_fits(M, N, K))
    return fail(MI355X_FP8_ENOTSUP,
                "skinny variant handles M <= %d, and M <= %d where 64x64 tiles give every CU at most one (got %lldx%lld)",
                kSkinnyMaxM, kNarrowMaxM, (long long)M, (long long)N);

  GemmParams p;
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b;
  p.a_scale = a_scale; p.b_scale = b_scale;
  p.bias = (const uint16_t*)bias; p.c = (uint16_t*)c;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.tiles_m = p.tiles_n = 0;
  p.splits = 1; p.steps_per_split = k_steps_of(K); p.partial = nullptr;
  p.m_sizes = nullptr; p.groups = 0; p.clear_rest = 0; p.out_f16 = out_type == MI355X_FP8_OUT_F16;
  p.div_tiles_mul = p.div_tiles_shift = p.div_group_mul = p.div_group_shift = 0; p.stamps = stamps;
  hipStream_t s = (hipStream_t)stream;

  switch (variant) {
    case MI355X_FP8_VARIANT_TILED:
      {
        // A caller that brought no (or too little) workspace gets the best plan that needs none,
        // unless it asked for a split factor by name.
        TiledPlan plan = known_plan(M, N, K, lda | ldb, plan_bits, kMaxSplits);
        const size_t need = plan.splits > 1 ? (size_t)plan.splits * M * N * sizeof(float) : 0;
        if (need && (!workspace || workspace_bytes < need)) {
          if ((plan_bits >> 16) & 0xff)
            return fail(MI355X_FP8_EINVAL, "split-K factor %d needs %zu bytes of workspace (got %zu)",
                        plan.splits, need, workspace ? workspace_bytes : (size_t)0);
          // the cheapest plan whose partial planes fit what the caller brought (none: the unsplit plans)
          const size_t plane = (size_t)M * (size_t)N * sizeof(float);
          const size_t fit = workspace ? workspace_bytes / plane : 0;
          plan = known_plan(M, N, K, lda | ldb, plan_bits, fit < 1 ? 1 : fit > (size_t)kMaxSplits ? kMaxSplits : (int)fit);
        }
        // (the partial sums of a tile are addressed with 32-bit byte offsets that must stay below 2^31)
        if (plan.splits > 1 && N * 512 > (int64_t)INT32_MAX) plan = known_plan(M, N, K, lda | ldb, plan_bits & 0xff00, 1);
        if (plan.splits > 1 && (reinterpret_cast<uintptr_t>(workspace) & 15))
          return fail(MI355X_FP8_EINVAL, "workspace must be 16-byte aligned");
        p.splits = plan.splits;
        p.steps_per_split = plan.steps_per_split;
        p.partial = plan.splits > 1 ? (float*)workspace : nullptr;
        switch (plan.config) {
          case 0: return mi355x_shared::tiled_config_0(p, s);
          case 1: return mi355x_shared::tiled_config_1(p, s);
          case 2: return mi355x_shared::tiled_config_2(p, s);
          case 3: return mi355x_shared::tiled_config_3(p, s);
          case 4: return mi355x_shared::tiled_config_4(p, s);
          case 5: return mi355x_shared::tiled_config_5(p, s);
          case 6: return mi355x_shared::tiled_config_6(p, s);
          default: return fail(MI355X_FP8_EINVAL, "unknown tile configuration %d", plan.config);
        }
      }
    case MI355X_FP8_VARIANT_SKINNY:
      // 16-row blocks of A | B tiles per wave | steps in flight per wave (sized to 128 VGPRs) | waves.
      // (Measured alternatives at M = 16: two B tiles per wave with 4, 6 or 8 steps in flight 17.8-19.9 us,
      // four waves 14.7-15.0 us, six steps in flight 16.4 us, against 14.4 us for this one.)
      if (plan_bits & MI355X_FP8_SKINNY_NARROW) {
        if (!narrow_fits(M, N, K))
          return fail(MI355X_FP8_ENOTSUP,
                      "the narrow-tile kernel takes M <= %d, and M <= %d where 64x64 tiles give every CU at most one (got %lldx%lld)",
                      kSkinnyMaxM, kNarrowMaxM, (long long)M, (long long)N);
        return launch_narrow_for<>(p, s);
      }
      if (M > kSkinnyMaxM) {
        if (plan_bits & MI355X_FP8_SKINNY_ONE_TILE)
          return fail(MI355X_FP8_ENOTSUP, "the one-tile-per-workgroup form takes M <= %d (got M=%lld)", kSkinnyMaxM, (long long)M);
        return launch_narrow_for<>(p, s);
      }
      if (!(plan_bits & (MI355X_FP8_SKINNY_ONE_TILE | MI355X_FP8_SKINNY_RESIDENT)) && narrow_preferred(M, N, K))
        return launch_narrow_for<>(p, s);
      if ((plan_bits & MI355X_FP8_SKINNY_RESIDENT) && !pair_skinny_fits(M, N, K) && !persistent_skinny_fits(M, N, K))
        return fail(MI355X_FP8_ENOTSUP, "neither form that keeps A on chip takes %lldx%lldx%lld", (long long)M, (long long)N, (long long)K);
      if ((pair_skinny_fits(M, N, K) || persistent_skinny_fits(M, N, K)) && !(plan_bits & MI355X_FP8_SKINNY_ONE_TILE)) {
        // 16-byte loads of b_scale, 8-byte loads of bias and 8-byte stores of C when everything is aligned for them
        const bool vec = (reinterpret_cast<uintptr_t>(b_scale) & 15) == 0 && (reinterpret_cast<uintptr_t>(bias) & 7) == 0 &&
                         (reinterpret_cast<uintptr_t>(c) & 7) == 0 && (ldc & 3) == 0;
        // (pinned, the forms that keep A on chip run wherever they fit; left to the library, where they are expected ahead)
        const bool resident = (plan_bits & MI355X_FP8_SKINNY_RESIDENT) || skinny_streaming_choice(M, N, K) != kStreamOneTile;
        // (the pair kernel addresses a workgroup's rows of B with 32-bit offsets below 2^31)
        if (resident && pair_skinny_fits(M, N, K) && ldb * 32 <= (int64_t)INT32_MAX)
          return vec ? launch_skinny_pair_form<true>(p, s) : launch_skinny_pair_form<false>(p, s);
        if (resident && persistent_skinny_fits(M, N, K))
          return vec ? launch_skinny_persistent_steps<true>(p, s) : launch_skinny_persistent_steps<false>(p, s);
      }
      if (M <= 16) return launch_skinny<1, 1, 4, 8>(p, s);
      if (M <= 32) return launch_skinny<2, 1, 2, 8>(p, s);
      if (M <= 48) return launch_skinny<3, 1, 2, 8>(p, s);
      return launch_skinny<4, 2, 2, 8>(p, s);  // 32 rows of B per workgroup: A passes L1 half as often
    case MI355X_FP8_VARIANT_GENERIC:
      {
        // (as many parts as the workspace holds planes; in one piece without one)
        const size_t planes = workspace && !(reinterpret_cast<uintptr_t>(workspace) & 15) ? workspace_bytes / ((size_t)M * (size_t)N * sizeof(float)) : 0;
        const GenericPlan plan = generic_plan(M, N, K, planes < 1 ? 1 : planes > (size_t)kMaxSplits ? kMaxSplits : (int)planes);
        p.splits = plan.splits;
        p.steps_per_split = plan.steps_per_split;
        p.partial = plan.splits > 1 ? (float*)workspace : nullptr;
        return launch_generic(p, s);
      }
    default:
      return fail(MI355X_FP8_EINVAL, "unknown variant %d", variant);
  }
}
}  // namespace

namespace {
constexpr int kWaveRows = 4;

// How a row's chunks of 16 bytes are dealt out by the quantiser and the fused front ends (rows that start 16-byte aligned): `lanes` of them,
// `chunks` rounds each that stay in registers; 64 lanes are a wave, kWaveRows rows a workgroup. Any form takes any row (what the registers don't
// hold is read again), so the rule is about speed alone, but for RMSNorm, whose lanes are those of the order of its sum or hand its chains on:
//  - no round is idle if it can be helped, for it loads and computes like any other: rows just above a power of two had up to half of them
//    idle (SiLU-mul 2048x19904 41.4 and 34.7; f32 8192x9472 72.7 and 60.6);
//  - up to one row a CU, what counts is the chain of a single row, and one round of as many lanes as that takes is the shortest (SiLU-mul
//    32x4096 4.89 as 8 of 64, 2.69 as one of 512). RMSNorm's second reduction makes that as long: cold 32x8192 3.49 us as 4 rounds of 256, 3.51
//    as 2 of 512 that hand on, 3.75 as one of 1024, 32x10240 3.78 as 3 of 512, 4.23 as 2 of 1024, so it keeps the lanes of its order;
//  - with more rows, fewer lanes with more rounds: RMSNorm 256x4 against 1024x1 is 35.5 and 53.0 us on 8192x8192, waves of 4 rounds against
//    256x1 11.0 and 14.3 on 8192x2048.
// Measured on 21 row lengths from 512 to 28672 with 1 to 8192 rows, every form whose rounds hold the row.
enum RowSource { kRowF32, kRowBf16, kRowRmsNorm, kRowSiluMul };
struct RowForm {
  int lanes, chunks;
};
constexpr bool row_form_exists(RowSource source, int lanes, int chunks) {
  if (source == kRowRmsNorm) return lanes <= 256 ? chunks <= 4 : lanes == 512 ? chunks == 8 || (chunks >= 3 && chunks <= 6) : chunks == 8;
  if (lanes == 64) return chunks <= 4 || (source == kRowF32 && (chunks == 6 || chunks == 8));
  if (lanes == 256) return chunks <= 5;
  if (lanes == 512) return chunks <= 8 && (chunks < 7 || source != kRowSiluMul);
  return chunks <= 4 || (source == kRowF32 && chunks <= 7) || (source != kRowBf16 && chunks == 8);
}
constexpr RowForm rms_row_form(int64_t R, int64_t chunks) {
  if (chunks > 4096) return {1024, 8};
  if (chunks > 256) {
    const int lanes = rms_sum_lanes(chunks), rounds = (int)((chunks + lanes - 1) / lanes);
    // (a round of its own at the end costs few rows more than an idle one, cold 32x20480 5.48 us as five, 4.78 as six, 32x28672 6.55 as seven, 5.42 as
    // eight; many rows not, 2048x20480 27.2 and 27.8, but for seven, 38.8 and 37.1)
    return {lanes, rounds == 7 || (rounds == 5 && R <= kNumCu) ? rounds + 1 : rounds};
  }
  if (chunks <= 64) return {64, 1};
  // (256x1 and 64x4 on rows of 2048: 512 rows 3.27 and 3.56 us, 1024 4.02 and 3.93, 2048 5.42 and 5.16; on rows of 1536 level with 512)
  if (R <= kNumCu || (chunks > 192 && R <= 2 * kNumCu)) return {256, 1};
  return {64, (int)((chunks + 63) / 64)};
}
constexpr RowForm row_form(RowSource source, int64_t R, int64_t chunks) {
  if (source == kRowRmsNorm) return rms_row_form(R, chunks);
  if (chunks > 4096) {  // (bf16 rows hold half the values in as many registers as f32 ones: more rounds than 4 halve their rate)
    if (source == kRowBf16) return {1024, 4};
    if (source == kRowF32 && chunks <= 7168) return {1024, (int)((chunks + 1023) / 1024)};
    return {1024, 8};
  }
  if (chunks <= 64) return {64, 1};
  if (R <= kNumCu) {
    if (chunks <= 256) return {256, 1};
    if (chunks <= 512) return {512, 1};
    return {1024, (int)((chunks + 1023) / 1024)};
  }
  const bool many = R > 2048;
  if (source == kRowBf16 && chunks <= 192 && R <= 1024) return {256, 1};  // (512 rows of 1536 3.07 us, in waves 3.67; 2048 4.91 and 4.96)
  if (chunks <= 192) return {64, chunks <= 128 ? 2 : 3};
  if (chunks <= 256) return many ? RowForm{64, 4} : RowForm{256, 1};
  if (chunks <= 512) return many && source == kRowF32 ? RowForm{64, chunks <= 384 ? 6 : 8} : RowForm{256, 2};
  if (chunks <= 768) return {256, 3};
  // (The quantiser: 2048 rows of 4096 f32 8.26 us as 256x4, 8.88 as 512x2, 1024 rows level; 8192 rows 28.8 and 27.5, of 3584 the other way
  // round. 2048 rows of 5120 f32 9.8 as 256x5, 10.4 as 512x3, 8192 35.2 and 34.1; bf16 keeps 256x5, 8192 of 8960 40.7 and 42.6.)
  if (source == kRowF32 && chunks > 960 && chunks <= 1024 && R > 4096) return {512, 2};
  if (chunks <= 1024) return many || (source != kRowSiluMul && R > 1024) ? RowForm{256, 4} : RowForm{512, 2};
  if (chunks <= 1280 && (many || (source == kRowF32 && R > 1024)) && !(source == kRowF32 && chunks > 1216 && R > 4096)) return {256, 5};
  if (chunks <= 3072) return {512, (int)((chunks + 511) / 512)};
  if (source == kRowSiluMul) return {1024, 4};
  return {512, chunks <= 3584 ? 7 : 8};
}
// Rows of a launch, which holds fewer than 2^32 lanes (256 a row: 16777212 rows). More of them are several launches of the same form.
constexpr int64_t rows_per_launch(int64_t lanes) { return (int64_t)UINT32_MAX / lanes / kWaveRows * kWaveRows; }
template <typename Launch>
void launch_by_rows(int64_t R, int64_t lanes, Launch&& launch) {
  for (int64_t row = 0; row < R; row += rows_per_launch(lanes)) launch(row, R - row < rows_per_launch(lanes) ? R - row : rows_per_launch(lanes));
}
constexpr bool row_forms_are_sound() {  // (the rule's lines lie at multiples of 64 chunks)
  for (int source = kRowF32; source <= kRowSiluMul; ++source) {
    bool chosen[17][9] = {};  // by 64 lanes and rounds
    for (int64_t R : {int64_t(1), int64_t(kNumCu), int64_t(kNumCu + 1), int64_t(1024), int64_t(1025), int64_t(2048), int64_t(2049), int64_t(4096), int64_t(4097)})
      for (int64_t chunks = 64; chunks <= 8192; chunks += 64)
        for (int64_t c : {chunks, chunks + 1}) {
          const RowForm f = row_form((RowSource)source, R, c);
          if (!row_form_exists((RowSource)source, f.lanes, f.chunks)) return false;
          chosen[f.lanes / 64][f.chunks] = true;
          if (!grid_fits(rows_per_launch(f.lanes), f.lanes)) return false;
          const int64_t held = (int64_t)f.lanes * f.chunks;
          if (source == kRowRmsNorm && c > held && rms_sum_lanes(held) != f.lanes) return false;
          if (source == kRowRmsNorm && rms_sum_lanes(held) != rms_sum_lanes(c)) return false;
          if (source == kRowRmsNorm && c <= 2048 && !rms_early_weights(f.lanes, f.chunks)) return false;
        }
    for (int lanes : {64, 256, 512, 1024})
      for (int chunks = 1; chunks <= 8; ++chunks)
        if (row_form_exists((RowSource)source, lanes, chunks) && !chosen[lanes / 64][chunks]) return false;
  }
  return true;
}
static_assert(row_forms_are_sound(), "a row without a kernel would not be quantised, and in another order of its sum not as among other rows; without "
                                     "its weights beside x it takes a second trip; a kernel without a row is code that nothing runs");

// Calls launch(lanes, chunks), as integral constants, for the form.
template <RowSource SOURCE, int LANES = 64, int CHUNKS = 1, typename Launch>
void with_row_form(RowForm f, Launch&& launch) {
  if constexpr (row_form_exists(SOURCE, LANES, CHUNKS)) {
    if (f.lanes == LANES && f.chunks == CHUNKS) return launch(std::integral_constant<int, LANES>{}, std::integral_constant<int, CHUNKS>{});
  }
  if constexpr (CHUNKS < 8) with_row_form<SOURCE, LANES, CHUNKS + 1>(f, launch);
  else if constexpr (LANES < 1024) with_row_form<SOURCE, LANES == 64 ? 256 : LANES * 2, 1>(f, launch);
}

// (more rows than a launch of 1024 lanes each holds keep 256 lanes, which read the rest of a long row twice)
constexpr bool quantize_any_long(int64_t R, int64_t chunks) { return chunks > 4 * 256 && grid_fits(R, 1024); }
static_assert(quantize_any_long(4194303, 1025) && !quantize_any_long(8388608, 1025), "512 lanes a row reach 2^32 at 8388608 rows");

template <RowSource SOURCE, typename SrcT>
void launch_quantize_rows(const SrcT* x, uint8_t* xq, float* inv_scale, int64_t R, int64_t K, int64_t ldx, int64_t ldq, hipStream_t s) {
  with_row_form<SOURCE>(row_form(SOURCE, R, K / VecTraits<SrcT>::EPV), [&](auto lanes, auto chunks) {
    constexpr int LANES = decltype(lanes)::value, ROWS = LANES == 64 ? kWaveRows : 1;
    launch_by_rows(R, LANES, [&](int64_t row, int64_t rows) {
      hipLaunchKernelGGL((quantize_rows_vec_kernel<SrcT, decltype(chunks)::value, LANES, ROWS>), dim3((unsigned)((rows + ROWS - 1) / ROWS)),
                         dim3(LANES * ROWS), 0, s, x + row * ldx, xq + row * ldq, inv_scale + row, (int)K, (long)ldx, (long)ldq, (long)rows);
    });
  });
}

// The quantiser on rows that do not start 16-byte aligned or do not hold whole 16-byte chunks: the vector kernel's
// unaligned forms, by the same lines as the aligned ones (fewer of them: this is the rare case). The element-by-element
// kernel, which ran them all before, is left for few or very short rows. Measured, sources rotated through memory, before
// -> now: f32 4096x8191 72 -> 28 us (2.3 -> 6.0 TB/s), 8192x2047 40 -> 15, 2048x20001 99 -> 36, 512x53247 181 -> 30; bf16
// 4096x8191 73 -> 22 (4.6 TB/s), 8192x2047 40 -> 15, 1024x28671 107 -> 23.
template <typename SrcT>
void launch_quantize_any(const SrcT* x, uint8_t* xq, float* inv_scale, int64_t R, int64_t K, int64_t ldx, int64_t ldq, hipStream_t s) {
  constexpr int epv = VecTraits<SrcT>::EPV;
  constexpr int very_long_cache = epv == 4 ? 8 : 4;
  const int64_t chunks = (K + epv - 1) / epv;
  auto go = [&](auto kern, int64_t grid, int threads) {
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3((unsigned)threads), 0, s, x, xq, inv_scale, (int)K, (long)ldx, (long)ldq, (long)R);
  };
  const bool long_row = quantize_any_long(R, chunks);
  // Rows of up to 64 chunks: a wave each with as few rounds of loads as they need. (256 lanes with four rounds, most of them idle,
  // lose to the element-by-element kernel there, f32 1985x51 3.1 -> 3.5 us, bf16 1624x106 3.3 -> 5.8; and so do eight rounds a
  // lane, bf16 13772x38 9.5 -> 15.7.) The same for many bf16 rows of up to 128: 2000x700 6.7 us on 256 lanes, 3.8 as waves.
  // Few very short bf16 rows stay with the latter kernel, which rounds a row's values to bf16 one by one on as many lanes
  // (115x20 2.7 us, a wave each 3.15).
  const bool few_short = epv == 8 && ((K <= 256 && R <= 512) || (K <= 64 && R <= 2048));
  const bool wave_each = chunks <= 64 || (epv == 8 && chunks <= 2 * 64 && R > 512);
  if (K < epv || few_short) {
    hipLaunchKernelGGL(quantize_rows_kernel<SrcT>, dim3((unsigned)R), dim3(256), 0, s, x, xq, inv_scale, (int)K, (long)ldx, (long)ldq);
  } else if (wave_each) {
    go(quantize_rows_vec_kernel<SrcT, 16 / epv, 64, kWaveRows, true>, (R + kWaveRows - 1) / kWaveRows, 64 * kWaveRows);
  } else if (chunks <= 8 * 64 && R > 2048) {
    go(quantize_rows_vec_kernel<SrcT, 8, 64, kWaveRows, true>, (R + kWaveRows - 1) / kWaveRows, 64 * kWaveRows);
  } else if (!long_row) {  // (no idle rounds where that is had without more forms than these)
    if (chunks <= 256) go(quantize_rows_vec_kernel<SrcT, 1, 256, 1, true>, R, 256);
    else if (chunks <= 512) go(quantize_rows_vec_kernel<SrcT, 2, 256, 1, true>, R, 256);
    else go(quantize_rows_vec_kernel<SrcT, 4, 256, 1, true>, R, 256);
  } else if (chunks <= 8 * 512) {
    go(quantize_rows_vec_kernel<SrcT, 8, 512, 1, true>, R, 512);
  } else {
    go(quantize_rows_vec_kernel<SrcT, very_long_cache, 1024, 1, true>, R, 1024);
  }
}
}  // namespace

extern "C" {

int mi355x_fp8_rowwise_gemm_noalloc(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                    const void* bias, void* c, int64_t M, int64_t N, int64_t K, int64_t lda,
                                    int64_t ldb, int64_t ldc, int variant, void* stream) {
  const int st = check_shape(M, N, K);
  if (st != MI355X_FP8_OK) return st;
  if (variant < 0 || (variant >> 24) || ((variant >> 8) & 0xff) > kNumTileConfigs)
    return fail(MI355X_FP8_EINVAL, "unknown variant 0x%x", variant);
  // host arithmetic only up to here: an oversized request is turned away before any device call
  const size_t need = mi355x_fp8_rowwise_workspace_bytes(M, N, K, variant);
  // A plan the buffer cannot hold is refused only when the caller named its split factor; left to
  // the library, the call runs the cheapest plan whose partial sums fit the buffer, as the workspace
  // form does with a workspace that is too small.
  if (need > kScratchBytes && ((variant >> 16) & 0xff))
    return fail(MI355X_FP8_ENOTSUP,
                "split-K factor %d on %lldx%lldx%lld needs %zu bytes of scratch, the built-in buffer holds %zu; "
                "call mi355x_fp8_rowwise_gemm with a workspace of that size instead",
                (variant >> 16) & 0xff, (long long)M, (long long)N, (long long)K, need, kScratchBytes);
  void* ws = nullptr;
  if (need) {
    if (const int ss = scratch_of_current_device(&ws)) return ss;
  }
  // Nothing in the buffer has to start at zero: every split stores its whole plane of partial sums
  // before the finalize kernel (stream-ordered behind it) reads any of it.
  // As many bytes as the workspace form would bring, though the buffer holds more: operands that send the call to another family than
  // the shape alone would (misaligned ones, to the generic family, which cuts K into as many parts as it gets planes) have to
  // find the same plan through both entries.
  return mi355x_fp8_rowwise_gemm_ex(a, b, a_scale, b_scale, bias, c, MI355X_FP8_OUT_BF16, M, N, K, lda, ldb, ldc,
                                    ws, need < kScratchBytes ? need : kScratchBytes, variant, stream);
}

int mi355x_fp8_rowwise_grouped_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                    const int32_t* m_sizes, void* c, int64_t G, int64_t M, int64_t N,
                                    int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int tile_config,
                                    void* stream) {
  return mi355x_fp8_rowwise_grouped_gemm_ex(a, b, a_scale, b_scale, m_sizes, c, G, M, N, K, lda, ldb, ldc, tile_config, 0, stream);
}

int mi355x_fp8_rowwise_grouped_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                       const int32_t* m_sizes, void* c, int64_t G, int64_t M, int64_t N,
                                       int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int tile_config,
                                       int clear_rest, void* stream) {
  int st = check_shape(M, N, K);
  if (st == MI355X_FP8_OK) st = check_fast_shape(K);
  if (st != MI355X_FP8_OK) return st;
  if (G < 1 || G > 65536) return fail(MI355X_FP8_EINVAL, "G must be in 1..65536 (got %lld)", (long long)G);
  if (G * N > INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "G*N exceeds 2^31-1");
  if (!a || !b || !a_scale || !b_scale || !m_sizes || !c) return fail(MI355X_FP8_EINVAL, "null operand pointer");
  if (lda < K || ldb < K || ldc < N) return fail(MI355X_FP8_EINVAL, "leading dimension smaller than the row length");
  if (lda % 16 || ldb % 16) return fail(MI355X_FP8_ENOTSUP, "lda and ldb must be multiples of 16");
  if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15))
    return fail(MI355X_FP8_ENOTSUP, "a and b must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(a_scale) & 3) || (reinterpret_cast<uintptr_t>(b_scale) & 3) ||
      (reinterpret_cast<uintptr_t>(c) & 1) || (reinterpret_cast<uintptr_t>(m_sizes) & 3))
    return fail(MI355X_FP8_EINVAL, "misaligned scale, size or output pointer");
  // (a tile's rows are addressed with 32-bit byte offsets that must stay below 2^31)
  if (lda * 256 > (int64_t)INT32_MAX || ldb * 256 > (int64_t)INT32_MAX || ldc * 512 > (int64_t)INT32_MAX)
    return fail(MI355X_FP8_ENOTSUP, "leading dimension too large");
  if (tile_config < -1 || tile_config >= kNumGroupedTileConfigs)
    return fail(MI355X_FP8_EINVAL, "unknown tile configuration %d", tile_config);

  GemmParams p;
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b;
  p.a_scale = a_scale; p.b_scale = b_scale;
  p.bias = nullptr; p.c = (uint16_t*)c;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.tiles_m = p.tiles_n = 0;
  p.splits = 1; p.steps_per_split = k_steps_of(K); p.partial = nullptr;
  p.m_sizes = m_sizes; p.groups = (int)G; p.clear_rest = clear_rest != 0; p.out_f16 = 0;
  p.div_tiles_mul = p.div_tiles_shift = p.div_group_mul = p.div_group_shift = 0; p.stamps = nullptr;
  hipStream_t s = (hipStream_t)stream;
  switch (tile_config < 0 ? grouped_form(G, M, N, K, ldb) : kGroupedTiles) {
    case kGroupedRows16: return launch_grouped_skinny<1, 2, 2, 4>(p, s);
    case kGroupedRows32: return launch_grouped_skinny<2, 2, 2, 8>(p, s);
    case kGroupedRows64: return launch_grouped_skinny<4, 2, 2, 8>(p, s);
    case kGroupedStream128: return launch_grouped_tiles<128, 128, kDefaultDist, true>(p, s);
    case kGroupedStream256: return launch_grouped_tiles<128, 256, kDefaultDist, true>(p, s);
    default: break;
  }
  // Large tiles when an average group fills most of one and there are enough of them for every
  // CU, small tiles otherwise (the group sizes themselves are on the device; M / G is what the
  // host knows). Where 256x256 tiles are too few and 256x128 tiles come to about one round of workgroups,
  // those, on rows long enough for their deeper ring to pay (measured, equal groups: G = 4, M = 1024,
  // N = K = 8192 78.8 -> 60.9 us; G = 2 ... 16, M = 4096, N = 2048, K = 7168 52-65 -> 49-60; at K = 2048
  // they are 1-3 % behind the small tiles).
  if (tile_config < 0) {
    const bool rows_fill = M / G >= 192;
    const int64_t tiles_256 = (M / 256) * (N / 256), tiles_128 = (M / 256) * (N / 128);
    tile_config = rows_fill && tiles_256 >= 192 ? 0 : rows_fill && tiles_128 >= 192 && tiles_128 <= 288 && K >= 4096 ? 2 : 1;
  }
  if (tile_config == 0) return launch_grouped_tiles<256, 256, kDefaultDist, false>(p, s);
  if (tile_config == 2) return launch_grouped_tiles<256, 128, 3, false>(p, s);
  return launch_grouped_tiles<128, 128, kDefaultDist, false>(p, s);
}

int mi355x_fp8_rowwise_grouped_form(int64_t G, int64_t M, int64_t N, int64_t K) {
  int st = check_shape(M, N, K);
  if (st == MI355X_FP8_OK) st = check_fast_shape(K);
  if (st != MI355X_FP8_OK) return st;
  if (G < 1 || G > 65536) return fail(MI355X_FP8_EINVAL, "G must be in 1..65536 (got %lld)", (long long)G);
  return grouped_form(G, M, N, K, K);
}

int mi355x_fp8_rowwise_generic_form(int64_t M, int64_t N, int64_t K, int dwords) {
  const int st = check_shape(M, N, K);
  if (st != MI355X_FP8_OK) return st;
  return generic_streams(M, N, K) ? MI355X_FP8_GENERIC_STREAM : generic_tiles(M, N, K, dwords != 0).tiles + 1;
}

int mi355x_fp8_blockwise_form(int64_t M, int64_t N, int64_t K) {
  int st = check_shape(M, N, K);
  if (st == MI355X_FP8_OK) st = check_fast_shape(K);
  if (st == MI355X_FP8_OK && K > 256 * kStepK)
    st = fail(MI355X_FP8_ENOTSUP, "block-scaled form handles K <= %d (got %lld)", 256 * kStepK, (long long)K);
  return st != MI355X_FP8_OK ? st : block_form(M, N, K, K % kStepK != 0);
}

int mi355x_fp8_blockwise_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale,
                              void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                              int64_t ldc, void* stream) {
  return mi355x_fp8_blockwise_gemm_ws(a, b, a_scale, b_scale, c, M, N, K, lda, ldb, ldc, nullptr, 0, -1, stream);
}

size_t mi355x_fp8_blockwise_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (check_shape(M, N, K) != MI355X_FP8_OK || check_fast_shape(K) != MI355X_FP8_OK || K > 256 * kStepK) return 0;
  const BlockPlan plan = known_block_plan(M, N, K, K, kMaxSplits);
  return plan.splits > 1 ? (size_t)plan.splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

int mi355x_fp8_blockwise_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                 void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                 int64_t ldc, int form, void* stream) {
  // (a form with a factor beside it is the entry's below: here it is none, refused where the others' operands have passed)
  return mi355x_fp8_blockwise_gemm_ws(a, b, a_scale, b_scale, c, M, N, K, lda, ldb, ldc, nullptr, 0, form > 0xff ? 0xff : form, stream);
}

int mi355x_fp8_blockwise_gemm_ws(const void* a, const void* b, const float* a_scale, const float* b_scale,
                                 void* c, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                 int64_t ldc, void* workspace, size_t workspace_bytes, int form, void* stream) {
  int st = check_shape(M, N, K);
  if (st == MI355X_FP8_OK) st = check_fast_shape(K);
  if (st != MI355X_FP8_OK) return st;
  if (K > 256 * kStepK) return fail(MI355X_FP8_ENOTSUP, "block-scaled form handles K <= %d (got %lld)",
                                    256 * kStepK, (long long)K);
  if (!a || !b || !a_scale || !b_scale || !c) return fail(MI355X_FP8_EINVAL, "null operand pointer");
  if (lda < K || ldb < K || ldc < N) return fail(MI355X_FP8_EINVAL, "leading dimension smaller than the row length");
  if (lda % 16 || ldb % 16) return fail(MI355X_FP8_ENOTSUP, "lda and ldb must be multiples of 16");
  if ((reinterpret_cast<uintptr_t>(a) & 15) || (reinterpret_cast<uintptr_t>(b) & 15))
    return fail(MI355X_FP8_ENOTSUP, "a and b must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(a_scale) & 3) || (reinterpret_cast<uintptr_t>(b_scale) & 3) ||
      (reinterpret_cast<uintptr_t>(c) & 1))
    return fail(MI355X_FP8_EINVAL, "misaligned scale or output pointer");
  // (a tile's rows are addressed with 32-bit byte offsets that must stay below 2^31)
  if (lda * 256 > (int64_t)INT32_MAX || ldb * 256 > (int64_t)INT32_MAX || ldc * 512 > (int64_t)INT32_MAX)
    return fail(MI355X_FP8_ENOTSUP, "leading dimension too large");
  GemmParams p;
  p.a = (const uint8_t*)a; p.b = (const uint8_t*)b;
  p.a_scale = a_scale; p.b_scale = b_scale;
  p.bias = nullptr; p.c = (uint16_t*)c;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.tiles_m = p.tiles_n = 0;
  p.splits = 1; p.steps_per_split = k_steps_of(K); p.partial = nullptr;
  p.m_sizes = nullptr; p.groups = 0; p.clear_rest = 0; p.out_f16 = 0;
  p.div_tiles_mul = p.div_tiles_shift = p.div_group_mul = p.div_group_shift = 0; p.stamps = nullptr;
  hipStream_t s = (hipStream_t)stream;
  const bool ktail = K % kStepK;
  // (a split factor pinned to TILES_128)
  const int want_splits = form < 0 ? 0 : form >> 8;
  if (form >= 0) form &= 0xff;
  if (want_splits && form != kBlockSmall) return fail(MI355X_FP8_EINVAL, "only the form of 128x128 tiles is split");
  const size_t plane = (size_t)M * (size_t)N * sizeof(float);
  if (form < 0 || want_splits) {
    // (a workspace that holds fewer planes than the best plan wants takes the best one that it does hold)
    const size_t planes = workspace ? workspace_bytes / plane : 0;
    BlockPlan plan = known_block_plan(M, N, K, ldb, kMaxSplits);
    if (plan.splits > 1 && (size_t)plan.splits > planes) plan = known_block_plan(M, N, K, ldb, planes < 2 ? 1 : (int)planes);
    if (want_splits) {
      plan.form = kBlockSmall;
      normalise_splits(p.steps_per_split, want_splits, plan.splits, plan.steps_per_split);
      if (plan.splits > 1 && ((size_t)plan.splits > planes || N * 512 > (int64_t)INT32_MAX))
        return fail(MI355X_FP8_EINVAL, "split-K factor %d needs %zu bytes of workspace (got %zu)", plan.splits, plan.splits * plane,
                    workspace ? workspace_bytes : (size_t)0);
    }
    if (plan.splits > 1) {
      if (reinterpret_cast<uintptr_t>(workspace) & 15) return fail(MI355X_FP8_EINVAL, "workspace must be 16-byte aligned");
      p.splits = plan.splits;
      p.steps_per_split = plan.steps_per_split;
      p.partial = (float*)workspace;
    }
    form = plan.form;
  } else if ((form == kBlockOneTile && M > kSkinnyMaxM) || (form == kBlockNarrow && !narrow_fits(M, N, K)) ||
             (form == kBlockResident && !pair_skinny_fits(M, N, K)))
    return fail(MI355X_FP8_ENOTSUP, "block-scaled form %d does not take %lldx%lld", form, (long long)M, (long long)N);
  switch (form) {
    case kBlockNarrow: return launch_narrow_for<true>(p, s);
    case kBlockResident: return launch_skinny_pair_block(p, s);
    case kBlockOneTile:
      if (M <= 16) return launch_skinny<1, 1, 4, 8, false, true>(p, s);
      if (M <= 32) return launch_skinny<2, 1, 2, 8, false, true>(p, s);
      if (M <= 48) return launch_skinny<3, 1, 2, 8, false, true>(p, s);
      return launch_skinny<4, 2, 2, 8, false, true>(p, s);
    case kBlockLarge: return launch_block(p, s);
    case kBlockSmallStream:
      return ktail ? launch_tiled<128, 128, 2, 2, true, kEpiPlain, false, true, kDefaultDist, true>(p, s)
                   : launch_tiled<128, 128, 2, 2, false, kEpiPlain, false, true, kDefaultDist, true>(p, s);
    case kBlockSmall: {
      // Loads three steps ahead where a CU has one work item and long rows of it, against two: 1047x1566x12800 in two 49.5 -> 42.7 us,
      // 1000x1000x28672 in four 54.5 -> 48.9, 64x4096x8192 in four 18.4 -> 17.4, level with fewer steps (unsplit,
      // 130x16384x16384 95 -> 82, 100x20000x8192 51.5 -> 48.3; 1500x2560x7168 34.6 -> 35.0, 1024^3 9.0 -> 9.2).
      const bool deep = ((M + 127) / 128) * ((N + 127) / 128) * p.splits <= kNumCu && p.steps_per_split >= (p.splits > 1 ? 16 : 64);
      if (p.splits > 1 && deep)
        return ktail ? launch_tiled<128, 128, 2, 2, true, kEpiPartial, false, true, 3>(p, s)
                     : launch_tiled<128, 128, 2, 2, false, kEpiPartial, false, true, 3>(p, s);
      if (p.splits > 1)
        return ktail ? launch_tiled<128, 128, 2, 2, true, kEpiPartial, false, true>(p, s)
                     : launch_tiled<128, 128, 2, 2, false, kEpiPartial, false, true>(p, s);
      if (deep)
        return ktail ? launch_tiled<128, 128, 2, 2, true, kEpiPlain, false, true, 3>(p, s)
                     : launch_tiled<128, 128, 2, 2, false, kEpiPlain, false, true, 3>(p, s);
      return ktail ? launch_tiled<128, 128, 2, 2, true, kEpiPlain, false, true>(p, s)
                   : launch_tiled<128, 128, 2, 2, false, kEpiPlain, false, true>(p, s);
    }
    default: return fail(MI355X_FP8_EINVAL, "unknown block-scaled form %d", form);
  }
}

int mi355x_fp8_rowwise_quantize(const void* x, int src_type, void* xq, float* inv_scale, int64_t R,
                                int64_t K, int64_t ldx, int64_t ldq, void* stream) {
  if (!x || !xq || !inv_scale) return fail(MI355X_FP8_EINVAL, "null pointer");
  if (R < 1 || K < 1 || ldx < K || ldq < K) return fail(MI355X_FP8_EINVAL, "bad shape or leading dimension");
  if (R > INT32_MAX || K > INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "dimension exceeds 2^31-1");
  hipStream_t s = (hipStream_t)stream;
  // source and destination rows that start 16-byte aligned and hold whole 16-byte source
  // chunks take the vector kernel
  const int esz = src_type == MI355X_FP8_SRC_BF16 ? 2 : 4;
  const int epv = 16 / esz;
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (ldx * esz) % 16 == 0 && K % epv == 0 &&
                   (reinterpret_cast<uintptr_t>(xq) & 15) == 0 && ldq % 16 == 0;
  if (vec && src_type == MI355X_FP8_SRC_F32) {
    launch_quantize_rows<kRowF32>((const float*)x, (uint8_t*)xq, inv_scale, R, K, ldx, ldq, s);
  } else if (vec && src_type == MI355X_FP8_SRC_BF16) {
    launch_quantize_rows<kRowBf16>((const uint16_t*)x, (uint8_t*)xq, inv_scale, R, K, ldx, ldq, s);
  } else if (src_type == MI355X_FP8_SRC_F32) {
    launch_quantize_any<float>((const float*)x, (uint8_t*)xq, inv_scale, R, K, ldx, ldq, s);
  } else if (src_type == MI355X_FP8_SRC_BF16) {
    launch_quantize_any<uint16_t>((const uint16_t*)x, (uint8_t*)xq, inv_scale, R, K, ldx, ldq, s);
  } else {
    return fail(MI355X_FP8_EINVAL, "unknown src_type %d", src_type);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "quantize kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

int mi355x_fp8_blockwise_quantize(const void* x, int src_type, void* xq, float* inv_scale, int64_t M, int64_t K,
                                  int64_t ldx, int64_t ldq, void* stream) {
  if (!x || !xq || !inv_scale) return fail(MI355X_FP8_EINVAL, "null pointer");
  if (M < 1 || K < 1 || ldx < K || ldq < K) return fail(MI355X_FP8_EINVAL, "bad shape or leading dimension");
  if (M > INT32_MAX || K > INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "dimension exceeds 2^31-1");
  if (src_type != MI355X_FP8_SRC_F32 && src_type != MI355X_FP8_SRC_BF16)
    return fail(MI355X_FP8_EINVAL, "unknown src_type %d", src_type);
  const int64_t grid_m = (M + kQuantBlock - 1) / kQuantBlock, grid_k = (K + kQuantBlock - 1) / kQuantBlock;
  if (grid_m > 65535) return fail(MI355X_FP8_ENOTSUP, "more than 65535 block rows");
  hipStream_t s = (hipStream_t)stream;
  const int esz = src_type == MI355X_FP8_SRC_BF16 ? 2 : 4;
  const int epv = 16 / esz;
  // whole 16-byte source chunks from 16-byte aligned rows, and stores of a chunk's codes (4 or 8 bytes) aligned
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (ldx * esz) % 16 == 0 && K % epv == 0 &&
                   (reinterpret_cast<uintptr_t>(xq) & (epv - 1)) == 0 && ldq % epv == 0;
  const dim3 grid((unsigned)grid_k, (unsigned)grid_m);
  if (src_type == MI355X_FP8_SRC_F32) {
    auto kern = vec ? quantize_blocks_kernel<float, true> : quantize_blocks_kernel<float, false>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, (const float*)x, (uint8_t*)xq, inv_scale, (int)M, (int)K, (long)ldx,
                       (long)ldq, (int)grid_k);
  } else {
    auto kern = vec ? quantize_blocks_kernel<uint16_t, true> : quantize_blocks_kernel<uint16_t, false>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, (const uint16_t*)x, (uint8_t*)xq, inv_scale, (int)M, (int)K,
                       (long)ldx, (long)ldq, (int)grid_k);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "block quantize kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}

namespace {
int launch_fused_quant(int op, const void* x1, const void* x2, float eps, void* xq, float* inv_scale, int64_t R,
                       int64_t K, int64_t ld1, int64_t ld2, int64_t ldq, void* stream) {
  if (!x1 || !x2 || !xq || !inv_scale) return fail(MI355X_FP8_EINVAL, "null pointer");
  if (R < 1 || K < 1 || ld1 < K || ldq < K || (op == kFusedSiluMul && ld2 < K))
    return fail(MI355X_FP8_EINVAL, "bad shape or leading dimension");
  if (R > INT32_MAX || K > INT32_MAX) return fail(MI355X_FP8_ENOTSUP, "dimension exceeds 2^31-1");
  // whole 16-byte chunks of bf16, rows that start 16-byte aligned (the GEMM that follows wants K a
  // multiple of 16 and 16-byte aligned rows of codes anyway)
  if (K % 8 || ld1 % 8 || (op == kFusedSiluMul && ld2 % 8) || ldq % 16 || (reinterpret_cast<uintptr_t>(x1) & 15) ||
      (reinterpret_cast<uintptr_t>(x2) & 15) || (reinterpret_cast<uintptr_t>(xq) & 15))
    return fail(MI355X_FP8_ENOTSUP, "rows must hold whole 16-byte chunks and start 16-byte aligned");
  if (!(eps >= 0.0f)) return fail(MI355X_FP8_EINVAL, "eps must be >= 0");
  hipStream_t s = (hipStream_t)stream;
  auto launch = [&](auto op_tag, RowForm form) {
    constexpr int OP = decltype(op_tag)::value;
    with_row_form<OP == kFusedRmsNorm ? kRowRmsNorm : kRowSiluMul>(form, [&](auto lanes, auto chunks) {
      constexpr int LANES = decltype(lanes)::value, ROWS = LANES == 64 ? kWaveRows : 1;
      launch_by_rows(R, LANES, [&](int64_t row, int64_t rows) {
        const uint16_t* second = (const uint16_t*)x2 + (OP == kFusedRmsNorm ? 0 : row * ld2);  // (RMSNorm: the weights of every row)
        hipLaunchKernelGGL((fused_rowwise_quant_kernel<OP, decltype(chunks)::value, LANES, ROWS>), dim3((unsigned)((rows + ROWS - 1) / ROWS)),
                           dim3(LANES * ROWS), 0, s, (const uint16_t*)x1 + row * ld1, second, eps, (uint8_t*)xq + row * ldq, inv_scale + row,
                           (int)K, (long)ld1, (long)ld2, (long)ldq, (long)rows);
      });
    });
  };
  if (op == kFusedRmsNorm) launch(std::integral_constant<int, kFusedRmsNorm>{}, row_form(kRowRmsNorm, R, K / 8));
  else launch(std::integral_constant<int, kFusedSiluMul>{}, row_form(kRowSiluMul, R, K / 8));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MI355X_FP8_ELAUNCH, "fused quantise kernel launch: %s", hipGetErrorString(e));
  return MI355X_FP8_OK;
}
}  // namespace

int mi355x_fp8_rmsnorm_rowwise_quantize(const void* x, const void* weight, float eps, void* xq, float* inv_scale,
                                        int64_t R, int64_t K, int64_t ldx, int64_t ldq, void* stream) {
  return launch_fused_quant(kFusedRmsNorm, x, weight, eps, xq, inv_scale, R, K, ldx, K, ldq, stream);
}

int mi355x_fp8_silu_mul_rowwise_quantize(const void* x1, const void* x2, void* xq, float* inv_scale, int64_t R,
                                         int64_t K, int64_t ldx1, int64_t ldx2, int64_t ldq, void* stream) {
  return launch_fused_quant(kFusedSiluMul, x1, x2, 0.0f, xq, inv_scale, R, K, ldx1, ldx2, ldq, stream);
}

}  // extern "C"
#endif  // !MI355X_TILED_PART
