// Backprojection of 16-bit slabs on the matrix cores of gfx950.
//
// For one tilt, the 16 voxels of a 4 x 4 (x, z) block read their two taps
// from at most seven consecutive detector positions: p = x c - z s + offset
// spans at most 3 |c| + 3 |s| <= 4.25 over the block. Interpolation of the
// block is therefore a product of a 16 x 8 matrix of weights (two non-zeros
// per voxel) with 8 positions x rows of the slab, and four tilts make the
// K = 32 of one v_mfma_f32_16x16x32_f16: 16 voxels x 16 detector rows x 4
// tilts per instruction, accumulated in FP32 over the tilts.
//
// Precision. The taps are the FP16 values of the slab (BF16 slabs are
// rounded to FP16 in LDS, as the direct kernel rounds them per tap). The
// weights stay FP32 quantities: each is split into an FP16 high part and the
// FP16 remainder of the exact product (not of its FP32 rounding), and both are
// multiplied, two matrix instructions per product. An instruction adds its
// four tilts to the accumulator one after another, each rounded to nearest
// even, so the small remainders go first. The error against FP64 sums is then
// no larger than that of FP32 weights and one FP32 fused multiply-add per tap
// (rel-L2 on the plan's own FP16 slabs, here / there: 6 tilts 7.1e-8 / 7.6e-8,
// 41 tilts 1.66e-7 / 1.69e-7, 121 tilts 2.81e-7 / 2.81e-7; BF16 1 to 15 %
// below). The weights of all tilts are scaled by one power
// of two that puts the largest in [2^13, 2^14), and the sum is scaled back at
// the end. The pairs end at 2^-24: where a tilt's weight lies more than
// 8192-fold below the largest, the series is computed tap by tap with FP32
// weights instead (k_bp_coefficients decides; with one scale for every series
// a 2^-40-fold weight was off by 8e-5 of its voxels). Detector position, tap
// and slab choice are the FP32 arithmetic of the direct kernel.
//
// Work split. A workgroup is a 16 x 16 (x, z) tile by RB row blocks of 32
// rows; each of its 8 waves holds two 4 x 4 blocks by all rows (64
// accumulator registers with RB = 4; four waves per SIMD). The weights of a
// block are built once (about 40 VALU instructions per 4 tilts) and used for
// all 32 RB rows, and the two 16-bit matrix instructions replace 2 FMAs per
// (voxel, row, tilt) on the vector units, which bound the former kernel at
// 0.96 of their issue rate.
//
// Measured (one launch, start to end): 121 tilts, 1024 x 256 x 1024 voxels,
// one slab, FP16: 2.10 ms with the staged kernel on the vector units, 1.05 ms
// here (3.1e13 updates/s); 61 tilts, 2048 x 512 x 2048, 16 slabs: 9.7 -> 6.9
// ms; 41 tilts, 1024 x 256 x 512, 4 slabs, BF16: 0.50 -> 0.36 ms. What binds
// now is instruction issue: the 16 matrix instructions of a block and four
// tilts take 16 cycles each, its other 57 vector instructions about 3, and
// on gfx950 the two hardly overlap (a probe: one 16x16x32 matrix instruction
// with 3 or 6 vector instructions takes 24 or 33 cycles, alone 19).
//
// LDS. Per (tilt, slab) a run of kPos = 24 positions of the tile's rows is
// loaded straight into LDS (the tile's taps span 15 |c| + 15 |s| <= 21.22
// positions), four tilts to a batch, two buffers: the loads of a batch are
// issued before the one before it is multiplied. A tile that spans two slabs
// at a tilt (two at most: they are 64 pixels or wider) takes a second run; a
// batch holds two of these and closes early for a third. The matrix operand
// needs 8 positions of one row in each lane, while a slab holds the rows of a
// position contiguously: the transposing LDS read (ds_read_b64_tr_b16) does
// that. Runs are laid out [32-row block][4 positions][16-row half][position]
// [16 rows], so that one read of 16 lanes is 4 consecutive positions x 32
// bytes in distinct banks and one 1 KiB load covers whole 64-byte pieces of
// the slab.
//
// Exceptional values. A zero weight times a NaN or an infinity would reach
// voxels that do not read it. The rows of a tile that end with a value that is
// not finite are therefore computed again tap by tap, so that such values
// reach exactly the voxels that read them; other rows keep their values.
#include <type_traits>

#include "gx_bp_geometry.hpp"
#include "gx_common.hpp"
#include "gx_kernels.hpp"

namespace gx {

namespace {

constexpr int kTile = 16;    // voxels of a tile in x and in z
constexpr int kPos = 24;     // staged positions
constexpr int kMaxBase = kPos - 8;
constexpr int kExtra = 2;    // runs of second slabs per batch
constexpr int kWaves = 8;
// order of the tiles (tile_of)
constexpr unsigned kStrip = 8;
constexpr unsigned kDeep = 32, kWide = 96;
constexpr size_t kFill = 256;
// window table: .y = first slab | (1 where there are two) << kSpanShift
constexpr int kSpanShift = 28;
constexpr int kSlabMask = (1 << kSpanShift) - 1;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4v mfma16(half8 a, half8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Eight positions of one row per lane, for the two 16-row tiles of a 32-row
// block at LDS address a + OFF: four transposing reads, in each of which 16
// lanes read 4 16-bit values and lane i receives value i % 4 of lanes i / 4,
// i / 4 + 4, ... of its group of 16. Written out, and waited for here,
// because the compiler makes an LDS read of a buffer wait for the direct
// loads into the other one that are still under way.
template <int OFF>
__device__ __forceinline__ void read_tr8x2(uint32_t a, half8 &h0, half8 &h1) {
  short4v v0, v1, v2, v3;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4 offset:%5\n\t"
      "ds_read_b64_tr_b16 %1, %4 offset:%6\n\t"
      "ds_read_b64_tr_b16 %2, %4 offset:%7\n\t"
      "ds_read_b64_tr_b16 %3, %4 offset:%8\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v0), "=&v"(v1), "=&v"(v2), "=&v"(v3)
      : "v"(a), "n"(OFF), "n"(OFF + 256), "n"(OFF + 128), "n"(OFF + 384)
      : "memory");
  typedef short short8v __attribute__((ext_vector_type(8)));
  h0 = __builtin_bit_cast(half8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
  h1 = __builtin_bit_cast(half8, __builtin_shufflevector(v2, v3, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Tile of block lb, and its row group (returned). The 64 tiles an XCD runs at
// a time share its L2: in a deep, wide volume they are 8 x 8 (strips of 8
// tiles in z, along x), whose taps of a tilt span 128 (|c| + |s|) positions at
// most, not one column of tiles through the depth, 16 |c| + Z |s|: 121 tilts,
// 4096 x 1024 x 4096 voxels, 32 slabs, 205 -> 140 GB fetched. Elsewhere a
// column's slab rows stay in the caches anyway, and walking x once beats
// reading them again for every strip. The time of strips over that of
// columns, 61 tilts: 512 wide 0.96 to 1.02 (192 to 512 deep); 1024 wide, one
// slab, 1.04 to 1.14 (272 to 1024 deep), 16 slabs 1.04 (272) to 0.97 (512);
// 1536 wide, 4 slabs, 1.05 (272), 0.99 (512), 0.96 (1536); 2048 wide 1.02 to
// 1.11 (272), 0.97 to 0.99 (512), 0.93 to 1.03 (1536 and 2048); 3072 wide
// 1.06 to 1.14 (272), 0.91 to 0.98 (2048 and 3072).
__device__ __forceinline__ int tile_of(unsigned lb, int nbx, int nbz, int &bx,
                                       int &bz) {
  const unsigned nz = (unsigned)nbz;
  const unsigned strip =
      nz >= kDeep && (unsigned)nbx >= kWide ? kStrip : nz;
  const unsigned nt = (unsigned)nbx * nz;
  const unsigned grp = lb / nt, r = lb - grp * nt;
  const unsigned s = r / (strip * (unsigned)nbx);
  const unsigned q = r - s * (strip * (unsigned)nbx);
  const unsigned h = min(strip, nz - s * strip);
  bx = (int)(q / h);
  bz = (int)(s * strip + q % h);
  return (int)grp;
}

// read_tr8x2 for two 32-row blocks.
template <int OFF, int STEP>
__device__ __forceinline__ void read_tr8x4(uint32_t a, half8 &h0, half8 &h1,
                                           half8 &h2, half8 &h3) {
  short4v v[8];
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%9\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%10\n\t"
      "ds_read_b64_tr_b16 %2, %8 offset:%11\n\t"
      "ds_read_b64_tr_b16 %3, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%13\n\t"
      "ds_read_b64_tr_b16 %5, %8 offset:%14\n\t"
      "ds_read_b64_tr_b16 %6, %8 offset:%15\n\t"
      "ds_read_b64_tr_b16 %7, %8 offset:%16\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]),
        "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(a), "n"(OFF), "n"(OFF + 256), "n"(OFF + 128), "n"(OFF + 384),
        "n"(OFF + STEP), "n"(OFF + STEP + 256), "n"(OFF + STEP + 128),
        "n"(OFF + STEP + 384)
      : "memory");
  half8 *out[4] = {&h0, &h1, &h2, &h3};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *out[i] = __builtin_bit_cast(
        half8, __builtin_shufflevector(v[2 * i], v[2 * i + 1], 0, 1, 2, 3, 4,
                                       5, 6, 7));
}

// Eight rows of two positions, at LDS addresses a0 and a1, in each of N
// 32-row blocks from OFF on, STEP bytes apart.
template <int OFF, int STEP, int N>
__device__ __forceinline__ void read_rows(uint32_t a0, uint32_t a1,
                                          half8 (&v0)[N], half8 (&v1)[N]) {
  if constexpr (N == 1)
    asm volatile(
        "ds_read_b128 %0, %2 offset:%4\n\t"
        "ds_read_b128 %1, %3 offset:%4\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v0[0]), "=&v"(v1[0])
        : "v"(a0), "v"(a1), "n"(OFF)
        : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %4 offset:%6\n\t"
        "ds_read_b128 %1, %5 offset:%6\n\t"
        "ds_read_b128 %2, %4 offset:%7\n\t"
        "ds_read_b128 %3, %5 offset:%7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(v0[0]), "=&v"(v1[0]), "=&v"(v0[1]), "=&v"(v1[1])
        : "v"(a0), "v"(a1), "n"(OFF), "n"(OFF + STEP)
        : "memory");
}

__device__ __forceinline__ uint32_t lds_address(const void *p) {
  typedef const __attribute__((address_space(3))) char *lp;
  return (uint32_t)(uintptr_t)(lp)(const char *)p;
}

// A lane's coefficients and window entry from a batch's tables in LDS
// (the entries 256 bytes after the coefficients); written out as read_tr8x2
// is.
__device__ __forceinline__ void read_tables(const uint4 *tables, int g,
                                            float4 &cf, int2 &w) {
  const uint32_t a = lds_address(tables);
  float4v c;
  typedef int int2v __attribute__((ext_vector_type(2)));
  int2v i;
  asm volatile(
      "ds_read_b128 %0, %2\n\t"
      "ds_read_b64 %1, %3 offset:256\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(c), "=&v"(i)
      : "v"(a + 16 * g), "v"(a + 8 * g)
      : "memory");
  cf = make_float4(c[0], c[1], c[2], c[3]);
  w = make_int2(i[0], i[1]);
}

// Smallest value over each group of 16 lanes, in all of them (four v_min with
// a rotation within the group as their DPP operand).
template <int CTRL>
__device__ __forceinline__ int min_rotated(int v) {
  return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, 0xf, 0xf,
                                            false));
}
__device__ __forceinline__ int min16(int v) {
  return min_rotated<0x121>(
      min_rotated<0x122>(min_rotated<0x124>(min_rotated<0x128>(v))));
}

template <int N>
using Int = std::integral_constant<int, N>;

typedef float float2v __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ half2v to_half2(float a, float b) {
  return __builtin_convertvector((float2v){a, b}, half2v);
}

__device__ __forceinline__ uint32_t bf16_pair_to_f16(uint32_t w) {
  return __builtin_bit_cast(
      uint32_t, to_half2(__uint_as_float(w << 16),
                         __uint_as_float(w & 0xffff0000u)));
}

// The 16 x 8 weights of one lane's voxel and tilt: w0 at position r, w1 at
// r + 1, zeros elsewhere. sel[r] holds, for each 32-bit word of the eight
// halves, the byte selector that places the pair (w0, w1).
__device__ __forceinline__ half8 place(uint4 sel, half2v w) {
  const uint32_t u = __builtin_bit_cast(uint32_t, w);
  const uint4 r = make_uint4(__builtin_amdgcn_perm(0u, u, sel.x),
                             __builtin_amdgcn_perm(0u, u, sel.y),
                             __builtin_amdgcn_perm(0u, u, sel.z),
                             __builtin_amdgcn_perm(0u, u, sel.w));
  return __builtin_bit_cast(half8, r);
}

}  // namespace

// ----------------------------------------------------------- window table --

// win[tile * Tpad + t], tile = bx * nbz + bz: over the tile's voxels, the
// smallest tap position, the first slab and how many slabs follow it. Both
// are monotone in x and in z, so the four corners decide.
template <bool MULTI>
__global__ void k_bp_mm_windows(const float4 *__restrict__ coef, int T,
                                int Tpad, int W, int Z, int nbx, int nbz,
                                float dscale, float doffset, int ndf,
                                int2 *__restrict__ win) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)nbx * nbz * Tpad) return;
  const int t = (int)(i % Tpad);
  const int tile = (int)(i / Tpad);
  const int bz = tile % nbz, bx = tile / nbz;
  int2 r = make_int2(0, 0);
  if (t < T) {
    const float4 cf = coef[t];
    int w = 0x7fffffff, k0 = 0x7fffffff, k1 = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float x = voxel_coord(
          (c & 1) ? min(bx * kTile + kTile, W) - 1 : bx * kTile, W);
      const float z = voxel_coord(
          (c & 2) ? min(bz * kTile + kTile, Z) - 1 : bz * kTile, Z);
      float tt;
      w = min(w, tap_index<false>(x, z, cf, tt));
      if constexpr (MULTI) {
        const int k = slab_of(x, z, cf, dscale, doffset, ndf);
        k0 = min(k0, k);
        k1 = max(k1, k);
      }
    }
    r = make_int2(w, MULTI ? k0 | (min(k1 - k0, 1) << kSpanShift) : 0);
  }
  win[i] = r;
}

size_t bp_mm_window_entries(int W, int Z, int T) {
  const size_t nbx = (W + kTile - 1) / kTile, nbz = (Z + kTile - 1) / kTile;
  return nbx * nbz * (size_t)bp_tilt_pad(T);
}

hipError_t launch_bp_mm_windows(const float4 *coef, int T, int W, int Z,
                                float dscale, float doffset, int ndf,
                                int2 *win, hipStream_t s) {
  const int nbx = (W + kTile - 1) / kTile, nbz = (Z + kTile - 1) / kTile;
  const size_t n = bp_mm_window_entries(W, Z, T);
  const dim3 g((unsigned)((n + 255) / 256)), b(256);
  if (ndf > 1)
    hipLaunchKernelGGL(k_bp_mm_windows<true>, g, b, 0, s, coef, T,
                       bp_tilt_pad(T), W, Z, nbx, nbz, dscale, doffset, ndf,
                       win);
  else
    hipLaunchKernelGGL(k_bp_mm_windows<false>, g, b, 0, s, coef, T,
                       bp_tilt_pad(T), W, Z, nbx, nbz, dscale, doffset, ndf,
                       win);
  return hipGetLastError();
}

// ----------------------------------------------------------------- kernel --

template <int RB, bool MULTI>
struct MmShape {
  static constexpr int kRun = kPos * 64 * RB;             // bytes of a run
  static constexpr int kLoads = (kRun + 1023) / 1024;     // 1 KiB loads
  // 128 bytes past whole 256: the runs of tilts g and g + 1, which one LDS
  // read takes together, then use the two halves of the 64 banks
  static constexpr int kRunStride = kLoads * 1024 + 128;
  static constexpr int kSlots = 4 + (MULTI ? kExtra : 0);
  static constexpr int kRT = 2 * RB;                      // 16-row tiles
  // the output staging of 16 rows: 16 x 16 voxels, rows padded by 16 bytes
  static constexpr int kOutRow = kTile * kTile + 4;       // floats
  static constexpr int kOut = 16 * kOutRow * 4;
  // after the runs: the batch's four coefficients and window entries
  static constexpr int kTables = (kSlots * kRunStride + 255) / 256 * 256;
  static constexpr int kStage = kTables + 512;
  static constexpr int kBuf = kStage > kOut ? kStage : kOut;
  // waves that share the loads of one run
  static constexpr int kSplit = kLoads % 2 == 0 && RB % 2 == 0 ? 2 : 1;
  static constexpr int kPer = kLoads / kSplit;            // loads per wave
};

template <int YB, int STORE, bool MULTI, int RB>
__global__ __launch_bounds__(kWaves * 64)
__attribute__((amdgpu_waves_per_eu(4, 4))) void k_bp_mm(
    const uint16_t *__restrict__ slab, const float4 *__restrict__ coef,
    const int2 *__restrict__ win, float dscale, float doffset, int ndf, int N,
    int T, int NYB, int W, int Z, int Y, int yb0, int yb1, int y_base,
    int slab_yb0, float *__restrict__ vol, int nbx, int nbz,
    unsigned nblocks) {
  using S = MmShape<RB, MULTI>;
  constexpr int kRT = S::kRT;
  constexpr int kYG = 32 * RB / YB;  // slab row blocks of a workgroup
  constexpr int kBufWords = S::kBuf / 16;
  __shared__ uint4 lds[2 * kBufWords];
  __shared__ uint4 sel[8];

  const unsigned lb = xcd_remap(blockIdx.x, nblocks);
  int bx, bz;
  const int byb = yb0 + kYG * tile_of(lb, nbx, nbz, bx, bz);
  const int lane = (int)(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int g = lane >> 4, m = lane & 15;  // tilt of the batch, voxel or row

  if (threadIdx.x < 32) {
    const int r = (int)threadIdx.x >> 2, j = (int)threadIdx.x & 3;
    uint32_t v = 0;
    for (int h = 0; h < 2; ++h) {
      const int d = 2 * j + h - r;
      v |= (d == 0 ? 0x0100u : d == 1 ? 0x0302u : 0x0c0cu) << (16 * h);
    }
    reinterpret_cast<uint32_t *>(sel)[threadIdx.x] = v;
  }

  // The wave's two blocks: 4 voxels in x at 4 (wave % 4), 8 in z at
  // 8 (wave / 4). Voxels past the volume repeat its last ones.
  const int ix = bx * kTile + 4 * (wave & 3) + (m & 3);
  const int iz = bz * kTile + 8 * (wave >> 2) + (m >> 2);
  const float x = voxel_coord(min(ix, W - 1), W);
  const float zb[2] = {voxel_coord(min(iz, Z - 1), Z),
                       voxel_coord(min(iz + 4, Z - 1), Z)};
  const int Tpad = bp_tilt_pad(T);
  const int2 *tw = win + (size_t)(bx * nbz + bz) * Tpad;
  const float up = kload(reinterpret_cast<const float *>(coef + Tpad), 0);
  const float down = kload(reinterpret_cast<const float *>(coef + Tpad), 1);
  // weights too far apart for FP16 pairs (k_bp_coefficients): all tap by tap
  const bool taps =
      kload(reinterpret_cast<const float *>(coef + Tpad), 2) != 0.0f;

  // Staging: a lane's position and byte offset in a run, for the loads of
  // its wave (16-byte chunk c of the layout above).
  const size_t row_len = (size_t)N * YB;
  const size_t tstride = (size_t)NYB * row_len;
  const uint16_t *rows = slab + (size_t)(byb - slab_yb0) * row_len;
  const int nyb = min(kYG, yb1 - byb);
  const bool many = nyb * YB > 64;
  const int records = nyb * (int)row_len * 2;
  const int part = S::kSplit == 2 ? wave & 1 : 0;
  const int slot_w = wave / S::kSplit;  // the slot this wave loads
  int cpos[S::kPer], coff[S::kPer];
#pragma unroll
  for (int i = 0; i < S::kPer; ++i) {
    const int c = 64 * (part * S::kPer + i) + lane;
    const int rb = c / (4 * kPos), q = c % (4 * kPos);
    const int p = (q >> 4) * 4 + ((q & 7) >> 1), half = (q >> 3) & 1;
    // slab row block (of the group) and 16-byte word within a position
    const int yb = YB == 32 ? rb : 2 * rb + half;
    const int word = (YB == 32 ? 2 * half : 0) + (q & 1);
    const bool ok = c < S::kRun / 16 && yb < nyb;
    cpos[i] = ok ? p : 0x40000000;
    coff[i] = ok ? (int)(yb * row_len * 2) + p * YB * 2 + word * 16 : 0;
  }
  const auto rs_coef = __builtin_amdgcn_make_buffer_rsrc(
      (void *)coef, (short)0, Tpad * 16, 0x00020000);
  const auto rs_win = __builtin_amdgcn_make_buffer_rsrc(
      (void *)tw, (short)0, Tpad * 8, 0x00020000);
  auto load_run = [&](int t, int k, int w0, bool ok, uint4 *dst) {
    const uint16_t *src =
        ok ? rows + ((size_t)k * T + t) * tstride : rows;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)src, (short)0, ok ? records : 0, 0x00020000);
    // positions outside [0, N) and rows past the group read as zeros
#pragma unroll
    for (int i = 0; i < S::kPer; ++i) {
      const bool in = (unsigned)(w0 + cpos[i]) < (unsigned)N;
      load_to_lds16(rs, dst + 64 * (part * S::kPer + i),
                    in ? coff[i] + w0 * (YB * 2) : -1);
    }
  };

  // A batch: tilts t0 .. t0 + nt - 1 and, per tilt j, the extra runs before
  // its own (4 bits each in ex).
  struct Batch {
    int t0, nt, ex;
  };
  auto next_batch = [&](int t0) {
    Batch b{t0, min(4, T - t0), 0};
    if constexpr (MULTI) {
      int n = 0, cum = 0, ex = 0;
      bool open = true;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int span = kload(tw, min(t0 + j, T - 1)).y >> kSpanShift;
        open = open && t0 + j < T && cum + span <= kExtra;
        ex |= cum << (4 * j);
        if (open) {
          ++n;
          cum += span;
        }
      }
      b.nt = n;  // at least one: a span is at most kExtra
      b.ex = ex | (cum << 16);
    }
    return b;
  };
  auto stage = [&](const Batch &b, uint4 *dst) {
    if (wave == kWaves - 1) {
      // 16 floats of coefficients and 8 words of windows, 4 bytes a lane;
      // entries past the tables read as zeros
      load_to_lds4(rs_coef, dst + S::kTables / 16,
                   lane < 16 ? b.t0 * 16 + lane * 4 : -1);
      load_to_lds4(rs_win, dst + S::kTables / 16 + 16,
                   lane < 8 ? b.t0 * 8 + lane * 4 : -1);
    }
    if (slot_w < 4) {
      const int2 w = kload(tw, min(b.t0 + slot_w, T - 1));
      load_run(b.t0 + slot_w, MULTI ? w.y & kSlabMask : 0, w.x,
               slot_w < b.nt, dst + slot_w * (S::kRunStride / 16));
    }
    if constexpr (MULTI) {
      // the extra runs, on the waves without a run of their own (or the
      // first ones)
      constexpr int kFirst = S::kSplit == 2 ? 0 : 4;
      const int e = slot_w - kFirst;
      if (e >= 0 && e < (b.ex >> 16)) {
        int j = 0;
#pragma unroll
        for (int i = 1; i < 4; ++i)
          if (i < b.nt && ((b.ex >> (4 * i)) & 15) <= e) j = i;
        const int2 w = kload(tw, b.t0 + j);
        load_run(b.t0 + j,
                 (w.y & kSlabMask) + 1 + e - ((b.ex >> (4 * j)) & 15), w.x,
                 true, dst + (4 + e) * (S::kRunStride / 16));
      }
    }
  };
  // BF16 runs to FP16, each chunk by the lane that loaded it.
  auto convert = [&](const Batch &b, uint4 *dst) {
    if constexpr (STORE == kBF16) {
      auto run = [&](uint4 *d) {
#pragma unroll
        for (int i = 0; i < S::kPer; ++i) {
          uint4 *q = d + 64 * (part * S::kPer + i) + lane;
          const uint4 v = *q;
          *q = make_uint4(bf16_pair_to_f16(v.x), bf16_pair_to_f16(v.y),
                          bf16_pair_to_f16(v.z), bf16_pair_to_f16(v.w));
        }
      };
      if (slot_w < 4) run(dst + slot_w * (S::kRunStride / 16));
      if constexpr (MULTI) {
        const int e = slot_w - (S::kSplit == 2 ? 0 : 4);
        if (e >= 0 && e < (b.ex >> 16))
          run(dst + (4 + e) * (S::kRunStride / 16));
      }
    }
  };

  // The lane's tilt of a batch staged at buf: its coefficients and window
  // entry (no weight and no extra runs past the batch).
  auto lane_tables = [&](const Batch &b, const uint4 *buf, float4 &cf,
                         int2 &w) {
    read_tables(buf + S::kTables / 16, g, cf, w);
    cf.w = g < b.nt ? cf.w * up : 0.0f;
    if (g >= b.nt) w.y = 0;
  };

  float4v acc[2][kRT];

  // One batch from `cur`.
  auto multiply = [&](const Batch &b, const uint4 *cur) {
    float4 cf;
    int2 w;
    lane_tables(b, cur, cf, w);
    const uint32_t run0 = lds_address(cur);
    const int lo_addr = (m & 3) * 8;
    const int e = m >> 2;
    const int exg = MULTI ? (b.ex >> (4 * g)) & 15 : 0;
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      float tt;
      const int i0 = tap_index<false>(x, zb[blk], cf, tt);
      const bool ok = (unsigned)i0 < (unsigned)(N - 1);
      int kr = 0;
      if constexpr (MULTI) {
        if (b.ex >> 16) {
          kr = slab_of(x, zb[blk], cf, dscale, doffset, ndf) -
               (w.y & kSlabMask);
          kr = min(max(kr, 0), w.y >> kSpanShift);
        }
      }
      const int rel = i0 - w.x;
      const int base = min(max(min16(rel), 0), kMaxBase);
      const uint4 sl = sel[(rel - base) & 7];
      // position p of a run at 256 (p / 4) + 32 (p % 4) = 64 p - 32 (p % 4)
      const int pos = base + e;
      const int addr = pos * 64 + lo_addr - __mul24(pos & 3, 32);
      const float s = ok ? cf.w : 0.0f;
      auto pass = [&](float sc, int slot) {
        const float w1 = sc * tt, w0 = sc - w1;
        const half2v hi = to_half2(w0, w1);
        // what the high parts leave of the exact weights
        const half2v lo = to_half2(fmaf(-sc, tt, sc - (float)hi[0]),
                                   fmaf(sc, tt, -(float)hi[1]));
        const half8 ah = place(sl, hi), al = place(sl, lo);
        const uint32_t q = run0 + slot * S::kRunStride + addr;
        auto tiles = [&](auto r0, auto n, half8(&bv)[decltype(n)::value]) {
          constexpr int R0 = decltype(r0)::value, KN = decltype(n)::value;
#pragma unroll
          for (int r = 0; r < KN; ++r)
            acc[blk][R0 + r] = mfma16(al, bv[r], acc[blk][R0 + r]);
#pragma unroll
          for (int r = 0; r < KN; ++r)
            acc[blk][R0 + r] = mfma16(ah, bv[r], acc[blk][R0 + r]);
        };
        constexpr int kBlock = 64 * kPos;  // bytes of a 32-row block
        if constexpr (RB == 1) {
          half8 bv[2];
          read_tr8x2<0>(q, bv[0], bv[1]);
          tiles(Int<0>(), Int<2>(), bv);
        } else {
          half8 bv[4];
          read_tr8x4<0, kBlock>(q, bv[0], bv[1], bv[2], bv[3]);
          tiles(Int<0>(), Int<4>(), bv);
          // (a last workgroup with at most 64 rows left has no more)
          if (RB == 4 && many) {
            read_tr8x4<2 * kBlock, kBlock>(q, bv[0], bv[1], bv[2], bv[3]);
            tiles(Int<4>(), Int<4>(), bv);
          }
        }
      };
      if constexpr (!MULTI) {
        pass(s, g);
      } else {
        // One pass, or two: each group of 16 lanes (one tilt) takes the
        // first slab that a voxel of the block reads, then the second one.
        int ks = 0;
        if (b.ex >> 16) ks = min16(kr);
        float sc = kr == ks ? s : 0.0f;
        int slot = ks != 0 ? 4 + exg : g;
        bool left = kr != ks;
#pragma unroll 1
        for (;;) {
          pass(sc, slot);
          if (__ballot(left) == 0) break;
          // (a tile within one slab at a tilt has no second run)
          sc = left ? s : 0.0f;
          slot = w.y >> kSpanShift ? 4 + exg : g;
          left = false;
        }
      }
    }
  };

  // Each lane holds, per block and 16-row tile, 4 voxels in x (row m, z =
  // g): 16 rows at a time pass through LDS and leave as 64-byte pieces.
  auto store_all = [&]() {
    const bool wide = W % 4 == 0 && (reinterpret_cast<uintptr_t>(vol) & 15) == 0;
#pragma unroll
    for (int r = 0; r < kRT; ++r) {
      float *out = reinterpret_cast<float *>(lds + (r & 1) * kBufWords);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float *q = out + m * S::kOutRow +
                   (8 * (wave >> 2) + 4 * i + g) * kTile + 4 * (wave & 3);
        float4v v = acc[i][r];
        *reinterpret_cast<float4v *>(q) = v * down;
      }
      lds_barrier();
      if (wide) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int row = 2 * wave + i;
          const int y = byb * YB + 16 * r + row;
          const int oz = bz * kTile + (lane >> 2);
          const int ox = bx * kTile + 4 * (lane & 3);
          if (y < Y && oz < Z && ox < W)
            *reinterpret_cast<float4v *>(
                vol + ((size_t)(y - y_base) * Z + oz) * W + ox) =
                *reinterpret_cast<const float4v *>(out + row * S::kOutRow +
                                                   4 * lane);
        }
      } else {
        // lines of W values are not whole 16-byte words: a lane per voxel
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int row = 2 * wave + (i >> 2);
          const int y = byb * YB + 16 * r + row;
          const int oz = bz * kTile + 4 * (i & 3) + (lane >> 4);
          const int ox = bx * kTile + (lane & 15);
          if (y < Y && oz < Z && ox < W)
            vol[((size_t)(y - y_base) * Z + oz) * W + ox] =
                out[row * S::kOutRow + 64 * (i & 3) + lane];
        }
      }
    }
  };

  // All batches through body(batch, its buffer): the next one's loads are
  // issued first, into the other buffer. (One copy of the loop body: two, one
  // for each buffer order, made the compiler keep the accumulators twice and
  // spill.)
  auto batches = [&](auto body) {
    Batch b = next_batch(0);
    stage(b, lds);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    convert(b, lds);
    lds_barrier();
    auto step = [&](const uint4 *cur, uint4 *nxt) {
      const int t1 = b.t0 + b.nt;
      Batch nb{t1, 0, 0};
      if (t1 < T) {
        nb = next_batch(t1);
        stage(nb, nxt);
      }
      body(b, cur);
      if (t1 < T) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        convert(nb, nxt);
      }
      lds_barrier();
      b = nb;
    };
    int odd = 0;
#pragma unroll 1
    while (b.t0 < T) {
      step(lds + odd * kBufWords, lds + (1 - odd) * kBufWords);
      odd = 1 - odd;
    }
  };

  unsigned bad = 0;  // bit r: a value of row 16 r + m is not finite
  bool redo = true;
  if (!taps) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < kRT; ++r) acc[i][r] = (float4v)(0.0f);
    batches(multiply);
#pragma unroll
    for (int r = 0; r < kRT; ++r) {
      bool b = false;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          b |= !(fabsf(acc[i][r][j]) < __builtin_inff());
      if (b && byb * YB + 16 * r + m < Y) bad |= 1u << r;
    }
    redo = __syncthreads_or((int)bad) != 0;
    store_all();
  }
  if (!redo) return;

  // The rows that are not finite, tap by tap on the vector units: FP32
  // weights, the taps of exactly the voxels that read them, added in tilt
  // order as k_bp_lds adds them. A thread takes two voxels (of z and z + 8)
  // and 8 of every 32 rows; four neighbouring lanes share a voxel, so that 16
  // lanes read four positions of all rows, 256 bytes in distinct banks.
  // 61 corrected projections of 1024^2, a NaN in one (all rows, no matrix
  // pass: k_bp_coefficients): 4.23 ms with a lane per row of its matrix tile
  // and 2-byte LDS reads, 1.49 here, 1.27 with k_bp_lds. The results are stored
  // over those of the matrix pass, once these have left.
  __shared__ uint32_t rows_bad[RB];  // a bit per row
  if (threadIdx.x < RB) rows_bad[threadIdx.x] = taps ? ~0u : 0u;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
#pragma unroll
  for (int r = 0; r < kRT; ++r)
    if ((bad >> r) & 1) atomicOr(&rows_bad[r >> 1], 1u << (16 * (r & 1) + m));
  lds_barrier();
  unsigned todo = 0;  // 32-row blocks with such rows
#pragma unroll
  for (int i = 0; i < RB; ++i)
    if (rows_bad[i] != 0 && byb * YB + 32 * i < Y) todo |= 1u << i;
  todo = (unsigned)__builtin_amdgcn_readfirstlane((int)todo);

  const int part8 = (int)threadIdx.x & 3;  // rows 8 part8 .. of a block
  const int vox = (int)threadIdx.x >> 2;
  const int vx = bx * kTile + (vox & 15), vz = bz * kTile + (vox >> 4);
  const float px = voxel_coord(min(vx, W - 1), W);
  const float pz[2] = {voxel_coord(min(vz, Z - 1), Z),
                       voxel_coord(min(vz + 8, Z - 1), Z)};
  const int lane_off = (part8 >> 1) * 128 + (part8 & 1) * 16;
  float sum[2][RB][8];
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int r = 0; r < 8; ++r) sum[v][i][r] = 0.0f;
  batches([&](const Batch &b, const uint4 *cur) {
    const uint32_t run0 = lds_address(cur) + lane_off;
#pragma unroll 1
    for (int j = 0; j < b.nt; ++j) {
      const float4 cf = kload(coef, b.t0 + j);
      const int2 w = kload(tw, b.t0 + j);
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        float tt;
        const int i0 = tap_index<false>(px, pz[v], cf, tt);
        if ((unsigned)i0 < (unsigned)(N - 1)) {
          int slot = j;
          if constexpr (MULTI) {
            // (a tile within one slab at a tilt has its own run alone)
            if (w.y >> kSpanShift &&
                slab_of(px, pz[v], cf, dscale, doffset, ndf) >
                    (w.y & kSlabMask))
              slot = 4 + ((b.ex >> (4 * j)) & 15);
          }
          const int p0 = min(max(i0 - w.x, 0), kPos - 2), p1 = p0 + 1;
          const uint32_t q = run0 + slot * S::kRunStride;
          const uint32_t a0 = q + (p0 >> 2) * 256 + (p0 & 3) * 32;
          const uint32_t a1 = q + (p1 >> 2) * 256 + (p1 & 3) * 32;
          const float w1 = cf.w * tt, w0 = cf.w - w1;
          auto blocks = [&](auto i, auto n) {
            constexpr int I = decltype(i)::value, KN = decltype(n)::value;
            constexpr int kBlock = 64 * kPos;
            if (((todo >> I) & ((1u << KN) - 1)) == 0) return;
            half8 v0[KN], v1[KN];
            read_rows<I * kBlock, kBlock>(a0, a1, v0, v1);
#pragma unroll
            for (int k = 0; k < KN; ++k)
#pragma unroll
              for (int r = 0; r < 8; ++r)
                sum[v][I + k][r] =
                    fmaf(w1, (float)v1[k][r],
                         fmaf(w0, (float)v0[k][r], sum[v][I + k][r]));
          };
          blocks(Int<0>(), Int<(RB > 1 ? 2 : 1)>());
          if constexpr (RB > 2) blocks(Int<2>(), Int<2>());
        }
      }
    }
  });
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const uint32_t rows8 = rows_bad[i] >> (8 * part8);
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int y = byb * YB + 32 * i + 8 * part8 + r, oz = vz + 8 * v;
        if (((rows8 >> r) & 1) && y < Y && oz < Z && vx < W)
          vol[((size_t)(y - y_base) * Z + oz) * W + vx] = sum[v][i][r];
      }
  }
}

// -------------------------------------------------------------- launchers --

template <int YB, int STORE, bool MULTI, int RB>
static hipError_t launch_mm(const BpArgs &a, hipStream_t s) {
  constexpr int kYG = 32 * RB / YB;
  const int nbx = (a.W + kTile - 1) / kTile;
  const int nbz = (a.Z + kTile - 1) / kTile;
  const int ng = (a.yb1 - a.yb0 + kYG - 1) / kYG;
  const size_t nb = (size_t)nbx * nbz * ng;
  if (nb > 0xffffffffu) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_bp_mm<YB, STORE, MULTI, RB>), dim3((unsigned)nb),
                     dim3(kWaves * 64), 0, s, (const uint16_t *)a.slab, a.coef,
                     a.win, a.dscale, a.doffset, a.ndf, a.N, a.T, a.NYB, a.W,
                     a.Z, a.Y, a.yb0, a.yb1, a.y_base, a.slab_yb0, a.vol, nbx,
                     nbz, (unsigned)nb);
  return hipGetLastError();
}

template <int YB, int STORE, bool MULTI>
static hipError_t launch_mm_rows(const BpArgs &a, hipStream_t s) {
  // Rows per workgroup: 128, so that a block's weights serve as many rows as
  // the registers hold; 64 or 32 where the volume has no more, or where
  // larger workgroups would leave CUs without one (256 of them). The result
  // does not depend on it.
  const int nrb = ((a.yb1 - a.yb0) * YB + 31) / 32;
  const size_t tiles = (size_t)((a.W + kTile - 1) / kTile) *
                       ((a.Z + kTile - 1) / kTile);
  if (nrb > 2 && tiles * ((nrb + 3) / 4) > kFill)
    return launch_mm<YB, STORE, MULTI, 4>(a, s);
  if (nrb > 1 && tiles * ((nrb + 1) / 2) > kFill)
    return launch_mm<YB, STORE, MULTI, 2>(a, s);
  return launch_mm<YB, STORE, MULTI, 1>(a, s);
}

// With one slab always (61 tilts, 16 to 1000 pixels, 1 to 256 rows: nowhere
// slower). With several, a workgroup's batches wait for window entries and
// second runs in turn, which takes other workgroups to hide, wide slabs to be
// rare, and full workgroups of 128 rows to pay. Its backprojection against the
// staged kernel's, 41 tilts, slabs of 64 to 300 pixels:
// - two workgroups per CU (512): 256 x 256 x 64 voxels (128) 0.79 to 1.04,
//   512 rows of it (256) 0.98 to 1.29, 1024 (512) 1.22 to 1.60; 512 x 128 x 128
//   (256) 0.90 to 1.24, 512 x 128 x 256 (512) 1.12 to 1.38;
// - 32-row blocks that cost the staged kernel, 4 for about the time of 3.5, or
//   of 2.75 where a last workgroup has 64 rows or less: of 512 x 256 and 1024 x
//   256 tiles' worth, 32 rows 0.61 to 0.88, 96 0.89 to 1.18, 128 1.12 to 1.47,
//   160 0.79 to 1.00, 192 0.92 to 1.18, 256 1.08 to 1.47, 320 0.98 to 1.27, 512
//   1.12 to 1.36;
// - slabs of at least 64 pixels (46: 1.10; 640 x 150 x 200, 53: 0.87);
// - lines of whole 16-byte words, as others cost it the rest (483 x 156 x 400,
//   161: the request 0.99).
// Of the volume's rows, not of a band's: the kernels differ in the last bit.
bool bp_mm_suits(int ndf, float dscale, int W, int Z, int Y) {
  if (ndf == 1) return true;
  const int rest = Y % 128;
  const size_t full = (size_t)Y / 128 + (rest > 64 ? 1 : 0);
  const size_t half = rest > 0 && rest <= 64 ? 1 : 0;
  const size_t tiles = (size_t)((W + kTile - 1) / kTile) *
                       ((Z + kTile - 1) / kTile);
  return tiles * (full + half) >= 512 &&
         4 * ((size_t)(Y + 31) / 32) >= 14 * full + 11 * half && W % 4 == 0 &&
         fabsf(dscale) * 64.0f <= 1.0f;
}

hipError_t launch_bp_mm(const BpArgs &a, int YB, int store, hipStream_t s) {
  if (a.yb1 <= a.yb0) return hipSuccess;
  if (a.win == nullptr) return hipErrorInvalidValue;
#define C_(yb, st)                                                          \
  if (YB == yb && store == st)                                              \
    return a.ndf > 1 ? launch_mm_rows<yb, st, true>(a, s)                   \
                     : launch_mm_rows<yb, st, false>(a, s);
  C_(32, kF16) C_(16, kF16) C_(32, kBF16) C_(16, kBF16)
#undef C_
  return hipErrorInvalidValue;
}

}  // namespace gx
