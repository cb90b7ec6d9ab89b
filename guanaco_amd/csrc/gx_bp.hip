// Voxel-driven backprojection on gfx950.
//
// Reference semantics (src/libguanaco/reconstructor.cpp:14-90): for every
// voxel (x, z) of a slice and every tilt t, p = x c - z s + offset; with
// several defocus slabs the slab is floor(h * dscale + doffset + 0.5) clamped,
// h = -x s - z c; the value (1-t) row[i0] + t row[i0+1] with i0 = floor(p -
// 0.5) is added, times the tilt's scale, only when 0 <= i0 < N-1.
//
// The geometry of a voxel column does not depend on the detector row y, so
// each thread owns one (x, z) and YB consecutive rows: the coordinate work is
// paid once per (voxel column, tilt) and the taps of all YB rows are one
// contiguous 2*YB-value read from the [k][t][y/YB][x][y%YB] layout. A
// workgroup is a 32 (x) by 8 (z) tile; consecutive logical workgroups are
// z-neighbours and are kept on one XCD so their overlapping row segments hit
// the same L2. The volume is written once, [y][z][x] with x fastest.
//
// kF32 reproduces the reference's FP32 operation order exactly (compiled
// without FMA contraction): per-tilt constants computed on the host as the
// reference does, tilt-outer accumulation order, no reassociation. kF16 and
// kBF16 (whose error budget is set by the storage) compute p with two fused
// multiply-adds from a table holding offset - 1/2 and the scale times the
// normalisation the filter pass divided out, and accumulate with FP32 fused
// multiply-adds (BF16 taps rounded to FP16 first: bf16_tap). The per-tilt
// tables are read with scalar loads. 16-bit plans with one slab, and large
// ones with wide slabs, run on the matrix cores instead (gx_bp_mm.hip).
#include <type_traits>

#include "gx_bp_geometry.hpp"
#include "gx_common.hpp"
#include "gx_kernels.hpp"

namespace gx {

constexpr int kTX = 32, kTZ = 8;
constexpr size_t kRowTiles = 2048;  // (launch_bp_rows_t)

template <int YB, int STORE>
struct Taps;

// BF16 taps enter the arithmetic rounded to FP16, as the staged kernel keeps
// them in LDS (bf16_pair_to_f16): exact for magnitudes in [2^-14, 65504]
// (eight significant bits fit FP16's eleven), and within 2^-25 below, where
// FP16 is subnormal. The normalised slabs stay far below 65504, as they must
// for FP16 storage. The staged kernel then interpolates with
// v_fma_mix_f32, one instruction per tap, like FP16, where BF16 would need a
// shift or mask before each FMA; the direct kernels round the same way so
// that every kernel gives the same bits.
__device__ __forceinline__ float bf16_tap(float v) {
  return (float)(_Float16)v;
}
__device__ __forceinline__ uint32_t bf16_pair_to_f16(uint32_t w) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  const f32x2 f = {__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
}
template <int STORE>
__device__ __forceinline__ float tap_value(typename StoreT<STORE>::T v) {
  if constexpr (STORE == kBF16) {
    return bf16_tap(StoreT<STORE>::unpack(v));
  } else {
    return StoreT<STORE>::unpack(v);
  }
}

template <int YB>
struct Taps<YB, kF32> {
  float v0[YB], v1[YB];
  // 16-byte word i of each tap: rows 4i .. 4i + 3
  __device__ __forceinline__ void unpack(int i, uint4 a, uint4 b) {
    v0[4 * i] = __uint_as_float(a.x); v0[4 * i + 1] = __uint_as_float(a.y);
    v0[4 * i + 2] = __uint_as_float(a.z); v0[4 * i + 3] = __uint_as_float(a.w);
    v1[4 * i] = __uint_as_float(b.x); v1[4 * i + 1] = __uint_as_float(b.y);
    v1[4 * i + 2] = __uint_as_float(b.z); v1[4 * i + 3] = __uint_as_float(b.w);
  }
  // The YB values of each tap as YB / 4 16-byte words at q0 and at q1
  // (global memory).
  __device__ __forceinline__ void load16(const uint4 *q0, const uint4 *q1) {
    static_assert(YB % 4 == 0, "16-byte taps need YB % 4 == 0");
#pragma unroll
    for (int i = 0; i < YB / 4; ++i) unpack(i, q0[i], q1[i]);
  }
  // word-major runs of the staged kernel: word i of position p at q[i SW]
  template <int SW>
  __device__ __forceinline__ void load16_strided(const uint4 *q) {
#pragma unroll
    for (int i = 0; i < YB / 4; ++i) unpack(i, q[i * SW], q[i * SW + 1]);
  }
  __device__ __forceinline__ void load(const float *p) {
    if constexpr (YB % 4 == 0) {
      const uint4 *q = (const uint4 *)__builtin_assume_aligned(p, 16);
      load16(q, q + YB / 4);
    } else {
#pragma unroll
      for (int i = 0; i < YB; ++i) {
        v0[i] = p[i];
        v1[i] = p[YB + i];
      }
    }
  }
};

template <int YB, int STORE>
struct Taps {
  using T = typename StoreT<STORE>::T;
  static_assert(YB % 8 == 0, "reduced storage needs YB % 8 == 0");
  float v0[YB], v1[YB];
  __device__ __forceinline__ void load(const T *p) {
    const uint4 *q = (const uint4 *)__builtin_assume_aligned(p, 16);
    load16(q, q + YB / 8);
  }
  // 16-byte word i of each tap: rows 8i .. 8i + 7, two to a 32-bit word
  __device__ __forceinline__ void unpack(int i, uint4 a, uint4 b) {
    const uint32_t wa[4] = {a.x, a.y, a.z, a.w};
    const uint32_t wb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v0[8 * i + 2 * j] = lo(wa[j]);
      v0[8 * i + 2 * j + 1] = hi(wa[j]);
      v1[8 * i + 2 * j] = lo(wb[j]);
      v1[8 * i + 2 * j + 1] = hi(wb[j]);
    }
  }
  __device__ __forceinline__ void load16(const uint4 *q0, const uint4 *q1) {
#pragma unroll
    for (int i = 0; i < YB / 8; ++i) unpack(i, q0[i], q1[i]);
  }
  // The staged kernel's word-major runs: word i of position p at q[i SW]
  // (q at position p), position p + 1 one word on.
  template <int SW>
  __device__ __forceinline__ void load16_strided(const uint4 *q) {
#pragma unroll
    for (int i = 0; i < YB / 8; ++i) unpack(i, q[i * SW], q[i * SW + 1]);
  }
  __device__ __forceinline__ static float lo(uint32_t w) {
    if constexpr (STORE == kF16) {
      return __half2float(__ushort_as_half((unsigned short)(w & 0xffffu)));
    } else {
      return bf16_tap(__uint_as_float(w << 16));
    }
  }
  __device__ __forceinline__ static float hi(uint32_t w) {
    if constexpr (STORE == kF16) {
      return __half2float(__ushort_as_half((unsigned short)(w >> 16)));
    } else {
      return bf16_tap(__uint_as_float(w & 0xffff0000u));
    }
  }
};

// ------------------------------------------------------- per-tilt tables --

// out[t] = (c, s, offset - 1/2, weight): the weight is the tilt's scale times
// the normalisation float(tmax[t]) * nrm_mul that the filter pass divided the
// stored values by (1 without tmax), and zero for a tilt whose largest value
// is zero: all it stored is zeros (or NaNs, which a zero weight keeps).
// Entries T .. Tpad - 1 are zero. Entry Tpad is launch_bp_mm's: (u, 1 / u, 0),
// the power of two u that takes the largest weight to [2^13, 2^14) (1 where
// there is none). Its FP16 pairs end at 2^-24, which is finer than the FP32
// rounding of a weight of at least 1; a series whose smallest weight falls
// below that after scaling (tilts that differ 8192-fold), or with one that is
// not finite, gets (1, 1, 1) and FP32 weights. One workgroup.
__global__ __launch_bounds__(256) void k_bp_coefficients(
    const float4 *__restrict__ coef, const uint32_t *__restrict__ tmax,
    float nrm_mul, int T, int Tpad, float4 *__restrict__ out) {
  __shared__ float red[4];
  float top = 0.0f, inv_low = 0.0f;  // (1 / the smallest, as a maximum)
  for (int t = threadIdx.x; t < Tpad; t += 256) {
    float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < T) {
      const float4 cf = coef[t];
      const float nrm =
          tmax != nullptr ? __uint_as_float(tmax[t]) * nrm_mul : 1.0f;
      r = make_float4(cf.x, cf.y, cf.z - 0.5f, cf.w * nrm);
      const float a = fabsf(r.w);
      if (!(a < __builtin_inff())) {
        inv_low = __builtin_inff();
      } else if (a > 0.0f) {
        top = fmaxf(top, a);
        inv_low = fmaxf(inv_low, 1.0f / a);
      }
    }
    out[t] = r;
  }
  top = block_max<256>(top, red);
  inv_low = block_max<256>(inv_low, red);
  if (threadIdx.x == 0) {
    int e = 0;
    if (top > 0.0f) {
      (void)frexpf(top, &e);  // top in [2^(e-1), 2^e)
      e = min(max(14 - e, -126), 126);
    }
    // smallest * u >= 1, also where 1 / smallest is infinite
    const float u = ldexpf(1.0f, e);
    out[Tpad] = inv_low <= u ? make_float4(u, ldexpf(1.0f, -e), 0.0f, 0.0f)
                             : make_float4(1.0f, 1.0f, 1.0f, 0.0f);
  }
}

hipError_t launch_bp_coefficients(const float4 *coef, const uint32_t *tmax,
                                  float nrm_mul, int T, float4 *out,
                                  hipStream_t s) {
  hipLaunchKernelGGL(k_bp_coefficients, dim3(1), dim3(256), 0, s, coef, tmax,
                     nrm_mul, T, bp_tilt_pad(T), out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// LDS-staged form.
//
// p is a chain of correctly rounded float operations, each monotone in x and
// in z, so over a 32 x 8 tile i0 is smallest at one of the four corners, and
// the exact range of p is at most 31|c| + 7|s| <= 31.79 sqrt(c^2 + s^2)
// (c^2 + s^2 = 1 / (cos^2 + sin^2) to rounding): the taps of one tilt lie in
// a window of 34 consecutive positions; kWPOS leaves a margin for rounding.
// Likewise h spans at most 31.79 units, so a tile touches at most
// ceil(31.79 |dscale|) + 1 consecutive slabs; the host picks KS, the slabs
// staged per tilt, no smaller than that. The window base and first slab of
// every (tile, tilt) come from a table computed once per plan with the same
// arithmetic as the kernel. For a batch of TB tilts the workgroup copies, per
// tilt and staged slab, kWPOS positions of its row block starting at the
// window base (one contiguous run of the slab, YB rows per position) into
// LDS, then interpolates from LDS with the same arithmetic per voxel as the
// direct kernel. LDS indices are clamped, so coefficients that break the
// bound (non-finite angles, which the host rejects) can only give wrong
// values, never an access outside the buffer.
//
// The runs are loaded straight into LDS (buffer_load ... lds), not through
// registers; BF16 runs are then converted to FP16 in place by the lanes that
// loaded them (bf16_tap). Two LDS buffers: the loads of batch b + 1 are
// issued before batch b is interpolated, one barrier per batch.
constexpr int kWPOS = 40;

template <int YB, int STORE, int KS>
struct Staging {
  using T = typename StoreT<STORE>::T;
  static constexpr int kPosBytes = YB * (int)sizeof(T);
  static constexpr int kPosWords = kPosBytes / 16;      // 16-byte words
  static constexpr int kTB = 256 / (kPosBytes * KS);    // tilts per batch
  static constexpr int kNSlot = kTB * KS;  // (tilt, slab) runs per batch
  static constexpr int kChunks = kWPOS * kPosWords;  // words per run
  static constexpr int kCPL = (kChunks + 63) / 64;   // words per lane per run
  static constexpr int kSPW = kNSlot / (kTX * kTZ / 64);  // runs per wave
  // buffer_load ... lds writes lane l of a load to slot l of a dense 1 KiB
  // block, so a run is kRunSlots 16-byte slots, slot s < kChunks holding
  // word s / kWPOS of position s % kWPOS. In this word-major order the reads
  // of lanes at consecutive positions are consecutive 16-byte words, which
  // gfx950 serves without bank conflicts (as it does a padded odd stride).
  static constexpr int kRunSlots = kCPL * 64;
  static constexpr int kBufWords = kNSlot * kRunSlots;
  static_assert(kPosBytes % 16 == 0, "a position is whole 16-byte words");
  static_assert(kTB >= 1 && kBpTiltPad % kTB == 0,
                "batches must tile the padded tilt tables");
  static_assert(kNSlot % (kTX * kTZ / 64) == 0, "runs split evenly on waves");
};

// Window of one tilt over the tile's active voxels [x0, x1] x [z0, z1]:
// smallest i0 and smallest k over the four corners, with kOneSlab set in .y
// when the largest k over the corners is the same: slab_of is monotone in x
// and in z like p, so every voxel of the tile then takes slab k.
constexpr int kOneSlab = 1 << 30;
constexpr int kSlabMask = kOneSlab - 1;

template <bool EXACT, bool MULTI>
__device__ __forceinline__ int2 tile_window(float4 cf, float x0, float x1,
                                            float z0, float z1, float dscale,
                                            float doffset, int ndf) {
  int w = 0x7fffffff, k = 0x7fffffff, kmax = -1;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float x = (c & 1) ? x1 : x0;
    const float z = (c & 2) ? z1 : z0;
    float tt;
    w = min(w, tap_index<EXACT>(x, z, cf, tt));
    if constexpr (MULTI) {
      const int kc = slab_of(x, z, cf, dscale, doffset, ndf);
      k = min(k, kc);
      kmax = max(kmax, kc);
    }
  }
  return make_int2(w, MULTI ? (k | (kmax == k ? kOneSlab : 0)) : 0);
}

// win[tile * Tpad + t], tile = bx * nbz + bz (the kernels' order).
template <bool EXACT, bool MULTI>
__global__ void k_bp_windows(const float4 *__restrict__ coef, int T, int Tpad,
                             int W, int Z, int nbx, int nbz, float dscale,
                             float doffset, int ndf, int2 *__restrict__ win) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i >= (size_t)nbx * nbz * Tpad) return;
  const int t = (int)(i % Tpad);
  const int tile = (int)(i / Tpad);
  const int bz = tile % nbz, bx = tile / nbz;
  int2 r = make_int2(0, 0);
  if (t < T) {
    const float x0 = voxel_coord(bx * kTX, W);
    const float x1 = voxel_coord(min(bx * kTX + kTX, W) - 1, W);
    const float z0 = voxel_coord(bz * kTZ, Z);
    const float z1 = voxel_coord(min(bz * kTZ + kTZ, Z) - 1, Z);
    r = tile_window<EXACT, MULTI>(coef[t], x0, x1, z0, z1, dscale, doffset,
                                  ndf);
  }
  win[i] = r;
}

size_t bp_window_entries(int W, int Z, int T) {
  const size_t nbx = (W + kTX - 1) / kTX, nbz = (Z + kTZ - 1) / kTZ;
  return nbx * nbz * (size_t)bp_tilt_pad(T);
}

hipError_t launch_bp_windows(const float4 *coef, int exact, int T, int W,
                             int Z, float dscale, float doffset, int ndf,
                             int2 *win, hipStream_t s) {
  const int nbx = (W + kTX - 1) / kTX, nbz = (Z + kTZ - 1) / kTZ;
  const size_t n = bp_window_entries(W, Z, T);
  const dim3 g((unsigned)((n + 255) / 256)), b(256);
  const int Tpad = bp_tilt_pad(T);
  const bool multi = ndf > 1;
  if (exact && multi)
    hipLaunchKernelGGL((k_bp_windows<true, true>), g, b, 0, s, coef, T, Tpad,
                       W, Z, nbx, nbz, dscale, doffset, ndf, win);
  else if (exact)
    hipLaunchKernelGGL((k_bp_windows<true, false>), g, b, 0, s, coef, T, Tpad,
                       W, Z, nbx, nbz, dscale, doffset, ndf, win);
  else if (multi)
    hipLaunchKernelGGL((k_bp_windows<false, true>), g, b, 0, s, coef, T, Tpad,
                       W, Z, nbx, nbz, dscale, doffset, ndf, win);
  else
    hipLaunchKernelGGL((k_bp_windows<false, false>), g, b, 0, s, coef, T, Tpad,
                       W, Z, nbx, nbz, dscale, doffset, ndf, win);
  return hipGetLastError();
}

// ------------------------------------------------------------ kernels -----

// Accumulate one tilt's taps (reconstructor.cpp:82-84).
template <int YB, int STORE>
__device__ __forceinline__ void accumulate(float (&acc)[YB],
                                           const Taps<YB, STORE> &tp,
                                           float4 cf, float tt) {
  if constexpr (STORE == kF32) {
    const float w0 = 1.0f - tt;
#pragma unroll
    for (int r = 0; r < YB; ++r)
      acc[r] = acc[r] + cf.w * (w0 * tp.v0[r] + tt * tp.v1[r]);
  } else {
    const float w1 = cf.w * tt;  // cf.w: scale x normalisation
    const float w0 = cf.w - w1;
#pragma unroll
    for (int r = 0; r < YB; ++r) {
      acc[r] = fmaf(w0, tp.v0[r], acc[r]);
      acc[r] = fmaf(w1, tp.v1[r], acc[r]);
    }
  }
}

template <int YB, int STORE, bool MULTI>
__global__ __launch_bounds__(kTX *kTZ) void k_bp(
    const typename StoreT<STORE>::T *__restrict__ slab,
    const float4 *__restrict__ coef, float dscale, float doffset, int ndf,
    int N, int T, int NYB, int W, int Z, int Y, int yb0, int y_base,
    int slab_yb0,
    float *__restrict__ vol, int nbx, int nbz, unsigned nblocks) {
  constexpr bool kExact = STORE == kF32;
  const unsigned lb = xcd_remap(blockIdx.x, nblocks);
  const int bz = (int)(lb % (unsigned)nbz);
  const int bx = (int)((lb / (unsigned)nbz) % (unsigned)nbx);
  const int byb = yb0 + (int)(lb / ((unsigned)nbz * (unsigned)nbx));
  const int ix = bx * kTX + (int)(threadIdx.x % kTX);
  const int iz = bz * kTZ + (int)(threadIdx.x / kTX);
  const bool active = ix < W && iz < Z;
  const float x = voxel_coord(ix, W);
  const float z = voxel_coord(iz, Z);

  float acc[YB];
#pragma unroll
  for (int r = 0; r < YB; ++r) acc[r] = 0.0f;

  const size_t row_len = (size_t)N * YB;
  const size_t kstride = (size_t)T * NYB * row_len;
  const typename StoreT<STORE>::T *yblock = slab + (size_t)(byb - slab_yb0) * row_len;

  for (int t = 0; t < T; ++t) {
    const float4 cf = kload(coef, t);
    int k = 0;
    if constexpr (MULTI) k = slab_of(x, z, cf, dscale, doffset, ndf);
    float tt;
    const int i0 = tap_index<kExact>(x, z, cf, tt);
    if (active && (unsigned)i0 < (unsigned)(N - 1)) {
      Taps<YB, STORE> tp;
      tp.load(yblock + (size_t)t * NYB * row_len + (size_t)k * kstride +
              (size_t)i0 * YB);
      accumulate<YB, STORE>(acc, tp, cf, tt);
    }
  }
  if (active) {
#pragma unroll
    for (int r = 0; r < YB; ++r) {
      const int y = byb * YB + r;
      if (y < Y) vol[((size_t)(y - y_base) * Z + iz) * W + ix] = acc[r];
    }
  }
}

// One slice of one detector row per slab (gx_recon, gx_project and their
// no-allocation form; slab [k][t][x]): a thread per voxel, so few waves that
// nothing hides the latency of a tilt's two loads but the loads of other
// tilts. kU tilts are therefore loaded together, unconditionally from clamped
// positions, and added in the reference's order. (With a branch and two loads
// a tilt, 61 tilts x 256 x 256 voxels took 25.5 us; here 13.9. Eight slabs over
// 1500 x 300 voxels, 90 tilts: 45 us either way, vector issue.)
template <bool MULTI>
__global__ __launch_bounds__(kTX *kTZ) void k_bp_slice(
    const float *__restrict__ slab, const float4 *__restrict__ coef,
    float dscale, float doffset, int ndf, int N, int T, int W, int Z,
    float *__restrict__ vol, int nbx) {
  constexpr int kU = 8;
  const int ix = (int)(blockIdx.x % (unsigned)nbx) * kTX +
                 (int)(threadIdx.x % kTX);
  const int iz = (int)(blockIdx.x / (unsigned)nbx) * kTZ +
                 (int)(threadIdx.x / kTX);
  const float x = voxel_coord(ix, W);
  const float z = voxel_coord(iz, Z);
  const size_t kstride = (size_t)T * N;
  const int next = N > 1 ? 1 : 0;
  float acc = 0.0f;
  for (int t0 = 0; t0 < T; t0 += kU) {
    float tt[kU], v0[kU], v1[kU], w[kU];
    bool in[kU];
#pragma unroll
    for (int j = 0; j < kU; ++j) {
      const int t = min(t0 + j, T - 1);
      const float4 cf = kload(coef, t);
      const int i0 = tap_index<true>(x, z, cf, tt[j]);
      in[j] = t0 + j < T && (unsigned)i0 < (unsigned)(N - 1);
      w[j] = cf.w;
      const float *row = slab + (size_t)t * N;
      if constexpr (MULTI)
        row += (size_t)slab_of(x, z, cf, dscale, doffset, ndf) * kstride;
      row += min(max(i0, 0), N - 1 - next);
      v0[j] = row[0];
      v1[j] = row[next];
    }
#pragma unroll
    for (int j = 0; j < kU; ++j) {
      float a = acc + w[j] * ((1.0f - tt[j]) * v0[j] + tt[j] * v1[j]);
      asm volatile("" : "+v"(a));  // (as in k_bp_rows)
      acc = in[j] ? a : acc;
    }
  }
  if (ix < W && iz < Z) vol[(size_t)iz * W + ix] = acc;
}

static hipError_t launch_bp_slice(const BpArgs &a, hipStream_t s) {
  if (a.yb1 <= a.yb0) return hipSuccess;
  // one row: the row block is the slab
  if (a.NYB != 1 || a.Y != 1 || a.yb0 != 0 || a.slab_yb0 != 0)
    return hipErrorInvalidValue;
  const int nbx = (a.W + kTX - 1) / kTX, nbz = (a.Z + kTZ - 1) / kTZ;
  const dim3 grid((unsigned)nbx * (unsigned)nbz), block(kTX * kTZ);
  if (a.ndf > 1)
    hipLaunchKernelGGL(k_bp_slice<true>, grid, block, 0, s,
                       (const float *)a.slab, a.coef, a.dscale, a.doffset,
                       a.ndf, a.N, a.T, a.W, a.Z, a.vol, nbx);
  else
    hipLaunchKernelGGL(k_bp_slice<false>, grid, block, 0, s,
                       (const float *)a.slab, a.coef, a.dscale, a.doffset,
                       a.ndf, a.N, a.T, a.W, a.Z, a.vol, nbx);
  return hipGetLastError();
}

// One slab value at a byte offset of a range-checked buffer.
template <int STORE>
__device__ __forceinline__ typename StoreT<STORE>::T buffer_tap(
    __amdgpu_buffer_rsrc_t rs, int off) {
  if constexpr (STORE == kF32) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
  } else {
    const uint16_t u = __builtin_amdgcn_raw_buffer_load_b16(rs, off, 0, 0);
    return __builtin_bit_cast(typename StoreT<STORE>::T, u);
  }
}

// Per-row rotation centres (one centre per slice, mp.py:144-154): each row
// has its own offset and so its own taps. The slab depends on h only, which
// no centre changes. kF32 keeps the reference's order: p = (x c - z s) +
// offset_y, then p - 1/2.
//
// A lane is a row here: the YB rows of a position are one contiguous run of
// 64 bytes (32 with the smaller blocks), and rows whose centres differ by
// little read the same or the next position, so a load of a wave touches a
// handful of cache lines. (With a lane per voxel, as in k_bp, each load
// touched one line per lane and the address unit bound the kernel: 61 tilts,
// 512 x 128 x 512 voxels, FP32: 4.94 ms; here 1.66e6 cycles, 0.69 ms at 2.4
// GHz.) A thread keeps 4 (x) by VZ (z) voxels; a workgroup is the same 32 x 8
// voxels by YB rows (VZ = YB / 4) or a part of them. The address and data units are busy 0.95 of that
// time, 6 cycles for each of the two loads of a wave's updates, and the vector
// units issue 15.7 instructions for an update: position, floor and fraction,
// address, range and the reference's five roundings, none of which
// rows share. A tile within one slab at a tilt (win) takes one buffer for
// all its voxels; elsewhere each voxel chooses its slab.
template <int YB, int STORE, bool MULTI, int VZ>
__global__ __launch_bounds__(kTX *kTZ) void k_bp_rows(
    const typename StoreT<STORE>::T *__restrict__ slab,
    const float4 *__restrict__ coef, const int2 *__restrict__ win,
    const float *__restrict__ row_off, int Y_tab, float dscale, float doffset,
    int ndf, int N, int T, int NYB, int W, int Z, int Y, int yb0, int y_base,
    int slab_yb0, float *__restrict__ vol, int nbx, int nbz,
    unsigned nblocks) {
  constexpr bool kExact = STORE == kF32;
  using ST = StoreT<STORE>;
  constexpr int VX = 4;               // (x) by VZ (z) voxels of a thread
  constexpr int GX = kTX / VX;        // thread groups of a tile in x
  constexpr int DZ = 32 * VZ / YB;    // z of a workgroup: kTZ, or a part
  static_assert(kTZ % DZ == 0, "workgroups split a tile");
  constexpr unsigned kParts = kTZ / DZ;
  const unsigned lp = xcd_remap(blockIdx.x, nblocks);
  const unsigned lb = lp / kParts, part = lp % kParts;
  const int bz = (int)(lb % (unsigned)nbz);
  const int bx = (int)((lb / (unsigned)nbz) % (unsigned)nbx);
  const int byb = yb0 + (int)(lb / ((unsigned)nbz * (unsigned)nbx));
  const int r = (int)threadIdx.x % YB, q = (int)threadIdx.x / YB;
  const int ix = bx * kTX + (q % GX) * VX;
  const int iz = bz * kTZ + (int)part * DZ + (q / GX) * VZ;
  const int y = byb * YB + r;
  float x[VX], z[VZ];
#pragma unroll
  for (int i = 0; i < VX; ++i) x[i] = voxel_coord(ix + i, W);
#pragma unroll
  for (int j = 0; j < VZ; ++j) z[j] = voxel_coord(iz + j, Z);

  float acc[VZ][VX];
#pragma unroll
  for (int j = 0; j < VZ; ++j)
#pragma unroll
    for (int i = 0; i < VX; ++i) acc[j][i] = 0.0f;

  const size_t row_len = (size_t)N * YB;
  const size_t kstride = (size_t)T * NYB * row_len;
  const typename ST::T *yblock = slab + (size_t)(byb - slab_yb0) * row_len;
  const int2 *tw = win + (size_t)(bx * nbz + bz) * bp_tilt_pad(T);
  const float *offs = row_off + min(y, Y_tab - 1);

  for (int t = 0; t < T; ++t) {
    const float4 cf = kload(coef, t);
    const float off = offs[(size_t)t * Y_tab];
    const typename ST::T *base = yblock + (size_t)t * NYB * row_len;
    bool one = true;  // the tile lies in one slab at this tilt
    if constexpr (MULTI) {
      const int k = kload(tw, t).y;
      one = (k & kOneSlab) != 0;
      if (one) base += (size_t)(k & kSlabMask) * kstride;
    }
    // One range-checked buffer over the row block: a position outside
    // [0, N) reads zeros (and its update is dropped).
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)base, (short)0, (int)(row_len * sizeof(*base)), 0x00020000);
    auto tilt = [&](auto one_slab) {
#pragma unroll
      for (int j = 0; j < VZ; ++j) {
        // the part of p that the voxels of one z share
        const float zs = kExact ? z[j] * cf.y : fmaf(-z[j], cf.y, off);
        float tt[VX], v0[VX], v1[VX];
        bool in[VX];
#pragma unroll
        for (int i = 0; i < VX; ++i) {
          float p;
          if constexpr (kExact) {
            p = x[i] * cf.x - zs;
            p = p + off;
            p = p - 0.5f;
          } else {
            p = fmaf(x[i], cf.x, zs);
          }
          const float fi = floorf(p);
          tt[i] = p - fi;
          const int i0 = (int)fi;
          in[i] = (unsigned)i0 < (unsigned)(N - 1);
          if constexpr (decltype(one_slab)::value) {
            const int o = (i0 * YB + r) * (int)sizeof(*base);
            v0[i] = tap_value<STORE>(buffer_tap<STORE>(rs, o));
            v1[i] = tap_value<STORE>(
                buffer_tap<STORE>(rs, o + YB * (int)sizeof(*base)));
          } else {
            const typename ST::T *s =
                base + (size_t)slab_of(x[i], z[j], cf, dscale, doffset, ndf) *
                           kstride +
                (size_t)(in[i] ? i0 : 0) * YB + r;
            v0[i] = tap_value<STORE>(s[0]);
            v1[i] = tap_value<STORE>(s[N > 1 ? YB : 0]);
          }
        }
#pragma unroll
        for (int i = 0; i < VX; ++i) {
          float a;
          if constexpr (kExact) {
            a = acc[j][i] + cf.w * ((1.0f - tt[i]) * v0[i] + tt[i] * v1[i]);
          } else {
            const float w1 = cf.w * tt[i];
            a = fmaf(w1, v1[i], fmaf(cf.w - w1, v0[i], acc[j][i]));
          }
          // computed whether it is in range or not: a branch around the
          // loads would serialise them
          asm volatile("" : "+v"(a));
          acc[j][i] = in[i] ? a : acc[j][i];
        }
      }
    };
    if (!MULTI || one)
      tilt(std::true_type());
    else
      tilt(std::false_type());
  }
  if (y >= Y) return;
  const bool wide = W % 4 == 0 && (reinterpret_cast<uintptr_t>(vol) & 15) == 0;
#pragma unroll
  for (int j = 0; j < VZ; ++j) {
    if (iz + j >= Z) continue;
    float *d = vol + ((size_t)(y - y_base) * Z + iz + j) * W + ix;
    if (wide) {
      if (ix < W)
        *reinterpret_cast<float4 *>(d) =
            make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
    } else {
#pragma unroll
      for (int i = 0; i < VX; ++i)
        if (ix + i < W) d[i] = acc[j][i];
    }
  }
}

template <int YB, int STORE, bool MULTI, int KS>
__global__ __launch_bounds__(kTX *kTZ) void k_bp_lds(
    const typename StoreT<STORE>::T *__restrict__ slab,
    const float4 *__restrict__ coef, const int2 *__restrict__ win,
    float dscale, float doffset, int ndf, int N, int T, int NYB, int W, int Z,
    int Y, int yb0, int y_base, int slab_yb0, float *__restrict__ vol,
    int nbx, int nbz,
    unsigned nblocks) {
  using S = Staging<YB, STORE, KS>;
  using ST = typename StoreT<STORE>::T;
  constexpr bool kExact = STORE == kF32;
  // BF16 runs are staged as FP16 (bf16_tap)
  constexpr int kLds = STORE == kBF16 ? kF16 : STORE;
  static_assert(MULTI || KS == 1, "one slab without defocus slabs");
  // Two buffers as two arrays: with distinct objects the compiler can tell
  // that reads of one do not wait for the direct loads into the other.
  __shared__ uint4 lds_a[S::kBufWords];
  __shared__ uint4 lds_b[S::kBufWords];

  const unsigned lb = xcd_remap(blockIdx.x, nblocks);
  const int bz = (int)(lb % (unsigned)nbz);
  const int bx = (int)((lb / (unsigned)nbz) % (unsigned)nbx);
  const int byb = yb0 + (int)(lb / ((unsigned)nbz * (unsigned)nbx));
  const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
  const int ix = bx * kTX + (int)(threadIdx.x % kTX);
  const int iz = bz * kTZ + (int)(threadIdx.x / kTX);
  const bool active = ix < W && iz < Z;
  const float x = voxel_coord(ix, W);
  const float z = voxel_coord(iz, Z);
  const int2 *tw = win + (size_t)(bx * nbz + bz) * bp_tilt_pad(T);

  const size_t row_len = (size_t)N * YB;
  const size_t tstride = (size_t)NYB * row_len;
  const size_t kstride = (size_t)T * tstride;
  const ST *yblock = slab + (size_t)(byb - slab_yb0) * row_len;

  // The staging runs of a wave are wave-uniform: with the wave index taken
  // from the first lane, each run's window entry is a scalar load and its
  // buffer descriptor lives in scalar registers.
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  // each lane's byte offset within a run past its window base (-1: the
  // slots past the run), the same for every batch
  int dslot[S::kCPL];
#pragma unroll
  for (int c = 0; c < S::kCPL; ++c) {
    const int s = lane + 64 * c;
    const int wi = s / kWPOS, p = s - wi * kWPOS;
    dslot[c] = s < S::kChunks
                   ? (p * YB + wi * (16 / (int)sizeof(ST))) * (int)sizeof(ST)
                   : -1;
  }
  auto load_batch = [&](int tb, uint4 *dst) {
#pragma unroll
    for (int i = 0; i < S::kSPW; ++i) {
      const int q = wave_u + (kTX * kTZ / 64) * i;
      const int j = q / KS, sl = q % KS;
      const int t = tb + j;
      const int2 w = kload(tw, t);
      const int k = MULTI ? (w.y & kSlabMask) + sl : 0;
      // a tile within one slab at this tilt reads only its first run
      const bool ok = t < T && k < ndf && (sl == 0 || !(w.y & kOneSlab));
      const ST *src = yblock + (size_t)t * tstride + (size_t)k * kstride;
      // One range-checked raw buffer per run: its N positions of YB values.
      // A load at an offset outside [0, N * YB * sizeof(T)) returns zeros
      // and touches no memory, so positions outside [0, N), the slots past
      // the window (offset -1) and runs past the last tilt or slab (no
      // records) all read as zero without branches.
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(
          (void *)(ok ? src : yblock), (short)0,
          ok ? (int)(row_len * sizeof(ST)) : 0, 0x00020000);
      // 64 slots of the run per load, lane l to slot l of its 1 KiB
      const int base = w.x * YB * (int)sizeof(ST);
#pragma unroll
      for (int c = 0; c < S::kCPL; ++c)
        load_to_lds16(rs, dst + q * S::kRunSlots + 64 * c,
                      dslot[c] >= 0 ? base + dslot[c] : -1);
    }
  };
  // After this wave's loads have landed: BF16 slots to FP16, each by the
  // lane that loaded it (no other wave touches them before the barrier).
  auto convert_batch = [&](uint4 *dst) {
    if constexpr (STORE == kBF16) {
#pragma unroll
      for (int i = 0; i < S::kSPW; ++i) {
        const int q = wave + (kTX * kTZ / 64) * i;
#pragma unroll
        for (int c = 0; c < S::kCPL; ++c) {
          uint4 *d = dst + q * S::kRunSlots + lane + 64 * c;
          const uint4 v = *d;
          *d = make_uint4(bf16_pair_to_f16(v.x), bf16_pair_to_f16(v.y),
                          bf16_pair_to_f16(v.z), bf16_pair_to_f16(v.w));
        }
      }
    }
  };

  float acc[YB];
#pragma unroll
  for (int r = 0; r < YB; ++r) acc[r] = 0.0f;

  // One batch: prefetch the next into `nxt`, interpolate from `cur`.
  auto batch = [&](int b, const uint4 *cur, uint4 *nxt) {
    const int tb = b * S::kTB;
    const bool more = tb + S::kTB < T;
    if (more) load_batch(tb + S::kTB, nxt);
#pragma unroll
    for (int j = 0; j < S::kTB; ++j) {
      const int t = tb + j;
      if (t < T) {
        const float4 cf = kload(coef, t);
        const int2 w = kload(tw, t);
        int ks = 0;
        if constexpr (MULTI) {
          // A tile within one slab at this tilt needs no per-voxel slab
          // choice (w is the workgroup's own entry: the branch is uniform).
          if (!(w.y & kOneSlab)) {
            const int kf = w.y & kSlabMask;
            if constexpr (KS == 2) {
              // The tile's voxels take slab kf or kf + 1 (<= ndf - 1, as the
              // tile spans two), and floor(d + 1/2) >= kf + 1 exactly when
              // d >= kf + 1/2: one comparison of the float d with a
              // representable bound decides as slab_of does.
              const float d = slab_coord(x, z, cf, dscale, doffset);
              ks = d >= (float)kf + 0.5f ? 1 : 0;
            } else {
              ks = slab_of(x, z, cf, dscale, doffset, ndf) - kf;
              ks = min(max(ks, 0), KS - 1);
            }
          }
        }
        float tt;
        const int i0 = tap_index<kExact>(x, z, cf, tt);
        if (active && (unsigned)i0 < (unsigned)(N - 1)) {
          const int rel = min(max(i0 - w.x, 0), kWPOS - 2);
          // word-major run: word wi of position p in slot wi kWPOS + p
          Taps<YB, kLds> tp;
          tp.template load16_strided<kWPOS>(cur + (j * KS + ks) * S::kRunSlots +
                                            rel);
          accumulate<YB, kLds>(acc, tp, cf, tt);
        }
      }
    }
    if (more) {
      // this wave's loads have landed; the barrier then covers the other
      // waves' too
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      convert_batch(nxt);
    }
    lds_barrier();
  };

  load_batch(0, lds_a);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  convert_batch(lds_a);
  lds_barrier();
  const int nb = (T + S::kTB - 1) / S::kTB;
  for (int b = 0; b < nb; b += 2) {
    batch(b, lds_a, lds_b);
    if (b + 1 < nb) batch(b + 1, lds_b, lds_a);
  }
  if (active) {
#pragma unroll
    for (int r = 0; r < YB; ++r) {
      const int y = byb * YB + r;
      if (y < Y) vol[((size_t)(y - y_base) * Z + iz) * W + ix] = acc[r];
    }
  }
}

// ------------------------------------------------------------ launchers ---
template <int YB, int STORE, bool MULTI, int KS>
static hipError_t launch_bp_lds_k(const BpArgs &a, hipStream_t s) {
  using ST = typename StoreT<STORE>::T;
  const int nbx = (a.W + kTX - 1) / kTX;
  const int nbz = (a.Z + kTZ - 1) / kTZ;
  if (a.yb1 <= a.yb0) return hipSuccess;
  if (a.win == nullptr) return hipErrorInvalidValue;
  const unsigned nb =
      (unsigned)nbx * (unsigned)nbz * (unsigned)(a.yb1 - a.yb0);
  hipLaunchKernelGGL((k_bp_lds<YB, STORE, MULTI, KS>), dim3(nb),
                     dim3(kTX * kTZ), 0, s, (const ST *)a.slab, a.coef, a.win,
                     a.dscale, a.doffset, a.ndf, a.N, a.T, a.NYB, a.W, a.Z,
                     a.Y, a.yb0, a.y_base, a.slab_yb0, a.vol, nbx, nbz, nb);
  return hipGetLastError();
}

template <int YB, int STORE>
static hipError_t launch_bp_lds_t(const BpArgs &a, hipStream_t s) {
  if (a.ndf == 1) {
    if constexpr (STORE == kF32)
      return launch_bp_lds_k<YB, STORE, false, 1>(a, s);
    return hipErrorInvalidValue;  // 16 bits, one slab: launch_bp_mm
  }
  switch (a.staged) {
    case 2: return launch_bp_lds_k<YB, STORE, true, 2>(a, s);
    case 4: return launch_bp_lds_k<YB, STORE, true, 4>(a, s);
    default: return hipErrorInvalidValue;
  }
}

template <int YB, int STORE>
static hipError_t launch_bp_t(const BpArgs &a, hipStream_t s) {
  using ST = typename StoreT<STORE>::T;
  const int nbx = (a.W + kTX - 1) / kTX;
  const int nbz = (a.Z + kTZ - 1) / kTZ;
  if (a.yb1 <= a.yb0) return hipSuccess;
  const unsigned nb =
      (unsigned)nbx * (unsigned)nbz * (unsigned)(a.yb1 - a.yb0);
  if (a.ndf > 1) {
    hipLaunchKernelGGL((k_bp<YB, STORE, true>), dim3(nb), dim3(kTX * kTZ), 0,
                       s, (const ST *)a.slab, a.coef, a.dscale, a.doffset,
                       a.ndf, a.N, a.T, a.NYB, a.W, a.Z, a.Y, a.yb0, a.y_base, a.slab_yb0,
                       a.vol, nbx, nbz, nb);
  } else if constexpr (STORE == kF32) {
    hipLaunchKernelGGL((k_bp<YB, STORE, false>), dim3(nb), dim3(kTX * kTZ), 0,
                       s, (const ST *)a.slab, a.coef, a.dscale, a.doffset,
                       a.ndf, a.N, a.T, a.NYB, a.W, a.Z, a.Y, a.yb0, a.y_base, a.slab_yb0,
                       a.vol, nbx, nbz, nb);
  } else {
    return hipErrorInvalidValue;  // 16 bits, one slab: launch_bp_mm
  }
  return hipGetLastError();
}

template <int YB, int STORE, bool MULTI, int VZ>
static hipError_t launch_bp_rows_v(const BpArgs &a, size_t tiles,
                                   hipStream_t s) {
  using ST = typename StoreT<STORE>::T;
  const size_t nb = tiles * (YB / 4 / VZ);
  if (nb > 0xffffffffu) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_bp_rows<YB, STORE, MULTI, VZ>), dim3((unsigned)nb),
                     dim3(kTX * kTZ), 0, s, (const ST *)a.slab, a.coef, a.win,
                     a.row_off, a.Y_tab, a.dscale, a.doffset, a.ndf, a.N, a.T,
                     a.NYB, a.W, a.Z, a.Y, a.yb0, a.y_base, a.slab_yb0, a.vol,
                     (a.W + kTX - 1) / kTX, (a.Z + kTZ - 1) / kTZ,
                     (unsigned)nb);
  return hipGetLastError();
}

// A thread takes 4 x YB / 4 voxels, or 4 x 1, of which a tile needs YB / 4
// workgroups: in a small volume few waves run, one after another of a thread's
// loads is waited for, and a partial row block leaves lanes idle. 41 tilts,
// backprojection alone, 4 x 1 over 4 x YB / 4 (and over a lane per voxel
// column): up to 16 tiles times row blocks 0.09 to 0.40 (0.13 to 0.65; without
// it 16-bit slabs took up to 5 times as long), 512 of them 0.33 to 1.04, 2048
// 0.96 to 1.03 (0.14 to 0.71), from 4096 on 1.00 to 1.19. With several 16-bit
// slabs at every size: 0.39 to 0.82 where neighbouring rows' centres lie
// close, 0.96 to 1.01 where they do not.
template <int YB, int STORE>
static hipError_t launch_bp_rows_t(const BpArgs &a, hipStream_t s) {
  if (a.yb1 <= a.yb0) return hipSuccess;
  const size_t tiles = (size_t)((a.W + kTX - 1) / kTX) *
                       ((a.Z + kTZ - 1) / kTZ) * (a.yb1 - a.yb0);
  if (a.ndf > 1) {
    if constexpr (STORE == kF32) {
      if (tiles > kRowTiles)
        return launch_bp_rows_v<YB, STORE, true, YB / 4>(a, tiles, s);
    }
    return launch_bp_rows_v<YB, STORE, true, 1>(a, tiles, s);
  }
  if (tiles > kRowTiles)
    return launch_bp_rows_v<YB, STORE, false, YB / 4>(a, tiles, s);
  return launch_bp_rows_v<YB, STORE, false, 1>(a, tiles, s);
}

hipError_t launch_bp(const BpArgs &a, int YB, int store, hipStream_t s) {
  if (a.mm) return launch_bp_mm(a, YB, store, s);
  if (a.row_off != nullptr) {
    if (store == kF32) {
      if (YB == 8) return launch_bp_rows_t<8, kF32>(a, s);
      if (YB == 16) return launch_bp_rows_t<16, kF32>(a, s);
    } else if (store == kF16) {
      if (YB == 16) return launch_bp_rows_t<16, kF16>(a, s);
      if (YB == 32) return launch_bp_rows_t<32, kF16>(a, s);
    } else if (store == kBF16) {
      if (YB == 16) return launch_bp_rows_t<16, kBF16>(a, s);
      if (YB == 32) return launch_bp_rows_t<32, kBF16>(a, s);
    }
    return hipErrorInvalidValue;
  }
  if (a.staged) {
    if (store == kF32) {
      if (YB == 8) return launch_bp_lds_t<8, kF32>(a, s);
      if (YB == 16) return launch_bp_lds_t<16, kF32>(a, s);
    } else if (store == kF16) {
      if (YB == 16) return launch_bp_lds_t<16, kF16>(a, s);
      if (YB == 32) return launch_bp_lds_t<32, kF16>(a, s);
    } else if (store == kBF16) {
      if (YB == 16) return launch_bp_lds_t<16, kBF16>(a, s);
      if (YB == 32) return launch_bp_lds_t<32, kBF16>(a, s);
    }
    return hipErrorInvalidValue;
  }
  if (store == kF32) {
    if (YB == 1) return launch_bp_slice(a, s);
    if (YB == 8) return launch_bp_t<8, kF32>(a, s);
    if (YB == 16) return launch_bp_t<16, kF32>(a, s);
  } else if (store == kF16) {
    if (YB == 16) return launch_bp_t<16, kF16>(a, s);
    if (YB == 32) return launch_bp_t<32, kF16>(a, s);
  } else if (store == kBF16) {
    if (YB == 16) return launch_bp_t<16, kBF16>(a, s);
    if (YB == 32) return launch_bp_t<32, kBF16>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace gx
