// Dense Linears at the two ends of the refiner forward, for gfx950.
//
//   bf16_linear   out = bf16(A W^T + b) [then bf16(gelu_tanh(out))]: the patch
//                 embedding (the Conv3d with kernel = stride = patch, as a
//                 GEMM, models.py:1551-1552) and the text embedding's two
//                 Linears and their tanh GELU (models.py:1860-1866)
//   linear_f32_modulated
//                 out = xin W^T + b in fp32, xin = f32(A) * s1 + m0: the head's
//                 modulation of its bf16 LayerNorm output and its fp32 Linear
//                 (models.py:1372-1384)
//   gemv_f32      out = x W^T + b in fp32: the time embedding and projection
//                 MLPs (models.py:1845-1849), whose input is one row
//
// Every product is exact and every accumulator is fp32, as torch's GEMMs on
// these dtypes; only the summation order differs.  Epilogues round where
// torch's separate ops round: the bias is added to the fp32 accumulator, the
// result rounds once to the output dtype, and the GELU acts on the rounded
// bf16 value and rounds again.
//
//   head_linear   linear_f32_modulated with bf16 weights on bf16 MFMAs, s1 and m0
//                 formed from the modulation and the timestep embedding
//   time_embed    the time MLP and projection on one timestep, sinusoid included
//
// bf16_linear on contiguous rows of whole 128-byte stages runs on the GEMM of
// fp8.hip, and large bf16-weight heads on the LDS-staged kernel below.  The other
// MFMA kernels here read their operands straight from global memory (L2), without
// LDS staging, for odd layouts, few rows or fp32 weights: one wave's 32-row operand
// slice is re-read by at most two waves of its workgroup.  Lanes 0-31 of an MFMA
// operand hold rows 0-31 of k-slice [k0, k0+8), lanes 32-63 the same rows at
// [k0+8, k0+16): a k index is paired the same way in A and W, so the sum over k is
// the GEMM's.
#include "common.h"

namespace srdit {
namespace {

typedef float f32x8v __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float x) {
  typedef float f32x2v __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
  return (uint16_t)__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2v{x, 0.f}, bf16x2v));
}

template <typename T>
__device__ __forceinline__ f32x8v load8_f32(const T* p);

template <>
__device__ __forceinline__ f32x8v load8_f32<float>(const float* p) {
  const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(p);
  const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(p + 4);
  return f32x8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

__device__ __forceinline__ f32x8v unpack_bf16x8(const uint4 v) {
  const uint32_t u[4] = {v.x, v.y, v.z, v.w};
  f32x8v f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(u[i] << 16);
    f[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
  }
  return f;
}

template <>
__device__ __forceinline__ f32x8v load8_f32<uint16_t>(const uint16_t* p) {
  return unpack_bf16x8(*reinterpret_cast<const uint4*>(p));
}

template <typename WT>
__device__ __forceinline__ float load1_f32(const WT* p, int i);
template <>
__device__ __forceinline__ float load1_f32<float>(const float* p, int i) { return p[i]; }
template <>
__device__ __forceinline__ float load1_f32<uint16_t>(const uint16_t* p, int i) {
  return bf16_bits_to_f32(p[i]);
}

// ---------------------------------------------------------------------------
// Tiling shared by the two GEMMs.  A wave owns a 32-row x 64-column output
// tile as two 32x32 MFMA accumulators (columns 0-31 and 32-63).  The MFMAs take
// W as their first operand and the activations as their second, so register v
// of lane l holds row l%32, column 32 t + 8 (v/4) + 4 (l/32) + v%4: four
// consecutive columns per register group.  A workgroup is 4 waves: with KS = 1
// they stack along rows (a 128 x 64 tile); with KS = 4 they share one 32 x 64
// tile and each sums a quarter of the k-steps (for grids too small to fill the
// chip, e.g. 512-row GEMMs).  The epilogue goes through LDS: each wave writes
// its accumulators as an fp32 tile, and the rows are read back 8 columns per
// lane (the KS partials summed in wave order, so results do not depend on
// timing) and stored as 16-byte pieces.
constexpr int WT_M = 32, WT_N = 64;
constexpr int EPI_LD = WT_N + 4;   // fp32 row stride of an LDS tile: rows start 4 banks apart
constexpr int EPI_TILE = WT_M * EPI_LD;
constexpr int RING = 4;            // k-steps of operands in flight per wave

__device__ __forceinline__ void acc_to_lds(float* tile, const f32x16_t& c0, const f32x16_t& c1,
                                           int lane) {
  float* row = tile + (lane & 31) * EPI_LD + 4 * (lane >> 5);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    *reinterpret_cast<f32x4_t*>(row + 8 * g) = f32x4_t{c0[4 * g], c0[4 * g + 1], c0[4 * g + 2], c0[4 * g + 3]};
    *reinterpret_cast<f32x4_t*>(row + 32 + 8 * g) =
        f32x4_t{c1[4 * g], c1[4 * g + 1], c1[4 * g + 2], c1[4 * g + 3]};
  }
}

template <typename OT>
__device__ __forceinline__ void store8(OT* p, const float v[8]);

template <>
__device__ __forceinline__ void store8<uint16_t>(uint16_t* p, const float v[8]) {
  uint32_t u[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    u[i] = (uint32_t)f32_to_bf16_bits(v[2 * i]) | ((uint32_t)f32_to_bf16_bits(v[2 * i + 1]) << 16);
  *reinterpret_cast<uint4*>(p) = make_uint4(u[0], u[1], u[2], u[3]);
}

template <>
__device__ __forceinline__ void store8<float>(float* p, const float v[8]) {
  *reinterpret_cast<f32x4_t*>(p) = f32x4_t{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
}

// The first nv (< 8, or rows not 16-byte aligned) values one at a time.
__device__ __forceinline__ void store1(uint16_t* p, float v) { *p = f32_to_bf16_bits(v); }
__device__ __forceinline__ void store1(float* p, float v) { *p = v; }

// After the LDS tiles are written and a barrier: wave w stores its own tile's
// 32 rows (KS = 1) or rows 8w..8w+7 of the shared tile (KS = 4).  Lane l takes
// row l/8 of each 8-row group, columns 8 (l%8) .. +8, as one 16-byte store
// where the piece is whole and the rows are 16-byte aligned (vec_out), else
// value by value (the last piece of a row whose length is not a multiple of 8).
template <int KS, int GELU, typename OT, typename BT>
__device__ __forceinline__ void epilogue(const float* lds, int wave, int lane, int m_tile, int n0,
                                         int M, int N, const BT* __restrict__ bias,
                                         OT* __restrict__ out, int64_t ldo, bool vec_out) {
  const int c = lane & 7, rr = lane >> 3;
  const int n = n0 + 8 * c;
  if (n >= N) return;
  const int nv = N - n < 8 ? N - n : 8;  // columns of this piece inside the matrix
  f32x8v b = {};
  if (bias) {
    if (nv == 8 && (reinterpret_cast<uintptr_t>(bias) & 15) == 0) {  // uniform
      b = load8_f32<BT>(bias + n);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = i < nv ? load1_f32<BT>(bias, n + i) : 0.f;
    }
  }
#pragma unroll
  for (int q = 0; q < (KS == 1 ? 4 : 1); ++q) {
    const int r = KS == 1 ? 8 * q + rr : 8 * wave + rr;
    const int m = m_tile + r;
    if (m >= M) break;   // rows only grow with q
    const float* src = lds + (KS == 1 ? wave : 0) * EPI_TILE + r * EPI_LD + 8 * c;
    f32x4_t lo = *reinterpret_cast<const f32x4_t*>(src);
    f32x4_t hi = *reinterpret_cast<const f32x4_t*>(src + 4);
#pragma unroll
    for (int p = 1; p < KS; ++p) {
      lo += *reinterpret_cast<const f32x4_t*>(src + p * EPI_TILE);
      hi += *reinterpret_cast<const f32x4_t*>(src + p * EPI_TILE + 4);
    }
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] += b[i];
      if (GELU) v[i] = gelu_tanh(bf16_rt(v[i]));
    }
    OT* dst = out + (int64_t)m * ldo + n;
    if (vec_out && nv == 8) {
      store8<OT>(dst, v);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < nv) store1(dst + i, v[i]);
    }
  }
}

// ---------------------------------------------------------------------------
// bf16 x bf16 -> fp32 accumulators -> bf16 (32x32x16 bf16 MFMAs).
template <int GELU, int KS>
__global__ __launch_bounds__(256) void bf16_linear_kernel(
    const uint16_t* __restrict__ a, int64_t lda, const uint16_t* __restrict__ w, int64_t ldw,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int64_t ldo, int M, int N,
    int K, bool vec_out) {
  __shared__ __attribute__((aligned(16))) float lds[4 * EPI_TILE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m_tile = blockIdx.y * (KS == 1 ? 4 * WT_M : WT_M) + (KS == 1 ? WT_M * wave : 0);
  const int n0 = blockIdx.x * WT_N;
  const int r = lane & 31, kh = (lane >> 5) * 8;
  // rows past the end read the last row (in bounds); their results are not stored
  const bf16x8_t* pa = reinterpret_cast<const bf16x8_t*>(a + (int64_t)min(m_tile + r, M - 1) * lda + kh);
  const bf16x8_t* pw0 = reinterpret_cast<const bf16x8_t*>(w + (int64_t)min(n0 + r, N - 1) * ldw + kh);
  const bf16x8_t* pw1 =
      reinterpret_cast<const bf16x8_t*>(w + (int64_t)min(n0 + 32 + r, N - 1) * ldw + kh);
  const int steps = K / 16;
  const int s_begin = KS == 1 ? 0 : wave * (steps / KS);
  const int s_end = KS == 1 ? steps : s_begin + steps / KS;
  const int groups = (s_end - s_begin) / RING;
  f32x16_t c0 = {}, c1 = {};
  bf16x8_t ra[RING], rw0[RING], rw1[RING];
  if (groups > 0) {
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      const int s = s_begin + j;
      ra[j] = pa[2 * s]; rw0[j] = pw0[2 * s]; rw1[j] = pw1[2 * s];
      __builtin_amdgcn_sched_barrier(0);   // slot by slot, as the refills
    }
    for (int g = 0; g < groups; ++g) {
#pragma unroll
      for (int j = 0; j < RING; ++j) {
        c0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rw0[j], ra[j], c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rw1[j], ra[j], c1, 0, 0, 0);
        const int s = min(s_begin + (g + 1) * RING + j, s_end - 1);   // past the end: reload
        ra[j] = pa[2 * s]; rw0[j] = pw0[2 * s]; rw1[j] = pw1[2 * s];
        // keep the refill here: clustered at the end of the group, the loads
        // would be waited for a few MFMAs after their issue
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (int s = s_begin + groups * RING; s < s_end; ++s) {
    const bf16x8_t va = pa[2 * s];
    c0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pw0[2 * s], va, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pw1[2 * s], va, c1, 0, 0, 0);
  }
  acc_to_lds(lds + wave * EPI_TILE, c0, c1, lane);
  __syncthreads();
  epilogue<KS, GELU, uint16_t, uint16_t>(lds, wave, lane, m_tile, n0, M, N, bias, out, ldo,
                                         vec_out);
}

// ---------------------------------------------------------------------------
// fp32 GEMM with the head's modulation applied to its bf16 input as it is
// read: xin = (f32(a) * s1[k]) + m0[k], rounded after the product and after the
// sum (torch's two elementwise kernels), as 32x32x2 fp32 MFMAs.
__device__ __forceinline__ float modulate(float x, float s1, float m0) {
#pragma clang fp contract(off)
  return x * s1 + m0;
}

template <typename WT>
struct WChunk;  // the raw 8 weights of one lane's k-slice
template <>
struct WChunk<uint16_t> {
  uint4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ f32x8v get() const { return unpack_bf16x8(v); }
};
template <>
struct WChunk<float> {
  f32x4_t lo, hi;
  __device__ __forceinline__ void load(const float* p) {
    lo = *reinterpret_cast<const f32x4_t*>(p);
    hi = *reinterpret_cast<const f32x4_t*>(p + 4);
  }
  __device__ __forceinline__ f32x8v get() const {
    return f32x8v{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
};

struct ModChunk {
  uint4 a;
  f32x4_t s_lo, s_hi, m_lo, m_hi;
  __device__ __forceinline__ void load(const uint16_t* pa, const float* s1, const float* m0) {
    a = *reinterpret_cast<const uint4*>(pa);
    s_lo = *reinterpret_cast<const f32x4_t*>(s1);
    s_hi = *reinterpret_cast<const f32x4_t*>(s1 + 4);
    m_lo = *reinterpret_cast<const f32x4_t*>(m0);
    m_hi = *reinterpret_cast<const f32x4_t*>(m0 + 4);
  }
};

template <typename WT>
__device__ __forceinline__ void mod_step(f32x16_t& c0, f32x16_t& c1, const ModChunk& x,
                                         const WChunk<WT>& w0, const WChunk<WT>& w1) {
  const f32x8v xa = unpack_bf16x8(x.a);
  const float sv[8] = {x.s_lo[0], x.s_lo[1], x.s_lo[2], x.s_lo[3], x.s_hi[0], x.s_hi[1], x.s_hi[2], x.s_hi[3]};
  const float mv[8] = {x.m_lo[0], x.m_lo[1], x.m_lo[2], x.m_lo[3], x.m_hi[0], x.m_hi[1], x.m_hi[2], x.m_hi[3]};
  const f32x8v b0 = w0.get(), b1 = w1.get();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float xin = modulate(xa[i], sv[i], mv[i]);
    c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(b0[i], xin, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_32x32x2f32(b1[i], xin, c1, 0, 0, 0);
  }
}

template <typename WT, int KS>
__global__ __launch_bounds__(256) void linear_f32_modulated_kernel(
    const uint16_t* __restrict__ a, int64_t lda, const float* __restrict__ s1,
    const float* __restrict__ m0, const WT* __restrict__ w, int64_t ldw,
    const WT* __restrict__ bias, float* __restrict__ out, int64_t ldo, int M, int N, int K,
    bool vec_out) {
  __shared__ __attribute__((aligned(16))) float lds[4 * EPI_TILE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m_tile = blockIdx.y * (KS == 1 ? 4 * WT_M : WT_M) + (KS == 1 ? WT_M * wave : 0);
  const int n0 = blockIdx.x * WT_N;
  const int r = lane & 31, kh = (lane >> 5) * 8;
  const uint16_t* pa = a + (int64_t)min(m_tile + r, M - 1) * lda + kh;
  const WT* pw0 = w + (int64_t)min(n0 + r, N - 1) * ldw + kh;
  const WT* pw1 = w + (int64_t)min(n0 + 32 + r, N - 1) * ldw + kh;
  const float* ps = s1 + kh;
  const float* pm = m0 + kh;
  const int steps = K / 16;
  const int s_begin = KS == 1 ? 0 : wave * (steps / KS);
  const int s_end = KS == 1 ? steps : s_begin + steps / KS;
  const int groups = (s_end - s_begin) / RING;
  f32x16_t c0 = {}, c1 = {};
  ModChunk rx[RING];
  WChunk<WT> rw0[RING], rw1[RING];
  if (groups > 0) {
#pragma unroll
    for (int j = 0; j < RING; ++j) {
      const int k = 16 * (s_begin + j);
      rx[j].load(pa + k, ps + k, pm + k);
      rw0[j].load(pw0 + k);
      rw1[j].load(pw1 + k);
      __builtin_amdgcn_sched_barrier(0);   // slot by slot, as the refills
    }
    for (int g = 0; g < groups; ++g) {
#pragma unroll
      for (int j = 0; j < RING; ++j) {
        mod_step<WT>(c0, c1, rx[j], rw0[j], rw1[j]);
        const int k = 16 * min(s_begin + (g + 1) * RING + j, s_end - 1);
        rx[j].load(pa + k, ps + k, pm + k);
        rw0[j].load(pw0 + k);
        rw1[j].load(pw1 + k);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (int s = s_begin + groups * RING; s < s_end; ++s) {
    ModChunk x;
    WChunk<WT> w0, w1;
    x.load(pa + 16 * s, ps + 16 * s, pm + 16 * s);
    w0.load(pw0 + 16 * s);
    w1.load(pw1 + 16 * s);
    mod_step<WT>(c0, c1, x, w0, w1);
  }
  acc_to_lds(lds + wave * EPI_TILE, c0, c1, lane);
  __syncthreads();
  epilogue<KS, 0, float, WT>(lds, wave, lane, m_tile, n0, M, N, bias, out, ldo, vec_out);
}

// ---------------------------------------------------------------------------
// The same product for bf16 weights on bf16 MFMAs, without rounding anything the
// fp32 MFMAs keep: xin is cut into three bf16 pieces of 8 significant bits each
// (its leading bits, those of the remainder, and the rest, all exact), every
// product of a piece with a bf16 weight is exact in fp32, and the sums stay fp32
// (the leading pieces in one accumulator, the others in a second).  An infinite
// xin keeps its infinity in the leading piece and zeros in the others; a NaN
// stays one.  Three bf16 MFMAs do the work of sixteen times as many fp32 ones.
//
// A workgroup owns 64 rows and 32 NT columns.  Its eight wavefronts are two row
// halves times four slices of 16 k in every 64-k stage, so each element of xin is
// formed and cut once and two wavefronts share a SIMD; the slices' sums meet in
// LDS at the end, in slice order.  Stages (128-byte rows, 16-byte chunk c of row r
// at c ^ ((r >> 1) & 7), which keeps the fragment reads of 16 lanes on distinct
// banks) stream through a ring of HM_NST; the next stage's fragments are read and
// cut while this one is multiplied.  s1 and m0 sit in LDS for the whole walk.  The
// weights are the MFMA's first operand: a lane holds runs of four columns of one row.
// Bound by its own chain: about 0.97 us per stage, 0.55 of it MFMAs (one workgroup
// per CU, 169 of them at 10800 rows); without the cut it is 0.82 us.
// Measured against the fp32 MFMAs, N = 192, K = 3072: 10800 rows 124.5 -> 59.0 us,
// 21600 rows 227.6 -> 115.6, 3000 rows 62.2 -> 54.8; relative error against 64
// bits 4.0e-7 -> 2.4e-7 (the sums are four chains of 48 x 3 additions, not of 384).
constexpr int HM_NST = 3;
constexpr int HM_ROWS = 64;
constexpr int HM_MAX_K = 4096;  // s1 and m0 take 8 K bytes of LDS

// Where s1 and m0 come from: given, or (mod != null) the head's adaLN vectors
// m0 = f32(mod[0]) + e and s1 = 1 + (f32(mod[1]) + e), rounded after each sum.
struct ModSource {
  const float* s1;
  const float* m0;
  const void* mod;  // [2, K], bf16 or fp32
  const float* e;   // [K]
  int mod_bf16;
};

__device__ __forceinline__ i32x4_t raw_rsrc(const void* p, int64_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return i32x4_t{static_cast<int>(static_cast<uint32_t>(a)),
                 static_cast<int>(static_cast<uint32_t>(a >> 32)), static_cast<int>(bytes),
                 0x00020000};
}

// 16 bytes per lane to LDS at lds + 16 lane; the compiler does not see the LDS
// write, so callers wait and synchronise before they read it.
__device__ __forceinline__ void dma16(i32x4_t rsrc, int voff, int soff, uint32_t lds) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(rsrc), "s"(soff),
               "{m0}"(lds)
               : "memory");
}

// At most N vector-memory operations in flight, LDS reads retired, then a barrier.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

struct Cut3 {
  bf16x8_t hi, mid, lo;
};

__device__ __forceinline__ uint32_t top_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// Eight bf16 of a row -> xin -> its three pieces.
__device__ __forceinline__ Cut3 modulate_cut(const i32x4_t a, const float* s1, const float* m0) {
#pragma clang fp contract(off)
  i32x4_t hi, mid, lo;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t w = static_cast<uint32_t>(a[p]);
    float x[2] = {__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
    float r[2], t[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x[i] = x[i] * s1[2 * p + i] + m0[2 * p + i];
      const float h = __uint_as_float(__float_as_uint(x[i]) & 0xffff0000u);
      r[i] = __builtin_fabsf(x[i]) == INFINITY ? 0.f : x[i] - h;
      t[i] = r[i] - __uint_as_float(__float_as_uint(r[i]) & 0xffff0000u);
    }
    hi[p] = static_cast<int>(top_halves(x[0], x[1]));
    mid[p] = static_cast<int>(top_halves(r[0], r[1]));
    lo[p] = static_cast<int>(top_halves(t[0], t[1]));
  }
  return Cut3{__builtin_bit_cast(bf16x8_t, hi), __builtin_bit_cast(bf16x8_t, mid),
              __builtin_bit_cast(bf16x8_t, lo)};
}

template <int NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void linear_f32_cut_kernel(const uint16_t* __restrict__ a, int64_t lda, ModSource ms,
                           const uint16_t* __restrict__ w, int64_t ldw,
                           const uint16_t* __restrict__ bias, float* __restrict__ out, int64_t ldo,
                           int M, int N, int K, bool vec_out) {
  constexpr int KB = 128;                          // bytes of k per stage
  constexpr int STAGE = (32 * NT + HM_ROWS) * KB;
  constexpr int WD = NT / 2;                       // weight DMAs per wavefront per stage
  constexpr int FILLS = WD + 1;
  constexpr int PART = 32 * 32 * NT;               // floats of one wavefront's sums
  constexpr int RING = HM_NST * STAGE > 4 * PART * 4 ? HM_NST * STAGE : 4 * PART * 4;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[RING + 8 * HM_MAX_K];
  float* ls1 = reinterpret_cast<float*>(smem + RING);
  float* lm0 = ls1 + K;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave & 1, slice = wave >> 1;
  const int m_base = blockIdx.y * HM_ROWS, n_base = blockIdx.x * 32 * NT;

  // Rows past the end read as zero through the descriptors' range check.
  const int rows = min(HM_ROWS, M - m_base), cols = min(32 * NT, N - n_base);
  const i32x4_t ra = raw_rsrc(a + (int64_t)m_base * lda, ((int64_t)(rows - 1) * lda + K) * 2);
  const i32x4_t rw = raw_rsrc(w + (int64_t)n_base * ldw, ((int64_t)(cols - 1) * ldw + K) * 2);
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
  // A DMA writes 8 rows of 128 bytes: lane l -> row l/8, position l%8 holding source
  // chunk (l%8) ^ ((row >> 1) & 7).  Wavefront w: activation rows [8 w, +8) and
  // weight rows [8 WD w, +8 WD).
  const int fr = lane >> 3, fp = lane & 7;
  auto fill = [&](int s, int slot) __attribute__((always_inline)) {
    const uint32_t base = lds_base + slot * STAGE;
#pragma unroll
    for (int q = 0; q < WD; ++q) {
      const int r = wave * 8 * WD + 8 * q + fr;
      const int off = r < cols ? (int)(r * ldw * 2) + ((fp ^ ((r >> 1) & 7)) * 16) : (int)0x80000000;
      dma16(rw, off, s * KB, base + (wave * 8 * WD + 8 * q) * KB);
    }
    const int r = wave * 8 + fr;
    const int off = r < rows ? (int)(r * lda * 2) + ((fp ^ ((r >> 1) & 7)) * 16) : (int)0x80000000;
    dma16(ra, off, s * KB, base + (32 * NT + wave * 8) * KB);
  };
  const int nst = K / 64;
#pragma unroll
  for (int s = 0; s < HM_NST; ++s)
    if (s < nst) fill(s, s);
  for (int k = threadIdx.x; k < K; k += 512) {
    if (ms.mod) {
      const float b0 = ms.mod_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(ms.mod)[k])
                                   : static_cast<const float*>(ms.mod)[k];
      const float b1 = ms.mod_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(ms.mod)[K + k])
                                   : static_cast<const float*>(ms.mod)[K + k];
      ls1[k] = 1.f + (b1 + ms.e[k]);
      lm0[k] = b0 + ms.e[k];
    } else {
      ls1[k] = ms.s1[k];
      lm0[k] = ms.m0[k];
    }
  }

  // Fragments of this wavefront's 16 k: lane l holds row l%32, k 8 (l/32) .. +8:
  // chunk 2 slice + l/32 of the row.
  const int frow = lane & 31, fg = lane >> 5;
  const int foff = frow * KB + (((2 * slice + fg) ^ ((frow >> 1) & 7)) * 16);
  const int kl = 16 * slice + 8 * fg;
  struct Frag {
    bf16x8_t w[NT];
    Cut3 x;
  };
  struct Raw {
    i32x4_t a;
    float s1[8], m0[8];
  };
  auto read = [&](int s, int slot, bf16x8_t (&wf)[NT]) __attribute__((always_inline)) -> Raw {
    const uint8_t* base = smem + slot * STAGE + foff;
    Raw r;
    r.a = *reinterpret_cast<const i32x4_t*>(base + (32 * NT + 32 * half) * KB);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4_t s4 = *reinterpret_cast<const f32x4_t*>(ls1 + 64 * s + kl + 4 * h);
      const f32x4_t m4 = *reinterpret_cast<const f32x4_t*>(lm0 + 64 * s + kl + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i) { r.s1[4 * h + i] = s4[i]; r.m0[4 * h + i] = m4[i]; }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) wf[t] = *reinterpret_cast<const bf16x8_t*>(base + 32 * t * KB);
    return r;
  };
  f32x16_t acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x16_t{};
  auto mma = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[t], f.x.lo, acc[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[t], f.x.mid, acc[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[t], f.x.hi, acc[t], 0, 0, 0);
  };
  __syncthreads();   // s1 and m0 are written
  stage_barrier<0>();  // the first stages landed
  Frag f0;
  {
    const Raw r = read(0, 0, f0.w);
    f0.x = modulate_cut(r.a, r.s1, r.m0);
  }
  int slot = 0;
  auto step = [&](int s, const Frag& fc, Frag& fn) __attribute__((always_inline)) {
    // stage s + 1 landed everywhere; stage s is in registers, its slot takes s + NST
    if (s + HM_NST - 1 < nst) stage_barrier<(HM_NST - 2) * FILLS>();
    else stage_barrier<0>();
    if (s + HM_NST < nst) fill(s + HM_NST, slot);
    slot = slot == HM_NST - 1 ? 0 : slot + 1;
    const Raw r = read(s + 1 < nst ? s + 1 : s, slot, fn.w);  // after the last stage: not used
    __builtin_amdgcn_sched_barrier(0);
    mma(fc);
    fn.x = modulate_cut(r.a, r.s1, r.m0);
    // the first MFMAs cover the reads' latency; the cut's vector operations then
    // fill the matrix pipe's 32 cycles per MFMA
    __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);     // MFMAs
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);  // nine VALU
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  Frag f1;
  int s = 0;
  for (; s + 1 < nst; s += 2) {
    step(s, f0, f1);
    step(s + 1, f1, f0);
  }
  if (s < nst) step(s, f0, f1);

  // The slices' sums: 2 and 3 to LDS, 0 and 1 add them; then 1 to LDS and 0 adds it.
  stage_barrier<0>();
  f32x4_t* part = reinterpret_cast<f32x4_t*>(smem);
  auto at = [&](int p, int t, int g) __attribute__((always_inline)) -> f32x4_t& {
    return part[((p * NT + t) * 4 + g) * 64 + lane];
  };
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    const int lo = round == 0 ? 2 : 1;  // slices [lo, 2 lo) are written, [0, lo) add them
    if (slice >= lo && slice < 2 * lo) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          at(2 * (slice - lo) + half, t, g) =
              f32x4_t{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
    }
    __syncthreads();
    if (slice < lo) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4_t v = at(2 * slice + half, t, g);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][4 * g + i] += v[i];
        }
    }
    __syncthreads();
  }
  // lane l: row l%32 of the half, columns 32 t + 8 g + 4 (l/32) .. +4
  const int m = m_base + 32 * half + frow;
  if (slice != 0 || m >= M) return;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n_base + 32 * t + 8 * g + 4 * fg;
      float* dst = out + (int64_t)m * ldo + n;
      f32x4_t v = {acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
      if (n + 4 <= N && vec_out) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += bias ? bf16_bits_to_f32(bias[n + i]) : 0.f;
        *reinterpret_cast<f32x4_t*>(dst) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) dst[i] = v[i] + (bias ? bf16_bits_to_f32(bias[n + i]) : 0.f);
      }
    }
}

// ---------------------------------------------------------------------------
// fp32 GEMV rows: out[m, n] = sum_k x[m, k] w[n, k] + b[n].  One wave per
// output (4 per workgroup); the lanes stride the row 8 elements at a time and
// the 64 partial sums reduce across the wave.
template <typename WT>
__device__ __forceinline__ float wave_dot(const float* x, const WT* __restrict__ w, int K, int lane) {
  float acc = 0.f;
  for (int k = lane * 8; k < K; k += 512) {
    const f32x8v xv = load8_f32<float>(x + k);
    const f32x8v wv = load8_f32<WT>(w + k);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = __builtin_fmaf(xv[i], wv[i], acc);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
  return acc;
}

// x / (1 + e^-x), as torch's fp32 silu.
__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + expf(-x)); }

// SILU: silu_out (beside out, which may be null) takes the result's silu.
template <typename WT, bool SILU>
__global__ __launch_bounds__(256) void gemv_f32_kernel(const float* __restrict__ x, int64_t ldx,
                                                       const WT* __restrict__ w, int64_t ldw,
                                                       const WT* __restrict__ bias,
                                                       float* __restrict__ out, int64_t ldo,
                                                       int N, int K, float* __restrict__ silu_out) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;  // whole waves: no barrier follows
  const int m = blockIdx.y;
  const float acc = wave_dot<WT>(x + (int64_t)m * ldx, w + (int64_t)n * ldw, K, lane);
  if (lane == 0) {
    const float v = acc + (bias ? load1_f32<WT>(bias, n) : 0.f);
    if (out) out[(int64_t)m * ldo + n] = v;
    if (SILU) silu_out[n] = silu_f32(v);
  }
}

// silu of the time MLP's first Linear on the sinusoid of one timestep.  Every
// workgroup forms the sinusoid in LDS, in 64 bits as the reference does (cos of
// t 10000^(-i / half), then sin, rounded to fp32), and takes TE_OUT outputs per
// wave, so that work is repeated 192 times at dim 3072, not 768.
constexpr int TE_OUT = 4;
constexpr int TE_MAX_FREQ = 2048;

template <typename WT>
__global__ __launch_bounds__(256) void time_sinusoid_gemv_kernel(
    const float* __restrict__ t, int freq, const WT* __restrict__ w, const WT* __restrict__ bias,
    float* __restrict__ silu_out, int N) {
  __shared__ __attribute__((aligned(16))) float x[TE_MAX_FREQ];
  const int half = freq / 2;
  const double pos = static_cast<double>(t[0]);
  for (int i = threadIdx.x; i < half; i += 256) {
    const double ang = pos * pow(10000.0, -static_cast<double>(i) / static_cast<double>(half));
    x[i] = static_cast<float>(cos(ang));
    x[half + i] = static_cast<float>(sin(ang));
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * TE_OUT;
  for (int n = n0; n < min(n0 + TE_OUT, N); ++n) {
    const float acc = wave_dot<WT>(x, w + (int64_t)n * freq, freq, lane);
    if (lane == 0) silu_out[n] = silu_f32(acc + (bias ? load1_f32<WT>(bias, n) : 0.f));
  }
}

bool aligned_rows16(const void* p, int64_t ld, int elem) {
  return aligned16(p) && (ld * elem) % 16 == 0;
}

}  // namespace
}  // namespace srdit

using namespace srdit;

namespace srdit {
namespace {

// Split k over the workgroup's 4 waves when 128 x 64 tiles would leave the
// grid under two workgroups per CU and every wave gets whole groups of steps.
int pick_ks(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 4 * WT_M - 1) / (4 * WT_M)) * ((N + WT_N - 1) / WT_N);
  const int64_t steps = K / 16;
  return (steps % 4 == 0 && steps >= 16 && tiles < 512) ? 4 : 1;
}

// bf16 weights over whole 64-k stages with s1 and m0 in LDS: the cut-operand kernel
// can take them.
bool cut_fits(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldw, int w_dtype) {
  return w_dtype == SRDIT_DTYPE_BF16 && K % 64 == 0 && K <= HM_MAX_K &&
         M <= 65535LL * HM_ROWS && HM_ROWS * lda * 2 < (1LL << 31) && 192 * ldw * 2 < (1LL << 31);
}

// It takes about 52 us for up to 256 workgroups (K = 3072, N = 192), the fp32
// kernel 34 us below 1000 rows and 62 us at 3000; with 64 columns 31 us against
// 34 at any row count.
bool cut_pays(int64_t M, int64_t N) { return N <= 64 || M * ((N + 191) / 192) >= 2560; }

void launch_cut(const void* a, int64_t lda, const ModSource& ms, const void* w, int64_t ldw,
                const void* bias, float* out, int64_t ldo, int64_t M, int64_t N, int64_t K,
                hipStream_t s) {
  const bool vec_out = aligned_rows16(out, ldo, 4);
  const uint16_t* ap = static_cast<const uint16_t*>(a);
  const uint16_t* wp = static_cast<const uint16_t*>(w);
  const uint16_t* bp = static_cast<const uint16_t*>(bias);
  const unsigned gy = (unsigned)((M + HM_ROWS - 1) / HM_ROWS);
  if (N <= 64)
    linear_f32_cut_kernel<2><<<dim3(1, gy), 512, 0, s>>>(ap, lda, ms, wp, ldw, bp, out, ldo,
                                                         (int)M, (int)N, (int)K, vec_out);
  else
    linear_f32_cut_kernel<6><<<dim3((unsigned)((N + 191) / 192), gy), 512, 0, s>>>(
        ap, lda, ms, wp, ldw, bp, out, ldo, (int)M, (int)N, (int)K, vec_out);
}

dim3 dense_grid(int64_t M, int64_t N, int ks) {
  const int64_t rows = ks == 1 ? 4 * WT_M : WT_M;
  return dim3((unsigned)((N + WT_N - 1) / WT_N), (unsigned)((M + rows - 1) / rows));
}

}  // namespace
}  // namespace srdit

extern "C" int srdit_bf16_linear(const void* a, int64_t lda, const void* w, int64_t ldw,
                                 const void* bias, void* out, int64_t ldo, int64_t M, int64_t N,
                                 int64_t K, int epilogue, void* stream) {
  const char* fn = "srdit_bf16_linear";
  SRDIT_REQUIRE(a && w && out, "%s: null operand", fn);
  SRDIT_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                "%s: bad sizes M=%lld N=%lld K=%lld", fn, (long long)M, (long long)N,
                (long long)K);
  SRDIT_REQUIRE(K % 16 == 0, "%s: K=%lld must be a multiple of 16", fn, (long long)K);
  SRDIT_REQUIRE(lda >= K && ldw >= K && ldo >= N, "%s: leading dimensions below the row length",
                fn);
  SRDIT_REQUIRE(aligned_rows16(a, lda, 2) && aligned_rows16(w, ldw, 2),
                "%s: A and W rows must be 16-byte aligned", fn);
  SRDIT_REQUIRE((reinterpret_cast<uintptr_t>(out) & 1) == 0 &&
                    (!bias || (reinterpret_cast<uintptr_t>(bias) & 1) == 0),
                "%s: misaligned bf16 output or bias", fn);
  const bool vec_out = aligned_rows16(out, ldo, 2);
  SRDIT_REQUIRE(epilogue == 0 || epilogue == 1, "%s: epilogue %d is not 0 (none) or 1 (gelu)", fn,
                epilogue);
  // Contiguous rows in whole 128-byte K stages take the LDS-pipelined GEMM
  // (fp8.hip, bf16 operands: persistent on large grids, small tiles on small
  // ones); the rest (odd layouts and widths) the kernel here.  512 x 3072 x 4096
  // runs 80.5 us on the kernel here and 24.7 us there.
  if (K % 64 == 0 && N % 16 == 0 && lda == K && ldw == K && aligned16(bias) &&
      aligned_rows16(out, ldo, 2) &&
      M * K * 2 < (1LL << 31) && N * K * 2 < (1LL << 31) && (255 * ldo + N) * 2 + 16 < (1LL << 31))
    return bf16_gemm_persistent(a, w, bias, out, M, N, K, ldo, epilogue, stream, fn);
  const int ks = pick_ks(M, N, K);
  const dim3 grid = dense_grid(M, N, ks);
  SRDIT_REQUIRE(grid.y < 65536u * 16, "%s: M=%lld too large", fn, (long long)M);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* ap = static_cast<const uint16_t*>(a);
  const uint16_t* wp = static_cast<const uint16_t*>(w);
  const uint16_t* bp = static_cast<const uint16_t*>(bias);
  uint16_t* op = static_cast<uint16_t*>(out);
#define SRDIT_BL(G, KS)                                                                      \
  bf16_linear_kernel<G, KS><<<grid, 256, 0, s>>>(ap, lda, wp, ldw, bp, op, ldo, (int)M, (int)N, \
                                                 (int)K, vec_out)
  if (epilogue && ks == 4) SRDIT_BL(1, 4);
  else if (epilogue) SRDIT_BL(1, 1);
  else if (ks == 4) SRDIT_BL(0, 4);
  else SRDIT_BL(0, 1);
#undef SRDIT_BL
  SRDIT_LAUNCH_CHECK("bf16_linear_kernel");
  return SRDIT_OK;
}

extern "C" int srdit_linear_f32_modulated(const void* a, int64_t lda, const float* s1,
                                          const float* m0, const void* w, int64_t ldw,
                                          const void* bias, int w_dtype, float* out, int64_t ldo,
                                          int64_t M, int64_t N, int64_t K, void* stream) {
  const char* fn = "srdit_linear_f32_modulated";
  SRDIT_REQUIRE(a && s1 && m0 && w && out, "%s: null operand", fn);
  SRDIT_REQUIRE(w_dtype == SRDIT_DTYPE_BF16 || w_dtype == SRDIT_DTYPE_FP32,
                "%s: w_dtype %d is not bf16 (0) or fp32 (2)", fn, w_dtype);
  SRDIT_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                "%s: bad sizes M=%lld N=%lld K=%lld", fn, (long long)M, (long long)N,
                (long long)K);
  SRDIT_REQUIRE(K % 16 == 0, "%s: K=%lld must be a multiple of 16", fn, (long long)K);
  SRDIT_REQUIRE(lda >= K && ldw >= K && ldo >= N, "%s: leading dimensions below the row length",
                fn);
  const int welem = w_dtype == SRDIT_DTYPE_FP32 ? 4 : 2;
  SRDIT_REQUIRE(aligned_rows16(a, lda, 2) && aligned_rows16(w, ldw, welem) && aligned16(s1) &&
                    aligned16(m0),
                "%s: A, W, s1 and m0 must be 16-byte aligned (rows included)", fn);
  SRDIT_REQUIRE((reinterpret_cast<uintptr_t>(out) & 3) == 0 &&
                    (!bias || (reinterpret_cast<uintptr_t>(bias) & (welem - 1)) == 0),
                "%s: misaligned output or bias", fn);
  const bool vec_out = aligned_rows16(out, ldo, 4);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (cut_fits(M, N, K, lda, ldw, w_dtype) && cut_pays(M, N)) {
    launch_cut(a, lda, ModSource{s1, m0, nullptr, nullptr, 0}, w, ldw, bias, out, ldo, M, N, K, s);
    SRDIT_LAUNCH_CHECK("linear_f32_cut_kernel");
    return SRDIT_OK;
  }
  const int ks = pick_ks(M, N, K);
  const dim3 grid = dense_grid(M, N, ks);
  SRDIT_REQUIRE(grid.y < 65536u * 16, "%s: M=%lld too large", fn, (long long)M);
  const uint16_t* ap = static_cast<const uint16_t*>(a);
#define SRDIT_LF(WT, KS)                                                                        \
  linear_f32_modulated_kernel<WT, KS><<<grid, 256, 0, s>>>(ap, lda, s1, m0,                     \
                                                           static_cast<const WT*>(w), ldw,      \
                                                           static_cast<const WT*>(bias), out,   \
                                                           ldo, (int)M, (int)N, (int)K, vec_out)
  if (w_dtype == SRDIT_DTYPE_FP32 && ks == 4) SRDIT_LF(float, 4);
  else if (w_dtype == SRDIT_DTYPE_FP32) SRDIT_LF(float, 1);
  else if (ks == 4) SRDIT_LF(uint16_t, 4);
  else SRDIT_LF(uint16_t, 1);
#undef SRDIT_LF
  SRDIT_LAUNCH_CHECK("linear_f32_modulated_kernel");
  return SRDIT_OK;
}

extern "C" int srdit_head_linear(const void* a, int64_t lda, const void* mod, int mod_dtype,
                                 const float* e, const void* w, int64_t ldw, const void* bias,
                                 float* out, int64_t ldo, int64_t M, int64_t N, int64_t K,
                                 void* stream) {
  const char* fn = "srdit_head_linear";
  SRDIT_REQUIRE(a && mod && e && w && out, "%s: null operand", fn);
  SRDIT_REQUIRE(mod_dtype == SRDIT_DTYPE_BF16 || mod_dtype == SRDIT_DTYPE_FP32,
                "%s: mod_dtype %d is not bf16 (0) or fp32 (2)", fn, mod_dtype);
  SRDIT_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                "%s: bad sizes M=%lld N=%lld K=%lld", fn, (long long)M, (long long)N,
                (long long)K);
  SRDIT_REQUIRE(lda >= K && ldw >= K && ldo >= N, "%s: leading dimensions below the row length",
                fn);
  SRDIT_REQUIRE(cut_fits(M, N, K, lda, ldw, SRDIT_DTYPE_BF16),
                "%s: K=%lld must be a multiple of 64, at most %d, and the rows below 2^31 bytes", fn,
                (long long)K, HM_MAX_K);
  SRDIT_REQUIRE(aligned_rows16(a, lda, 2) && aligned_rows16(w, ldw, 2),
                "%s: A and W rows must be 16-byte aligned", fn);
  SRDIT_REQUIRE((reinterpret_cast<uintptr_t>(out) & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(e) & 3) == 0 &&
                    (reinterpret_cast<uintptr_t>(mod) & 3) == 0 &&
                    (!bias || (reinterpret_cast<uintptr_t>(bias) & 1) == 0),
                "%s: misaligned vector or output", fn);
  launch_cut(a, lda, ModSource{nullptr, nullptr, mod, e, mod_dtype == SRDIT_DTYPE_BF16}, w, ldw,
             bias, out, ldo, M, N, K, static_cast<hipStream_t>(stream));
  SRDIT_LAUNCH_CHECK("linear_f32_cut_kernel");
  return SRDIT_OK;
}

extern "C" int srdit_gemv_f32(const float* x, int64_t ldx, const void* w, int64_t ldw,
                              const void* bias, int w_dtype, float* out, int64_t ldo, int64_t M,
                              int64_t N, int64_t K, void* stream) {
  const char* fn = "srdit_gemv_f32";
  SRDIT_REQUIRE(x && w && out, "%s: null operand", fn);
  SRDIT_REQUIRE(w_dtype == SRDIT_DTYPE_BF16 || w_dtype == SRDIT_DTYPE_FP32,
                "%s: w_dtype %d is not bf16 (0) or fp32 (2)", fn, w_dtype);
  SRDIT_REQUIRE(M > 0 && M < 65536 && N > 0 && N < (1LL << 31) && K > 0 && K < (1LL << 31),
                "%s: bad sizes M=%lld N=%lld K=%lld", fn, (long long)M, (long long)N,
                (long long)K);
  SRDIT_REQUIRE(K % 8 == 0, "%s: K=%lld must be a multiple of 8", fn, (long long)K);
  SRDIT_REQUIRE(ldx >= K && ldw >= K && ldo >= N, "%s: leading dimensions below the row length",
                fn);
  const int welem = w_dtype == SRDIT_DTYPE_FP32 ? 4 : 2;
  SRDIT_REQUIRE(aligned_rows16(x, ldx, 4) && aligned_rows16(w, ldw, welem),
                "%s: x and W rows must be 16-byte aligned", fn);
  SRDIT_REQUIRE((reinterpret_cast<uintptr_t>(out) & 3) == 0 &&
                    (!bias || (reinterpret_cast<uintptr_t>(bias) & (welem - 1)) == 0),
                "%s: misaligned output or bias", fn);
  const dim3 grid((unsigned)((N + 3) / 4), (unsigned)M);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (w_dtype == SRDIT_DTYPE_FP32)
    gemv_f32_kernel<float, false><<<grid, 256, 0, s>>>(x, ldx, static_cast<const float*>(w), ldw,
                                                       static_cast<const float*>(bias), out, ldo,
                                                       (int)N, (int)K, nullptr);
  else
    gemv_f32_kernel<uint16_t, false><<<grid, 256, 0, s>>>(
        x, ldx, static_cast<const uint16_t*>(w), ldw, static_cast<const uint16_t*>(bias), out, ldo,
        (int)N, (int)K, nullptr);
  SRDIT_LAUNCH_CHECK("gemv_f32_kernel");
  return SRDIT_OK;
}

namespace srdit {
namespace {
template <typename WT>
void launch_time_embed(const float* t, int64_t freq, const void* w0, const void* b0, const void* w2,
                       const void* b2, const void* wp, const void* bp, float* hidden, float* e,
                       float* e0, int64_t dim, int64_t n_out, hipStream_t s) {
  const int per = 4 * TE_OUT;
  float* h2 = hidden + dim;
  time_sinusoid_gemv_kernel<WT><<<(unsigned)((dim + per - 1) / per), 256, 0, s>>>(
      t, (int)freq, static_cast<const WT*>(w0), static_cast<const WT*>(b0), hidden, (int)dim);
  gemv_f32_kernel<WT, true><<<(unsigned)((dim + 3) / 4), 256, 0, s>>>(
      hidden, dim, static_cast<const WT*>(w2), dim, static_cast<const WT*>(b2), e, dim, (int)dim,
      (int)dim, h2);
  gemv_f32_kernel<WT, false><<<(unsigned)((n_out + 3) / 4), 256, 0, s>>>(
      h2, dim, static_cast<const WT*>(wp), dim, static_cast<const WT*>(bp), e0, n_out, (int)n_out,
      (int)dim, nullptr);
}
}  // namespace
}  // namespace srdit

extern "C" int srdit_time_embed(const float* t, int64_t freq, const void* w0,
                                const void* b0, const void* w2, const void* b2, const void* wp,
                                const void* bp, int w_dtype, float* hidden, float* e, float* e0,
                                int64_t dim, int64_t n_out, void* stream) {
  const char* fn = "srdit_time_embed";
  SRDIT_REQUIRE(t && w0 && w2 && wp && hidden && e && e0, "%s: null operand", fn);
  SRDIT_REQUIRE(w_dtype == SRDIT_DTYPE_BF16 || w_dtype == SRDIT_DTYPE_FP32,
                "%s: w_dtype %d is not bf16 (0) or fp32 (2)", fn, w_dtype);
  SRDIT_REQUIRE(freq > 0 && freq % 8 == 0 && freq <= TE_MAX_FREQ && dim > 0 && dim % 8 == 0 &&
                    n_out > 0 && dim < (1LL << 31) && n_out < (1LL << 31),
                "%s: freq=%lld (at most %d) and dim=%lld must be positive multiples of 8, n_out=%lld "
                "positive", fn, (long long)freq, TE_MAX_FREQ, (long long)dim, (long long)n_out);
  const uintptr_t bmask = w_dtype == SRDIT_DTYPE_FP32 ? 3 : 1;
  SRDIT_REQUIRE(aligned16(w0) && aligned16(w2) && aligned16(wp) && aligned16(hidden) &&
                    (reinterpret_cast<uintptr_t>(t) & 3) == 0 &&
                    ((reinterpret_cast<uintptr_t>(b0) | reinterpret_cast<uintptr_t>(b2) |
                      reinterpret_cast<uintptr_t>(bp)) & bmask) == 0 &&
                    ((reinterpret_cast<uintptr_t>(e) | reinterpret_cast<uintptr_t>(e0)) & 3) == 0,
                "%s: weights and hidden must be 16-byte aligned, the rest to their elements", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (w_dtype == SRDIT_DTYPE_FP32)
    launch_time_embed<float>(t, freq, w0, b0, w2, b2, wp, bp, hidden, e, e0, dim, n_out, s);
  else
    launch_time_embed<uint16_t>(t, freq, w0, b0, w2, b2, wp, bp, hidden, e, e0, dim, n_out, s);
  SRDIT_LAUNCH_CHECK("time embedding");
  return SRDIT_OK;
}
