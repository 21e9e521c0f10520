// tq_qjl.hip -- the QJL products of TurboQuantProd above padded size 128
// (256 .. 1024) on the matrix cores: sign(S r) of the quantize and z S of the
// dequantize (reference turboquant/qjl.py:36-63), S a dim x dim Gaussian
// matrix.
//
// Both are C = X W^T with K (= dim) contiguous in X and W, in tiles of 128
// vectors x 128 outputs per workgroup of four waves (each 64 x 64, 2 x 2
// blocks of v_mfma_f32_32x32x16_f16), K in steps of 32 through two LDS
// buffers.  fp32 operands enter as fp16 hi + lo halves:
//  * quantize: X = the unit residual times 4096 (exact; it keeps lo out of the
//    fp16 subnormals, and a sign does not see it), W = S; three products
//    hi hi + hi lo + lo hi.  What is dropped is 2^-22 of |S_j| |r|, under the
//    rounding of an fp32 sum of these terms.
//  * dequantize: X = z (int8, exact in fp16), W = S^T; two products.
// The halves of one K step feed 12 (8) MFMAs from 8 (6) LDS reads, so the
// kernels are MFMA-bound where a plain fp16 product of this tile is
// LDS-bound.  Tiles are copied with direct-to-LDS loads, 16-byte chunks
// XOR-swizzled by row ((row / 2) % 4), so the 16-byte operand reads of 8
// consecutive rows hit all bank groups once.  Blocks of one XCD take
// neighbouring tiles, the output blocks of one vector tile first: X is read
// into one L2 once.
//
// Measured at 20,011 vectors of dim 1000: sign(S r) 123 us (126 GFLOP issued:
// 1.0 PFLOP/s; a plain 8192^3 library product reaches 1.23 on this card), z S
// 102 us; as fp32 library products they took 377 and 357 us, plus 130 us of
// compares, conversions and sign arithmetic around them.  What bounds them is
// the wait per K step (MFMAs fill half of it) and the last round of tiles, so
// as many workgroups per CU as fit hide each other's barrier: two of the
// quantize (64 KB of LDS each), three of the dequantize (48 KB, 132 VGPRs; two
// of them 112 us).  The signs of a step are in registers a step ahead and go
// to LDS behind the copies' own wait (loaded and waited for inside the step:
// 125 us).
#include "tq_qjl.h"

namespace tq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBT = 128;           // tile edge (vectors, outputs)
constexpr int kBK = 32;            // K step: 64 bytes of a row
constexpr int kSide = kBT * kBK * 2;  // bytes of one operand half in LDS

struct QjlGemmParams {
  const _Float16* xh;   // quantize: residual halves [n][ldk]
  const _Float16* xl;
  const int8_t* z;      // dequantize: signs [n][dim]
  const _Float16* wh;   // S (quantize) or S^T (dequantize) halves [ldk][ldk]
  const _Float16* wl;
  int8_t* zout;         // quantize: [n][dim]
  float* term;          // dequantize: [n][dim]
  int64_t n;
  int dim, ldk;
  int ntn;              // output tiles
  int64_t tiles;
};

// byte offset of 16-byte chunk c of row r in a tile of 64-byte rows
__device__ __forceinline__ int chunk_at(int r, int c) {
  return r * (kBK * 2) + ((c ^ ((r >> 1) & 3)) * 16);
}

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const _Float16* base, int64_t row,
                                                            int64_t rows, int ldk) {
  const uint64_t a = (uint64_t)(uintptr_t)(base + row * ldk);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const int64_t live = rows - row < kBT ? rows - row : kBT;
  const int nrec = __builtin_amdgcn_readfirstlane((int)live * ldk * 2);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)hi << 32) | lo), (short)0,
                                           nrec, 0x00020000);
}
#endif

// four int8 as fp16 (exact: 1024 + (z + 128) - 1152)
__device__ __forceinline__ void z_to_half(uint32_t w, uint32_t& lo, uint32_t& hi) {
  const uint32_t u = w ^ 0x80808080u;
  const half2_t b = {(_Float16)1152.0f, (_Float16)1152.0f};
  lo = __builtin_bit_cast(uint32_t, (half2_t)(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(
                                        0x64646464u, u, 0x04010400u)) - b));
  hi = __builtin_bit_cast(uint32_t, (half2_t)(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(
                                        0x64646464u, u, 0x04030402u)) - b));
}

template <bool QUANT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(QUANT ? 2 : 3)))
void qjl_gemm_kernel(QjlGemmParams p) {
  // quantize: xh, xl, wh, wl; dequantize: z as fp16, wh, wl
  constexpr int kNS = QUANT ? 4 : 3;
  __shared__ __attribute__((aligned(16))) uint8_t buf0[kNS * kSide];
  __shared__ __attribute__((aligned(16))) uint8_t buf1[kNS * kSide];

  // tiles in runs per XCD (workgroups go to the XCDs round robin)
  const int64_t per = (p.tiles + 7) / 8;
  const int64_t id = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int64_t)(blockIdx.x >> 3) >= per || id >= p.tiles) return;
  const int64_t m0 = id / p.ntn * kBT;        // first vector
  const int n0 = (int)(id % p.ntn) * kBT;     // first output

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int hh = lane >> 5, ln = lane & 31;
  const int wm = 64 * (w & 1), wn = 64 * (w >> 1);  // the wave's vectors / outputs

  // copies: 1 KB = 16 rows of 64 bytes; wave w takes copies w and w + 4 of each
  // half (8 per half).  Lane l writes row l / 4, physical chunk l % 4.
  const int crow = lane >> 2;
  uint32_t coff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int row = 16 * (w + 4 * i) + crow;
    coff[i] = (uint32_t)(row * p.ldk * 2 + (((lane & 3) ^ ((row >> 1) & 3)) * 16));
  }
  // dequantize: thread t stages signs of vector t / 2, 16 of a step's 32
  const int zr = threadIdx.x >> 1, zk = 16 * (threadIdx.x & 1);
  const int8_t* zrow = QUANT ? nullptr : p.z + (m0 + zr < p.n ? m0 + zr : 0) * p.dim;
  const bool zlive = !QUANT && m0 + zr < p.n;
  const bool zvec = !QUANT && (p.dim & 7) == 0;  // rows 8-byte aligned (the entry checks z)
  const int64_t zend = p.n * p.dim;
  // four K steps at a time: a thread's pieces of one 128-byte line go out
  // together (4% at dim 1024 against a step at a time)
  uint32_t zreg[4][4];
  auto load_z = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int h = i & 1, k = (t0 + i / 2) * kBK + zk + 8 * h;
      uint2 v = {0u, 0u};
      if (zlive && k < p.dim) {
        if (zvec) {
          v = *reinterpret_cast<const uint2*>(zrow + k);
        } else if ((m0 + zr) * p.dim + k + 8 <= zend) {
          // unaligned; what lies past the row's end meets zero rows of W
          __builtin_memcpy(&v, zrow + k, 8);
        } else {
          for (int e = 0; e < 8 && k + e < p.dim; e++)
            (e < 4 ? v.x : v.y) |= (uint32_t)(uint8_t)zrow[k + e] << (8 * (e & 3));
        }
      }
      zreg[i / 2][2 * h] = v.x;
      zreg[i / 2][2 * h + 1] = v.y;
    }
  };
  auto store_z = [&](uint8_t* b, const uint32_t* zr4) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      u32x4 v;
      uint32_t a, c;
      z_to_half(zr4[2 * h], a, c);
      v[0] = a;
      v[1] = c;
      z_to_half(zr4[2 * h + 1], a, c);
      v[2] = a;
      v[3] = c;
      *reinterpret_cast<u32x4*>(b + chunk_at(zr, 2 * (threadIdx.x & 1) + h)) = v;
    }
  };
  auto issue = [&](int k0, uint8_t* b) {
#if defined(__HIP_DEVICE_COMPILE__)
    auto half = [&](const __amdgpu_buffer_rsrc_t& r, int side) {
#pragma unroll
      for (int i = 0; i < 2; i++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (void*)(b + side * kSide + 1024 * (w + 4 * i)),
                                                 16, coff[i], k0 * 2, 0, 0);
    };
    if constexpr (QUANT) {
      half(rows_rsrc(p.xh, m0, p.n, p.ldk), 0);
      half(rows_rsrc(p.xl, m0, p.n, p.ldk), 1);
    }
    half(rows_rsrc(p.wh, n0, p.ldk, p.ldk), kNS - 2);
    half(rows_rsrc(p.wl, n0, p.ldk, p.ldk), kNS - 1);
#else
    (void)k0;
    (void)b;
#endif
  };

  f32x16 acc[2][2];  // [vector block][output block]
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

  auto mma = [&](half8_t x, half8_t wv, f32x16 c) {
    // quantize: outputs are the C rows (a lane then holds runs of four outputs
    // of one vector); dequantize: vectors are (32 lanes hold 32 outputs)
    if constexpr (QUANT) return __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, x, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, wv, c, 0, 0, 0);
  };
  auto step = [&](const uint8_t* b) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      auto frag = [&](int side, int r) {
        return *reinterpret_cast<const half8_t*>(b + side * kSide + chunk_at(r + ln, 2 * s + hh));
      };
      half8_t xh[2], xl[2], wh[2], wl[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        xh[i] = frag(0, wm + 32 * i);
        if constexpr (QUANT) xl[i] = frag(1, wm + 32 * i);
        wh[i] = frag(kNS - 2, wn + 32 * i);
        wl[i] = frag(kNS - 1, wn + 32 * i);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = mma(xh[i], wl[j], acc[i][j]);
      if constexpr (QUANT) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = mma(xl[i], wh[j], acc[i][j]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = mma(xh[i], wh[j], acc[i][j]);
    }
  };

  const int nk = (p.dim + kBK - 1) / kBK;
  issue(0, buf0);
  if constexpr (!QUANT) {
    load_z(0);
    store_z(buf0, zreg[0]);
  }
  auto iter = [&](int t, int j, uint8_t* cur, uint8_t* nxt) {  // j = t % 4
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's copies of step t
    __syncthreads();
    if (t + 1 < nk) {
      // the signs of step t + 1 are in registers: loaded at the latest a step
      // ago, they arrived with the copies just waited for
      if constexpr (!QUANT) store_z(nxt, zreg[(j + 1) & 3]);
      issue((t + 1) * kBK, nxt);
      if constexpr (!QUANT)
        if (j == 2) load_z(t + 2);  // (past the last step: zeros)
    }
    step(cur);
  };
  for (int t = 0; t < nk; t += 4) {
    iter(t, 0, buf0, buf1);
    if (t + 1 < nk) iter(t + 1, 1, buf1, buf0);
    if (t + 2 < nk) iter(t + 2, 2, buf0, buf1);
    if (t + 3 < nk) iter(t + 3, 3, buf1, buf0);
  }

  if constexpr (QUANT) {
    // signs of the tile staged in LDS as bytes ([vector][output], rows of 144
    // bytes), then written as runs of a row
    constexpr int kRS = kBT + 16;
    static_assert(kBT * kRS <= kNS * kSide, "stage fits");
    __syncthreads();  // the last step's reads
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          uint32_t pk = 0;
#pragma unroll
          for (int e = 0; e < 4; e++)  // +1 for >= 0 (sign() with 0 -> +1), else -1
            pk |= (acc[i][j][4 * q + e] >= 0.0f ? 0x01u : 0xffu) << (8 * e);
          *reinterpret_cast<uint32_t*>(buf0 + (wm + 32 * i + ln) * kRS + wn + 32 * j + 8 * q +
                                       4 * hh) = pk;
        }
    __syncthreads();
    const int cols = p.dim - n0 < kBT ? p.dim - n0 : kBT;
    if ((p.dim & 7) == 0) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int r = 16 * i + (threadIdx.x >> 4), c = 8 * (threadIdx.x & 15);
        if (m0 + r < p.n && c < cols)
          *reinterpret_cast<uint2*>(p.zout + (m0 + r) * p.dim + n0 + c) =
              *reinterpret_cast<const uint2*>(buf0 + r * kRS + c);
      }
    } else {
      for (int i = threadIdx.x; i < kBT * kBT; i += 256) {
        const int r = i / kBT, c = i % kBT;
        if (m0 + r < p.n && c < cols)
          p.zout[(m0 + r) * p.dim + n0 + c] = (int8_t)buf0[r * kRS + c];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = n0 + wn + 32 * j + ln;
        if (col >= p.dim) continue;
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int64_t row = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * hh + (e & 3);
          if (row < p.n) p.term[row * p.dim + col] = acc[i][j][e];
        }
      }
  }
}

// S [dim][dim] and its transpose as fp16 hi + lo halves, zero-padded: out is
// [4][pd][pd], S hi, S lo, S^T hi, S^T lo.  32 x 32 tiles through LDS; one
// launch where torch took a dozen small ones (120 us of a first call).
__global__ __launch_bounds__(256) void split_halves_kernel(const float* __restrict__ s, int dim,
                                                           int pd, _Float16* __restrict__ out) {
  __shared__ float tile[32][33];
  const int r0 = 32 * (int)blockIdx.y, c0 = 32 * (int)blockIdx.x;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const int64_t sq = (int64_t)pd * pd;
  auto put = [&](int64_t at, float v) {
    const _Float16 hi = (_Float16)v;
    out[at] = hi;
    out[at + sq] = (_Float16)(v - (float)hi);
  };
#pragma unroll
  for (int i = y; i < 32; i += 8) {
    const int r = r0 + i, c = c0 + x;
    const float v = r < dim && c < dim ? s[(int64_t)r * dim + c] : 0.0f;
    tile[i][x] = v;
    put((int64_t)r * pd + c, v);
  }
  __syncthreads();
#pragma unroll
  for (int i = y; i < 32; i += 8)  // row c0 + i of S^T
    put(2 * sq + (int64_t)(c0 + i) * pd + r0 + x, tile[x][i]);
}

}  // namespace

hipError_t launch_qjl(bool quant, const _Float16* xh, const _Float16* xl, const int8_t* z,
                      const _Float16* wh, const _Float16* wl, int8_t* zout, float* term, int64_t n,
                      int dim, int ldk, hipStream_t st) {
  QjlGemmParams p;
  p.xh = xh;
  p.xl = xl;
  p.z = z;
  p.wh = wh;
  p.wl = wl;
  p.zout = zout;
  p.term = term;
  p.n = n;
  p.dim = dim;
  p.ldk = ldk;
  p.ntn = (dim + kBT - 1) / kBT;
  p.tiles = (n + kBT - 1) / kBT * p.ntn;
  const int64_t grid = (p.tiles + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  if (quant)
    hipLaunchKernelGGL((qjl_gemm_kernel<true>), dim3((unsigned)grid), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((qjl_gemm_kernel<false>), dim3((unsigned)grid), dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace tq

extern "C" int tq_qjl_halves(const float* s, int32_t dim, int32_t padded_dim, void* halves,
                             tq_stream_t stream) {
  using namespace tq;
  if (padded_dim < 64 || padded_dim > 1024 || (padded_dim & (padded_dim - 1)) != 0 || dim < 1 ||
      dim > padded_dim) {
    set_error("qjl_halves: padded_dim %d must be a power of two 64..1024, dim %d at most that",
              padded_dim, dim);
    return kEinval;
  }
  if (!s || !halves) {
    set_error("qjl_halves: null pointer");
    return kEinval;
  }
  hipLaunchKernelGGL(split_halves_kernel, dim3(padded_dim / 32, padded_dim / 32), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), s, dim, padded_dim,
                     static_cast<_Float16*>(halves));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) set_error("qjl_halves: launch failed: %s", hipGetErrorString(e));
  return (int)e;
}
