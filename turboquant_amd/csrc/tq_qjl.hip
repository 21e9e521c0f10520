// tq_qjl.hip -- the QJL products of TurboQuantProd above padded size 128
// (256 .. 1024) on the matrix cores: sign(S r) of the quantize and z S of the
// dequantize (reference turboquant/qjl.py:36-63), S a dim x dim Gaussian
// matrix.
//
// Both are C = X W^T with K (= dim) contiguous in X and W, in tiles of 128
// vectors x 128 outputs per workgroup of four waves (each 64 x 64, 2 x 2
// blocks of v_mfma_f32_32x32x16_f16; 64 x 64 tiles of one block per wave where
// 128 x 128 ones leave CUs idle, and a split-K kernel for the smallest
// quantizes: launch_qjl has the rule), K in steps of 32 through two LDS
// buffers.  fp32 operands enter as fp16 hi + lo halves:
//  * quantize: X = the unit residual times 4096 (exact; it keeps lo out of the
//    fp16 subnormals, and a sign does not see it), W = S; three products
//    hi hi + hi lo + lo hi.  What is dropped is 2^-22 of |S_j| |r|, under the
//    rounding of an fp32 sum of these terms.
//  * dequantize: X = z (int8, exact in fp16), W = S^T; two products.
// Each row of W comes scaled by a power of two that takes its largest entry to
// [2^14, 2^15) (qjl_operand), so that S has fp32's range here too and hi + lo its
// 22 bits for every entry down to 2^-17 of its row's largest: without the scale
// 10% of a Gaussian S (|S| < 2^-3) had a subnormal lo of fewer bits.  A sign does
// not see the scale; the dequantize takes it out of the sum, exactly.
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
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 32;  // K step: 64 bytes of a row

struct QjlGemmParams {
  const _Float16* xh;   // quantize: residual halves [n][ldk]
  const _Float16* xl;
  const int8_t* z;      // dequantize: signs [n][dim]
  const _Float16* wh;   // S (quantize) or S^T (dequantize) halves [ldk][ldk]
  const _Float16* wl;
  const float* wscale;  // dequantize: what the rows of W were divided by [ldk], or null
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
template <int ROWS>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const _Float16* base, int64_t row,
                                                            int64_t rows, int ldk) {
  const uint64_t a = (uint64_t)(uintptr_t)(base + row * ldk);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const int64_t live = rows - row < ROWS ? rows - row : ROWS;
  const int nrec = __builtin_amdgcn_readfirstlane((int)live * ldk * 2);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)hi << 32) | lo), (short)0,
                                           nrec, 0x00020000);
}
#endif

// BT: the tile's edge, 128 or 64 (vectors, outputs).
template <bool QUANT, int BT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(QUANT ? 2 : 3)))
void qjl_gemm_kernel(QjlGemmParams p) {
  constexpr int kSide = BT * kBK * 2;  // bytes of one operand half in LDS
  constexpr int WB = BT / 64;          // 32 x 32 blocks per wave and direction
  constexpr int NC = BT / 64;          // copies per wave and half, 8-sign pieces per thread
  // quantize: xh, xl, wh, wl; dequantize: z as fp16, wh, wl
  constexpr int kNS = QUANT ? 4 : 3;
  __shared__ __attribute__((aligned(16))) uint8_t buf0[kNS * kSide];
  __shared__ __attribute__((aligned(16))) uint8_t buf1[kNS * kSide];

  // tiles in runs per XCD (workgroups go to the XCDs round robin)
  const int64_t per = (p.tiles + 7) / 8;
  const int64_t id = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int64_t)(blockIdx.x >> 3) >= per || id >= p.tiles) return;
  const int64_t m0 = id / p.ntn * BT;        // first vector
  const int n0 = (int)(id % p.ntn) * BT;     // first output

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int hh = lane >> 5, ln = lane & 31;
  const int wm = BT / 2 * (w & 1), wn = BT / 2 * (w >> 1);  // the wave's vectors / outputs

  // copies: 1 KB = 16 rows of 64 bytes; wave w takes copies w (and w + 4) of
  // each half.  Lane l writes row l / 4, physical chunk l % 4.
  const int crow = lane >> 2;
  uint32_t coff[NC];
#pragma unroll
  for (int i = 0; i < NC; i++) {
    const int row = 16 * (w + 4 * i) + crow;
    coff[i] = (uint32_t)(row * p.ldk * 2 + (((lane & 3) ^ ((row >> 1) & 3)) * 16));
  }
  // dequantize: a thread stages 8 * NC of a step's 32 signs of one vector
  constexpr int TPV = 4 / NC;  // threads per vector
  const int zr = threadIdx.x / TPV, zk = 8 * NC * (threadIdx.x % TPV);
  const int8_t* zrow = QUANT ? nullptr : p.z + (m0 + zr < p.n ? m0 + zr : 0) * p.dim;
  const bool zlive = !QUANT && m0 + zr < p.n;
  const bool zvec = !QUANT && (p.dim & 7) == 0;  // rows 8-byte aligned (the entry checks z)
  const int64_t zend = p.n * p.dim;
  // four K steps at a time: a thread's pieces of one 128-byte line go out
  // together (4% at dim 1024 against a step at a time)
  uint32_t zreg[4][2 * NC];
  auto load_z = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 4 * NC; i++) {
      const int h = i % NC, k = (t0 + i / NC) * kBK + zk + 8 * h;
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
      zreg[i / NC][2 * h] = v.x;
      zreg[i / NC][2 * h + 1] = v.y;
    }
  };
  auto store_z = [&](uint8_t* b, const uint32_t* zr4) {
#pragma unroll
    for (int h = 0; h < NC; h++) {
      u32x4 v;
      uint32_t a, c;
      z_to_half(zr4[2 * h], a, c);
      v[0] = a;
      v[1] = c;
      z_to_half(zr4[2 * h + 1], a, c);
      v[2] = a;
      v[3] = c;
      *reinterpret_cast<u32x4*>(b + chunk_at(zr, NC * (threadIdx.x % TPV) + h)) = v;
    }
  };
  auto issue = [&](int k0, uint8_t* b) {
#if defined(__HIP_DEVICE_COMPILE__)
    auto half = [&](const __amdgpu_buffer_rsrc_t& r, int side) {
#pragma unroll
      for (int i = 0; i < NC; i++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (void*)(b + side * kSide + 1024 * (w + 4 * i)),
                                                 16, coff[i], k0 * 2, 0, 0);
    };
    if constexpr (QUANT) {
      half(rows_rsrc<BT>(p.xh, m0, p.n, p.ldk), 0);
      half(rows_rsrc<BT>(p.xl, m0, p.n, p.ldk), 1);
    }
    half(rows_rsrc<BT>(p.wh, n0, p.ldk, p.ldk), kNS - 2);
    half(rows_rsrc<BT>(p.wl, n0, p.ldk, p.ldk), kNS - 1);
#else
    (void)k0;
    (void)b;
#endif
  };

  f32x16 acc[WB][WB];  // [vector block][output block]
#pragma unroll
  for (int i = 0; i < WB; i++)
#pragma unroll
    for (int j = 0; j < WB; j++)
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
      half8_t xh[WB], xl[WB], wh[WB], wl[WB];
#pragma unroll
      for (int i = 0; i < WB; i++) {
        xh[i] = frag(0, wm + 32 * i);
        if constexpr (QUANT) xl[i] = frag(1, wm + 32 * i);
        wh[i] = frag(kNS - 2, wn + 32 * i);
        wl[i] = frag(kNS - 1, wn + 32 * i);
      }
#pragma unroll
      for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WB; j++) acc[i][j] = mma(xh[i], wl[j], acc[i][j]);
      if constexpr (QUANT) {
#pragma unroll
        for (int i = 0; i < WB; i++)
#pragma unroll
          for (int j = 0; j < WB; j++) acc[i][j] = mma(xl[i], wh[j], acc[i][j]);
      }
#pragma unroll
      for (int i = 0; i < WB; i++)
#pragma unroll
        for (int j = 0; j < WB; j++) acc[i][j] = mma(xh[i], wh[j], acc[i][j]);
    }
  };

  // the lane's output scales, loaded ahead of the K loop (loaded at its end
  // 20,011 vectors of dim 1000 take 132 us against 124)
  float wsc[WB];
#pragma unroll
  for (int j = 0; j < WB; j++) wsc[j] = 1.0f;
  if constexpr (!QUANT)
    if (p.wscale)
#pragma unroll
      for (int j = 0; j < WB; j++) wsc[j] = p.wscale[n0 + wn + 32 * j + ln];  // < ldk

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
    // signs of the tile staged in LDS as bytes ([vector][output], rows of BT + 16
    // bytes), then written as runs of a row
    constexpr int kRS = BT + 16;
    static_assert(BT * kRS <= kNS * kSide, "stage fits");
    __syncthreads();  // the last step's reads
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
      for (int j = 0; j < WB; j++)
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
    const int cols = p.dim - n0 < BT ? p.dim - n0 : BT;
    if ((p.dim & 7) == 0) {
#pragma unroll
      for (int i = threadIdx.x; i < BT * BT / 8; i += 256) {
        const int r = i / (BT / 8), c = 8 * (i % (BT / 8));
        if (m0 + r < p.n && c < cols)
          *reinterpret_cast<uint2*>(p.zout + (m0 + r) * p.dim + n0 + c) =
              *reinterpret_cast<const uint2*>(buf0 + r * kRS + c);
      }
    } else {
      for (int i = threadIdx.x; i < BT * BT; i += 256) {
        const int r = i / BT, c = i % BT;
        if (m0 + r < p.n && c < cols)
          p.zout[(m0 + r) * p.dim + n0 + c] = (int8_t)buf0[r * kRS + c];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < WB; i++)
#pragma unroll
      for (int j = 0; j < WB; j++) {
        const int col = n0 + wn + 32 * j + ln;
        if (col >= p.dim) continue;
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int64_t row = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * hh + (e & 3);
          if (row < p.n) p.term[row * p.dim + col] = acc[i][j][e] * wsc[j];
        }
      }
  }
}

// sign(S r) of a small launch: 32 vectors x 32 outputs per workgroup, K split
// over its waves (wave w takes the runs of 64 elements w, w + waves, ...), the
// operands straight from memory into registers.  What bounds such a launch is
// latency: a 128 x 128 tile walks K (dim 1000) in 32 dependent steps of 0.7 us
// whatever n is, a 64 x 64 tile in 32 of 0.45; here every load of a wave's two
// runs is in flight at once (the products of 16 vectors 8 us, 23 and 14 in
// tiles), and up to 16 times as many workgroups fetch.  K is
// taken in an order of its own, the same in both operands: the 16-byte pieces
// hh * 64 + 16 i of a run's 128-byte line feed MFMA i, so a lane pair reads
// whole lines.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2)))
void qjl_signs_small_kernel(QjlGemmParams p) {
  constexpr int kT = 32, kRow = kT + 4;
  __shared__ __attribute__((aligned(16))) float part[WAVES][kT * kRow];
  const int nt = (p.dim + kT - 1) / kT;
  const int64_t m0 = (int64_t)(blockIdx.x / nt) * kT;
  const int n0 = (int)(blockIdx.x % nt) * kT;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int hh = lane >> 5, ln = lane & 31;
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.0f;
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t rs[4] = {
      rows_rsrc<kT>(p.xh, m0, p.n, p.ldk), rows_rsrc<kT>(p.xl, m0, p.n, p.ldk),
      rows_rsrc<kT>(p.wh, n0, p.ldk, p.ldk), rows_rsrc<kT>(p.wl, n0, p.ldk, p.ldk)};
  const int runs = (p.dim + 63) / 64;  // (ldk is a multiple of 64, zeros past dim)
  for (int g = w; g < runs; g += 2 * WAVES) {
    half8_t f[2][4][4];  // [run][operand][piece]
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int o = 0; o < 4; o++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          // (a second run past K: out of range, zeros)
          f[r][o][i] = __builtin_bit_cast(
              half8_t, __builtin_amdgcn_raw_buffer_load_b128(
                           rs[o],
                           g + r * WAVES < runs
                               ? (uint32_t)(ln * p.ldk * 2 + (g + r * WAVES) * 128 + hh * 64 + i * 16)
                               : 0x80000000u,
                           0, 0));
    __builtin_amdgcn_sched_barrier(0);  // all of them in flight before the first wait
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[r][3][i], f[r][0][i], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[r][2][i], f[r][1][i], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[r][2][i], f[r][0][i], acc, 0, 0, 0);
      }
  }
#endif
  // the waves' sums, [vector][output]
#pragma unroll
  for (int q = 0; q < 4; q++)
    *reinterpret_cast<float4*>(&part[w][ln * kRow + 8 * q + 4 * hh]) =
        float4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
  for (int t = threadIdx.x; t < kT * kT / 4; t += 64 * WAVES) {
    const int v = t / (kT / 4), c = 4 * (t % (kT / 4));
    float4 s = *reinterpret_cast<const float4*>(&part[0][v * kRow + c]);
#pragma unroll
    for (int k = 1; k < WAVES; k++) {
      const float4 a = *reinterpret_cast<const float4*>(&part[k][v * kRow + c]);
      s.x += a.x;
      s.y += a.y;
      s.z += a.z;
      s.w += a.w;
    }
    if (m0 + v >= p.n) continue;
    int8_t* z = p.zout + (m0 + v) * p.dim + n0 + c;
    // +1 for >= 0 (sign() with 0 -> +1), else -1
    const uint32_t pk = (s.x >= 0.0f ? 0x01u : 0xffu) | (s.y >= 0.0f ? 0x0100u : 0xff00u) |
                        (s.z >= 0.0f ? 0x010000u : 0xff0000u) |
                        (s.w >= 0.0f ? 0x01000000u : 0xff000000u);
    if ((p.dim & 7) == 0) {
      if (n0 + c < p.dim) *reinterpret_cast<uint32_t*>(z) = pk;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (n0 + c + e < p.dim) z[e] = (int8_t)(pk >> (8 * e));
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

// The power of two that takes m (the largest magnitude of a row) to [2^14,
// 2^15), as far as it and its inverse are normal floats.
__device__ __forceinline__ float row_scale(float m, float& inv) {
  const int e = min(253, max(1, 268 - (int)(__float_as_uint(m) >> 23)));
  inv = __uint_as_float((uint32_t)(254 - e) << 23);
  return __uint_as_float((uint32_t)e << 23);
}

__device__ __forceinline__ void put_halves(_Float16* out, int64_t at, int64_t sq, float v) {
  const _Float16 hi = (_Float16)v;
  out[at] = hi;
  // (an infinite entry: lo 0 instead of inf - inf)
  out[at + sq] = __builtin_isinf((float)hi) ? (_Float16)0.0f : (_Float16)(v - (float)hi);
}

// W = S as hi + lo [2][pd][pd], rows scaled, zero-padded; one wave per row.
__global__ __launch_bounds__(256) void operand_rows_kernel(const float* __restrict__ s, int dim,
                                                           int pd, _Float16* __restrict__ out,
                                                           float* __restrict__ scales) {
  const int lane = threadIdx.x & 63, r = 4 * (int)blockIdx.x + (threadIdx.x >> 6);
  float v[16], m = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int c = 64 * i + lane;
    v[i] = r < dim && c < dim ? s[(int64_t)r * dim + c] : 0.0f;
    m = fmaxf(m, fabsf(v[i]));
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  float inv;
  const float sc = row_scale(m, inv);
  if (lane == 0) scales[r] = inv;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int c = 64 * i + lane;
    if (c < pd) put_halves(out, (int64_t)r * pd + c, (int64_t)pd * pd, v[i] * sc);
  }
}

// The same for W = S^T: a workgroup reads 32 columns of S whole (thread:
// column tid % 32, rows tid / 32 + 32 i, all loads in flight) for their scales
// and writes every eighth 32 x 32 tile of them as rows of W, through LDS.
// Eight workgroups read the same strip (out of L2) so that the few strips do
// not leave most CUs idle: dim 1024 6.3 us with the launch, 9.8 with one
// workgroup per strip (W = S 3.7 us).
__global__ __launch_bounds__(1024) void operand_cols_kernel(const float* __restrict__ s, int dim,
                                                            int pd, _Float16* __restrict__ out,
                                                            float* __restrict__ scales) {
  __shared__ float tile[32][33];
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5, c0 = 32 * (int)blockIdx.x;
  float v[32], m = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) {
    const int r = 32 * i + y;
    v[i] = r < dim && c0 + x < dim ? s[(int64_t)r * dim + c0 + x] : 0.0f;
    m = fmaxf(m, fabsf(v[i]));
  }
  tile[y][x] = m;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 32; k++) m = fmaxf(m, tile[k][x]);
  float inv;
  const float sc = row_scale(m, inv);
  if (y == 0 && blockIdx.y == 0) scales[c0 + x] = inv;
#pragma unroll
  for (int i = 0; i < 32; i++) {
    if ((i & 7) != (int)blockIdx.y || 32 * i >= pd) continue;  // uniform
    __syncthreads();
    tile[x][y] = v[i] * sc;
    __syncthreads();
    put_halves(out, (int64_t)(c0 + y) * pd + 32 * i + x, (int64_t)pd * pd, tile[y][x]);
  }
}

}  // namespace

hipError_t launch_qjl(bool quant, const _Float16* xh, const _Float16* xl, const int8_t* z,
                      const _Float16* wh, const _Float16* wl, const float* wscale, int8_t* zout,
                      float* term, int64_t n, int dim, int ldk, hipStream_t st) {
  QjlGemmParams p;
  p.xh = xh;
  p.xl = xl;
  p.z = z;
  p.wh = wh;
  p.wl = wl;
  p.wscale = wscale;
  p.zout = zout;
  p.term = term;
  p.n = n;
  p.dim = dim;
  p.ldk = ldk;
  // The form by the number of tiles.  Up to one 32 x 32 tile per CU the split-K
  // kernel: quantize, dim 1000, n = 16 / 256 / 512 16.6 / 19.3 / 29 us against 22.8
  // / 24 / 26.5 with 64 x 64 tiles and 31.5 / 33.2 / 34 with 128 x 128 (the whole
  // call but for the 4 .. 6 us of the operand's launch; the products alone 8
  // against 23 us at n = 16).  Then 64 x 64 tiles while
  // few enough to fill a round or two of the card: 2.5 per CU for the quantize (n
  // = 2500 41.3 against 43.5, n = 4096 60 against 50; dim 256, n = 8192 19.8
  // against 22.0), 5 for the dequantize, more of which fit a CU (dim 1000, n =
  // 2500 31.5 against 43.0, n = 4096 41.3 against 45.8; dim 256, n = 12000 20.8
  // against 23.6; dim 1000, n = 8192 72 against 61).
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  const int64_t t32 = (n + 31) / 32 * ((dim + 31) / 32);
  if (quant && t32 <= cus) {
    if (dim > 256)
      hipLaunchKernelGGL((qjl_signs_small_kernel<8>), dim3((unsigned)t32), dim3(512), 0, st, p);
    else
      hipLaunchKernelGGL((qjl_signs_small_kernel<4>), dim3((unsigned)t32), dim3(256), 0, st, p);
    return hipGetLastError();
  }
  const int64_t t64 = (n + 63) / 64 * ((dim + 63) / 64);
  const int bt = t64 <= (quant ? 5 : 10) * cus / 2 ? 64 : 128;
  p.ntn = (dim + bt - 1) / bt;
  p.tiles = (n + bt - 1) / bt * p.ntn;
  const int64_t grid = (p.tiles + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const dim3 g((unsigned)grid), wg(256);
  if (quant && bt == 64)
    hipLaunchKernelGGL((qjl_gemm_kernel<true, 64>), g, wg, 0, st, p);
  else if (quant)
    hipLaunchKernelGGL((qjl_gemm_kernel<true, 128>), g, wg, 0, st, p);
  else if (bt == 64)
    hipLaunchKernelGGL((qjl_gemm_kernel<false, 64>), g, wg, 0, st, p);
  else
    hipLaunchKernelGGL((qjl_gemm_kernel<false, 128>), g, wg, 0, st, p);
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

extern "C" int tq_qjl_operand(const float* s, int32_t dim, int32_t padded_dim, int32_t transposed,
                              void* halves, float* scales, tq_stream_t stream) {
  using namespace tq;
  if ((padded_dim != 256 && padded_dim != 512 && padded_dim != 1024) || dim < 1 ||
      dim > padded_dim) {
    set_error("qjl_operand: padded_dim %d must be 256, 512 or 1024, dim %d at most that",
              padded_dim, dim);
    return kEinval;
  }
  if (!s || !halves || !scales) {
    set_error("qjl_operand: null pointer");
    return kEinval;
  }
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  _Float16* const out = static_cast<_Float16*>(halves);
  if (transposed)
    hipLaunchKernelGGL(operand_cols_kernel, dim3(padded_dim / 32, 8), dim3(1024), 0, st, s, dim,
                       padded_dim, out, scales);
  else
    hipLaunchKernelGGL(operand_rows_kernel, dim3(padded_dim / 4), dim3(256), 0, st, s, dim,
                       padded_dim, out, scales);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) set_error("qjl_operand: launch failed: %s", hipGetErrorString(e));
  return (int)e;
}
