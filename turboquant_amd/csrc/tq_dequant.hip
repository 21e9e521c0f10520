// tq_dequant.hip -- packed cache pages -> fp16 K/V rows in the original domain.
//
// Used by the prefill of a chunk whose sequence already has cached context:
// the context is read back from the quantized cache, as the decode reads it
// (dequantize-then-attend, turboquant/triton_decode_ref.py:89-131), and
// rotated back to the original domain so that it can be attended together
// with the chunk's fresh K/V.  Entry layout as written by
// quantize_write_kernel.cuh:332-431: pd/2 code bytes (dim 2k in the high
// nibble of byte k), then the fp16 norm.  Per vector:
//   x = s * FWHT(c[code]) * norm / pd
// (the inverse of the write's rotation, its two 1/sqrt(pd) taken together).
//
// tq_dequant_paged reads back one sequence; tq_prefill_gather assembles the
// keys and values of all requests of a prefill step in one launch: each
// request's cached context read back, followed by its fresh rows converted to
// fp16, both padded to pd elements.
//
// One pass over the entries, L = pd/32 lanes per vector (32 dims = 16 code
// bytes per lane, one 16-byte load), four vectors per thread with every load
// issued first, the output staged in LDS and written 1 KB per wave store.
// Bound by its VALU work (12 instructions per dim: two to index the codebook,
// 5 + log2 L butterflies, the scale, conversion and sign), the HBM bytes are
// 2 x 68 read and 4 pd written per token and head.  30,720 tokens x 8 heads x
// 128: 41 us, 3.9 TB/s (a copy of those bytes 30 us); 49 us with the codebook
// value scaled before the transform, two instructions per cross-lane butterfly
// and 64-bit divisions for the token and page of each vector.
#include "tq_common.h"

namespace tq {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__constant__ float kCodebook[16] = {
    -2.7326368f, -2.0693470f, -1.6180345f, -1.2562491f, -0.9423684f, -0.6567591f,
    -0.3880823f, -0.1284154f, 0.1284154f,  0.3880823f,  0.6567591f,  0.9423684f,
    1.2562491f,  1.6180345f,  2.0693470f,  2.7326368f};

constexpr int kVecsPerThread = 4;
constexpr int kMaxReqs = 64;

// one request of a gather: ctx cached tokens (page-table row bt_row), then
// fresh rows from src_row of key / value, to output rows dst_row ..
struct GatherReq {
  int ctx, fresh, dst_row, src_row, bt_row;
  int ctx_blk, fresh_blk;  // first workgroup of each part
};

struct ReadBackParams {
  const uint8_t* k_slab;
  const uint8_t* v_slab;
  const int32_t* pages;
  int64_t page_stride;  // page-table row stride
  const float* signs;
  _Float16* out_k;
  _Float16* out_v;
  int64_t out_stride_tok;
  int64_t num_blocks;
  uint32_t hmul;  // ceil(2^32 / H) for 1 < H <= 32768 (exact for r < H + 1024), else 0
  int H, head_dim, block_size, block_shift, ebs;
  int row_dim;    // elements written per head: head_dim, or pd (zero past head_dim)
  bool vec_store;  // row_dim == pd and 16-byte aligned rows
  // gather
  const void* key;
  const void* value;
  int dtype;
  int64_t k_st, k_sh, v_st, v_sh;
  bool vec_load;  // rows in whole aligned 8-element pieces
  int nreq, ctx_blocks;
  GatherReq reqs[kMaxReqs];
};

// x[k] += sg * (x[k] of lane l ^ D), D in {1, 2}, for 8 registers: one
// v_fmac_f32 with a DPP quad-permuted operand each
template <int D>
__device__ __forceinline__ void fmac_quad8(float* x, float sg) {
#if defined(__HIP_DEVICE_COMPILE__)
#define TQ_Q(I, CTL) "v_fmac_f32_dpp %" #I ", %" #I ", %8 " CTL " row_mask:0xf bank_mask:0xf\n\t"
#define TQ_Q8(CTL)                                                                          \
  asm volatile("s_nop 1\n\t" TQ_Q(0, CTL) TQ_Q(1, CTL) TQ_Q(2, CTL) TQ_Q(3, CTL)           \
                   TQ_Q(4, CTL) TQ_Q(5, CTL) TQ_Q(6, CTL) TQ_Q(7, CTL)                       \
               : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]),     \
                 "+v"(x[6]), "+v"(x[7])                                                      \
               : "v"(sg))
  if constexpr (D == 1) TQ_Q8("quad_perm:[1,0,3,2]");
  else TQ_Q8("quad_perm:[2,3,0,1]");
#undef TQ_Q8
#undef TQ_Q
#else
  (void)x;
  (void)sg;
#endif
}

// value of lane (lane ^ 4): two masked row shifts (banks 0, 2 take lane + 4,
// banks 1, 3 lane - 4)
__device__ __forceinline__ float lane_xor4(float x) {
  const int xi = __float_as_int(x);
  int r = __builtin_amdgcn_update_dpp(xi, xi, 0x104, 0xf, 0x5, false);  // row_shl:4
  r = __builtin_amdgcn_update_dpp(r, xi, 0x114, 0xf, 0xa, false);       // row_shr:4
  return __int_as_float(r);
}

__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, half2_t));
}

// r / H for r < H + 1024
__device__ __forceinline__ uint32_t div_heads(const ReadBackParams& p, uint32_t r) {
  return p.hmul ? __umulhi(r, p.hmul) : r / (uint32_t)p.H;
}

// the request whose workgroup range holds `blk` (first[i] ascending; requests
// without blocks share the next one's first and are passed over)
template <class First>
__device__ __forceinline__ int find_request(int n, int blk, First first) {
  int lo = 0, hi = n - 1;  // last i with first(i) <= blk
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first(mid) <= blk) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Cached vectors [block's range) of tokens 0 .. num_tokens - 1 (`pages` their
// page-table row) to out (token 0's row).  blk: workgroup within the range.
template <int PD>
__device__ __forceinline__ void read_back(const ReadBackParams& p, const int32_t* pages,
                                          int num_tokens, int blk, _Float16* out,
                                          const float* cb, _Float16* stage) {
  constexpr int L = PD / 32;  // lanes per vector, 32 dims (16 code bytes) each
  constexpr int VPB = 256 / L, NV = kVecsPerThread;
  const int lane = threadIdx.x % L;
  const uint8_t* slab = blockIdx.y ? p.v_slab : p.k_slab;
  const int64_t nvec = (int64_t)num_tokens * p.H;
  const int64_t vb = (int64_t)blk * (NV * VPB);  // the workgroup's first vector (uniform)
  const uint32_t tb = (uint32_t)(vb / p.H);      // its token and head
  const uint32_t hb = (uint32_t)(vb - (int64_t)tb * p.H);

  // every load of the thread's NV vectors goes out before any math
  uint32_t tv[NV], hv[NV];
  int pg[NV];
  bool live[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const uint32_t i = (uint32_t)(j * VPB) + threadIdx.x / L;
    live[j] = vb + i < nvec;  // all L lanes of a vector agree
    const uint32_t r = hb + i;
    const uint32_t dt = div_heads(p, r);
    tv[j] = tb + dt;
    hv[j] = r - dt * (uint32_t)p.H;
    const uint32_t page = p.block_shift >= 0 ? tv[j] >> p.block_shift
                                             : tv[j] / (uint32_t)p.block_size;
    pg[j] = live[j] ? pages[page] : -1;
    tv[j] -= page * (uint32_t)p.block_size;  // from here the token within its page
  }
  u32x4 w[NV];
  float nrm[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    w[j] = u32x4{0u, 0u, 0u, 0u};
    nrm[j] = 0.0f;
    if (pg[j] >= 0 && pg[j] < p.num_blocks) {
      const uint8_t* e =
          slab + (((int64_t)pg[j] * p.block_size + tv[j]) * p.H + hv[j]) * (int64_t)p.ebs;
      w[j] = *reinterpret_cast<const u32x4*>(e + 16 * lane);
      nrm[j] = (float)__builtin_bit_cast(_Float16, *reinterpret_cast<const uint16_t*>(e + PD / 2));
    }
  }
  uint32_t sm[16];  // sign bits of the lane's dim pairs as fp16 masks
#pragma unroll
  for (int i = 0; i < 16; i++) sm[i] = 0u;
  if (p.signs) {
    const float4* sp = reinterpret_cast<const float4*>(p.signs + 32 * lane);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float4 s = sp[i];
      sm[2 * i] = __builtin_amdgcn_perm(__float_as_uint(s.y), __float_as_uint(s.x), 0x070c030cu) &
                  0x80008000u;
      sm[2 * i + 1] =
          __builtin_amdgcn_perm(__float_as_uint(s.w), __float_as_uint(s.z), 0x070c030cu) &
          0x80008000u;
    }
  }
  __syncthreads();  // codebook ready
  // packed full rows (row stride H * row_dim): a wave's 64 / L vectors are
  // 4 KB of consecutive output, staged in LDS and written with whole-wave
  // 1 KB stores instead of 16-byte pieces at a 64-byte stride
  const bool packed = p.vec_store && p.out_stride_tok == (int64_t)p.H * p.row_dim;  // uniform
  const int wv = threadIdx.x >> 6;
#pragma unroll 1
  for (int j = 0; j < NV; j++) {
    if (!packed && !live[j]) continue;  // whole vector (L lanes of one DPP row) together
    float y[32];  // dims 32 * lane + i
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const uint32_t b = w[j][k / 4] >> (8 * (k % 4));
      y[2 * k] = cb[(b >> 4) & 15u];
      y[2 * k + 1] = cb[b & 15u];
    }
    float sc;
    if (p.signs) {
      // FWHT: stages 1 .. 16 in-lane, then across the vector's lanes; a DPP
      // stage keeps own + sg * partner, which is the butterfly's value negated
      // on the upper lane: tau, folded into the scale
#pragma unroll
      for (int hh = 1; hh < 32; hh <<= 1)
#pragma unroll
        for (int i = 0; i < 32; i++)
          if (!(i & hh)) {
            const float a = y[i], c = y[i + hh];
            y[i] = a + c;
            y[i + hh] = a - c;
          }
      if constexpr (L >= 2)
#pragma unroll
        for (int i = 0; i < 32; i += 8) fmac_quad8<1>(y + i, (lane & 1) ? -1.0f : 1.0f);
      if constexpr (L >= 4)
#pragma unroll
        for (int i = 0; i < 32; i += 8) fmac_quad8<2>(y + i, (lane & 2) ? -1.0f : 1.0f);
      if constexpr (L >= 8) {
        const float s = (lane & 4) ? -1.0f : 1.0f;  // upper lane: partner - own
#pragma unroll
        for (int i = 0; i < 32; i++) y[i] = __builtin_fmaf(y[i], s, lane_xor4(y[i]));
      }
      const bool neg = L >= 2 && ((lane ^ (L >= 4 ? lane >> 1 : 0)) & 1);
      sc = nrm[j] * (neg ? -1.0f / PD : 1.0f / PD);
    } else {
      sc = nrm[j] * (1.0f / __builtin_sqrtf((float)PD));
    }
    uint32_t h[16];
#pragma unroll
    for (int i = 0; i < 16; i++) h[i] = pack_h2(y[2 * i] * sc, y[2 * i + 1] * sc) ^ sm[i];
    if (p.head_dim < p.row_dim) {  // zero past head_dim (uniform)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int d = 32 * lane + 2 * i;
        h[i] = d + 1 < p.head_dim ? h[i] : d < p.head_dim ? h[i] & 0xffffu : 0u;
      }
    }
    if (packed) {
      uint32_t* st = reinterpret_cast<uint32_t*>(stage + wv * 64 * 32 + 32 * (threadIdx.x & 63));
#pragma unroll
      for (int c = 0; c < 4; c++)
        *reinterpret_cast<u32x4*>(st + 4 * c) =
            u32x4{h[4 * c], h[4 * c + 1], h[4 * c + 2], h[4 * c + 3]};
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // the wave's vectors: vec0 .. vec0 + 64 / L - 1, the live ones first
      const int64_t vec0 = vb + j * VPB + wv * (64 / L);
      const int64_t n = nvec - vec0 < 64 / L ? nvec - vec0 : 64 / L;
      if (n > 0) {
        const int bytes = (int)n * PD * 2;
        uint8_t* const dst0 = reinterpret_cast<uint8_t*>(out + vec0 * PD);
        const uint8_t* const src0 = reinterpret_cast<const uint8_t*>(stage + wv * 64 * 32);
        const int lb = 16 * (threadIdx.x & 63);
#pragma unroll
        for (int k = 0; k < 4; k++)
          if (lb + 1024 * k < bytes)
            *reinterpret_cast<u32x4*>(dst0 + lb + 1024 * k) =
                *reinterpret_cast<const u32x4*>(src0 + lb + 1024 * k);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the next vectors rewrite the stage
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      continue;
    }
    const uint32_t r = hb + (uint32_t)(j * VPB) + threadIdx.x / L;
    const uint32_t dt = div_heads(p, r);
    _Float16* dst = out + (int64_t)(tb + dt) * p.out_stride_tok + (int64_t)hv[j] * p.row_dim +
                    32 * lane;
    if (p.vec_store) {  // 8 dims per 16-byte store
#pragma unroll
      for (int c = 0; c < 4; c++)
        *reinterpret_cast<u32x4*>(dst + 8 * c) =
            u32x4{h[4 * c], h[4 * c + 1], h[4 * c + 2], h[4 * c + 3]};
    } else {
#pragma unroll
      for (int i = 0; i < 32; i++)
        if (32 * lane + i < p.row_dim)
          dst[i] = __builtin_bit_cast(_Float16, (uint16_t)(h[i / 2] >> (16 * (i & 1))));
    }
  }
}

constexpr int kFreshPieces = 4;  // 8-element pieces per thread of a fresh-row workgroup

// fresh rows of a request, converted to fp16 (round to nearest) and padded
template <int PD>
__device__ __forceinline__ void copy_fresh(const ReadBackParams& p, const GatherReq& r, int blk) {
  constexpr int C = PD / 8;  // pieces per vector
  const int64_t pieces = (int64_t)r.fresh * p.H * C;
  const void* src = blockIdx.y ? p.value : p.key;
  const int64_t st = blockIdx.y ? p.v_st : p.k_st, sh = blockIdx.y ? p.v_sh : p.k_sh;
  _Float16* out = (blockIdx.y ? p.out_v : p.out_k) +
                  (int64_t)(r.dst_row + r.ctx) * p.out_stride_tok;
  const int64_t b0 = (int64_t)blk * (256 * kFreshPieces);
  const uint32_t tb = (uint32_t)(b0 / (p.H * C));  // first token of the workgroup (uniform)
  const uint32_t rb = (uint32_t)(b0 - (int64_t)tb * (p.H * C));
#pragma unroll
  for (int j = 0; j < kFreshPieces; j++) {
    const uint32_t i = (uint32_t)(j * 256) + threadIdx.x;
    if (b0 + i >= pieces) continue;
    const uint32_t x = rb + i, vec = x / C;  // vector from token tb on
    const uint32_t dt = div_heads(p, vec);
    const uint32_t head = vec - dt * (uint32_t)p.H;
    const int d = 8 * (int)(x % C);
    const int64_t off = (int64_t)(r.src_row + tb + dt) * st + (int64_t)head * sh + d;
    float f[8];
    u32x4 o = {0u, 0u, 0u, 0u};
    if (d < p.head_dim) {
      if (p.vec_load && p.dtype == TQ_F16) {
        o = *reinterpret_cast<const u32x4*>(static_cast<const _Float16*>(src) + off);
      } else {
        if (p.vec_load && p.dtype == TQ_BF16) {
          const u32x4 b = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(src) + off);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            f[2 * e] = __uint_as_float(b[e] << 16);
            f[2 * e + 1] = __uint_as_float(b[e] & 0xffff0000u);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            f[e] = 0.0f;
            if (d + e < p.head_dim)
              f[e] = p.dtype == TQ_F16 ? (float)static_cast<const _Float16*>(src)[off + e]
                     : p.dtype == TQ_BF16
                         ? __uint_as_float((uint32_t)static_cast<const uint16_t*>(src)[off + e] << 16)
                         : static_cast<const float*>(src)[off + e];
          }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = pack_h2(f[2 * e], f[2 * e + 1]);
      }
    }
    *reinterpret_cast<u32x4*>(out + (int64_t)(tb + dt) * p.out_stride_tok +
                              (int64_t)head * PD + d) = o;
  }
}

template <int PD, bool GATHER>
__global__ __launch_bounds__(256) void read_back_kernel(ReadBackParams p, int num_tokens) {
  __shared__ float cb[16];  // the codebook, indexed per lane
  __shared__ __attribute__((aligned(16))) _Float16 stage[4 * 64 * 32];
  if (threadIdx.x < 16) cb[threadIdx.x] = kCodebook[threadIdx.x];
  _Float16* out = blockIdx.y ? p.out_v : p.out_k;
  if constexpr (!GATHER) {
    read_back<PD>(p, p.pages, num_tokens, blockIdx.x, out, cb, stage);
  } else {
    const int blk = (int)blockIdx.x - p.ctx_blocks;
    if (blk < 0) {
      const int i = find_request(p.nreq, (int)blockIdx.x, [&](int r) { return p.reqs[r].ctx_blk; });
      const GatherReq& r = p.reqs[i];
      read_back<PD>(p, p.pages + (int64_t)r.bt_row * p.page_stride, r.ctx,
                    (int)blockIdx.x - r.ctx_blk, out + (int64_t)r.dst_row * p.out_stride_tok, cb,
                    stage);
    } else {
      const int i = find_request(p.nreq, blk, [&](int r) { return p.reqs[r].fresh_blk; });
      copy_fresh<PD>(p, p.reqs[i], blk - p.reqs[i].fresh_blk);
    }
  }
}

int check_geometry(const char* what, int pd, int head_dim, int H, int block_size,
                   int64_t num_blocks, int ebs) {
  if (pd != 64 && pd != 128 && pd != 256) {
    set_error("%s: padded_dim must be 64, 128 or 256, got %d", what, pd);
    return kEinval;
  }
  if (head_dim <= 0 || head_dim > pd || H <= 0 || block_size <= 0 || num_blocks < 0) {
    set_error("%s: bad sizes", what);
    return kEinval;
  }
  if (ebs % 16 != 0 || ebs < pd / 2 + 2 * (pd / 64)) {
    set_error("%s: ebs %d must be a multiple of 16 and >= %d", what, ebs, pd / 2 + 2 * (pd / 64));
    return kEinval;
  }
  return 0;
}

void fill_geometry(ReadBackParams& p, const uint8_t* k_slab, const uint8_t* v_slab,
                   const int32_t* pages, const float* signs, int H, int head_dim, int block_size,
                   int ebs, int64_t num_blocks) {
  p.k_slab = k_slab;
  p.v_slab = v_slab;
  p.pages = pages;
  p.page_stride = 0;
  p.signs = signs;
  p.num_blocks = num_blocks;
  p.H = H;
  p.hmul = H == 1 || H > 32768 ? 0u : (uint32_t)((((uint64_t)1 << 32) + H - 1) / H);
  p.head_dim = head_dim;
  p.block_size = block_size;
  p.block_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  p.ebs = ebs;
  p.key = p.value = nullptr;
  p.dtype = TQ_F16;
  p.k_st = p.k_sh = p.v_st = p.v_sh = 0;
  p.vec_load = false;
  p.nreq = p.ctx_blocks = 0;
}

template <bool GATHER>
hipError_t launch_read_back(int pd, dim3 grid, hipStream_t s, const ReadBackParams& p, int tokens) {
  if (pd == 64)
    hipLaunchKernelGGL((read_back_kernel<64, GATHER>), grid, dim3(256), 0, s, p, tokens);
  else if (pd == 128)
    hipLaunchKernelGGL((read_back_kernel<128, GATHER>), grid, dim3(256), 0, s, p, tokens);
  else
    hipLaunchKernelGGL((read_back_kernel<256, GATHER>), grid, dim3(256), 0, s, p, tokens);
  return hipGetLastError();
}

int64_t ctx_block_count(int64_t tokens, int H, int pd) {
  const int per = kVecsPerThread * (256 / (pd / 32));
  return (tokens * H + per - 1) / per;
}

}  // namespace
}  // namespace tq

extern "C" int tq_dequant_paged(const uint8_t* k_slab, const uint8_t* v_slab,
                                const int32_t* pages, int64_t num_tokens, int32_t num_kv_heads,
                                int32_t head_dim, int32_t padded_dim, int32_t block_size,
                                int32_t ebs, int64_t num_blocks, const float* signs,
                                void* out_k, void* out_v, int64_t out_stride_tok,
                                tq_stream_t stream) {
  using namespace tq;
  const int pd = padded_dim;
  const int rc = check_geometry("dequant", pd, head_dim, num_kv_heads, block_size, num_blocks, ebs);
  if (rc) return rc;
  if (num_tokens < 0) {
    set_error("dequant: bad sizes");
    return kEinval;
  }
  if (out_stride_tok < (int64_t)num_kv_heads * head_dim) {
    set_error("dequant: out_stride_tok %lld < num_kv_heads * head_dim", (long long)out_stride_tok);
    return kEinval;
  }
  if (num_tokens == 0) return 0;
  if (!k_slab || !v_slab || !pages || !out_k || !out_v) {
    set_error("dequant: null pointer");
    return kEinval;
  }
  const int64_t blocks = num_tokens > INT32_MAX ? INT64_MAX
                                                : ctx_block_count(num_tokens, num_kv_heads, pd);
  if (blocks > 0x7fffffffLL) {
    set_error("dequant: too many tokens");
    return kEinval;
  }
  ReadBackParams p;
  fill_geometry(p, k_slab, v_slab, pages, signs, num_kv_heads, head_dim, block_size, ebs,
                num_blocks);
  p.out_k = static_cast<_Float16*>(out_k);
  p.out_v = static_cast<_Float16*>(out_v);
  p.out_stride_tok = out_stride_tok;
  p.row_dim = head_dim;
  // full rows with 16-byte aligned dims: vector stores
  p.vec_store = head_dim == pd && out_stride_tok % 8 == 0 && (uintptr_t)out_k % 16 == 0 &&
                (uintptr_t)out_v % 16 == 0;
  const hipError_t e = launch_read_back<false>(pd, dim3((unsigned)blocks, 2),
                                               reinterpret_cast<hipStream_t>(stream), p,
                                               (int)num_tokens);
  if (e != hipSuccess) {
    set_error("dequant: launch failed: %s", hipGetErrorString(e));
    return (int)e;
  }
  return 0;
}

extern "C" int tq_prefill_gather(
    const uint8_t* k_slab, const uint8_t* v_slab, const int32_t* block_table,
    int64_t block_table_stride, int32_t num_kv_heads, int32_t head_dim, int32_t padded_dim,
    int32_t block_size, int32_t ebs, int64_t num_blocks, const float* signs, const void* key,
    const void* value, int32_t in_dtype, int64_t k_stride_tok, int64_t k_stride_head,
    int64_t v_stride_tok, int64_t v_stride_head, const int32_t* table_rows, const int32_t* ctx_lens,
    const int32_t* fresh_starts, const int32_t* fresh_lens, const int32_t* out_starts,
    int32_t num_requests, void* out_k, void* out_v, tq_stream_t stream) {
  using namespace tq;
  const char* what = "prefill_gather";
  const int pd = padded_dim;
  const int rc = check_geometry(what, pd, head_dim, num_kv_heads, block_size, num_blocks, ebs);
  if (rc) return rc;
  if (in_dtype != TQ_F32 && in_dtype != TQ_F16 && in_dtype != TQ_BF16) {
    set_error("%s: unsupported input dtype %d", what, in_dtype);
    return kEinval;
  }
  if (num_requests < 0) {
    set_error("%s: bad sizes", what);
    return kEinval;
  }
  if (num_requests == 0) return 0;
  if (!key || !value || !table_rows || !ctx_lens || !fresh_starts || !fresh_lens || !out_starts ||
      !out_k || !out_v) {
    set_error("%s: null pointer", what);
    return kEinval;
  }
  if ((((uintptr_t)out_k | (uintptr_t)out_v) & 15) != 0) {
    set_error("%s: out_k / out_v must be 16-byte aligned", what);
    return kEinval;
  }
  for (int i = 0; i < num_requests; i++) {
    if (ctx_lens[i] < 0 || fresh_lens[i] < 0 || fresh_starts[i] < 0 || out_starts[i] < 0 ||
        table_rows[i] < 0) {
      set_error("%s: bad request %d", what, i);
      return kEinval;
    }
    if (ctx_lens[i] > 0 && (!k_slab || !v_slab || !block_table)) {
      set_error("%s: null pointer", what);
      return kEinval;
    }
  }
  ReadBackParams p;
  fill_geometry(p, k_slab, v_slab, block_table, signs, num_kv_heads, head_dim, block_size, ebs,
                num_blocks);
  p.page_stride = block_table_stride;
  p.out_k = static_cast<_Float16*>(out_k);
  p.out_v = static_cast<_Float16*>(out_v);
  p.out_stride_tok = (int64_t)num_kv_heads * pd;
  p.row_dim = pd;
  p.vec_store = true;
  p.key = key;
  p.value = value;
  p.dtype = in_dtype;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.vec_load = in_dtype != TQ_F32 && head_dim % 8 == 0 && k_stride_tok % 8 == 0 &&
               k_stride_head % 8 == 0 && v_stride_tok % 8 == 0 && v_stride_head % 8 == 0 &&
               (((uintptr_t)key | (uintptr_t)value) & 15) == 0;
  for (int a = 0; a < num_requests; a += kMaxReqs) {
    p.nreq = num_requests - a < kMaxReqs ? num_requests - a : kMaxReqs;
    int64_t cblk = 0, fblk = 0;
    for (int i = 0; i < p.nreq; i++) {
      GatherReq& r = p.reqs[i];
      r.ctx = ctx_lens[a + i];
      r.fresh = fresh_lens[a + i];
      r.dst_row = out_starts[a + i];
      r.src_row = fresh_starts[a + i];
      r.bt_row = table_rows[a + i];
      r.ctx_blk = (int)cblk;
      r.fresh_blk = (int)fblk;
      cblk += ctx_block_count(r.ctx, num_kv_heads, pd);
      fblk += ((int64_t)r.fresh * num_kv_heads * (pd / 8) + 256 * kFreshPieces - 1) /
              (256 * kFreshPieces);
      if (cblk + fblk > 0x7fffffffLL) {
        set_error("%s: too many tokens", what);
        return kEinval;
      }
    }
    if (cblk + fblk == 0) continue;
    p.ctx_blocks = (int)cblk;
    const hipError_t e = launch_read_back<true>(pd, dim3((unsigned)(cblk + fblk), 2),
                                                reinterpret_cast<hipStream_t>(stream), p, 0);
    if (e != hipSuccess) {
      set_error("%s: launch failed: %s", what, hipGetErrorString(e));
      return (int)e;
    }
  }
  return 0;
}
