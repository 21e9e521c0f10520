// tq_prefill.hip -- causal GQA flash attention of a prefill chunk (fp16 K/V,
// head size 64, 128 or 256).
//
// Semantics: o[i, h] = softmax_j(q[i, h] . k[j, h / ratio] * sm_scale) v[j, h / ratio]
// over keys j <= (Lk - Lq) + i (causal, aligned to the end of the keys: a
// chunk of Lq new tokens whose keys are the Lk - Lq earlier tokens of its
// sequence followed by its own).  This is the attention the backend's prefill
// path needs (reference turboquant/vllm_backend_fused.py:335-371 runs it over
// the fresh chunk only, in flash-attn; TurboQuantFusedImpl here prepends the
// cached context read back from the quantized cache).
//
// gfx950 design:
//  * One workgroup = 32 NW query rows of one q head (NW waves x 32 rows,
//    NW = 8 when the grid of such blocks still fills the CUs, else 4); grid
//    (q heads, query blocks): the longest (last) query blocks are dispatched
//    first, and the q heads of one kv head are neighbours (their K/V tiles
//    are shared in L2).  Eight waves (one workgroup per CU at two waves per
//    SIMD) copy each K/V tile into LDS once for 256 rows instead of twice
//    for two workgroups of 128, and take 128-key tiles in the LDS that frees
//    (half the per-tile max, rescale and barrier steps): 7-9% faster on long
//    prompts than the four-wave, 64-key shape.
//  * Scores are computed transposed, S^T = K Q^T, with
//    v_mfma_f32_32x32x16_f16 (A = K rows from LDS, B = q columns held in
//    registers for the whole kernel): the C layout then gives each lane one
//    query row (lane % 32) and 16 key rows per 32-key block, so the softmax
//    max and sum are in-lane plus one permlane32 swap, and the lane's
//    probabilities are, in order, the B operand of O^T = V^T P^T (the MFMA's
//    reduction order is the C layout's row order; V^T is read in the same
//    order).  O^T's C layout again gives each lane its own query row, so the
//    online-softmax rescale is a per-lane scalar.
//  * K and V tiles (64 or 128 keys) stream into LDS as rows with
//    direct-to-LDS 16-byte copies, their 16-byte chunks XOR-swizzled by row:
//    the K reads (16 bytes of one row per lane, issued four MFMAs ahead of
//    their use) and the V transpose reads (ds_read_b64_tr_b16: four keys of
//    one dim per lane, the V^T operand without a transposing copy) are
//    conflict-free.  Two buffers of each (distinct LDS arrays, so the
//    compiler does not wait for the copies in flight into the other buffer),
//    one barrier per tile.
//  * The requests of a scheduler step run as one launch of work items (batch
//    mode, tq_prefill_attention_batch): five prompts of 229 .. 1326 tokens at
//    32 q heads take 52 us where five launches with their key splits and
//    merges took 125 us, chunks of 309 and 867 tokens over 5000 cached 140 against
//    175.
//  * Short chunks over long contexts (too few query blocks to fill the
//    CUs): each query block's tiles are split over several workgroups
//    (grid z), which leave their normalised O (fp16), reference max and row
//    sum in a caller-owned workspace; prefill_merge_kernel combines them.
//  * Online softmax in the exp2 domain with a lazy rescale (the running max
//    moves only when a tile exceeds it by more than 8 / scale); probabilities
//    enter the PV MFMA as fp16 (round to nearest), accumulation is fp32;
//    at head size 64 the row sum is taken from those fp16 values.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "tq_common.h"

namespace tq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// two floats as an fp16 pair, round to nearest even (one v_cvt_pk_f16_f32)
__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, half2_t));
}

constexpr int kBNmax = 128;  // largest tile (keys)

struct PrefillParams {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  _Float16* o;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, o_st, o_sh;  // strides in elements
  int lq, lk, ratio, nqb;
  float c;  // sm_scale * log2(e)
  // split-KV mode: workgroup z of a (head, query block) covers its tiles
  // [z tps, (z + 1) tps) and leaves its rows' O / row sum (fp16) and
  // (reference max in log2 units, row sum) in the workspace for
  // prefill_merge_kernel
  int nsplit, tps;
  _Float16* ws_o;  // [nsplit][lq][Hq][D]
  float* ws_ml;    // [nsplit][lq][Hq][2]
};

// Batch mode: the query blocks of several requests in one launch, as a list of
// work items (a kernel argument, so no device copy of the plan is needed).
// Item: query block qb (kBM rows) of request req over its key tiles [t0, t1);
// ws_row >= 0: the tiles are a share of the block's, O and (max, sum) of its
// rows go to the workspace rows from there for prefill_batch_merge_kernel.
//
// More items than the list holds (160: a prompt of 40,960 tokens, less where
// few heads need splits) go as one run of blocks per request, one workgroup row
// per block and grid z for its shares, which the workgroup works out by itself:
// still one launch, where lists of 160 one after the other leave the card to
// drain in between (48,000 tokens at 4 q heads 2.42 -> 2.26 ms, 30,000 at two
// 0.72 -> 0.49, 60,000 at one 1.83 -> 0.96).
struct PrefillReq {
  int q0, lq;  // first row in q and o, query rows
  int k0, lk;  // first row in the K / V source, keys
  int src;     // 0: k, v; 1: k2, v2
};
struct PrefillItem {
  uint32_t req_qb;  // req | qb << 6
  int t0, t1, ws_row;
};
struct PrefillRun {  // the blocks of a request, the last (longest) first
  int first, req;    // its first workgroup row
  int ws_row;        // share z of its query row i: workspace row ws_row + z lq + i
};
constexpr int kBatchReqs = 64, kBatchItems = 160;

// the shares of a block of `tiles` key tiles, of `unit` each but the last (0:
// blocks stay whole)
__host__ __device__ inline int split_shares(int tiles, int unit) {
  return unit == 0 ? 1 : (tiles + unit - 1) / unit;
}

// the run of workgroup row y: the last that starts at or before it
__device__ __forceinline__ PrefillRun find_run(const PrefillRun* runs, int n, int y) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (runs[mid].first <= y) lo = mid;
    else hi = mid - 1;
  }
  return runs[lo];
}

// key tiles that any row of query block qb sees
template <int kBM, int kBN>
__device__ __forceinline__ int block_tiles(const PrefillReq& rq, int qb) {
  return (rq.lk - rq.lq + min((qb + 1) * kBM, rq.lq) + kBN - 1) / kBN;
}
struct PrefillBatch {
  const void* q;
  const _Float16* k;
  const _Float16* v;
  const _Float16* k2;
  const _Float16* v2;
  void* o;
  int64_t q_st, q_sh, k_st, k_sh, v_st, v_sh, k2_st, k2_sh, o_st, o_sh;  // in elements
  int ratio, hd;      // hd <= kD: dims of q and o rows (zero padded to kD here)
  int q_bf16, o_bf16;  // q / o element type (else fp16)
  float c;             // sm_scale * log2(e)
  float* ws_o;         // [row][Hq][kD]
  float* ws_ml;        // [row][Hq][2]
  int nruns, unit, y0;  // runs (0: items), their split_shares unit, this launch's first row
  PrefillReq reqs[kBatchReqs];
  union {
    PrefillItem items[kBatchItems];
    PrefillRun runs[kBatchReqs];
  };
};
static_assert(sizeof(PrefillBatch) <= 4096, "kernel argument");
// The same argument read as runs: a type of its own, so that the list's kernels
// hold neither the search nor the choice (five prompts of 229 .. 1326 tokens
// 51.1 us; 51.8 with both in one kernel).
struct PrefillRuns : PrefillBatch {};

// eight bf16 as eight fp16, round to nearest even (exact in fp16's range)
__device__ __forceinline__ u32x4 bf16_to_f16(u32x4 x) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++)
    r[i] = pack_h2(__uint_as_float(x[i] << 16), __uint_as_float(x[i] & 0xffff0000u));
  return r;
}

// two floats as a bf16 pair, round to nearest even
__device__ __forceinline__ uint32_t pack_b2(float a, float b) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf2));
}

// max / sum of x over lanes l and l ^ 32: v_permlane32_swap of x with
// itself returns (x, x of lane l ^ 32) in some order in every lane
__device__ __forceinline__ float max32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// what one workgroup computes: rows qb kBM .. of a request (query rows from
// q_row0) over its key tiles [t0, t1)
struct PrefillWork {
  int qb, q_row0, lq, lk, t0, t1, ws_row, hd;  // t1 < 0: nothing
  const _Float16* k;
  const _Float16* v;
  int64_t k_st, k_sh, v_st, v_sh;
};

template <int kBM, int kBN, bool SPLIT>
__device__ __forceinline__ PrefillWork prefill_work(const PrefillParams& p) {
  PrefillWork r;
  r.qb = p.nqb - 1 - (int)blockIdx.y;
  r.q_row0 = 0;
  r.lq = p.lq;
  r.lk = p.lk;
  r.ws_row = -1;
  r.hd = 0;
  r.k = p.k;
  r.v = p.v;
  r.k_st = p.k_st;
  r.k_sh = p.k_sh;
  r.v_st = p.v_st;
  r.v_sh = p.v_sh;
  const int q0 = r.qb * kBM;
  const int kend = min(p.lk, p.lk - p.lq + min(q0 + kBM, p.lq));  // keys any row here sees
  r.t0 = 0;
  r.t1 = (kend + kBN - 1) / kBN;
  if constexpr (SPLIT) {
    r.t0 = (int)blockIdx.z * p.tps;
    r.t1 = min(r.t1, r.t0 + p.tps);
  }
  return r;
}

// the rows of the request that r's workgroup serves
__device__ __forceinline__ void request_of_work(const PrefillBatch& p, const PrefillReq& rq,
                                                PrefillWork& r) {
  r.q_row0 = rq.q0;
  r.lq = rq.lq;
  r.lk = rq.lk;
  r.hd = p.hd;
  r.k_st = rq.src ? p.k2_st : p.k_st;
  r.k_sh = rq.src ? p.k2_sh : p.k_sh;
  r.v_st = rq.src ? p.k2_st : p.v_st;
  r.v_sh = rq.src ? p.k2_sh : p.v_sh;
  r.k = (rq.src ? p.k2 : p.k) + (int64_t)rq.k0 * r.k_st;
  r.v = (rq.src ? p.v2 : p.v) + (int64_t)rq.k0 * r.v_st;
}

template <int kBM, int kBN, bool SPLIT>
__device__ __forceinline__ PrefillWork prefill_work(const PrefillBatch& p) {
  PrefillWork r;
  const PrefillItem it = p.items[blockIdx.y];
  r.qb = (int)(it.req_qb >> 6);
  r.t0 = it.t0;
  r.t1 = it.t1;
  r.ws_row = it.ws_row;
  request_of_work(p, p.reqs[it.req_qb & 63u], r);
  return r;
}

template <int kBM, int kBN, bool SPLIT>
__device__ __forceinline__ PrefillWork prefill_work(const PrefillRuns& p) {
  PrefillWork r;
  const int y = p.y0 + (int)blockIdx.y, z = (int)blockIdx.z;
  const PrefillRun run = find_run(p.runs, p.nruns, y);
  const PrefillReq rq = p.reqs[run.req];
  r.qb = (rq.lq + kBM - 1) / kBM - 1 - (y - run.first);
  const int tiles = block_tiles<kBM, kBN>(rq, r.qb), ns = split_shares(tiles, p.unit);
  r.t0 = z * p.unit;
  r.t1 = z >= ns ? -1 : ns > 1 ? min(tiles, r.t0 + p.unit) : tiles;
  r.ws_row = ns > 1 ? run.ws_row + z * rq.lq + r.qb * kBM : -1;
  request_of_work(p, rq, r);
  return r;
}

// The head of a workgroup.  Workgroups go to the 8 XCDs round robin, so with
// head = blockIdx.x the q heads of one kv head land on different XCDs and each
// of their L2s fetches the same K and V; taken this way an XCD serves
// consecutive heads, one kv head at 32 / 8.  Where few rows meet many keys that
// traffic is what bounds the kernel: 256 rows over 32,512 keys 168 -> 147 us (with
// fp16 partials then; 150 .. 153 with the fp32 ones of today), four chunks of 300
// over 8,000 with 64 / 8 heads 479 -> 397, six prompts of 1,300 121 -> 112; a 32k
// prompt is the same within noise, nothing slower.  Head counts off the 8 XCDs
// keep the plain order (no head order keeps them apart).
__device__ __forceinline__ int head_of_block() {
  const int x = blockIdx.x, hq = gridDim.x;
  return (hq & 7) == 0 ? (x & 7) * (hq >> 3) + (x >> 3) : x;
}

// WPE: waves per SIMD the register budget is sized for (2 at head size 64
// and 128; 1 at 256, whose q operand and output accumulators alone take 192
// registers per lane)
//
// PP: PrefillParams (one request, SPLIT: its split-KV mode), PrefillBatch or
// PrefillRuns.
template <int kD, int NW, int kBN, bool SPLIT, int WPE = 2, class PP = PrefillParams>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void prefill_kernel(PP p) {
  constexpr bool kBatch = std::is_base_of_v<PrefillBatch, PP>;
  constexpr int kKRow = kD * 2;       // bytes of one K row in LDS
  constexpr int kCH = kD / 8;         // 16-byte chunks per K row
  constexpr int kRPC = 1024 / kKRow;  // K rows per 1 KB copy
  constexpr int kBM = 32 * NW;  // query rows per workgroup
  constexpr int kNU = kBN / 32, kNS = kBN / 16;  // 32-key score blocks, 16-key PV steps
  // 64-byte quarters of a row the V swizzle rotates over (D >= 128: four;
  // 64: two)
  constexpr int kQS = kD >= 128 ? 0 : 1;  // row % 4 >> kQS selects the quarter
  __shared__ __attribute__((aligned(16))) uint8_t kbuf0[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t kbuf1[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t vbuf0[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t vbuf1[kBN * kKRow];

  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int hh = lane >> 5, n = lane & 31;
  const int head = head_of_block(), g = head / p.ratio;
  const PrefillWork wk = prefill_work<kBM, kBN, SPLIT>(p);
  if (std::is_same_v<PP, PrefillRuns> && wk.t1 < 0) return;
  const int q0 = wk.qb * kBM;
  const int off = wk.lk - wk.lq;
  const int qrow = q0 + 32 * w + n;  // this lane's query row (of its request)

  // q^T as the B operand of S^T = K Q^T: k-step s covers dims 16s .. 16s+15,
  // lane (hh, n) holds dims 16s + 8hh .. +7 of query row qrow
  half8_t qB[kD / 16];
  {
    const int64_t qo = (int64_t)(wk.q_row0 + qrow) * p.q_st + (int64_t)head * p.q_sh + 8 * hh;
    const _Float16* qp = static_cast<const _Float16*>(p.q) + qo;  // (bf16: the same size)
#pragma unroll
    for (int s = 0; s < kD / 16; s++) {
      u32x4 x = {0u, 0u, 0u, 0u};
      if (qrow < wk.lq && (!kBatch || 16 * s + 8 * hh < wk.hd))
        x = *reinterpret_cast<const u32x4*>(qp + 16 * s);
      if constexpr (kBatch)
        if (p.q_bf16) x = bf16_to_f16(x);
      qB[s] = __builtin_bit_cast(half8_t, x);
    }
  }

  // K and V copies: copy j fills LDS bytes [1024 j, 1024 j + 1024) of a
  // buffer = rows kRPC j .. kRPC j + kRPC - 1; lane l writes row
  // kRPC j + l / kCH, physical 16-byte chunk l % kCH.  K rows hold logical
  // chunk (l % kCH) ^ (row % kCH) there (the score MFMAs' A reads, 16 bytes
  // of one row per lane, hit distinct chunks); V rows hold logical chunk
  // (l % kCH) ^ 4 ((row % 4) >> kQS), which moves the 64-byte quarters of
  // four consecutive rows apart for the transpose reads of the PV MFMAs (and
  // lets their addresses be a per-lane base xor 64 d plus an immediate).
  // Wave w issues copies j = w + NW i of both.
  constexpr int kKC = (kBN / kRPC) / NW;  // copies per wave, tile and tensor
  const int kst_b = (int)(wk.k_st * 2), vst_b = (int)(wk.v_st * 2);
  uint32_t koff[kKC], voff[kKC];  // per-lane byte offsets of this wave's copies in a tile
#pragma unroll
  for (int i = 0; i < kKC; i++) {
    const int j = w + NW * i, row = kRPC * j + lane / kCH;
    koff[i] = (uint32_t)(row * kst_b + (((lane % kCH) ^ (row % kCH)) * 16));
    voff[i] = (uint32_t)(row * vst_b + (((lane % kCH) ^ (4 * ((row & 3) >> kQS))) * 16));
  }
  // buffer resource over rows [kb, Lk) of a K or V tile (wave-uniform base
  // and size; rows past Lk read as zeros)
  auto tile_rsrc = [&](const _Float16* base, int64_t st, int kb) {
    const int rows = min(kBN, wk.lk - kb);
    const uint64_t a = (uint64_t)(uintptr_t)(base + (int64_t)kb * st);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const int nrec = __builtin_amdgcn_readfirstlane(rows * (int)(st * 2));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)hi << 32) | lo),
                                             (short)0, nrec, 0x00020000);
  };
  const _Float16* const kbase = wk.k + (int64_t)g * wk.k_sh;
  const _Float16* const vbase = wk.v + (int64_t)g * wk.v_sh;
  auto issue = [&](int kt, uint8_t* kb, uint8_t* vb) {
#if defined(__HIP_DEVICE_COMPILE__)  // the LDS-copy builtin has no host form
    const __amdgpu_buffer_rsrc_t rk = tile_rsrc(kbase, wk.k_st, kt * kBN);
    const __amdgpu_buffer_rsrc_t rv = tile_rsrc(vbase, wk.v_st, kt * kBN);
#pragma unroll
    for (int i = 0; i < kKC; i++) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (void*)(kb + 1024 * (w + NW * i)), 16,
                                               koff[i], 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (void*)(vb + 1024 * (w + NW * i)), 16,
                                               voff[i], 0, 0, 0);
    }
#else
    (void)kt;
    (void)kb;
    (void)vb;
    (void)tile_rsrc;
    (void)kbase;
    (void)vbase;
#endif
  };
  // PV transpose reads (ds_read_b64_tr_b16): in each 16-lane group gq, source
  // lane s reads 4 halves V[K0 + s/4][D0 + 4 (s % 4) .. +3] and result lane i
  // receives V^T[D0 + i][K0 .. K0 + 3] (D0 = 32 d + 16 (gq % 2), K0 = 16 st +
  // 4 hh, plus 8 for the second read): the A operand of O^T = V^T P^T.
  // vread_base is this lane's byte offset for d = 0, st = 0.
  const int vgq = lane >> 4, vsl = lane & 15, vt4 = vsl >> 2;
  const uint32_t vread_base =
      (uint32_t)((4 * hh + vt4) * kKRow +
                 ((2 * (vgq & 1) + ((vsl & 3) >> 1)) ^ (4 * (vt4 >> kQS))) * 16 + 8 * (vsl & 1));

  f32x16 oacc[kD / 32];
#pragma unroll
  for (int d = 0; d < kD / 32; d++)
#pragma unroll
    for (int j = 0; j < 16; j++) oacc[d][j] = 0.0f;
  float m = -INFINITY, mc = -INFINITY, lsum = 0.0f;
  const int qlim = off + qrow;  // last key of this lane's row

  auto tile = [&](int kt, const uint8_t* kbuf, const uint8_t* vt) {
    const int kb = kt * kBN;
    // the wave's rows are q0 + 32w .. +31: nothing to do when all its keys
    // in this tile are beyond every row (uniform)
    if (kb > off + q0 + 32 * w + 31) return;
    // S^T blocks: MFMA i = s * kNU + u adds k-step s of key block u.  The K
    // fragments are read kKP ahead of their MFMA and the schedule is pinned
    // (one MFMA, then one read): left to itself the compiler issued each
    // read one or two MFMAs ahead and waited for it in full (1.5-2.5% slower)
    constexpr int kKP = 4;
    constexpr int kNI = kNU * (kD / 16);
    f32x16 sacc[kNU];
#pragma unroll
    for (int u = 0; u < kNU; u++)
#pragma unroll
      for (int j = 0; j < 16; j++) sacc[u][j] = 0.0f;
    auto kfrag = [&](int i) {
      const int u = i % kNU, s = i / kNU, row = 32 * u + n;
      return *reinterpret_cast<const u32x4*>(kbuf + row * kKRow +
                                             (((2 * s + hh) ^ (row % kCH)) * 16));
    };
    u32x4 fr[kKP];
#pragma unroll
    for (int j = 0; j < kKP; j++) fr[j] = kfrag(j);
#pragma unroll
    for (int i = 0; i < kNI; i++) {
      const u32x4 a = fr[i % kKP];
      if (i + kKP < kNI) fr[i % kKP] = kfrag(i + kKP);
      sacc[i % kNU] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          __builtin_bit_cast(half8_t, a), qB[i / kNU], sacc[i % kNU], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, kKP, 0);  // the first kKP reads
#pragma unroll
    for (int i = 0; i < kNI; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA i
      if (i + kKP < kNI) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // read i + kKP
    }
    // mask keys beyond the row (causal) or beyond Lk (uniform test): lim is
    // the lane's last visible key relative to key 4 hh of the tile, and the
    // score at tile key 4 hh + kk gets -inf (the sign bits of lim - kk spread
    // into 0xff800000) or +0 added; no compare masks, so no scalar registers
    // for them
    if (kb + kBN - 1 > off + q0 + 32 * w || kb + kBN > wk.lk) {
      const int lim = min(qlim, wk.lk - 1) - kb - 4 * hh;
#pragma unroll
      for (int u = 0; u < kNU; u++)
#pragma unroll
        for (int j = 0; j < 16; j++) {
          const int kk = 32 * u + 8 * (j >> 2) + (j & 3);
          sacc[u][j] += __int_as_float(((lim - kk) >> 31) & (int)0xff800000u);
        }
    }
    float tmax = -INFINITY;
#if defined(TQ_PREFILL_PROBE) && TQ_PREFILL_PROBE >= 2
    tmax = sacc[0][0];  // measurement probe: no row max
#else
#pragma unroll
    for (int u = 0; u < kNU; u++)
#pragma unroll
      for (int j = 0; j < 16; j++) tmax = fmaxf(tmax, sacc[u][j]);
    tmax = max32(tmax);
#endif
    const float m_new = fmaxf(m, tmax);
    // lazy rescale: p = exp2((s - m) c) stays below 2^8 between rescales
    if (__builtin_amdgcn_ballot_w64(m_new * p.c > mc + 8.0f) != 0) {
      const float alpha = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mc - m_new * p.c);
#pragma unroll
      for (int d = 0; d < kD / 32; d++) oacc[d] *= alpha;
      lsum *= alpha;
      m = m_new;
      mc = m_new * p.c;
    }
    // a row with no visible key yet (possible in split mode, where a split's
    // first tiles can lie wholly beyond a row) keeps mc = -inf while the
    // wave's ballot above may fire for other rows: its exponent offset is
    // then 0, so its probabilities are exp2(-inf) = 0 instead of NaN, and
    // the split leaves sum 0 and O = 0 for it
    const float mce = mc == -INFINITY ? 0.0f : mc;
    half8_t pB[kNS];  // B operand of O^T = V^T P^T for k-steps (u, t)
#pragma unroll
    for (int u = 0; u < kNU; u++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
        float pr[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
#if defined(TQ_PREFILL_PROBE) && TQ_PREFILL_PROBE >= 1
          pr[i] = __builtin_fmaf(sacc[u][8 * t + i], p.c, -mce);  // measurement probe: no exp2
#else
          pr[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[u][8 * t + i], p.c, -mce));
#endif
          if constexpr (kD != 64) lsum += pr[i];
        }
        u32x4 pk;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const half2_t h = __builtin_convertvector(f32x2{pr[2 * i], pr[2 * i + 1]}, half2_t);
          // head size 64 (two scores per MFMA, the softmax weighs more): the
          // row sum of the fp16 probabilities the PV MFMAs take, two per
          // v_dot2 against (1, 1) with an fp32 accumulator.  (Dot2 of an
          // element extracted from a u32x4 miscompiled here: the same source
          // register for all four; the sum reads the half2 values.)
          if constexpr (kD == 64)
            lsum = __builtin_amdgcn_fdot2(h, half2_t{(_Float16)1.0f, (_Float16)1.0f}, lsum, false);
          pk[i] = __builtin_bit_cast(uint32_t, h);
        }
        pB[2 * u + t] = __builtin_bit_cast(half8_t, pk);
      }
    // O^T += V^T P^T: k-step (u, t) reduces keys 32u + 16t + {4hh + 0..3,
    // 8 + 4hh + 0..3} (the C-layout rows of the lane's probabilities)
#pragma unroll
    for (int st = 0; st < kNS; st++) {
#pragma unroll
      for (int d = 0; d < kD / 32; d++) {
        typedef __attribute__((address_space(3))) uint8_t lds_u8;
        typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
        lds_u8* const pd = (lds_u8*)vt + (vread_base ^ (uint32_t)(64 * d)) + 16 * st * kKRow;
        const u32x2 a0 =
            __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)pd));
        const u32x2 a1 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(pd + 8 * kKRow)));
        const u32x4 a = {a0[0], a0[1], a1[0], a1[1]};
        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), pB[st],
                                                         oacc[d], 0, 0, 0);
      }
    }
  };

  // this workgroup's tiles: all of them, or split z's share
  const int t0 = wk.t0, t1 = wk.t1;
  if (t0 < t1) issue(t0, kbuf0, vbuf0);
  for (int kt = t0; kt < t1; kt += 2) {
    // tile kt: buffers 0
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's copies of tile kt
    __syncthreads();                     // everyone's copies of tile kt
    if (kt + 1 < t1) issue(kt + 1, kbuf1, vbuf1);
    tile(kt, kbuf0, vbuf0);
    if (kt + 1 >= t1) break;
    // tile kt + 1: buffers 1
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 2 < t1) issue(kt + 2, kbuf0, vbuf0);
    tile(kt + 1, kbuf1, vbuf1);
  }

  lsum = sum32(lsum);
  const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
  if (SPLIT || (kBatch && wk.ws_row >= 0)) {
    // this split's O / row sum and (mc, row sum); a split that held no visible
    // key for a row leaves mc = -inf, sum 0, O = 0.  One request: as fp16 (a
    // convex combination of V rows: safe).  Batch mode splits blocks that one
    // launch per request left whole, so what was a sum in fp32 stays one: fp32.
    if (qrow < wk.lq) {
      const int64_t r = (kBatch ? (int64_t)wk.ws_row + 32 * w + n
                                : (int64_t)blockIdx.z * wk.lq + qrow) * gridDim.x + head;
      if constexpr (kBatch) {
        float* const wo = p.ws_o + r * kD + 4 * hh;
#pragma unroll
        for (int d = 0; d < kD / 32; d++)
#pragma unroll
          for (int jq = 0; jq < 4; jq++)
            *reinterpret_cast<f32x4*>(wo + 32 * d + 8 * jq) =
                f32x4{oacc[d][4 * jq] * inv, oacc[d][4 * jq + 1] * inv, oacc[d][4 * jq + 2] * inv,
                      oacc[d][4 * jq + 3] * inv};
      } else {
        _Float16* const wo = p.ws_o + r * kD + 4 * hh;
#pragma unroll
        for (int d = 0; d < kD / 32; d++)
#pragma unroll
          for (int jq = 0; jq < 4; jq++) {
            const uint32_t lo = pack_h2(oacc[d][4 * jq] * inv, oacc[d][4 * jq + 1] * inv);
            const uint32_t hi = pack_h2(oacc[d][4 * jq + 2] * inv, oacc[d][4 * jq + 3] * inv);
            *reinterpret_cast<u32x2*>(wo + 32 * d + 8 * jq) = u32x2{lo, hi};
          }
      }
      if (hh == 0) *reinterpret_cast<f32x2*>(p.ws_ml + 2 * r) = f32x2{mc, lsum};
    }
    return;
  }

  // o = O / sum, lane (hh, n) holds dims 32d + 8jq + 4hh + 0..3 of row qrow
  if (qrow < wk.lq) {
    _Float16* op = static_cast<_Float16*>(p.o) + (int64_t)(wk.q_row0 + qrow) * p.o_st +
                   (int64_t)head * p.o_sh + 4 * hh;
#pragma unroll
    for (int d = 0; d < kD / 32; d++)
#pragma unroll
      for (int jq = 0; jq < 4; jq++) {
        const float f0 = oacc[d][4 * jq] * inv, f1 = oacc[d][4 * jq + 1] * inv;
        const float f2 = oacc[d][4 * jq + 2] * inv, f3 = oacc[d][4 * jq + 3] * inv;
        if (kBatch && 32 * d + 8 * jq + 4 * hh >= wk.hd) continue;
        u32x2 r = {pack_h2(f0, f1), pack_h2(f2, f3)};
        if constexpr (kBatch)
          if (p.o_bf16) r = u32x2{pack_b2(f0, f1), pack_b2(f2, f3)};
        *reinterpret_cast<u32x2*>(op + 32 * d + 8 * jq) = r;
      }
  }
}

// The same attention with RB row blocks of 32 query rows per wave: each K
// fragment and each V^T fragment read from LDS feeds RB MFMAs instead of
// one, so a tile's LDS reads per MFMA drop by RB.  Non-split only.  Row block
// rb of wave w holds rows q0 + 32 (RB w + rb) + n.  Used at head size 64
// (RB 2, 64-key tiles: 217 VGPRs, two waves per SIMD), where the registers
// of two row blocks fit; at head size 128 they do not (one wave per SIMD,
// measured slower).
template <int kD, int NW, int kBN, int RB, int WPE, class PP = PrefillParams>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void prefill_rb_kernel(PP p) {
  constexpr bool kBatch = std::is_base_of_v<PrefillBatch, PP>;
  constexpr int kKRow = kD * 2;
  constexpr int kCH = kD / 8;
  constexpr int kRPC = 1024 / kKRow;
  constexpr int kBM = 32 * NW * RB;
  constexpr int kNU = kBN / 32, kNS = kBN / 16;
  constexpr int kQS = kD >= 128 ? 0 : 1;
  __shared__ __attribute__((aligned(16))) uint8_t kbuf0[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t kbuf1[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t vbuf0[kBN * kKRow];
  __shared__ __attribute__((aligned(16))) uint8_t vbuf1[kBN * kKRow];

  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int hh = lane >> 5, n = lane & 31;
  const int head = head_of_block(), g = head / p.ratio;
  const PrefillWork wk = prefill_work<kBM, kBN, false>(p);
  const int q0 = wk.qb * kBM;
  const int off = wk.lk - wk.lq;
  const int wrow0 = q0 + 32 * RB * w;  // the wave's first row
  const int ntiles = wk.t1;

  half8_t qB[RB][kD / 16];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
    const int qrow = wrow0 + 32 * rb + n;
    const int64_t qo = (int64_t)(wk.q_row0 + qrow) * p.q_st + (int64_t)head * p.q_sh + 8 * hh;
    const _Float16* qp = static_cast<const _Float16*>(p.q) + qo;  // (bf16: the same size)
#pragma unroll
    for (int s = 0; s < kD / 16; s++) {
      u32x4 x = {0u, 0u, 0u, 0u};
      if (qrow < wk.lq && (!kBatch || 16 * s + 8 * hh < wk.hd))
        x = *reinterpret_cast<const u32x4*>(qp + 16 * s);
      if constexpr (kBatch)
        if (p.q_bf16) x = bf16_to_f16(x);
      qB[rb][s] = __builtin_bit_cast(half8_t, x);
    }
  }

  constexpr int kKC = (kBN / kRPC) / NW;
  const int kst_b = (int)(wk.k_st * 2), vst_b = (int)(wk.v_st * 2);
  uint32_t koff[kKC], voff[kKC];
#pragma unroll
  for (int i = 0; i < kKC; i++) {
    const int j = w + NW * i, row = kRPC * j + lane / kCH;
    koff[i] = (uint32_t)(row * kst_b + (((lane % kCH) ^ (row % kCH)) * 16));
    voff[i] = (uint32_t)(row * vst_b + (((lane % kCH) ^ (4 * ((row & 3) >> kQS))) * 16));
  }
  auto tile_rsrc = [&](const _Float16* base, int64_t st, int kb) {
    const int rows = min(kBN, wk.lk - kb);
    const uint64_t a = (uint64_t)(uintptr_t)(base + (int64_t)kb * st);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const int nrec = __builtin_amdgcn_readfirstlane(rows * (int)(st * 2));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)hi << 32) | lo),
                                             (short)0, nrec, 0x00020000);
  };
  const _Float16* const kbase = wk.k + (int64_t)g * wk.k_sh;
  const _Float16* const vbase = wk.v + (int64_t)g * wk.v_sh;
  auto issue = [&](int kt, uint8_t* kb, uint8_t* vb) {
#if defined(__HIP_DEVICE_COMPILE__)
    const __amdgpu_buffer_rsrc_t rk = tile_rsrc(kbase, wk.k_st, kt * kBN);
    const __amdgpu_buffer_rsrc_t rv = tile_rsrc(vbase, wk.v_st, kt * kBN);
#pragma unroll
    for (int i = 0; i < kKC; i++) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (void*)(kb + 1024 * (w + NW * i)), 16,
                                               koff[i], 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (void*)(vb + 1024 * (w + NW * i)), 16,
                                               voff[i], 0, 0, 0);
    }
#else
    (void)kt;
    (void)kb;
    (void)vb;
    (void)tile_rsrc;
    (void)kbase;
    (void)vbase;
#endif
  };
  const int vgq = lane >> 4, vsl = lane & 15, vt4 = vsl >> 2;
  const uint32_t vread_base =
      (uint32_t)((4 * hh + vt4) * kKRow +
                 ((2 * (vgq & 1) + ((vsl & 3) >> 1)) ^ (4 * (vt4 >> kQS))) * 16 + 8 * (vsl & 1));

  f32x16 oacc[RB][kD / 32];
  float m[RB], mc[RB], lsum[RB];
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
#pragma unroll
    for (int d = 0; d < kD / 32; d++)
#pragma unroll
      for (int j = 0; j < 16; j++) oacc[rb][d][j] = 0.0f;
    m[rb] = -INFINITY;
    mc[rb] = -INFINITY;
    lsum[rb] = 0.0f;
  }

  auto tile = [&](int kt, const uint8_t* kbuf, const uint8_t* vt) {
    const int kb = kt * kBN;
    if (kb > off + wrow0 + 32 * RB - 1) return;  // beyond every row of the wave
    constexpr int kKP = 4;
    constexpr int kNI = kNU * (kD / 16);
    f32x16 sacc[RB][kNU];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
      for (int u = 0; u < kNU; u++)
#pragma unroll
        for (int j = 0; j < 16; j++) sacc[rb][u][j] = 0.0f;
    auto kfrag = [&](int i) {
      const int u = i % kNU, s = i / kNU, row = 32 * u + n;
      return *reinterpret_cast<const u32x4*>(kbuf + row * kKRow +
                                             (((2 * s + hh) ^ (row % kCH)) * 16));
    };
    u32x4 fr[kKP];
#pragma unroll
    for (int j = 0; j < kKP; j++) fr[j] = kfrag(j);
#pragma unroll
    for (int i = 0; i < kNI; i++) {
      const u32x4 a = fr[i % kKP];
      if (i + kKP < kNI) fr[i % kKP] = kfrag(i + kKP);
#pragma unroll
      for (int rb = 0; rb < RB; rb++)
        sacc[rb][i % kNU] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            __builtin_bit_cast(half8_t, a), qB[rb][i / kNU], sacc[rb][i % kNU], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, kKP, 0);
#pragma unroll
    for (int i = 0; i < kNI; i++) {
      __builtin_amdgcn_sched_group_barrier(0x008, RB, 0);  // the RB MFMAs of read i
      if (i + kKP < kNI) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    half8_t pB[RB][kNS];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      const int rfirst = wrow0 + 32 * rb;
      if (kb + kBN - 1 > off + rfirst || kb + kBN > wk.lk) {
        const int lim = min(off + rfirst + n, wk.lk - 1) - kb - 4 * hh;
#pragma unroll
        for (int u = 0; u < kNU; u++)
#pragma unroll
          for (int j = 0; j < 16; j++) {
            const int kk = 32 * u + 8 * (j >> 2) + (j & 3);
            sacc[rb][u][j] += __int_as_float(((lim - kk) >> 31) & (int)0xff800000u);
          }
      }
      float tmax = -INFINITY;
#pragma unroll
      for (int u = 0; u < kNU; u++)
#pragma unroll
        for (int j = 0; j < 16; j++) tmax = fmaxf(tmax, sacc[rb][u][j]);
      tmax = max32(tmax);
      const float m_new = fmaxf(m[rb], tmax);
      if (__builtin_amdgcn_ballot_w64(m_new * p.c > mc[rb] + 8.0f) != 0) {
        const float alpha =
            m[rb] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mc[rb] - m_new * p.c);
#pragma unroll
        for (int d = 0; d < kD / 32; d++) oacc[rb][d] *= alpha;
        lsum[rb] *= alpha;
        m[rb] = m_new;
        mc[rb] = m_new * p.c;
      }
      const float mce = mc[rb] == -INFINITY ? 0.0f : mc[rb];
#pragma unroll
      for (int u = 0; u < kNU; u++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
          float pr[8];
#pragma unroll
          for (int i = 0; i < 8; i++) {
            pr[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[rb][u][8 * t + i], p.c, -mce));
            if constexpr (kD != 64) lsum[rb] += pr[i];
          }
          u32x4 pk;
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const half2_t h = __builtin_convertvector(f32x2{pr[2 * i], pr[2 * i + 1]}, half2_t);
            if constexpr (kD == 64)
              lsum[rb] = __builtin_amdgcn_fdot2(h, half2_t{(_Float16)1.0f, (_Float16)1.0f},
                                                lsum[rb], false);
            pk[i] = __builtin_bit_cast(uint32_t, h);
          }
          pB[rb][2 * u + t] = __builtin_bit_cast(half8_t, pk);
        }
    }
#pragma unroll
    for (int st = 0; st < kNS; st++) {
#pragma unroll
      for (int d = 0; d < kD / 32; d++) {
        typedef __attribute__((address_space(3))) uint8_t lds_u8;
        typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
        lds_u8* const pd = (lds_u8*)vt + (vread_base ^ (uint32_t)(64 * d)) + 16 * st * kKRow;
        const u32x2 a0 =
            __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)pd));
        const u32x2 a1 = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(pd + 8 * kKRow)));
        const u32x4 a = {a0[0], a0[1], a1[0], a1[1]};
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
          oacc[rb][d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              __builtin_bit_cast(half8_t, a), pB[rb][st], oacc[rb][d], 0, 0, 0);
      }
    }
  };

  if (ntiles > 0) issue(0, kbuf0, vbuf0);
  for (int kt = 0; kt < ntiles; kt += 2) {
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 1 < ntiles) issue(kt + 1, kbuf1, vbuf1);
    tile(kt, kbuf0, vbuf0);
    if (kt + 1 >= ntiles) break;
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (kt + 2 < ntiles) issue(kt + 2, kbuf0, vbuf0);
    tile(kt + 1, kbuf1, vbuf1);
  }

#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
    const int qrow = wrow0 + 32 * rb + n;
    const float ls = sum32(lsum[rb]);
    if (qrow < wk.lq) {
      const float inv = ls > 0.0f ? 1.0f / ls : 0.0f;
      _Float16* op = static_cast<_Float16*>(p.o) + (int64_t)(wk.q_row0 + qrow) * p.o_st +
                     (int64_t)head * p.o_sh + 4 * hh;
#pragma unroll
      for (int d = 0; d < kD / 32; d++)
#pragma unroll
        for (int jq = 0; jq < 4; jq++) {
          const float f0 = oacc[rb][d][4 * jq] * inv, f1 = oacc[rb][d][4 * jq + 1] * inv;
          const float f2 = oacc[rb][d][4 * jq + 2] * inv, f3 = oacc[rb][d][4 * jq + 3] * inv;
          if (kBatch && 32 * d + 8 * jq + 4 * hh >= wk.hd) continue;
          u32x2 r = {pack_h2(f0, f1), pack_h2(f2, f3)};
          if constexpr (kBatch)
            if (p.o_bf16) r = u32x2{pack_b2(f0, f1), pack_b2(f2, f3)};
          *reinterpret_cast<u32x2*>(op + 32 * d + 8 * jq) = r;
        }
    }
  }
}

// Merge of the splits of split-KV mode: one wave per (query row, q head),
// o = sum_z w_z (O_z / l_z) / sum_z w_z, w_z = 2^(mc_z - M) l_z, fp16 out.
template <int kD>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillParams p, int hq) {
  constexpr int V = kD / 64;  // dims per lane
  const int lane = threadIdx.x & 63;
  const int64_t idx = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // row * hq + head
  if (idx >= (int64_t)p.lq * hq) return;
  const int row = (int)(idx / hq), head = (int)(idx % hq);
  const int64_t zs = (int64_t)p.lq * hq;  // rows of one split
  float mx = -INFINITY;
  for (int z = 0; z < p.nsplit; z++) mx = fmaxf(mx, p.ws_ml[2 * (z * zs + idx)]);
  float den = 0.0f, acc[V];
#pragma unroll
  for (int i = 0; i < V; i++) acc[i] = 0.0f;
  for (int z = 0; z < p.nsplit; z++) {
    const f32x2 ml = *reinterpret_cast<const f32x2*>(p.ws_ml + 2 * (z * zs + idx));
    if (ml[0] == -INFINITY) continue;  // no visible key in this split
    const float wgt = __builtin_amdgcn_exp2f(ml[0] - mx) * ml[1];
    den += wgt;
    const _Float16* const src = p.ws_o + (z * zs + idx) * kD + V * lane;
#pragma unroll
    for (int i = 0; i < V; i++) acc[i] += wgt * (float)src[i];
  }
  const float inv = den > 0.0f ? 1.0f / den : 0.0f;
  _Float16* const op = p.o + (int64_t)row * p.o_st + (int64_t)head * p.o_sh + V * lane;
#pragma unroll
  for (int i = 0; i < V; i++) op[i] = (_Float16)(acc[i] * inv);
}

// Merge of the split query blocks of a batch: D / 8 lanes per (row, q head), 8
// dims (16 bytes) each, the same weights as above.
struct PrefillGroup {
  int q_row, ws_row;  // the block's first row in o, and in the workspace
  int stride;         // workspace rows from one share to the next
  uint16_t nsplit, rows;
};
struct PrefillMerge {
  void* o;
  int64_t o_st, o_sh;
  int hq, hd, o_bf16;
  const float* ws_o;
  const float* ws_ml;
  int nruns, unit, y0;  // as in PrefillBatch
  union {
    PrefillGroup groups[kBatchItems];
    struct {
      PrefillReq reqs[kBatchReqs];
      PrefillRun runs[kBatchReqs];
    };
  };
};

template <int kD>
__global__ __launch_bounds__(256) void prefill_batch_merge_kernel(PrefillMerge p) {
  constexpr int L = kD / 8, kVecs = 256 / L;
  PrefillGroup g;
  if (p.nruns == 0) {
    g = p.groups[blockIdx.y];
  } else {
    constexpr int kBM = 128, kBN = 64;  // what splits blocks
    const int y = p.y0 + (int)blockIdx.y;
    const PrefillRun run = find_run(p.runs, p.nruns, y);
    const PrefillReq rq = p.reqs[run.req];
    const int qb = (rq.lq + kBM - 1) / kBM - 1 - (y - run.first);
    g.nsplit = (uint16_t)split_shares(block_tiles<kBM, kBN>(rq, qb), p.unit);
    if (g.nsplit < 2) return;
    g.q_row = rq.q0 + qb * kBM;
    g.ws_row = run.ws_row + qb * kBM;
    g.stride = rq.lq;
    g.rows = (uint16_t)min(kBM, rq.lq - qb * kBM);
  }
  const int idx = (int)blockIdx.x * kVecs + (int)threadIdx.x / L;  // row * hq + head
  const int c = 8 * ((int)threadIdx.x % L);
  if (idx >= g.rows * p.hq) return;
  const int row = idx / p.hq, head = idx % p.hq;
  const int64_t zs = (int64_t)g.stride * p.hq;  // vectors from share to share
  const int64_t v0 = (int64_t)g.ws_row * p.hq + idx;
  float mx = -INFINITY;
  for (int z = 0; z < g.nsplit; z++) mx = fmaxf(mx, p.ws_ml[2 * (v0 + z * zs)]);
  float den = 0.0f, acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++) acc[i] = 0.0f;
#pragma unroll 4
  for (int z = 0; z < g.nsplit; z++) {
    const f32x2 ml = *reinterpret_cast<const f32x2*>(p.ws_ml + 2 * (v0 + z * zs));
    const f32x4* const x = reinterpret_cast<const f32x4*>(p.ws_o + (v0 + z * zs) * kD + c);
    const f32x4 x0 = x[0], x1 = x[1];
    // a split without a visible key for the row has weight 0 (its O is 0)
    const float wgt = ml[0] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[0] - mx) * ml[1];
    den += wgt;
#pragma unroll
    for (int i = 0; i < 8; i++) acc[i] = __builtin_fmaf(wgt, i < 4 ? x0[i] : x1[i - 4], acc[i]);
  }
  if (c >= p.hd) return;
  const float inv = den > 0.0f ? 1.0f / den : 0.0f;
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; i++)
    r[i] = p.o_bf16 ? pack_b2(acc[2 * i] * inv, acc[2 * i + 1] * inv)
                    : pack_h2(acc[2 * i] * inv, acc[2 * i + 1] * inv);
  *reinterpret_cast<u32x4*>(static_cast<_Float16*>(p.o) + (int64_t)(g.q_row + row) * p.o_st +
                            (int64_t)head * p.o_sh + c) = r;
}

// the workgroup shapes, at head size 64 or 128: 256 query rows (eight waves
// with 128-key tiles at head size 128; four waves of two row blocks with
// 64-key tiles at head size 64); four waves, 64-key tiles; four waves split
// over the keys (then merged).
// Head size 256: four waves, 64-key tiles (128 KB of LDS for the K and V
// double buffers), one wave per SIMD, split or not.
template <int D>
hipError_t launch_prefill(int nw, int heads, hipStream_t st, const PrefillParams& p) {
  if constexpr (D == 256) {
    (void)nw;
    if (p.nsplit <= 1) {
      hipLaunchKernelGGL((prefill_kernel<D, 4, 64, false, 1>), dim3(heads, p.nqb), dim3(256), 0,
                         st, p);
    } else {
      hipLaunchKernelGGL((prefill_kernel<D, 4, 64, true, 1>), dim3(heads, p.nqb, p.nsplit),
                         dim3(256), 0, st, p);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      const int64_t waves = (int64_t)p.lq * heads;
      hipLaunchKernelGGL((prefill_merge_kernel<D>), dim3((unsigned)((waves + 3) / 4)), dim3(256),
                         0, st, p, heads);
    }
  } else if (nw == 8) {
    if constexpr (D == 64)  // four waves of 64 rows (two row blocks each), 64-key tiles
      hipLaunchKernelGGL((prefill_rb_kernel<D, 4, 64, 2, 2>), dim3(heads, p.nqb), dim3(256), 0, st,
                         p);
    else
      hipLaunchKernelGGL((prefill_kernel<D, 8, 128, false>), dim3(heads, p.nqb), dim3(512), 0, st,
                         p);
  } else if (p.nsplit <= 1) {
    hipLaunchKernelGGL((prefill_kernel<D, 4, 64, false>), dim3(heads, p.nqb), dim3(256), 0, st,
                       p);
  } else {
    hipLaunchKernelGGL((prefill_kernel<D, 4, 64, true>), dim3(heads, p.nqb, p.nsplit), dim3(256),
                       0, st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t waves = (int64_t)p.lq * heads;
    hipLaunchKernelGGL((prefill_merge_kernel<D>), dim3((unsigned)((waves + 3) / 4)), dim3(256),
                       0, st, p, heads);
  }
  return hipGetLastError();
}


// Launch plan of one call: the workgroup shape and, when the grid would
// leave CUs idle (short chunks over long contexts), a split of the keys.
struct PrefillPlan {
  int nw = 4, nqb = 0, nsplit = 1, tps = 0;
  int64_t ws_bytes = 0;  // workspace the split needs (0: none)
};
PrefillPlan plan_prefill(int q_len, int kv_len, int heads, int head_dim) {
  PrefillPlan sp;
  const int cus = device_cus();
  const int64_t nqb8 = (q_len + 255) / 256;
  if (head_dim != 256 && (int64_t)heads * nqb8 >= (int64_t)cus) {
    // 256-row workgroups (8 waves, one per CU) when they still give every CU one
    sp.nw = 8;
    sp.nqb = (int)nqb8;
    return sp;
  }
  // else 128-row workgroups (4 waves, two per CU; one at head size 256);
  // with fewer than two per CU, the keys of each query block are split so that the grid fills the
  // chip, each split at least 8 tiles (512 keys)
  sp.nqb = (q_len + 127) / 128;
  const int64_t wgs = (int64_t)heads * sp.nqb;
  const int ntl = (kv_len + 63) / 64;  // tiles of the last (longest) query block
  if (cus > 0 && wgs < 2LL * cus && ntl >= 16) {
    int64_t S = (2LL * cus + wgs - 1) / wgs;
    if (S > ntl / 8) S = ntl / 8;
    if (S > 64) S = 64;
    if (S >= 2) {
      sp.tps = (int)((ntl + S - 1) / S);
      sp.nsplit = (ntl + sp.tps - 1) / sp.tps;
      sp.ws_bytes = (int64_t)sp.nsplit * q_len * heads * (head_dim * 2 + 8);
    }
  }
  return sp;
}

// Plan of one batch of at most kBatchReqs requests: its items (longest first)
// and the split query blocks, or its runs.
struct BatchPlan {
  int nw = 4;
  int ws_rows = 0;
  std::vector<PrefillItem> items;
  std::vector<PrefillGroup> groups;  // q_row: of the request (group_req)
  std::vector<int> group_req;
  std::vector<PrefillRun> runs;  // not empty: instead of items and groups
  int unit = 0, shares = 1, rows = 0;  // of the runs: unit, most shares of a block, blocks
};

struct QueryBlock {
  int req, qb, tiles;
};

// Time of a list of items (tiles each, longest first) in tiles: `groups` sets
// of workgroup slots, one workgroup per q head in each, take the items in
// turn as they fall free; an item costs its tiles and about one for its start.
template <class Tiles>
double batch_time(size_t n, double groups, Tiles tiles) {
  if (groups < 1.0) groups = 1.0;
  double total = 0.0;
  if (n > 512 || n <= groups) {
    for (size_t i = 0; i < n; i++) total += tiles(i) + 1.0;
    return n == 0 ? 0.0 : std::max(tiles(0) + 1.0, total / groups);
  }
  std::vector<double> busy((size_t)groups, 0.0);  // a heap, the first to fall free on top
  auto later = [](double x, double y) { return x > y; };
  for (size_t i = 0; i < n; i++) {
    std::pop_heap(busy.begin(), busy.end(), later);
    busy.back() += tiles(i) + 1.0;
    total = std::max(total, busy.back());
    std::push_heap(busy.begin(), busy.end(), later);
  }
  return total;
}

std::vector<QueryBlock> query_blocks(const int32_t* q_lens, const int32_t* kv_lens, int nreq,
                                     int bm, int bn) {
  std::vector<QueryBlock> blocks;
  for (int i = 0; i < nreq; i++)
    for (int qb = 0; (int64_t)qb * bm < q_lens[i]; qb++) {
      const int kend = kv_lens[i] - q_lens[i] + std::min((qb + 1) * bm, q_lens[i]);
      blocks.push_back({i, qb, (kend + bn - 1) / bn});
    }
  std::stable_sort(blocks.begin(), blocks.end(),
                   [](const QueryBlock& x, const QueryBlock& y) { return x.tiles > y.tiles; });
  return blocks;
}

// Shape and splits by estimated time.  Measured at 32 q heads, head size 128
// on 256 CUs: a 256-row, 128-key tile takes 3.84 us of a CU (one workgroup),
// a 128-row, 64-key tile 2.1 us (two resident); at head size 64 both shapes
// run two workgroups per CU, 2.15 and 1.15 us a tile.  So 256-row blocks win
// where they waste few rows and fill whole rounds (2048 tokens over 30k: 947
// against 1008 us; a 4096-token prompt 140 against 152 us) and 128-row blocks
// elsewhere (five prompts of 229 .. 1326 tokens 55 against 61 us; six of 1300
// 126 against 147 us).  Splitting the keys of 128-row blocks pays where few
// blocks leave slots idle (256 tokens over 32k: 155 against 669 us) and costs
// the merge, 4 .. 9 us.
BatchPlan plan_batch(const int32_t* q_lens, const int32_t* kv_lens, int nreq, int heads,
                     int head_dim) {
  BatchPlan bp;
  const double cus = device_cus() > 0 ? device_cus() : 256;
  std::vector<QueryBlock> blocks = query_blocks(q_lens, kv_lens, nreq, 128, 64);
  const double groups = (head_dim == 256 ? 1.0 : 2.0) * cus / heads;
  int64_t total = 0;
  for (const QueryBlock& b : blocks) total += b.tiles;
  // the parts of a block of t tiles at most `unit` tiles each
  auto parts = [](int t, double unit) {
    return t > 1.25 * unit ? (int)std::ceil(t / unit) : 1;
  };
  double best = batch_time(blocks.size(), groups, [&](size_t i) { return blocks[i].tiles; });
  double unit = 1e30;
  int run_unit = 0;                              // not 0: split in runs, by this unit
  bool long_list = blocks.size() > kBatchItems;  // a split does not fit the list
  if (!blocks.empty() && !long_list && blocks.size() <= 4 * groups) {
    const double even = std::max(8.0, total / groups);  // tiles per slot, at least 512 keys
    for (const double f : {1.5, 1.05, 0.8, 0.5}) {
      const double u = std::max(8.0, f * even);
      int slots = 0;
      std::vector<double> cost;
      for (const QueryBlock& b : blocks) {
        const int ns = parts(b.tiles, u);
        if (ns > 1) slots += ns;
        cost.insert(cost.end(), ns, (double)((b.tiles + ns - 1) / ns));
      }
      if (slots == 0) continue;
      if (cost.size() > kBatchItems) {
        long_list = true;
        continue;
      }
      std::sort(cost.begin(), cost.end(), [](double x, double y) { return x > y; });
      // the merge: its launch and the slots' rows written and read
      const double t = batch_time(cost.size(), groups, [&](size_t i) { return cost[i]; }) + 2.0 +
                       0.3 * slots * heads / 32.0;
      if (t < best) {
        best = t;
        unit = u;
      }
    }
  }
  const int64_t wgs = (int64_t)blocks.size() * heads;
  if (long_list && wgs < 2 * cus && blocks[0].tiles >= 16) {
    // splits in runs: as many shares of the longest block as give every CU two
    // workgroups, each at least 8 tiles; shares of one size start longest
    // first and the remainders fill in behind them
    const int most = blocks[0].tiles;
    const int ns = (int)std::min<int64_t>(((int64_t)(2 * cus) + wgs - 1) / wgs, most / 8);
    const int u = (most + ns - 1) / ns;
    int slots = 0, items = 0;
    for (const QueryBlock& b : blocks) {
      const int n = split_shares(b.tiles, u);
      items += n;
      if (n > 1) slots += n;
    }
    // (so many shares that the merge is bound by their bytes, 0.04 us per 128
    // rows of a head written and read)
    const double t = std::max(u + 1.0, (total + items) / groups) + 2.0 + 0.6 * slots * heads / 32.0;
    if (slots > 0 && t < best) {
      best = t;
      run_unit = u;
    }
  }
  if (head_dim != 256) {
    const std::vector<QueryBlock> wide =
        query_blocks(q_lens, kv_lens, nreq, 256, head_dim == 128 ? 128 : 64);
    const double t = batch_time(wide.size(), (head_dim == 128 ? 1.0 : 2.0) * cus / heads,
                                [&](size_t i) { return wide[i].tiles; });
    if (head_dim == 128 ? t * 3.84 <= best * 2.1 : t * 2.15 <= best * 1.15) {
      bp.nw = 8;
      unit = 1e30;
      run_unit = 0;
      blocks = wide;
    }
  }
  const int bm = bp.nw == 8 ? 256 : 128;
  if (run_unit || blocks.size() > kBatchItems) {
    bp.unit = run_unit;
    std::vector<int> shares(nreq, 0);  // of a request's longest block, which comes first
    for (const QueryBlock& b : blocks) {
      if (shares[b.req]) continue;
      const int ns = shares[b.req] = split_shares(b.tiles, bp.unit);
      bp.runs.push_back({bp.rows, b.req, bp.ws_rows});
      bp.rows += (q_lens[b.req] + bm - 1) / bm;
      bp.shares = std::max(bp.shares, ns);
      if (ns > 1) bp.ws_rows += ns * q_lens[b.req];
    }
    return bp;
  }
  for (const QueryBlock& b : blocks) {
    int ns = parts(b.tiles, unit);
    const int per = (b.tiles + ns - 1) / ns;
    ns = (b.tiles + per - 1) / per;
    const int row0 = bp.ws_rows, rows = std::min(bm, q_lens[b.req] - b.qb * bm);
    for (int z = 0; z < ns; z++)
      bp.items.push_back({(uint32_t)b.req | (uint32_t)b.qb << 6, z * per,
                          std::min(b.tiles, (z + 1) * per), ns > 1 ? row0 + rows * z : -1});
    if (ns > 1) {
      bp.ws_rows += rows * ns;
      bp.groups.push_back({b.qb * bm, row0, rows, (uint16_t)ns, (uint16_t)rows});
      bp.group_req.push_back(b.req);
    }
  }
  std::stable_sort(bp.items.begin(), bp.items.end(), [](const PrefillItem& x, const PrefillItem& y) {
    return x.t1 - x.t0 > y.t1 - y.t0;
  });
  return bp;
}

constexpr int kGridRows = 65535;  // workgroup rows of one launch

template <int D, class PP>
void launch_batch_kernel(int nw, dim3 grid, hipStream_t st, const PP& p) {
  if (nw == 8) {
    if constexpr (D == 64)
      hipLaunchKernelGGL((prefill_rb_kernel<D, 4, 64, 2, 2, PP>), grid, dim3(256), 0, st, p);
    else if constexpr (D == 128)
      hipLaunchKernelGGL((prefill_kernel<D, 8, 128, false, 2, PP>), grid, dim3(512), 0, st, p);
  } else {
    hipLaunchKernelGGL((prefill_kernel<D, 4, 64, false, D == 256 ? 1 : 2, PP>), grid, dim3(256), 0,
                       st, p);
  }
}

template <int D>
hipError_t launch_batch(const BatchPlan& bp, int heads, hipStream_t st, PrefillBatch& p) {
  const int nrows = bp.runs.empty() ? (int)bp.items.size() : bp.rows;
  p.nruns = (int)bp.runs.size();
  p.unit = bp.unit;
  if (p.nruns) std::copy(bp.runs.begin(), bp.runs.end(), p.runs);
  else std::copy(bp.items.begin(), bp.items.end(), p.items);
  for (p.y0 = 0; p.y0 < nrows; p.y0 += kGridRows) {
    const dim3 grid(heads, std::min(kGridRows, nrows - p.y0), bp.shares);
    if (p.nruns) launch_batch_kernel<D>(bp.nw, grid, st, PrefillRuns{p});
    else launch_batch_kernel<D>(bp.nw, grid, st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (bp.ws_rows == 0) return hipSuccess;
  PrefillMerge m = {};
  m.o = p.o;
  m.o_st = p.o_st;
  m.o_sh = p.o_sh;
  m.hq = heads;
  m.hd = p.hd;
  m.o_bf16 = p.o_bf16;
  m.ws_o = p.ws_o;
  m.ws_ml = p.ws_ml;
  m.nruns = p.nruns;
  m.unit = p.unit;
  int ngroups = bp.rows, rows = 128;
  if (p.nruns) {
    std::copy(p.reqs, p.reqs + kBatchReqs, m.reqs);
    std::copy(bp.runs.begin(), bp.runs.end(), m.runs);
  } else {
    ngroups = (int)bp.groups.size();
    rows = 0;
    for (int i = 0; i < ngroups; i++) {
      m.groups[i] = bp.groups[i];
      m.groups[i].q_row += p.reqs[bp.group_req[i]].q0;
      rows = std::max<int>(rows, m.groups[i].rows);
    }
  }
  constexpr int kVecs = 256 / (D / 8);
  for (m.y0 = 0; m.y0 < ngroups; m.y0 += kGridRows) {
    hipLaunchKernelGGL((prefill_batch_merge_kernel<D>),
                       dim3((rows * heads + kVecs - 1) / kVecs, std::min(kGridRows, ngroups - m.y0)),
                       dim3(256), 0, st, m);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// workspace of a plan: O rows, then (max, sum) pairs
int64_t batch_ws_bytes(const BatchPlan& bp, int heads, int head_dim) {
  return (int64_t)bp.ws_rows * heads * (head_dim * 4 + 8);
}

bool batch_sizes_ok(const int32_t* q_lens, const int32_t* kv_lens, int32_t nreq, int32_t heads,
                    int32_t head_dim) {
  if (nreq < 0 || heads <= 0 || (nreq > 0 && (!q_lens || !kv_lens)) ||
      (head_dim != 64 && head_dim != 128 && head_dim != 256))
    return false;
  for (int i = 0; i < nreq; i++)
    if (q_lens[i] < 0 || kv_lens[i] < q_lens[i] || q_lens[i] > (1 << 26)) return false;
  return true;
}

}  // namespace
}  // namespace tq

extern "C" int64_t tq_prefill_batch_workspace_bytes(const int32_t* q_lens, const int32_t* kv_lens,
                                                    int32_t num_requests, int32_t num_qo_heads,
                                                    int32_t padded_dim) {
  using namespace tq;
  if (!batch_sizes_ok(q_lens, kv_lens, num_requests, num_qo_heads, padded_dim)) return 0;
  int64_t most = 0;
  try {
    for (int a = 0; a < num_requests; a += kBatchReqs)
      most = std::max(most, batch_ws_bytes(plan_batch(q_lens + a, kv_lens + a,
                                                      std::min(kBatchReqs, num_requests - a),
                                                      num_qo_heads, padded_dim),
                                           num_qo_heads, padded_dim));
  } catch (...) {
    return 0;
  }
  return most;
}

extern "C" int tq_prefill_attention_batch(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, int32_t q_dtype, const void* k,
    int64_t k_stride_tok, int64_t k_stride_head, const void* v, int64_t v_stride_tok,
    int64_t v_stride_head, const void* k2, const void* v2, int64_t k2_stride_tok,
    int64_t k2_stride_head, void* o, int64_t o_stride_tok, int64_t o_stride_head, int32_t o_dtype,
    const int32_t* q_starts, const int32_t* q_lens, const int32_t* kv_starts,
    const int32_t* kv_lens, const int32_t* kv_sources, int32_t num_requests, int32_t num_qo_heads,
    int32_t num_kv_heads, int32_t head_dim, int32_t padded_dim, float sm_scale, void* workspace,
    int64_t workspace_bytes, tq_stream_t stream) {
  using namespace tq;
  const char* what = "prefill_attention_batch";
  if (!batch_sizes_ok(q_lens, kv_lens, num_requests, num_qo_heads, padded_dim)) {
    set_error("%s: bad sizes (padded_dim 64, 128 or 256; 0 <= q_len <= kv_len)", what);
    return kEinval;
  }
  if (num_kv_heads <= 0 || num_qo_heads % num_kv_heads != 0) {
    set_error("%s: num_qo_heads %d not a multiple of num_kv_heads %d", what, num_qo_heads,
              num_kv_heads);
    return kEinval;
  }
  if (head_dim <= 0 || head_dim > padded_dim || head_dim % 8 != 0) {
    set_error("%s: head_dim %d must be a multiple of 8 up to padded_dim", what, head_dim);
    return kEinval;
  }
  if ((q_dtype != TQ_F16 && q_dtype != TQ_BF16) || (o_dtype != TQ_F16 && o_dtype != TQ_BF16)) {
    set_error("%s: q and o must be fp16 or bf16", what);
    return kEinval;
  }
  if (num_requests == 0) return 0;
  if (!q || !o || !q_starts || !kv_starts || !kv_sources) {
    set_error("%s: null pointer", what);
    return kEinval;
  }
  bool use1 = false, use2 = false;
  for (int i = 0; i < num_requests; i++) {
    if (q_starts[i] < 0 || kv_starts[i] < 0 || q_starts[i] > INT32_MAX - q_lens[i] - 256 ||
        kv_starts[i] > INT32_MAX - kv_lens[i]) {
      set_error("%s: bad request %d", what, i);
      return kEinval;
    }
    (kv_sources[i] ? use2 : use1) = true;
  }
  if ((use1 && (!k || !v)) || (use2 && (!k2 || !v2))) {
    set_error("%s: null pointer", what);
    return kEinval;
  }
  const int64_t strides[10] = {q_stride_tok,  q_stride_head, o_stride_tok,  o_stride_head,
                               k_stride_tok,  k_stride_head, v_stride_tok,  v_stride_head,
                               k2_stride_tok, k2_stride_head};
  for (int i = 0; i < 10; i++) {
    if (i >= 4 && i < 8 && !use1) continue;
    if (i >= 8 && !use2) continue;
    if (strides[i] < 0 || strides[i] % 8 != 0) {
      set_error("%s: strides must be non-negative multiples of 8 elements", what);
      return kEinval;
    }
  }
  // K and V rows are read to padded_dim
  const int64_t lim = INT32_MAX / 2 / kBNmax;
  if ((use1 && (k_stride_tok < padded_dim || v_stride_tok < padded_dim || k_stride_tok > lim ||
                v_stride_tok > lim)) ||
      (use2 && (k2_stride_tok < padded_dim || k2_stride_tok > lim))) {
    set_error("%s: k / v token strides out of range", what);
    return kEinval;
  }
  uintptr_t al = (uintptr_t)q | (uintptr_t)o | (uintptr_t)workspace;
  if (use1) al |= (uintptr_t)k | (uintptr_t)v;
  if (use2) al |= (uintptr_t)k2 | (uintptr_t)v2;
  if (al & 15) {
    set_error("%s: tensors must be 16-byte aligned", what);
    return kEinval;
  }
  PrefillBatch p = {};
  p.q = q;
  p.k = static_cast<const _Float16*>(k);
  p.v = static_cast<const _Float16*>(v);
  p.k2 = static_cast<const _Float16*>(k2);
  p.v2 = static_cast<const _Float16*>(v2);
  p.o = o;
  p.q_st = q_stride_tok;
  p.q_sh = q_stride_head;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.k2_st = k2_stride_tok;
  p.k2_sh = k2_stride_head;
  p.o_st = o_stride_tok;
  p.o_sh = o_stride_head;
  p.ratio = num_qo_heads / num_kv_heads;
  p.hd = head_dim;
  p.q_bf16 = q_dtype == TQ_BF16;
  p.o_bf16 = o_dtype == TQ_BF16;
  p.c = sm_scale * 1.4426950408889634f;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  try {
    for (int a = 0; a < num_requests; a += kBatchReqs) {
      const int n = std::min(kBatchReqs, num_requests - a);
      const BatchPlan bp = plan_batch(q_lens + a, kv_lens + a, n, num_qo_heads, padded_dim);
      if (batch_ws_bytes(bp, num_qo_heads, padded_dim) > (workspace ? workspace_bytes : 0)) {
        set_error("%s: workspace smaller than tq_prefill_batch_workspace_bytes", what);
        return kEinval;
      }
      p.ws_o = static_cast<float*>(workspace);
      p.ws_ml = p.ws_o + (int64_t)bp.ws_rows * num_qo_heads * padded_dim;
      for (int i = 0; i < n; i++)
        p.reqs[i] = {q_starts[a + i], q_lens[a + i], kv_starts[a + i], kv_lens[a + i],
                     kv_sources[a + i] ? 1 : 0};
      hipError_t e;
      if (padded_dim == 64) e = launch_batch<64>(bp, num_qo_heads, st, p);
      else if (padded_dim == 128) e = launch_batch<128>(bp, num_qo_heads, st, p);
      else e = launch_batch<256>(bp, num_qo_heads, st, p);
      if (e != hipSuccess) {
        set_error("%s: launch failed: %s", what, hipGetErrorString(e));
        return (int)e;
      }
    }
  } catch (...) {
    set_error("%s: out of host memory", what);
    return (int)hipErrorOutOfMemory;
  }
  return 0;
}

extern "C" int64_t tq_prefill_workspace_bytes(int32_t q_len, int32_t kv_len, int32_t num_qo_heads,
                                              int32_t num_kv_heads, int32_t head_dim) {
  if (q_len <= 0 || kv_len < q_len || num_qo_heads <= 0 || num_kv_heads <= 0 ||
      (head_dim != 64 && head_dim != 128 && head_dim != 256))
    return 0;
  (void)num_kv_heads;
  return tq::plan_prefill(q_len, kv_len, num_qo_heads, head_dim).ws_bytes;
}

extern "C" int tq_prefill_attention_ws(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, const void* k,
    int64_t k_stride_tok, int64_t k_stride_head, const void* v, int64_t v_stride_tok,
    int64_t v_stride_head, void* o, int64_t o_stride_tok, int64_t o_stride_head, int32_t q_len,
    int32_t kv_len, int32_t num_qo_heads, int32_t num_kv_heads, int32_t head_dim, float sm_scale,
    void* workspace, int64_t workspace_bytes, tq_stream_t stream) {
  using namespace tq;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) {
    set_error("prefill_attention: head_dim %d unsupported (64, 128 or 256 only)", head_dim);
    return kEinval;
  }
  if (num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads != 0) {
    set_error("prefill_attention: num_qo_heads %d not a multiple of num_kv_heads %d",
              num_qo_heads, num_kv_heads);
    return kEinval;
  }
  if (q_len < 0 || kv_len < q_len) {
    set_error("prefill_attention: need 0 <= q_len (%d) <= kv_len (%d)", q_len, kv_len);
    return kEinval;
  }
  if (!q || !k || !v || !o) {
    set_error("prefill_attention: null pointer");
    return kEinval;
  }
  const int64_t strides[8] = {q_stride_tok, q_stride_head, k_stride_tok, k_stride_head,
                              v_stride_tok, v_stride_head, o_stride_tok, o_stride_head};
  for (int i = 0; i < 8; i++) {
    if (strides[i] < 0 || strides[i] % 8 != 0) {
      set_error("prefill_attention: strides must be non-negative multiples of 8 elements");
      return kEinval;
    }
  }
  if (k_stride_tok < head_dim || v_stride_tok < head_dim ||
      (k_stride_tok > v_stride_tok ? k_stride_tok : v_stride_tok) * 2 * (int64_t)kBNmax > INT32_MAX) {
    set_error("prefill_attention: k / v token strides out of range");
    return kEinval;
  }
  const uintptr_t al = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o;
  if (al & 15) {
    set_error("prefill_attention: tensors must be 16-byte aligned");
    return kEinval;
  }
  if (q_len == 0) return 0;
  PrefillParams p;
  p.q = static_cast<const _Float16*>(q);
  p.k = static_cast<const _Float16*>(k);
  p.v = static_cast<const _Float16*>(v);
  p.o = static_cast<_Float16*>(o);
  p.q_st = q_stride_tok;
  p.q_sh = q_stride_head;
  p.k_st = k_stride_tok;
  p.k_sh = k_stride_head;
  p.v_st = v_stride_tok;
  p.v_sh = v_stride_head;
  p.o_st = o_stride_tok;
  p.o_sh = o_stride_head;
  p.lq = q_len;
  p.lk = kv_len;
  p.ratio = num_qo_heads / num_kv_heads;
  p.c = sm_scale * 1.4426950408889634f;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const PrefillPlan sp = plan_prefill(q_len, kv_len, num_qo_heads, head_dim);
  p.nqb = sp.nqb;
  p.nsplit = 1;
  p.tps = 0;
  p.ws_o = nullptr;
  p.ws_ml = nullptr;
  // the split runs only with a workspace that holds it (else one workgroup
  // per query block, the same result)
  if (sp.nsplit > 1 && workspace && workspace_bytes >= sp.ws_bytes &&
      ((uintptr_t)workspace & 15) == 0) {
    p.nsplit = sp.nsplit;
    p.tps = sp.tps;
    p.ws_o = static_cast<_Float16*>(workspace);
    p.ws_ml = reinterpret_cast<float*>(p.ws_o + (int64_t)sp.nsplit * q_len * num_qo_heads *
                                                    head_dim);
  }
  if (head_dim == 64) return (int)launch_prefill<64>(sp.nw, num_qo_heads, st, p);
  if (head_dim == 128) return (int)launch_prefill<128>(sp.nw, num_qo_heads, st, p);
  return (int)launch_prefill<256>(sp.nw, num_qo_heads, st, p);
}

extern "C" int tq_prefill_attention(const void* q, int64_t q_stride_tok, int64_t q_stride_head,
                                    const void* k, int64_t k_stride_tok, int64_t k_stride_head,
                                    const void* v, int64_t v_stride_tok, int64_t v_stride_head,
                                    void* o, int64_t o_stride_tok, int64_t o_stride_head,
                                    int32_t q_len, int32_t kv_len, int32_t num_qo_heads,
                                    int32_t num_kv_heads, int32_t head_dim, float sm_scale,
                                    tq_stream_t stream) {
  return tq_prefill_attention_ws(q, q_stride_tok, q_stride_head, k, k_stride_tok, k_stride_head,
                                 v, v_stride_tok, v_stride_head, o, o_stride_tok, o_stride_head,
                                 q_len, kv_len, num_qo_heads, num_kv_heads, head_dim, sm_scale,
                                 nullptr, 0, stream);
}
