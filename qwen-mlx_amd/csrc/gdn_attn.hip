// gdn_attn.hip -- the attention layers' step on a paged KV cache
// (Qwen35Attention::forward_with_cache, qwen3_5.rs:377-455), for a packed
// batch of tokens from any number of sequences, each at its own position.
//
// The reference stacks per-sequence KV caches by zero-padding them to the
// longest and runs decode attention with no mask and one RoPE offset for the
// whole batch (mlx_executor.rs:57-88, qwen3_5.rs:410,443-447), so with B > 1
// a shorter sequence attends to padding and is rotated at the wrong
// position. Here every token carries its own sequence, position and KV page,
// keys are masked at each token's own position, and RoPE uses that position.
//
// Launches per layer step (T tokens, Hq query heads, Hkv kv heads, G = Hq/Hkv
// query heads per kv head, head dim 256, pages of 64 tokens):
//   attn_prep_kernel    q, k rms-norm (qwen3_5.rs:399-407), partial RoPE
//                       (:411-417), K/V rows into the token's page
//   attn_tile_kernel    prompts: a work-group takes 128 (token, query head)
//                       columns through all of their keys and writes the
//                       gated rows
//   attn_block_kernel   decode tokens and short prompts: one wave per worker of
//                       an even split of all (token group, kv head, key
//                       chunk) work, one partial per chunk
//   attn_combine_kernel merge those tokens' partials, output gate sigmoid(gate)
//                       * attn (:452-454), bf16 rows for o_proj
// Both attention kernels run scores and P.V on MFMA with an online softmax over
// 32-key blocks inside chunks of 384 keys, and merge the chunks' results in
// order with the same operations (scaled_dot_product_attention, :427-446): a
// token's output is the same bits in either, in any batch and however its
// prompt was cut into steps.
//
// Page layout. A page holds 64 positions of one layer: [2 (K, V)][Hkv][16384]
// bf16, each 16384-element tile stored in the order the MFMA operands are
// loaded, so that every load instruction of a wave reads 1 KiB of contiguous
// memory (s = (kk/32) XOR (page % 2), the 32-key block's slot; its 16 operands of
// 1 KiB in the order f XOR (page/2 % 16)):
//   K (key kk, dim d): [s][f = (kk/16)%2 d/32][(d/8)%4][kk%16][d%8] -- A operand
//       of v_mfma_f32_16x16x32_bf16, rows = 16 keys, 32-deep k = dims
//   V (key kk, dim d): [s][f = d/16][(kk/4)%4][d%16][(kk/16)%2][kk%4] -- A operand
//       of the same, rows = 16 dims, 32-deep k = keys: a lane group's eight are
//       4 keys of the block's first half, then the same 4 of its second, as the
//       two score accumulators hold them
#include "gdn_common.h"

namespace gdn {

namespace {

constexpr int kHd = 256;            // head dim = threads of the prep / combine work-groups
constexpr int kPage = 64;           // tokens per KV page
constexpr int kTile = kPage * kHd;  // elements of one page's K (or V) tile of one kv head
constexpr int kPartLd = 4 + kHd;    // partial row: m, l, 2 pad, 256 outputs (f32)
constexpr int kBlock = 32;          // keys per online-softmax block
constexpr int kBlockElems = kBlock * kHd;
constexpr int kChunkBlocks = 12;    // blocks per chunk (384 keys): one partial each

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// rows of q_full, k, v and out are only known to be 2-byte aligned
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

// Slot of 32-key block b (0, 1) of page `page`, and position in the slot of its
// 1 KiB operand f (0..15): both XOR-swizzled by the page id, so that workers
// which start at the same block of different pages (and move in step) read
// different parts of the pages' 128 KiB.
__device__ __forceinline__ int block_slot(int b, int page) { return b ^ (page & 1); }
__device__ __forceinline__ int frag_pos(int f, int page) { return f ^ ((page >> 1) & 15); }
__device__ __forceinline__ int k_off(int kk, int d, int page) {
  const int f = ((kk >> 4) & 1) * 8 + (d >> 5);
  return (block_slot(kk >> 5, page) * 16 + frag_pos(f, page)) * 512 + ((d >> 3) & 3) * 128 +
         (kk & 15) * 8 + (d & 7);
}
__device__ __forceinline__ int v_off(int kk, int d, int page) {
  return (block_slot(kk >> 5, page) * 16 + frag_pos(d >> 4, page)) * 512 + ((kk >> 2) & 3) * 128 +
         (d & 15) * 8 + ((kk >> 4) & 1) * 4 + (kk & 3);
}

__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Maximum over the four lanes of a column (lane ^ 16, lane ^ 32, both), on
// VALU swaps.
__device__ __forceinline__ float max_xor16_32(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// One 32-key block's online softmax for the 16 columns of a tile pair (s0, s1:
// scores of keys 4 g4 + r and 16 + 4 g4 + r of the block, g4 = lane / 16, for
// column lane % 16), in the log2 domain; keys past cpos are masked. rescale(c)
// multiplies the column's accumulators by c; it runs only when some column's
// running maximum m grows. (The hardware exp2 flushes results below 2^-126,
// which a sum of at least 1 in float32 does not see.) p comes out split exactly into three bf16 parts
// (together its 24 significant bits) in the B operand layout.
template <typename F>
__device__ __forceinline__ void softmax_block(const f32x4& s0, const f32x4& s1, int key0, int cpos,
                                              float scale_log2, float& m, float& lsum, F rescale,
                                              u32x4& ph, u32x4& pm, u32x4& pl) {
  float x[8];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    x[r] = key0 + r <= cpos ? s0[r] * scale_log2 : -INFINITY;
    x[4 + r] = key0 + 16 + r <= cpos ? s1[r] * scale_log2 : -INFINITY;
  }
  float bm = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                   fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
  bm = max_xor16_32(bm);
  const float mnew = fmaxf(m, bm);
  if (__any(mnew > m)) {
    const float corr = mnew > m ? __builtin_amdgcn_exp2f(m - mnew) : 1.0f;  // m = -inf: 0
    lsum *= corr;
    rescale(corr);
    m = mnew;
  }
  const float mref = m == -INFINITY ? 0.f : m;
  float p[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) p[r] = __builtin_amdgcn_exp2f(x[r] - mref);  // masked: 0
  lsum += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
#pragma unroll
  for (int e = 0; e < 4; ++e) {  // each part takes the next 8 significant bits
    const float a = p[2 * e], b = p[2 * e + 1];
    ph[e] = f2bf2(a, b);
    const float a1 = a - bf_lo(ph[e]), b1 = b - bf_hi(ph[e]);
    pm[e] = f2bf2(a1, b1);
    pl[e] = f2bf2(a1 - bf_lo(pm[e]), b1 - bf_hi(pm[e]));
  }
}

// V operand of a block with the keys from nkeys on zeroed (those rows of a page
// may hold anything); key0 = the block's first key + 4 g4.
__device__ __forceinline__ u32x4 mask_v(u32x4 v, int key0, int nkeys) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int k = key0 + (e >> 1) * 16 + (e & 1) * 2;
    v[e] &= (k < nkeys ? 0xffffu : 0u) | (k + 1 < nkeys ? 0xffff0000u : 0u);
  }
  return v;
}

// Factors that merge a chunk's result (maximum m) into the running one (M):
// R <- R * a + r * b. A chunk with no key of the column changes nothing.
__device__ __forceinline__ void merge_factors(float& M, float m, float& a, float& b) {
  const float Mn = fmaxf(M, m);
  const bool none = m == -INFINITY;
  a = none ? 1.0f : exp2f(M - Mn);  // M = -inf: 0
  b = none ? 0.0f : exp2f(m - Mn);
  M = Mn;
}

// bf16(bf16(o) * bf16(sigmoid(gate)))
__device__ __forceinline__ uint16_t gated(float o, float gate) {
  return f2bf(rbf(o) * rbf(sigmoid_f32(gate)));
}

}  // namespace

// grid (T, ceil((Hq + Hkv) / hpg)), block 256: a work-group takes hpg heads of
// one token, a wave one head at a time, four dimensions per lane. Heads < Hq
// are query heads (the first 256 of the head's 512 q_proj outputs; the other
// 256 are its output gate), the rest kv heads. The token's RoPE angles are
// formed once per work-group. The token's page comes with the step metadata;
// the first token of a page also records it in the sequence's page table,
// which the attention kernels read. Bound by the latency of its few loads and
// of the angles: prompts take all heads of a token in one group (one sincos
// pass per token; 2,048 tokens: 43 us before, with a group per head and token),
// decode batches spread them (4 heads a group).
__global__ __launch_bounds__(kHd) void attn_prep_kernel(
    const uint16_t* __restrict__ q_full, int64_t qs, const uint16_t* __restrict__ k, int64_t ks,
    const uint16_t* __restrict__ v, int64_t vs, const uint16_t* __restrict__ q_norm_w,
    const uint16_t* __restrict__ k_norm_w, float eps, int rot_dim, float log2_base, int Hq,
    int Hkv, int hpg, const int32_t* __restrict__ meta, int T, int32_t* __restrict__ ptab,
    int max_pages, uint16_t* __restrict__ pages, uint16_t* __restrict__ q_rot) {
  __shared__ float cs[kHd / 2], sn[kHd / 2];
  __shared__ float xs[4][kHd];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h1 = min((int)(blockIdx.y + 1) * hpg, Hq + Hkv);
  const int d0 = 4 * lane;
  // a head's row and norm weight (and v), the first head's before the angles
  u32x2_a2 xr = {0u, 0u}, wr = {0u, 0u}, vr = {0u, 0u};
  auto load = [&](int h) {
    const bool isq = h < Hq;
    const int j = h - Hq;  // kv head
    const uint16_t* src =
        isq ? q_full + (size_t)t * qs + (size_t)h * 2 * kHd : k + (size_t)t * ks + (size_t)j * kHd;
    xr = *reinterpret_cast<const u32x2_a2*>(src + d0);
    wr = *reinterpret_cast<const u32x2_a2*>((isq ? q_norm_w : k_norm_w) + d0);
    if (!isq) vr = *reinterpret_cast<const u32x2_a2*>(v + (size_t)t * vs + (size_t)j * kHd + d0);
  };
  int h = blockIdx.y * hpg + wave;
  if (h < h1) load(h);
  const int slot = meta[t], pos = meta[T + t], page = meta[2 * T + t];
  const int half = rot_dim >> 1;
  if (tid < half) {
    const float inv_freq = exp2f(-(2.0f * (float)tid / (float)rot_dim) * log2_base);
    sincosf((float)pos * inv_freq, &sn[tid], &cs[tid]);
  }
  lds_barrier();
  for (; h < h1; h += 4) {
    const bool isq = h < Hq;
    const int j = h - Hq;
    const float x[4] = {bf_lo(xr.x), bf_hi(xr.x), bf_lo(xr.y), bf_hi(xr.y)};
    const float w[4] = {bf_lo(wr.x), bf_hi(wr.x), bf_lo(wr.y), bf_hi(wr.y)};
    const uint32_t vh[2] = {vr.x, vr.y};
    if (h + 4 < h1) load(h + 4);
    const float ss = wave_sum((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]));
    const float rn = 1.0f / sqrtf(ss / (float)kHd + eps);
    // RoPE, rotate-half form over the first rot_dim dimensions: pairs (i, i + rot_dim/2),
    // exchanged through the wave's own row of xs
#pragma unroll
    for (int e = 0; e < 4; ++e) xs[wave][d0 + e] = rbf(w[e] * rbf(x[e] * rn));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    float yv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = d0 + e;
      const float xn = xs[wave][d];
      yv[e] = xn;
      if (d < rot_dim) {
        const int i = d < half ? d : d - half;
        yv[e] = d < half ? xn * cs[i] - xs[wave][d + half] * sn[i]
                         : xs[wave][d - half] * sn[i] + xn * cs[i];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    const uint2 yb = make_uint2(f2bf2(yv[0], yv[1]), f2bf2(yv[2], yv[3]));
    if (isq) {
      *reinterpret_cast<uint2*>(q_rot + ((size_t)t * Hq + h) * kHd + d0) = yb;
    } else {
      const int kk = pos & (kPage - 1);
      const size_t tile = ((size_t)page * 2 * Hkv + j) * kTile;
      *reinterpret_cast<uint2*>(pages + tile + k_off(kk, d0, page)) = yb;  // K: 4 dims side by side
      uint16_t* vt = pages + tile + (size_t)Hkv * kTile;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        vt[v_off(kk, d0 + e, page)] = (uint16_t)(vh[e >> 1] >> (16 * (e & 1)));
      if (j == 0 && lane == 0 && kk == 0) ptab[(size_t)slot * max_pages + pos / kPage] = page;
    }
  }
}

// One wave per work-group; work-group w is worker w of P. The work is every
// (token group, kv head) segment's keys (segment s = group * Hkv + j) cut at
// fixed points into chunks of kChunkBlocks 32-key blocks; the flat list of
// all chunks, in segment order, goes to the workers in equal runs of k
// (worker w: chunks [w k, (w+1) k)), which may span several segments. Every
// chunk writes its own partial, so a token's result depends only on its own
// keys: the same in any batch, and when a prompt's tokens are grouped
// differently.
//
// A token group is up to 16/G consecutive tokens of one sequence: the 16
// columns of the MFMA tiles are (token, query head) pairs, column c = token
// c / G of the group, head j G + c % G. Per 32-key block:
//   S^T (2 x 16 keys x 16 columns) = K_blk (32 x 256) . Q^T (256 x 16): 16
//     MFMAs, K straight from the page, Q^T re-read from LDS;
//   online softmax per column (softmax_block);
//   O^T (256 dims x 16 columns) += V^T_blk . P^T: three 32-deep MFMAs per 16
//     dims, against P's hi, mid and lo parts (the products are those of
//     float32 P). The score accumulators are the B operand as they are.
// The next block's K is loaded as soon as this block's scores are formed, its V
// after this block's P.V, across chunk boundaries within a segment. HBM-bound
// at decode: 32 KiB of K/V per block in flight per wave.
//
// Schedule tables (int32, built by the host for the step):
//   grp[NG][4]  first token, tokens, first position, sequence slot
//   seg[NS][4]  first chunk (= its partial), chunks, -, -
//   wseg[P]     segment of the worker's first chunk
// Partials [chunks][16][kPartLd] f32: running max (log2 domain), sum, output.
template <int G, bool STREAM>
__global__ __launch_bounds__(64, 2) void attn_block_kernel(
    const uint16_t* __restrict__ q_rot, int Hq, int Hkv, const int32_t* __restrict__ grp,
    const int32_t* __restrict__ seg, const int32_t* __restrict__ wseg, int NC, int k,
    const int32_t* __restrict__ ptab, int max_pages, const uint16_t* __restrict__ pages,
    float scale_log2, float* __restrict__ part) {
  static_assert(16 % G == 0, "whole tokens per 16 columns");
  __shared__ u32x4 qlds[8][64];  // this wave's Q^T operand
  const int w = blockIdx.x, lane = threadIdx.x;
  const int g4 = lane >> 4, c = lane & 15;
  const int gw1 = min(NC, (w + 1) * k);
  int g = w * k;  // next chunk
  int s = wseg[w];
  const size_t page_stride = (size_t)2 * Hkv * kTile;
  const size_t v_shift = (size_t)Hkv * kTile;
  while (g < gw1) {
    const int gi = s / Hkv, j = s - gi * Hkv;
    const int t0 = grp[4 * gi], ntok = grp[4 * gi + 1], pos0 = grp[4 * gi + 2],
              slot = grp[4 * gi + 3];
    const int cs0 = seg[4 * s], nch = seg[4 * s + 1];
    const int nkeys = pos0 + ntok;  // the group's last position + 1
    const int nblk = (nkeys + kBlock - 1) / kBlock;
    const int gend = min(gw1, cs0 + nch);  // this worker's chunks of the segment: [g, gend)
    const int kb0 = (g - cs0) * kChunkBlocks;
    const int kb1 = min(nblk, (gend - cs0) * kChunkBlocks);
    const int ctok = c / G;
    const bool cvalid = ctok < ntok;
    const int cpos = cvalid ? pos0 + ctok : -1;  // keys <= cpos are attended
    // Q^T: lane l holds column c, dims 32 ks + 8 g4 .. +7, kept in LDS
    {
      const u32x4* qsrc = reinterpret_cast<const u32x4*>(
          q_rot + ((size_t)(t0 + (cvalid ? ctok : 0)) * Hq + j * G + c % G) * kHd + 8 * g4);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        qlds[ks][lane] = cvalid ? qsrc[4 * ks] : (u32x4){0u, 0u, 0u, 0u};
    }
    // the piece's page ids, one per lane (64 pages = 4096 keys per reload)
    const int32_t* prow = ptab + (size_t)slot * max_pages;
    const int npages = (nblk + 1) >> 1;
    int pbase = kb0 >> 1;
    int pid = pbase + lane < npages ? prow[pbase + lane] : 0;
    const uint16_t* kv_head = pages + (size_t)j * kTile;

    float m = -INFINITY, lsum = 0.f;
    f32x4 O[16];
#pragma unroll
    for (int db = 0; db < 16; ++db) O[db] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // K of block kb (V lies v_shift behind); page ids are reloaded as needed
    auto block_ptr = [&](int kb, int& x) {
      int idx = (kb >> 1) - pbase;
      if (idx >= 64) {  // wave-uniform: the next 64 page ids
        pbase += 64;
        idx -= 64;
        pid = pbase + lane < npages ? prow[pbase + lane] : 0;
      }
      const int page = __builtin_amdgcn_readlane(pid, idx);
      x = frag_pos(0, page);
      return kv_head + (size_t)page * page_stride + (size_t)block_slot(kb & 1, page) * kBlockElems;
    };
    // STREAM (each block read about once in the step): non-temporal loads
    // stream past the caches; otherwise plain loads keep the blocks that
    // later token groups of the same prompt read again
    auto load16 = [&](const uint16_t* src, int x, u32x4(&f)[16]) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const u32x4* p = reinterpret_cast<const u32x4*>(src + (i ^ x) * 512) + lane;
        f[i] = STREAM ? __builtin_nontemporal_load(p) : *p;
      }
    };
    // the partial of the chunk that block kb ends, then a fresh state
    auto flush = [&](int kb) {
      const float l4 = lsum + __shfl_xor(lsum, 16, 64);
      const float lt = l4 + __shfl_xor(l4, 32, 64);
      if (cvalid) {
        float* pr = part + ((size_t)(cs0 + kb / kChunkBlocks) * 16 + c) * kPartLd;
        if (g4 == 0) {
          pr[0] = m;
          pr[1] = lt;
        }
#pragma unroll
        for (int db = 0; db < 16; ++db)
          *reinterpret_cast<f32x4*>(pr + 4 + 16 * db + 4 * g4) = O[db];
      }
      m = -INFINITY;
      lsum = 0.f;
#pragma unroll
      for (int db = 0; db < 16; ++db) O[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };

    u32x4 kf[16], vf[16];
    int x = 0;
    const uint16_t* cur = block_ptr(kb0, x);
    load16(cur, x, kf);
    load16(cur + v_shift, x, vf);
    // block kb, with the next block's loads behind its products; the range's
    // last block (a call of its own) has none to issue
    auto block = [&](int kb, auto lastc) {
      constexpr bool last = decltype(lastc)::value;
      const uint16_t* nxt = nullptr;
      if constexpr (!last) nxt = block_ptr(kb + 1, x);
      f32x4 S[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      // Q^T is re-read from LDS for every block rather than held in registers:
      // an empty asm with a memory clobber keeps the compiler from hoisting
      // the reads (a volatile read would also drain the memory counters).
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const u32x4 q = qlds[ks][lane];
        S[0] = mfma32(kf[ks], q, S[0]);
        S[1] = mfma32(kf[8 + ks], q, S[1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!last) load16(nxt, x, kf);
      __builtin_amdgcn_sched_barrier(0);
      u32x4 ph, pm, pl;
      const int key0 = kBlock * kb + 4 * g4;
      softmax_block(
          S[0], S[1], key0, cpos, scale_log2, m, lsum,
          [&](float corr) {
#pragma unroll
            for (int db = 0; db < 16; ++db) O[db] *= corr;
          },
          ph, pm, pl);
      if (kBlock * (kb + 1) > nkeys) {  // wave-uniform: rows past the group's last key
#pragma unroll
        for (int db = 0; db < 16; ++db) vf[db] = mask_v(vf[db], key0, nkeys);
      }
#pragma unroll
      for (int db = 0; db < 16; ++db) {
        O[db] = mfma32(vf[db], ph, O[db]);
        O[db] = mfma32(vf[db], pm, O[db]);
        O[db] = mfma32(vf[db], pl, O[db]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!last) load16(nxt + v_shift, x, vf);
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int kb = kb0; kb + 1 < kb1; ++kb) {
      block(kb, std::false_type{});
      if ((kb + 1) % kChunkBlocks == 0) flush(kb);
    }
    block(kb1 - 1, std::true_type{});
    flush(kb1 - 1);
    g = gend;
    ++s;
  }
}

// Prompts. Work-group (tile, kv head j) takes a tile of up to 128 / G
// consecutive tokens of one sequence, 128 (token, query head) columns, through
// all of their keys; wave w owns columns 16 w .. +15 (a token group of
// attn_block_kernel) and holds the running chunk's O^T and the merged O^T in
// registers, their Q^T in LDS. A 32-key block of K and V (32 KiB) is copied into
// LDS by DMA one block ahead, two buffers, and read by all eight waves: a key
// block is fetched once per 128 columns. Scores, softmax, chunks and merges are attn_block_kernel's and
// attn_combine_kernel's, operation by operation, so the bits are theirs; no
// partials go through memory.
//
// What bounds it: LDS reads, 40 KiB per wave and block (2,500 cycles for the
// eight waves), beside 64 MFMAs per wave (2,048 cycles for the two waves of a
// SIMD; three quarters of them P's hi, mid and lo parts). Two waves per SIMD let
// one's softmax meet the other's products; four waves of 32 columns (half the
// LDS reads, one wave per SIMD) took 3.4 us per block.
template <int G>
__global__ __launch_bounds__(512, 2) void attn_tile_kernel(
    const uint16_t* __restrict__ q_rot, int Hq, int Hkv, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ ptab, int max_pages, const uint16_t* __restrict__ pages,
    float scale_log2, const uint16_t* __restrict__ q_full, int64_t qs, uint16_t* __restrict__ out,
    int64_t os) {
  constexpr int TG = 16 / G;  // tokens per 16-column group
  __shared__ u32x4 lk0[1024], lk1[1024], lv0[1024], lv1[1024];  // K and V blocks, two of each
  __shared__ u32x4 lq[8][8][64];  // each wave's Q^T operands
  const int lane = threadIdx.x & 63, g4 = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ti = blockIdx.x / Hkv, j = blockIdx.x - ti * Hkv;
  const int t0 = tiles[4 * ti], ntok = tiles[4 * ti + 1], pos0 = tiles[4 * ti + 2],
            slot = tiles[4 * ti + 3];
  const int nblk = (pos0 + ntok + kBlock - 1) / kBlock;
  const int32_t* prow = ptab + (size_t)slot * max_pages;
  const size_t page_stride = (size_t)2 * Hkv * kTile;
  const size_t v_shift = (size_t)Hkv * kTile;
  const uint16_t* kv_head = pages + (size_t)j * kTile;

  // the wave's column group: tokens gt .. of the tile
  const int gt = w * TG, tok = gt + c / G;
  const bool valid = tok < ntok;
  const int cpos = valid ? pos0 + tok : -1;
  const int nkeys = pos0 + min(gt + TG, ntok);  // the group's last position + 1
  {
    const u32x4* qsrc = reinterpret_cast<const u32x4*>(
        q_rot + ((size_t)(t0 + (valid ? tok : 0)) * Hq + j * G + c % G) * kHd + 8 * g4);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) lq[w][ks][lane] = valid ? qsrc[4 * ks] : (u32x4){0u, 0u, 0u, 0u};
  }

  // block kb's K and V into buffer b: wave w copies 2 KiB of each
  auto copy = [&](int kb, auto bc) {
    constexpr int b = decltype(bc)::value;
    const int page = prow[kb >> 1];
    const uint16_t* src = kv_head + (size_t)page * page_stride +
                          (size_t)block_slot(kb & 1, page) * kBlockElems + lane * 8;
    u32x4* const dk = (b ? lk1 : lk0) + 2 * w * 64;
    u32x4* const dv = (b ? lv1 : lv0) + 2 * w * 64;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(
          (const void __attribute__((address_space(1)))*)(src + frag_pos(2 * w + i, page) * 512),
          (void __attribute__((address_space(3)))*)(dk + i * 64), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(
          (const void __attribute__((address_space(1)))*)(src + v_shift + frag_pos(2 * w + i, page) * 512),
          (void __attribute__((address_space(3)))*)(dv + i * 64), 16, 0, 0);
  };

  float m = -INFINITY, lsum = 0.f, M = -INFINITY, L = 0.f;
  f32x4 O[16], R[16];
#pragma unroll
  for (int db = 0; db < 16; ++db) O[db] = R[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // the chunk's result into the merged one, then a fresh chunk
  auto merge = [&]() {
    const float l4 = lsum + __shfl_xor(lsum, 16, 64);
    const float lt = l4 + __shfl_xor(l4, 32, 64);
    float a, b;
    merge_factors(M, m, a, b);
    L = fmaf(L, a, lt * b);
#pragma unroll
    for (int db = 0; db < 16; ++db) {
      R[db] = __builtin_elementwise_fma(R[db], (f32x4){a, a, a, a}, O[db] * b);
      O[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    m = -INFINITY;
    lsum = 0.f;
  };

  auto block = [&](int kb, auto bc) {
    constexpr int b = decltype(bc)::value;
    // this wave's copies of block kb have landed and its reads of the other
    // buffer have returned (lds_barrier waits for them): after the barrier
    // everyone's have, and the other buffer may be copied over
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    lds_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "global");
    copy(min(kb + 1, nblk - 1), std::integral_constant<int, 1 - b>{});
    __builtin_amdgcn_sched_barrier(0);
    const u32x4* const lk = b ? lk1 : lk0;
    const u32x4* const lv = b ? lv1 : lv0;
    f32x4 S[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    asm volatile("" ::: "memory");  // Q^T is re-read from LDS for every block
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const u32x4 q = lq[w][ks][lane];
      S[0] = mfma32(lk[ks * 64 + lane], q, S[0]);
      S[1] = mfma32(lk[(8 + ks) * 64 + lane], q, S[1]);
    }
    const int key0 = kBlock * kb + 4 * g4;
    u32x4 ph, pm, pl;
    softmax_block(
        S[0], S[1], key0, cpos, scale_log2, m, lsum,
        [&](float corr) {
#pragma unroll
          for (int db = 0; db < 16; ++db) O[db] *= corr;
        },
        ph, pm, pl);
    auto pv = [&](auto masked) {
#pragma unroll
      for (int db = 0; db < 16; ++db) {
        u32x4 v = lv[db * 64 + lane];
        if constexpr (decltype(masked)::value) v = mask_v(v, key0, nkeys);
        O[db] = mfma32(v, ph, O[db]);
        O[db] = mfma32(v, pm, O[db]);
        O[db] = mfma32(v, pl, O[db]);
      }
    };
    if (kBlock * (kb + 1) > nkeys)  // wave-uniform: keys past the group's last one
      pv(std::true_type{});
    else
      pv(std::false_type{});
    if ((kb + 1) % kChunkBlocks == 0 || kb + 1 == nblk) merge();
  };

  copy(0, std::integral_constant<int, 0>{});
  int kb = 0;
#pragma nounroll
  for (; kb + 2 <= nblk; kb += 2) {
    block(kb, std::integral_constant<int, 0>{});
    block(kb + 1, std::integral_constant<int, 1>{});
  }
  if (kb < nblk) block(kb, std::integral_constant<int, 0>{});
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the last copies (a repeat) land before the LDS is given back

  if (!valid) return;
  const int h = j * G + c % G;
  const float inv = 1.0f / L;
  const uint16_t* gr = q_full + (size_t)(t0 + tok) * qs + (size_t)h * 2 * kHd + kHd + 4 * g4;
  uint16_t* orow = out + (size_t)(t0 + tok) * os + (size_t)h * kHd + 4 * g4;
#pragma unroll
  for (int db = 0; db < 16; ++db) {
    const u32x2_a2 gv = *reinterpret_cast<const u32x2_a2*>(gr + 16 * db);
    const f32x4 r = R[db];
    u32x2_a2 o;
    o.x = gated(r[0] * inv, bf_lo(gv.x)) | (uint32_t)gated(r[1] * inv, bf_hi(gv.x)) << 16;
    o.y = gated(r[2] * inv, bf_lo(gv.y)) | (uint32_t)gated(r[3] * inv, bf_hi(gv.y)) << 16;
    *reinterpret_cast<u32x2_a2*>(orow + 16 * db) = o;
  }
}

// grid (T, Hq / DPL), block 256: out[t, hq 256 + d] = bf16(bf16(o) *
// bf16(sigmoid(gate))) with o the normalised merge of the token's chunks, in
// order, for query head hq; gate is the second half of the head's q_proj
// outputs. tokseg[t] = the token's group (-1: attn_tile_kernel wrote the token),
// tokseg[T + t] = its first column. A wave takes one head with four dimensions
// per lane (DPL = 4), or a quarter of one with one (DPL = 1); the merge factors
// of 64 chunks are formed at a time, a chunk per lane, so that the chunks' rows
// are independent loads, 64 / DPL in flight. Bound by the latency of those
// loads: with few chunks wide loads (64 tokens at 4,096 keys, 11 chunks), with
// many (kLongChunks) more of them in flight.
template <int G, int DPL>
__global__ __launch_bounds__(kHd) void attn_combine_kernel(
    const float* __restrict__ part, const int32_t* __restrict__ tokseg,
    const int32_t* __restrict__ seg, int T, int Hkv, const uint16_t* __restrict__ q_full,
    int64_t qs, uint16_t* __restrict__ out, int64_t os) {
  constexpr int kAhead = 64 / DPL;
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hq = DPL == 4 ? blockIdx.y * 4 + wave : blockIdx.y;
  const int d0 = DPL == 4 ? 4 * lane : 64 * wave + lane;  // the lane's dimensions d0 ..
  const int ts = tokseg[t];
  if (ts < 0) return;
  const int j = hq / G, g = hq - j * G;
  const int s = ts * Hkv + j;
  const int p0 = seg[4 * s], np = seg[4 * s + 1];
  const float* pc = part + ((size_t)p0 * 16 + tokseg[T + t] + g) * kPartLd;
  constexpr size_t kStride = (size_t)16 * kPartLd;  // consecutive chunks
  const uint16_t* gr = q_full + (size_t)t * qs + (size_t)hq * 2 * kHd + kHd + d0;
  float gate[DPL];
  if constexpr (DPL == 4) {
    const u32x2_a2 gv = *reinterpret_cast<const u32x2_a2*>(gr);
    gate[0] = bf_lo(gv.x), gate[1] = bf_hi(gv.x), gate[2] = bf_lo(gv.y), gate[3] = bf_hi(gv.y);
  } else {
    gate[0] = bf2f(*gr);
  }
  typedef float fvec __attribute__((ext_vector_type(DPL)));
  float M = -INFINITY, L = 0.f;
  fvec A = (fvec)(0.f);
  for (int c0 = 0; c0 < np; c0 += 64) {
    const int n = min(64, np - c0);
    const float* ps = pc + (size_t)c0 * kStride;
    const float mi = lane < n ? ps[lane * kStride] : -INFINITY;
    const float li = lane < n ? ps[lane * kStride + 1] : 0.f;
    fvec v[kAhead];
    auto rows = [&](int i0) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
        v[i] = *reinterpret_cast<const fvec*>(ps + min(i0 + i, n - 1) * kStride + 4 + d0);
    };
    rows(0);
    float sm = mi;  // running maximum, this chunk's included
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float u = __shfl_up(sm, off, 64);
      sm = lane >= off ? fmaxf(sm, u) : sm;
    }
    float a, b, Mi = fmaxf(M, __shfl_up(sm, 1, 64));
    if (lane == 0) Mi = M;
    merge_factors(Mi, mi, a, b);
    const float lb = li * b;
    for (int i0 = 0; i0 < n; i0 += kAhead) {
      if (i0) rows(i0);
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
        if (i0 + i < n) {
          const float ai = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(a), i0 + i));
          const float bi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b), i0 + i));
          const float li_b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lb), i0 + i));
          L = fmaf(L, ai, li_b);
          A = __builtin_elementwise_fma(A, (fvec)(ai), v[i] * bi);
        }
    }
    M = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(Mi), n - 1));
  }
  const float inv = 1.0f / L;
  uint16_t* orow = out + (size_t)t * os + (size_t)hq * kHd + d0;
  if constexpr (DPL == 4) {
    u32x2_a2 o;
    o.x = gated(A[0] * inv, gate[0]) | (uint32_t)gated(A[1] * inv, gate[1]) << 16;
    o.y = gated(A[2] * inv, gate[2]) | (uint32_t)gated(A[3] * inv, gate[3]) << 16;
    *reinterpret_cast<u32x2_a2*>(orow) = o;
  } else {
    *orow = gated(A[0] * inv, gate[0]);
  }
}

// grid (pages of the sequence, Hkv, 2), block 256: a sequence's cached K (z =
// 0) or V (z = 1) rows of one layer into dst [Hkv][len][256].
__global__ __launch_bounds__(kHd) void kv_gather_kernel(const uint16_t* __restrict__ pages,
                                                       const int32_t* __restrict__ prow, int Hkv,
                                                       int64_t len, uint16_t* __restrict__ k_out,
                                                       uint16_t* __restrict__ v_out) {
  const int p = blockIdx.x, j = blockIdx.y, isv = blockIdx.z, d = threadIdx.x;
  uint16_t* dst = isv ? v_out : k_out;
  if (!dst) return;
  const int page = prow[p];
  const uint16_t* tile = pages + ((size_t)page * 2 * Hkv + (size_t)isv * Hkv + j) * kTile;
  for (int kk = 0; kk < kPage; ++kk) {
    const int64_t pos = (int64_t)p * kPage + kk;
    if (pos >= len) break;
    dst[((size_t)j * len + pos) * kHd + d] = tile[isv ? v_off(kk, d, page) : k_off(kk, d, page)];
  }
}

size_t attn_part_offset(int T, int Hq) { return ((size_t)T * Hq * kHd * 2 + 255) & ~(size_t)255; }

size_t attn_workspace_bytes(int T, int Hq, int64_t chunks) {
  return attn_part_offset(T, Hq) + (size_t)chunks * 16 * kPartLd * sizeof(float);
}

int attn_chunk_keys() { return kChunkBlocks * kBlock; }
int attn_block_keys() { return kBlock; }

// Heads per work-group of attn_prep_kernel: with at least this many tokens all
// heads of a token (the tokens alone fill the chip), below it four.
constexpr int kPrepWholeTokens = 512;
// Chunks of the step's longest sequence above which a combine wave takes a
// quarter of a head (four times the loads in flight).
constexpr int kLongChunks = 32;

hipError_t launch_attn(const AttnArgs& a) {
  if (a.T <= 0) return hipSuccess;
  const int G = a.Hq / a.Hkv;
  if (G != 4 && G != 8) return hipErrorInvalidValue;
  uint16_t* q_rot = static_cast<uint16_t*>(a.workspace);
  float* part =
      reinterpret_cast<float*>(static_cast<char*>(a.workspace) + attn_part_offset(a.T, a.Hq));
  const int heads = a.Hq + a.Hkv, hpg = a.T >= kPrepWholeTokens ? heads : 4;
  hipLaunchKernelGGL(attn_prep_kernel, dim3(a.T, (heads + hpg - 1) / hpg), dim3(kHd), 0, a.stream,
                     a.q_full, a.qs, a.k, a.ks, a.v, a.vs, a.q_norm_w, a.k_norm_w, a.eps, a.rot_dim,
                     a.log2_base, a.Hq, a.Hkv, hpg, a.meta, a.T, a.ptab, a.max_pages, a.pages,
                     q_rot);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const float scale_log2 = 1.4426950408889634f / sqrtf((float)kHd);  // log2(e) / sqrt(256)
  if (a.NT > 0) {
    auto tile = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(a.NT * a.Hkv), dim3(512), 0, a.stream, q_rot, a.Hq, a.Hkv,
                         a.tiles, a.ptab, a.max_pages, a.pages, scale_log2, a.q_full, a.qs, a.out,
                         a.os);
    };
    if (G == 8)
      tile(attn_tile_kernel<8>);
    else
      tile(attn_tile_kernel<4>);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (a.NC <= 0) return hipSuccess;
  auto blocks = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(a.P), dim3(64), 0, a.stream, q_rot, a.Hq, a.Hkv, a.grp, a.seg,
                       a.wseg, a.NC, a.kpw, a.ptab, a.max_pages, a.pages, scale_log2, part);
  };
  const int dpl = a.max_chunks > kLongChunks ? 1 : 4;
  auto combine = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(a.T, a.Hq / dpl), dim3(kHd), 0, a.stream, part, a.tokseg, a.seg, a.T,
                       a.Hkv, a.q_full, a.qs, a.out, a.os);
  };
  if (G == 8) {
    if (a.stream_keys)
      blocks(attn_block_kernel<8, true>);
    else
      blocks(attn_block_kernel<8, false>);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    dpl == 4 ? combine(attn_combine_kernel<8, 4>) : combine(attn_combine_kernel<8, 1>);
  } else {
    if (a.stream_keys)
      blocks(attn_block_kernel<4, true>);
    else
      blocks(attn_block_kernel<4, false>);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    dpl == 4 ? combine(attn_combine_kernel<4, 4>) : combine(attn_combine_kernel<4, 1>);
  }
  return hipGetLastError();
}

hipError_t launch_kv_gather(const uint16_t* pages, const int32_t* prow, int Hkv, int64_t len,
                            uint16_t* k_out, uint16_t* v_out, hipStream_t s) {
  if (len <= 0) return hipSuccess;
  const int np = (int)((len + kPage - 1) / kPage);
  hipLaunchKernelGGL(kv_gather_kernel, dim3(np, Hkv, 2), dim3(kHd), 0, s, pages, prow, Hkv, len,
                     k_out, v_out);
  return hipGetLastError();
}

}  // namespace gdn
