// Paged attention over the slot pool [num_slots, KVH, D] (slot = block * 16 + offset), GQA with
// query head h reading KV head h / (H / KVH), scale applied to q.k, softmax over the visible keys.
//
// Decode (one new token per sequence): a workgroup of four wavefronts per (sequence, KV head);
// the wavefronts interleave the sequence's 16-token blocks, read straight from the pool through
// the block table -- no gathered copy. The G = H / KVH query heads of the KV head share every K/V
// load. The arithmetic runs on bf16 pairs with v_dot2_f32_bf16 (the kernel is otherwise bound by
// VALU issue, not HBM); the wavefronts merge through LDS. Only when sequences x KV heads are too
// few to fill the GPU does the host add workgroup-level splits; those write (acc, max, sum) to a
// workspace and a second small kernel merges them -- no workgroup ever waits for another (a
// sequence whose keys fit one split is written directly).
//
// Prefill (any number of new tokens, fresh or after cached keys): flash-attention on MFMA. A
// workgroup owns one KV head and 64 / G query tokens in three key groups of four wavefronts;
// wavefront w of a group takes query head w % G and 16 of the tokens. Per 32-key tile a key group
// stages K and V (both key-major) in LDS, then each wavefront computes S^T = K Q^T
// (v_mfma_f32_16x16x32_bf16, 2 x 4 instructions) so each lane holds 8 scores of ONE query, applies
// the causal mask and an online softmax with lane-local statistics, and accumulates
// O^T += V^T P^T (8 instructions, V^T fragments through gfx950's transposing LDS reads) with P in
// bf16; the softmax denominators accumulate on MFMA too (a ones matrix times P).
#include <mutex>

#include "common.h"

namespace msa {

constexpr int kHeadDim = 128;
constexpr int kBlock = 16;

struct DecodeArgs {
  const uint16_t* q;
  int64_t ldq;
  const uint16_t* kc;
  const uint16_t* vc;
  int64_t num_blocks;
  int heads;
  int kv_heads;
  const int32_t* bt;
  int max_blocks;
  const int32_t* ctx;
  const int32_t* qrows;
  int part_tokens;  // keys per workgroup-level split (multiple of 16)
  int splits;       // workgroups per (sequence, KV head)
  int serpentine;   // plan rows taken in serpentine order (kDecodeSerpentineRows)
  float scale_log2;
  uint16_t* out;
  int64_t ldo;
  float* ws_o;   // [num_seqs][heads][splits][128] unnormalized output of each split
  float* ws_ml;  // [num_seqs][heads][splits][2]   (running max, sum of exp) of each split
  // Fused front half (the QKV template flag): q points at the projection rows [q | k | v] and the
  // kernel applies the per-head RMSNorm and RoPE of model/qwen3.py:95-98 itself, writes the new
  // token's key and value into the cache and attends to them from registers.
  const uint16_t* qn_w;
  const uint16_t* kn_w;
  float qk_eps;
  const float* cos_t;  // [max_pos, 128] float32, a row per position (ROWS: per row of q)
  const float* sin_t;
  int64_t max_pos;
  const int64_t* slots;  // [T] cache slot of each row's new token (< 0: not written)
};

__device__ __forceinline__ void unpack8(const uint4& v, float (&f)[8]) {
  f[0] = bf16lo(v.x); f[1] = bf16hi(v.x);
  f[2] = bf16lo(v.y); f[3] = bf16hi(v.y);
  f[4] = bf16lo(v.z); f[5] = bf16hi(v.z);
  f[6] = bf16lo(v.w); f[7] = bf16hi(v.w);
}

// Keys a sequence may read: its context, clamped to its block-table row (memory safety when a
// caller passes inconsistent sizes; correct calls never hit the clamp).
__device__ __forceinline__ int decode_context(const DecodeArgs& a, int seq) {
  const int ctx = a.ctx[seq];
  const int cap = a.max_blocks * kBlock;
  // the same in every lane; saying so keeps the block loop's control flow scalar (a loop the
  // compiler takes as divergent gets conservative waits on its loads)
  return __builtin_amdgcn_readfirstlane(ctx < cap ? ctx : cap);
}

// Workgroup = W wavefronts for one (sequence, KV head, split). Wave w takes blocks b0 + w,
// b0 + w + W, ... of the split, keeping the next block's K and V in flight while it computes one.
// The grid is (KV head, split, sequence) with the KV head fastest, so the workgroups that read the
// other head slices of the same token rows are dispatched together.
//
// Lane (rp, dg) = (lane / 8, lane % 8) owns key rows 2rp and 2rp + 1 of each 16-token block and
// dims [8dg, 8dg + 8) and [64 + 8dg, 64 + 8dg + 8) of each row: one load instruction covers the
// same 128 contiguous bytes of eight rows. bf16 pairs are multiplied with v_dot2_f32_bf16 (exact
// products, float32 sums): q.k takes 8 dot2 per (row, head) plus a 3-step DPP sum over the 8
// lanes of the row; p.v pairs the two rows' values of each dim with v_perm and takes 16 dot2 per
// head, with p rounded to bf16 as the MFMA prefill path does. The running maximum of each head is
// wave-uniform (the accumulators are rescaled only when it grows); sums and accumulators are
// lane-local (this lane's rows) and merged over the row pairs, then the wavefronts, at the end.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}
// Sum over the 8 lanes of an aligned 8-lane group (quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror).
__device__ __forceinline__ float group8_sum(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  return v;
}
// Across the 8 row-pair groups of a wavefront (values are uniform within each 8-lane group).
__device__ __forceinline__ float rowpair_max(float v) {
  v = fmaxf(v, dpp<0x140>(v));  // row_mirror: group g <-> the other group of its 16-lane row
  return xrow_max(v);
}
__device__ __forceinline__ float rowpair_sum(float v) {
  v += dpp<0x128>(v);  // row_ror:8 -- lane l ^ 8 within its 16-lane row
  return xrow_sum(v);
}

// Per-head RMSNorm then RoPE (model/layers.py:18-22, 56-65 rounding) of the 16 dims this lane holds
// -- [8dg, 8dg + 8) in v[0..3] and their rotary partners [64 + 8dg, 64 + 8dg + 8) in v[4..7], as
// bf16 pairs -- given the norm weights of those dims and the float32 cos / sin of the position.
// The sum of squares is completed over the 8 lanes of the lane's group (one head row).
__device__ __forceinline__ void norm_rope16(uint32_t (&v)[8], const uint4& wlo, const uint4& whi, const float (&c)[16],
                                            const float (&sn)[16], float eps) {
  float x[16];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    x[2 * (e & 3) + 8 * (e >> 2)] = bf16lo(v[e]);
    x[2 * (e & 3) + 1 + 8 * (e >> 2)] = bf16hi(v[e]);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) ss += x[i] * x[i];
  ss = group8_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)kHeadDim + eps);
  const uint32_t ww[8] = {wlo.x, wlo.y, wlo.z, wlo.w, whi.x, whi.y, whi.z, whi.w};
  float y[16];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    y[2 * (e & 3) + 8 * (e >> 2)] = round_bf16(bf16lo(ww[e]) * round_bf16(x[2 * (e & 3) + 8 * (e >> 2)] * r));
    y[2 * (e & 3) + 1 + 8 * (e >> 2)] = round_bf16(bf16hi(ww[e]) * round_bf16(x[2 * (e & 3) + 1 + 8 * (e >> 2)] * r));
  }
  float o[16];
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // dim 8dg + i pairs with 64 + 8dg + i
    const float x0 = y[i], x1 = y[8 + i];
    o[i] = round_bf16(round_bf16(x0 * round_bf16(c[i])) + round_bf16(-x1 * round_bf16(sn[i])));
    o[8 + i] = round_bf16(round_bf16(x1 * round_bf16(c[8 + i])) + round_bf16(x0 * round_bf16(sn[8 + i])));
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = pack_bf16x2(o[2 * (e & 3) + 8 * (e >> 2)], o[2 * (e & 3) + 1 + 8 * (e >> 2)]);
}

// ROWS (of QKV): the new token's rotary row is its own of rows the caller gathered, not position ctx - 1's.
template <int G, int W, bool QKV, bool ROWS = false>
__global__ __launch_bounds__(64 * W) void paged_decode_kernel(DecodeArgs a) {
  __shared__ float s_acc[W][G][kHeadDim];
  __shared__ float s_ml[W][G][2];
  const int kvh = blockIdx.x, split = blockIdx.z;
  int seq = blockIdx.y;
  if (a.serpentine) {  // alternate passes of 32 plan rows reversed (see kDecodeSerpentineRows)
    const int base = seq & ~31, cnt = min(32, (int)gridDim.y - base);
    if ((seq >> 5) & 1) seq = base + cnt - 1 - (seq - base);
  }
  const int start = split * a.part_tokens;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar control flow
  const int rp = lane >> 3, dg = lane & 7;
  const int32_t* btr = a.bt + (int64_t)seq * a.max_blocks;
  const int64_t tok_stride = (int64_t)a.kv_heads * kHeadDim;
  const int64_t lane_off = (int64_t)(2 * rp) * tok_stride + (int64_t)kvh * kHeadDim + 8 * dg;
  // Lane i holds the table entry of this wavefront's i-th block, bfirst + i * W (a split has at
  // most 64 blocks per wavefront, checked on the host), read with the context length, not after
  // it: indices are clamped into the table row, and a block past the context (a padding entry) is
  // loaded but never used. The block loop then reads entries with readlane and issues no table
  // loads of its own. Every load below is issued unconditionally -- indices are clamped and dead
  // loads masked to one address instead of branched around -- so that the compiler's in-order
  // load counter stays exact and waiting for one block never waits for the next one's loads.
  const int bfirst = start / kBlock + wave;
  const int tab = btr[min(bfirst + lane * W, a.max_blocks - 1)];
  const int ph0 = __builtin_amdgcn_readlane(tab, 0);
  const int64_t qrow = a.qrows[seq];
  const int ctx = decode_context(a, seq);

  // q of this lane's 16 dims for each head of the group, as bf16 pairs
  uint32_t qv[G][8];
  uint32_t kn[8], vn[8];  // fused: the new token's key (normed, rotated) and value, this KV head
  auto load8 = [&](const uint16_t* p, uint32_t (&v)[8]) {
    const uint4 lo = *(const uint4*)p, hi = *(const uint4*)(p + 64);
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
    v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  };
  // [row rr][half]: rows 2rp + rr, dims 8dg.. (half 0) and 64 + 8dg.. (half 1) of physical block
  // phys. A dead load (live false) reads the cache's first 16 bytes at every lane: one cache line.
  auto load_block = [&](int phys, bool live, uint4 (&kr)[2][2], uint4 (&vr)[2][2]) {
    phys = ((uint32_t)phys < (uint64_t)a.num_blocks) ? phys : 0;  // out-of-range table entries read block 0
    const int64_t mask = -(int64_t)live;
    const int64_t base = ((int64_t)phys * kBlock * tok_stride + lane_off) & mask;
    const int64_t rs = tok_stride & mask, hs = 64 & mask;
#pragma unroll
    for (int rr = 0; rr < 2; ++rr)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        kr[rr][hf] = load_once16(a.kc + base + rr * rs + hf * hs);
        vr[rr][hf] = load_once16(a.vc + base + rr * rs + hf * hs);
      }
  };
  uint4 ka[2][2], va[2][2], kb[2][2], vb[2][2];
  const uint16_t* qrow_p = a.q + qrow * a.ldq;
  if constexpr (!QKV) {
#pragma unroll
    for (int h = 0; h < G; ++h) load8(qrow_p + (int64_t)(kvh * G + h) * kHeadDim + 8 * dg, qv[h]);
  } else {
    // Fused front half: the new token sits at position ctx - 1 (model_runner.py:186-189). The G
    // query heads and the key are normed and rotated once per workgroup lane group: vector v of
    // the G + 1 is done by the row-pair group rp == v (of its round), then every lane gathers
    // all of them from those groups' lanes with the same dims.
    load8(qrow_p + (int64_t)(a.heads + a.kv_heads + kvh) * kHeadDim + 8 * dg, vn);
    int64_t pos = ROWS ? qrow : (int64_t)ctx - 1;
    pos = pos < 0 ? 0 : (pos >= a.max_pos ? a.max_pos - 1 : pos);  // memory safety only
    float c[16], sn[16];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const float4* cp = (const float4*)(a.cos_t + pos * kHeadDim + 64 * hf + 8 * dg);
      const float4* sp = (const float4*)(a.sin_t + pos * kHeadDim + 64 * hf + 8 * dg);
      const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
      c[8 * hf + 0] = c0.x; c[8 * hf + 1] = c0.y; c[8 * hf + 2] = c0.z; c[8 * hf + 3] = c0.w;
      c[8 * hf + 4] = c1.x; c[8 * hf + 5] = c1.y; c[8 * hf + 6] = c1.z; c[8 * hf + 7] = c1.w;
      sn[8 * hf + 0] = s0.x; sn[8 * hf + 1] = s0.y; sn[8 * hf + 2] = s0.z; sn[8 * hf + 3] = s0.w;
      sn[8 * hf + 4] = s1.x; sn[8 * hf + 5] = s1.y; sn[8 * hf + 6] = s1.z; sn[8 * hf + 7] = s1.w;
    }
    constexpr int kRounds = (G + 1 + 7) / 8;
    // Round 0's vector and norm weights are loaded before the first K / V block, which then
    // streams in while the norms and RoPE are computed (the loads complete in issue order, so
    // waiting for these does not wait for the block).
    uint32_t mine0[8];
    uint4 nw0lo, nw0hi;
    {
      const int vi = min(rp, G);
      const bool is_k = vi == G;
      load8(qrow_p + (int64_t)(is_k ? a.heads + kvh : kvh * G + vi) * kHeadDim + 8 * dg, mine0);
      const uint16_t* nw = is_k ? a.kn_w : a.qn_w;
      nw0lo = *(const uint4*)(nw + 8 * dg);
      nw0hi = *(const uint4*)(nw + 64 + 8 * dg);
    }
    __builtin_amdgcn_sched_barrier(0);
    load_block(ph0, bfirst < a.max_blocks, ka, va);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int round = 0; round < kRounds; ++round) {
      const int vi = min(round * 8 + rp, G);  // groups past the last vector redo the key (unused)
      const bool is_k = vi == G;
      uint32_t mine[8];
      if (round == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) mine[e] = mine0[e];
        norm_rope16(mine, nw0lo, nw0hi, c, sn, a.qk_eps);
      } else {
        load8(qrow_p + (int64_t)(is_k ? a.heads + kvh : kvh * G + vi) * kHeadDim + 8 * dg, mine);
        const uint16_t* nw = is_k ? a.kn_w : a.qn_w;
        norm_rope16(mine, *(const uint4*)(nw + 8 * dg), *(const uint4*)(nw + 64 + 8 * dg), c, sn, a.qk_eps);
      }
#pragma unroll
      for (int v = round * 8; v < min(round * 8 + 8, G + 1); ++v) {
        const int src = (v - round * 8) * 8 + dg;  // lane holding vector v's dims for this dg
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t x = (uint32_t)__shfl((int)mine[e], src);
          if (v < G) qv[v][e] = x; else kn[e] = x;
        }
      }
    }
  }
  float m[G], l[G], acc[G][16];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[h][e] = 0.f;
  }
  if constexpr (!QKV) load_block(ph0, bfirst < a.max_blocks, ka, va);  // before the context length is checked
  if (start >= ctx) return;  // the reduce kernel merges only splits that hold keys
  // Fused: the cache is read for the keys before the new token, which comes from registers.
  const int end = min(QKV ? ctx - 1 : ctx, start + a.part_tokens);
  const int b1 = (end + kBlock - 1) / kBlock;

  // One block of q.k, online softmax and p.v on K/V registers kr, vr (wave-uniform block index).
  auto process = [&](int blk, const uint4 (&kr)[2][2], uint4 (&vr)[2][2]) {
    float sc[G][2];
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      const uint32_t kw[8] = {kr[rr][0].x, kr[rr][0].y, kr[rr][0].z, kr[rr][0].w,
                              kr[rr][1].x, kr[rr][1].y, kr[rr][1].z, kr[rr][1].w};
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d = dot2(kw[e], qv[h][e], d);
        sc[h][rr] = group8_sum(d) * a.scale_log2;
      }
    }
    if (blk * kBlock + kBlock > end) {  // the split's last, partial block
#pragma unroll
      for (int rr = 0; rr < 2; ++rr) {
        if (blk * kBlock + 2 * rp + rr >= end) {
#pragma unroll
          for (int h = 0; h < G; ++h) sc[h][rr] = -INFINITY;
          vr[rr][0] = uint4{0, 0, 0, 0};  // masked rows contribute exactly zero even if stale
          vr[rr][1] = uint4{0, 0, 0, 0};
        }
      }
    }
    uint32_t pp[G];
#pragma unroll
    for (int h = 0; h < G; ++h) {
      // the block's max over its rows, the same in every lane (finite: row 0 of the block is visible)
      const float bm = __builtin_bit_cast(
          float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, rowpair_max(fmaxf(sc[h][0], sc[h][1])))));
      if (bm > m[h]) {  // wave-uniform
        const float alpha = exp2f(m[h] - bm);
        m[h] = bm;
        l[h] *= alpha;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[h][e] *= alpha;
      }
      pp[h] = pack_bf16x2(exp2f(sc[h][0] - m[h]), exp2f(sc[h][1] - m[h]));
      l[h] += bf16lo(pp[h]) + bf16hi(pp[h]);  // the weights actually applied
    }
    const uint32_t v0[8] = {vr[0][0].x, vr[0][0].y, vr[0][0].z, vr[0][0].w,
                            vr[0][1].x, vr[0][1].y, vr[0][1].z, vr[0][1].w};
    const uint32_t v1[8] = {vr[1][0].x, vr[1][0].y, vr[1][0].z, vr[1][0].w,
                            vr[1][1].x, vr[1][1].y, vr[1][1].z, vr[1][1].w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t lo = __builtin_amdgcn_perm(v1[e], v0[e], 0x05040100u);  // (v0[2e], v1[2e])
      const uint32_t hi = __builtin_amdgcn_perm(v1[e], v0[e], 0x07060302u);  // (v0[2e+1], v1[2e+1])
#pragma unroll
      for (int h = 0; h < G; ++h) {
        acc[h][2 * e] = dot2(lo, pp[h], acc[h][2 * e]);
        acc[h][2 * e + 1] = dot2(hi, pp[h], acc[h][2 * e + 1]);
      }
    }
  };

  // Two register buffers in turn, the next block's loads in flight while one is processed: pairs
  // of blocks per iteration and the odd last block after the loop -- a loop with a single exit, so
  // the compiler's wait counting sees every buffer consumed before it is reloaded. Entry j of the
  // table (this wavefront's block bfirst + j * W) is lane j of tab.
  const int nb = bfirst < b1 ? (b1 - bfirst + W - 1) / W : 0;  // this wavefront's blocks
  auto entry = [&](int j) { return __builtin_amdgcn_readlane(tab, min(j, 63)); };
  int i = 0;  // block i (ka) is loaded at the top of each iteration
  for (; i + 2 <= nb; i += 2) {
    load_block(entry(i + 1), true, kb, vb);
    process(bfirst + i * W, ka, va);
    load_block(entry(i + 2), i + 2 < nb, ka, va);
    process(bfirst + (i + 1) * W, kb, vb);
  }
  if (i < nb) process(bfirst + i * W, ka, va);
  if constexpr (QKV) {
    // The new token: the last wavefront of the split holding position ctx - 1 attends to it (row 0
    // of its lanes' first row pair only) and writes its key and value into the cache. Blocks are
    // dealt to the wavefronts from wavefront 0 on, so the last one never holds more of them than
    // another (a step of 64 sequences measured 7 us faster than with the work on wavefront 0).
    if (wave == W - 1 && ctx - 1 < start + a.part_tokens) {
      float sc[G];
#pragma unroll
      for (int h = 0; h < G; ++h) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d = dot2(kn[e], qv[h][e], d);
        sc[h] = group8_sum(d) * a.scale_log2;  // the same in every row pair
      }
#pragma unroll
      for (int h = 0; h < G; ++h) {
        if (sc[h] > m[h]) {  // wave-uniform
          const float alpha = exp2f(m[h] - sc[h]);
          m[h] = sc[h];
          l[h] *= alpha;
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[h][e] *= alpha;
        }
        if (rp == 0) {
          const float p = round_bf16(exp2f(sc[h] - m[h]));
          l[h] += p;
#pragma unroll
          for (int e = 0; e < 8; ++e) {  // acc[h][e]: dim 8dg + e (e < 8), 64 + 8dg + e - 8 (e >= 8)
            const int x = 2 * (e & 3) + 8 * (e >> 2);
            acc[h][x] += bf16lo(vn[e]) * p;
            acc[h][x + 1] += bf16hi(vn[e]) * p;
          }
        }
      }
      if (rp == 0) {
        const int64_t slot = a.slots[qrow];
        if (slot >= 0 && slot < a.num_blocks * kBlock) {
          const int64_t off = slot * tok_stride + (int64_t)kvh * kHeadDim + 8 * dg;
          *(uint4*)(const_cast<uint16_t*>(a.kc) + off) = uint4{kn[0], kn[1], kn[2], kn[3]};
          *(uint4*)(const_cast<uint16_t*>(a.kc) + off + 64) = uint4{kn[4], kn[5], kn[6], kn[7]};
          *(uint4*)(const_cast<uint16_t*>(a.vc) + off) = uint4{vn[0], vn[1], vn[2], vn[3]};
          *(uint4*)(const_cast<uint16_t*>(a.vc) + off + 64) = uint4{vn[4], vn[5], vn[6], vn[7]};
        }
      }
    }
  }
  // Merge the row pairs of the wavefront (lanes dg, dg + 8, ...), then the wavefronts through LDS.
  // acc[h][e]: dim 8dg + e for e < 8, 64 + 8dg + (e - 8) for e >= 8.
#pragma unroll
  for (int h = 0; h < G; ++h) {
    l[h] = rowpair_sum(l[h]);  // the 8 row pairs; each lane of a pair already holds the pair's sum
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[h][e] = rowpair_sum(acc[h][e]);
    if (rp == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s_acc[wave][h][8 * dg + e] = acc[h][e];
        s_acc[wave][h][64 + 8 * dg + e] = acc[h][8 + e];
      }
    }
    if (lane == 0) {
      s_ml[wave][h][0] = m[h];  // -inf for a wavefront that got no block
      s_ml[wave][h][1] = l[h];
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < G * kHeadDim; idx += 64 * W) {
    const int h = idx / kHeadDim, d = idx % kHeadDim;
    float mx = s_ml[0][h][0];  // -inf for a wavefront with no key; some wavefront holds one
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_ml[w][h][0]);
    float den = 0.f, num = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float f = exp2f(s_ml[w][h][0] - mx);
      den += f * s_ml[w][h][1];
      num += f * s_acc[w][h][d];
    }
    const int head = kvh * G + h;
    // A sequence whose keys fit one split is finished here (the merge kernel skips it: with one
    // split its factor would be exp2(0) = 1, so the value is the same).
    if (a.splits == 1 || ctx <= a.part_tokens) {
      a.out[qrow * a.ldo + (int64_t)head * kHeadDim + d] = f32_to_bf16(num / den);
    } else {
      const int64_t slot = ((int64_t)seq * a.heads + head) * a.splits + split;
      a.ws_o[slot * kHeadDim + d] = num;
      if (d == 0) *(float2*)(a.ws_ml + slot * 2) = float2{mx, den};
    }
  }
}

// Merge of the workgroup-level splits of each (sequence, query head): one thread per dim. Every load
// -- the context, lane p's (maximum, sum) of split p, the splits' partial values -- is issued at once,
// unconditionally (slots past the sequence's splits hold anything and are not used), so the kernel
// waits for memory once instead of four times in a row: 7.8 -> 4.8 us for one sequence of 18
// splits at 32 heads, 6.7 -> 4.7 for three of 15 (traced durations).
constexpr int kReduceSplits = 64;  // a wavefront's lanes
template <int CH>
__global__ __launch_bounds__(kHeadDim) void paged_decode_reduce_kernel(DecodeArgs a) {
  const int seq = blockIdx.x, head = blockIdx.y, d = threadIdx.x, lane = threadIdx.x & 63;
  const int64_t base = ((int64_t)seq * a.heads + head) * a.splits;
  const float* po = a.ws_o + base * kHeadDim + d;
  const float2 ml = *(const float2*)(a.ws_ml + (base + min(lane, a.splits - 1)) * 2);
  float o[CH];
#pragma unroll
  for (int p = 0; p < CH; ++p) o[p] = po[min(p, a.splits - 1) * kHeadDim];
  const int qrow = a.qrows[seq];
  const int ctx = decode_context(a, seq);
  const int nsplit = min(a.splits, (ctx + a.part_tokens - 1) / a.part_tokens);
  if (nsplit <= 1) return;  // one split (or none): the attention kernel wrote the output itself
  const float mx = wave_max(lane < nsplit ? ml.x : -INFINITY);
  const float f = lane < nsplit ? exp2f(ml.x - mx) : 0.f;
  const float den = wave_sum(lane < nsplit ? f * ml.y : 0.f);
  float num = 0.f;
#pragma unroll
  for (int p = 0; p < CH; ++p) {
    const float fp = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), p));
    if (p < nsplit) num += fp * o[p];
  }
  for (int p = CH; p < nsplit; ++p)
    num += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), p)) * po[p * kHeadDim];
  a.out[(int64_t)qrow * a.ldo + (int64_t)head * kHeadDim + d] = f32_to_bf16(num / den);
}

// The merge for more splits than kReduceSplits, one after another.
__global__ __launch_bounds__(kHeadDim) void paged_decode_reduce_many_kernel(DecodeArgs a) {
  const int seq = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  const int ctx = decode_context(a, seq);
  const int nsplit = min(a.splits, (ctx + a.part_tokens - 1) / a.part_tokens);
  if (nsplit <= 1) return;  // one split (or none): the attention kernel wrote the output itself
  const int64_t base = ((int64_t)seq * a.heads + head) * a.splits;
  float mx = -INFINITY;
  for (int p = 0; p < nsplit; ++p) mx = fmaxf(mx, a.ws_ml[(base + p) * 2]);
  float den = 0.f, num = 0.f;
  for (int p = 0; p < nsplit; ++p) {
    const float2 ml = *(const float2*)(a.ws_ml + (base + p) * 2);
    const float f = exp2f(ml.x - mx);
    den += f * ml.y;
    num += f * a.ws_o[(base + p) * kHeadDim + d];
  }
  a.out[(int64_t)a.qrows[seq] * a.ldo + (int64_t)head * kHeadDim + d] = f32_to_bf16(num / den);
}

static void launch_reduce(const DecodeArgs& a, int num_seqs, hipStream_t s) {
  const dim3 grid(num_seqs, a.heads), block(kHeadDim);
  if (a.splits <= 8) hipLaunchKernelGGL(paged_decode_reduce_kernel<8>, grid, block, 0, s, a);
  else if (a.splits <= kReduceSplits) hipLaunchKernelGGL(paged_decode_reduce_kernel<32>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(paged_decode_reduce_many_kernel, grid, block, 0, s, a);
}

// ---------------------------------------------------------------------------------------------

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;  // an LDS pointer for the transposing reads

constexpr int kKeyTile = 32;              // keys per LDS tile
constexpr int kKsStride = kHeadDim + 8;   // bf16 elements per K row in LDS
constexpr int kVsStride = kHeadDim + 16;  // per V row: 288 bytes, so the 4 rows x 32 bytes a
                                          // transposing read gathers per 16 lanes hit distinct banks
constexpr int kKsTile = kKeyTile * kKsStride;
constexpr int kVsTile = kKeyTile * kVsStride;
constexpr int kKeyGroups = 3;  // groups of four wavefronts splitting a workgroup's key tiles
// Per key group two buffers of K and V (both key-major): 107,520 bytes, one workgroup of twelve
// wavefronts per CU, which leaves room for one four-wavefront decode workgroup beside it.
constexpr size_t kPrefillLds = (size_t)kKeyGroups * 2 * (kKsTile + kVsTile) * 2;
constexpr int kXchFloats = 34 * 64;  // per wavefront at the merge: 32 accumulators, m, l per lane
static_assert((size_t)4 * (kKeyGroups - 1) * kXchFloats * 4 <= kPrefillLds, "merge exchange fits the tile buffers");

struct PrefillArgs {
  const uint16_t* q;
  int64_t ldq;
  const uint16_t* kc;
  const uint16_t* vc;
  int64_t num_blocks;
  int heads;
  int kv_heads;
  const int32_t* bt;
  int max_blocks;
  const int32_t* seq_info;  // [S][3] flat start, num_new, num_cached
  const int32_t* work;      // [W][2] sequence, first new-token index of the tile
  float scale_log2;
  uint16_t* out;
  int64_t ldo;
};

// Three key groups of four wavefronts: group kg takes key tiles kg, kg + 3, ... of the workgroup's
// query tile, with its own double-buffered K / V tiles, and hands its softmax state to group 0
// through LDS at the end -- a third of the chain of key tiles of the longest query tile, which
// sets the time of a causal chunk (1984-token chunk: 50.9 µs, against 52.1 with four groups and
// 55.0 with two groups at two workgroups per CU). Twelve wavefronts of 118 VGPRs leave each SIMD
// room for one more wavefront: the decode rows of a mixed batch (four-wavefront workgroups, on
// another stream) run beside the chunk instead of after it.
template <int G, bool OFF32>
__global__ __launch_bounds__(256 * kKeyGroups) __attribute__((amdgpu_waves_per_eu(4, 4))) void paged_prefill_kernel(PrefillArgs a) {
  constexpr int kSub = 4 / G;       // 16-token query sub-tiles per workgroup
  constexpr int kQTok = 16 * kSub;  // query tokens per workgroup
  extern __shared__ __attribute__((aligned(16))) uint16_t psm[];
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // key group
  const int tg = threadIdx.x & 255;                                  // thread within the key group
  uint16_t* Ks = psm + kg * 2 * (kKsTile + kVsTile);  // [2][kKeyTile][kKsStride]
  uint16_t* Vs = Ks + 2 * kKsTile;                     // [2][kKeyTile][kVsStride]

  // KV head fastest in dispatch order: workgroups go round-robin over the 8 XCDs, so with 8 KV
  // heads each XCD serves one head and its L2 holds that head's keys and values for every query
  // tile (work items stay longest first).
  const int lin = blockIdx.x + gridDim.x * blockIdx.y;
  const int kvh = lin % a.kv_heads, wi = lin / a.kv_heads;
  const int seq = a.work[2 * wi], tstart = a.work[2 * wi + 1];
  const int flat = a.seq_info[3 * seq], nnew = a.seq_info[3 * seq + 1], ncached = a.seq_info[3 * seq + 2];
  const int lane = threadIdx.x & 63, wave = tg >> 6;  // wavefront within the key group
  const int g = wave % G, st = wave / G;
  const int head = kvh * G + g;
  const int j = lane & 15, grp = lane >> 4;

  const int qi = tstart + st * 16 + j;
  const bool qvalid = qi < nnew;
  const int qi_c = qvalid ? qi : nnew - 1;
  const int qpos = ncached + qi_c;
  const int wave_last = ncached + min(tstart + st * 16 + 15, nnew - 1);
  const int wave_first = ncached + min(tstart + st * 16, nnew - 1);  // the wave's lowest query position

  bf16x8 qfrag[4];
  {
    const uint16_t* qp = a.q + (int64_t)(flat + qi_c) * a.ldq + (int64_t)head * kHeadDim + 8 * grp;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qfrag[ks] = *(const bf16x8*)(qp + 32 * ks);
  }

  const int kend = ncached + min(tstart + kQTok, nnew);
  const int ntiles = (kend + kKeyTile - 1) / kKeyTile;
  const int niter = (ntiles + kKeyGroups - 1) / kKeyGroups;  // tiles per key group (the last ones may idle once)
  const int32_t* btr = a.bt + (int64_t)seq * a.max_blocks;
  const int64_t tok_stride = (int64_t)a.kv_heads * kHeadDim;

  // Loader role within the key group: keys 2la and 2la + 1 of the tile (both in block
  // tile * 2 + la / 8, rows 2 (la % 8) and 2 (la % 8) + 1 of it), 8-wide dim chunk lb. A tile's
  // table entry is read one tile before its keys and values, so the keys never wait on a table
  // read; every load is issued unconditionally (a dead key's address masked to the cache's first
  // row). Dead keys (past kend, only in the last tile) are masked out of the scores by the causal
  // mask; their values are zeroed where they are stored, so the probability 0 they get multiplies
  // a zero. The dim chunk is the fast index: 16 consecutive lanes read one key's 256 contiguous
  // bytes and store one LDS row, which no two of them share a bank in (with the key as the fast
  // index the V rows' 288-byte pitch put four lanes on each bank: 1984-token chunk 51.8 -> 44.5 us).
  const int la = tg >> 4, lb = tg & 15;
  const int64_t thread_off = (int64_t)(2 * (la % 8)) * tok_stride + (int64_t)kvh * kHeadDim + 8 * lb;
  // OFF32 (a cache of under 4 GB, checked on the host): 32-bit byte offsets from the cache base --
  // one 24-bit multiply per tile instead of 64-bit address arithmetic per load.
  const uint32_t thread_off_b = (uint32_t)thread_off * 2u;
  const uint32_t row_b = (uint32_t)tok_stride * 2u, block_b = (uint32_t)kBlock * row_b;
  uint4 kr[2], vr[2];  // [key rr]
  int dead_from = 2;   // keys rr >= dead_from of this thread's pair are dead
  auto tile_of = [&](int i) { return kg + kKeyGroups * i; };  // the group's i-th tile
  auto table_entry = [&](int tile) {
    return btr[min(tile * (kKeyTile / kBlock) + la / 8, a.max_blocks - 1)];
  };
  auto load_tile = [&](int tile, int phys) {
    phys = ((uint32_t)phys < (uint64_t)a.num_blocks) ? phys : 0;
    const int key = tile * kKeyTile + 2 * la;
    const bool blk_ok = tile * (kKeyTile / kBlock) + la / 8 < a.max_blocks;
    dead_from = !blk_ok || key >= kend ? 0 : (key + 1 >= kend ? 1 : 2);
    // loaded as vector values, not struct copies (which the compiler keeps in scratch)
    u32x4 k0, v0, k1, v1;
    if constexpr (OFF32) {
      const uint32_t base = __umul24((unsigned)phys, block_b) + thread_off_b;
      const uint32_t off0 = (blk_ok && key < kend) ? base : 0u;
      const uint32_t off1 = (blk_ok && key + 1 < kend) ? base + row_b : 0u;
      k0 = *(const u32x4*)((const char*)a.kc + off0);
      v0 = *(const u32x4*)((const char*)a.vc + off0);
      k1 = *(const u32x4*)((const char*)a.kc + off1);
      v1 = *(const u32x4*)((const char*)a.vc + off1);
    } else {
      const int64_t base = (int64_t)phys * kBlock * tok_stride + thread_off;
      const int64_t off0 = (blk_ok && key < kend) ? base : 0;
      const int64_t off1 = (blk_ok && key + 1 < kend) ? base + tok_stride : 0;
      k0 = *(const u32x4*)(a.kc + off0);
      v0 = *(const u32x4*)(a.vc + off0);
      k1 = *(const u32x4*)(a.kc + off1);
      v1 = *(const u32x4*)(a.vc + off1);
    }
    kr[0] = uint4{k0.x, k0.y, k0.z, k0.w};
    vr[0] = uint4{v0.x, v0.y, v0.z, v0.w};
    kr[1] = uint4{k1.x, k1.y, k1.z, k1.w};
    vr[1] = uint4{v1.x, v1.y, v1.z, v1.w};
  };
  auto store_tile = [&](int buf, bool last) {
    uint16_t* K = Ks + buf * kKsTile;
    uint16_t* V = Vs + buf * kVsTile;
    if (last) {  // wave-uniform: only the sequence's last tile holds dead keys
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
        if (rr >= dead_from) vr[rr] = uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      *(uint4*)&K[(2 * la + rr) * kKsStride + 8 * lb] = kr[rr];
      *(uint4*)&V[(2 * la + rr) * kVsStride + 8 * lb] = vr[rr];
    }
  };
  auto is_last = [&](int tile) { return (tile + 1) * kKeyTile > kend; };
  // The PV product's A operand (V^T fragments) straight from the key-major V tile with gfx950's
  // transposing LDS read: in each 16-lane group, lane i names 4 dims of one key row (row i / 4 of
  // the group's 4, dims 4 (i % 4)..+3) and lane 4a + c receives dim c of rows a, a + 4, a + 8,
  // a + 12 -- so lane (grp, j) gets dim dt * 16 + j of keys 4grp..4grp + 3 (and, from the second
  // read, 16 + 4grp..), the key order of its probabilities.
  const int vt_off = (4 * grp + (j >> 2)) * kVsStride + 4 * (j & 3);  // element offset, half 0, dt 0

  f32x4 acc[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Row sums of the probabilities on MFMA: ones (16 x 32) times P gives every lane its query's sum
  // over the tile's keys, accumulated like the outputs (and rescaled with them).
  f32x4 lsum = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
  float m = -INFINITY;

  // Pipeline per key group: its tile i is computed from LDS buffer i % 2 while the registers
  // receive its tile i + 1; those are written to the other buffer after the MFMAs, then tile i + 2
  // is requested. All groups run niter iterations, so every barrier is reached by all wavefronts.
  load_tile(tile_of(0), table_entry(tile_of(0)));
  const int ph1 = table_entry(tile_of(1));
  store_tile(0, is_last(tile_of(0)));
  if (niter > 1) load_tile(tile_of(1), ph1);
  int ph_next = table_entry(tile_of(2));  // the entry of the group's tile i + 2 at the top of iteration i
  __syncthreads();
  for (int i = 0; i < niter; ++i) {
    const int buf = i & 1;
    const int key0 = tile_of(i) * kKeyTile;
    if (key0 <= wave_last) {  // else every query of this wavefront precedes the tile (or it is past kend)
      const uint16_t* K = Ks + buf * kKsTile;
      const uint16_t* V = Vs + buf * kVsTile;
      f32x4 sT[2];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        sT[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const bf16x8 kf = *(const bf16x8*)&K[(mt * 16 + j) * kKsStride + 32 * ks + 8 * grp];
          sT[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qfrag[ks], sT[mt], 0, 0, 0);
        }
      }
      // this lane's 8 raw scores q.k: keys mt * 16 + 4grp + rr (s8[mt * 4 + rr])
      float s8[8];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) s8[mt * 4 + rr] = sT[mt][rr];
      if (key0 + kKeyTile - 1 > wave_first) {  // wave-uniform: a tile on the diagonal
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr)
            if (key0 + mt * 16 + 4 * grp + rr > qpos) s8[mt * 4 + rr] = -INFINITY;
      }
      float bm = fmaxf(fmaxf(fmaxf(s8[0], s8[1]), fmaxf(s8[2], s8[3])), fmaxf(fmaxf(s8[4], s8[5]), fmaxf(s8[6], s8[7])));
      bm = xrow_max(bm) * a.scale_log2;  // the scale is positive: the maximum of the scaled scores
      // group 0 sees key 0 first, so its maximum is finite from the first tile on; a later group's
      // wavefront whose first visible tile masks a whole row keeps -inf there and adds zeros
      const float mn = fmaxf(m, bm);
      // Rescale only when some row's maximum grew: elsewhere the factor is exp2(0) = 1 exactly.
      if (__builtin_amdgcn_ballot_w64(mn > m)) {
        const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);  // 0 from m = -inf
        lsum *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) acc[dt] *= alpha;
      }
      m = mn;
      // p = exp2(s * scale - mn) with one rounding (fma); a row still at -inf subtracts 0 and
      // gets exp2(-inf) = 0. The hardware exp2: arguments are <= 0 and results below 2^-126 are
      // negligible against the row's largest weight, 1.
      const float mb = mn == -INFINITY ? 0.0f : mn;
      bf16x8 pb;
#pragma unroll
      for (int e = 0; e < 8; ++e) pb[e] = (__bf16)__builtin_amdgcn_exp2f(__builtin_fmaf(s8[e], a.scale_log2, -mb));
      lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb, lsum, 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(V + vt_off + dt * 16));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(V + vt_off + 16 * kVsStride + dt * 16));
        const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb, acc[dt], 0, 0, 0);
      }
    }
    if (i + 1 < niter) {
      store_tile(buf ^ 1, is_last(tile_of(i + 1)));  // buffer of the group's tile i - 1: every wavefront passed the barrier after it
      if (i + 2 < niter) load_tile(tile_of(i + 2), ph_next);
      ph_next = table_entry(tile_of(i + 3));
    }
    __syncthreads();
  }
  float l = lsum[0];  // the query's sum over every key this group saw (the same in all four)

  // Merge: groups 1.. leave their state in LDS (over the tile buffers, free after the last
  // barrier); group 0 combines them with its own in group order, lane by lane (the groups' lanes
  // hold the same rows and dims), and writes the output.
  if (kg > 0) {
    float* xw = (float*)psm + ((kg - 1) * 4 + wave) * kXchFloats;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) xw[(dt * 4 + r) * 64 + lane] = acc[dt][r];
    xw[32 * 64 + lane] = m;
    xw[33 * 64 + lane] = l;
  }
  __syncthreads();
  if (kg > 0) return;
  float mm = m;  // finite: group 0 saw key 0
#pragma unroll
  for (int o = 1; o < kKeyGroups; ++o) mm = fmaxf(mm, ((float*)psm + ((o - 1) * 4 + wave) * kXchFloats)[32 * 64 + lane]);
  const float f0 = __builtin_amdgcn_exp2f(m - mm);
  float fo[kKeyGroups];
  l = l * f0;
#pragma unroll
  for (int o = 1; o < kKeyGroups; ++o) {
    const float* xw = (float*)psm + ((o - 1) * 4 + wave) * kXchFloats;
    const float mo = xw[32 * 64 + lane];
    fo[o] = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - mm);
    l += xw[33 * 64 + lane] * fo[o];
  }
  if (!qvalid) return;
  const float inv = 1.0f / l;
  uint16_t* orow = a.out + (int64_t)(flat + qi) * a.ldo + (int64_t)head * kHeadDim;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = acc[dt][r] * f0;
#pragma unroll
      for (int oo = 1; oo < kKeyGroups; ++oo)
        v += ((float*)psm + ((oo - 1) * 4 + wave) * kXchFloats)[(dt * 4 + r) * 64 + lane] * fo[oo];
      o[r] = v * inv;
    }
    const int d = dt * 16 + 4 * grp;
    *(uint2*)(orow + d) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  }
}

// The same attention on 32-query wavefront tiles (v_mfma_f32_32x32x16_bf16): every K and V^T fragment
// read from LDS feeds twice the queries, and a query's keys lie in two lanes instead of four. The
// 16-query kernel is bound by LDS and VALU (per 32-key tile and wavefront 41 ns of LDS reads, its share
// of the stores and ~40 ns of softmax against 33 ns of MFMA); here the reads, the maxima and the tile's
// bookkeeping serve two times the MFMAs: 2000 tokens after 6000 at 32 / 8 heads 376 -> 272 us (0.61 ->
// 0.84 PFLOP/s), 2 x 2048 fresh tokens 152 -> 106. 163 registers: three wavefronts per SIMD and no room
// for a decode wavefront beside them. Taken when it gives enough workgroups (the caller's rule).
constexpr int kVsStride32 = kHeadDim + 32;  // 320 bytes: a transposing read's 4 rows x 64 bytes on distinct banks
constexpr int kVsTile32 = kKeyTile * kVsStride32;
constexpr int kXchFloats32 = 66 * 64;  // per wavefront at the merge: 64 accumulators, m, l per lane
constexpr size_t kPrefillTiles32 = (size_t)kKeyGroups * 2 * (kKsTile + kVsTile32) * 2;
constexpr size_t kPrefillXch32 = (size_t)4 * (kKeyGroups - 1) * kXchFloats32 * 4;
constexpr size_t kPrefillLds32 = kPrefillTiles32 > kPrefillXch32 ? kPrefillTiles32 : kPrefillXch32;

template <int G, bool OFF32>
__global__ __launch_bounds__(256 * kKeyGroups) __attribute__((amdgpu_waves_per_eu(3, 3))) void paged_prefill32_kernel(PrefillArgs a) {
  constexpr int kSub = 4 / G;       // 32-token query sub-tiles per workgroup
  constexpr int kQTok = 32 * kSub;  // query tokens per workgroup
  extern __shared__ __attribute__((aligned(16))) uint16_t psm[];
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // key group
  const int tg = threadIdx.x & 255;                                  // thread within the key group
  uint16_t* Ks = psm + kg * 2 * (kKsTile + kVsTile32);  // [2][kKeyTile][kKsStride]
  uint16_t* Vs = Ks + 2 * kKsTile;                       // [2][kKeyTile][kVsStride32]

  const int lin = blockIdx.x + gridDim.x * blockIdx.y;  // KV head fastest, as in the 16-query kernel
  const int kvh = lin % a.kv_heads, wi = lin / a.kv_heads;
  const int seq = a.work[2 * wi], tstart = a.work[2 * wi + 1];
  const int flat = a.seq_info[3 * seq], nnew = a.seq_info[3 * seq + 1], ncached = a.seq_info[3 * seq + 2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(tg >> 6);  // wavefront within the key group
  const int st = wave / G, head = kvh * G + wave % G;
  const int qc = lane & 31, h = lane >> 5;  // this lane's query column; its half of each 16-wide K slice

  const int qi = tstart + st * 32 + qc;
  const bool qvalid = qi < nnew;
  const int qi_c = qvalid ? qi : nnew - 1;
  const int qpos = ncached + qi_c;
  const int wave_last = ncached + min(tstart + st * 32 + 31, nnew - 1);
  const int wave_first = ncached + min(tstart + st * 32, nnew - 1);

  bf16x8 qfrag[8];  // Q^T, the B operand: dims 16 ks + 8h .. + 7 of query qc
  {
    const uint16_t* qp = a.q + (int64_t)(flat + qi_c) * a.ldq + (int64_t)head * kHeadDim + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qfrag[ks] = *(const bf16x8*)(qp + 16 * ks);
  }

  const int kend = ncached + min(tstart + kQTok, nnew);
  const int ntiles = (kend + kKeyTile - 1) / kKeyTile;
  const int niter = (ntiles + kKeyGroups - 1) / kKeyGroups;
  const int32_t* btr = a.bt + (int64_t)seq * a.max_blocks;
  const int64_t tok_stride = (int64_t)a.kv_heads * kHeadDim;

  const int la = tg >> 4, lb = tg & 15;
  const int64_t thread_off = (int64_t)(2 * (la % 8)) * tok_stride + (int64_t)kvh * kHeadDim + 8 * lb;
  const uint32_t thread_off_b = (uint32_t)thread_off * 2u;
  const uint32_t row_b = (uint32_t)tok_stride * 2u, block_b = (uint32_t)kBlock * row_b;
  u32x4 kr[2], vr[2];
  int dead_from = 2;
  auto tile_of = [&](int i) { return kg + kKeyGroups * i; };
  auto table_entry = [&](int tile) { return btr[min(tile * (kKeyTile / kBlock) + la / 8, a.max_blocks - 1)]; };
  auto load_tile = [&](int tile, int phys) {
    phys = ((uint32_t)phys < (uint64_t)a.num_blocks) ? phys : 0;
    const int key = tile * kKeyTile + 2 * la;
    const bool blk_ok = tile * (kKeyTile / kBlock) + la / 8 < a.max_blocks;
    dead_from = !blk_ok || key >= kend ? 0 : (key + 1 >= kend ? 1 : 2);
    if constexpr (OFF32) {
      const uint32_t base = __umul24((unsigned)phys, block_b) + thread_off_b;
      const uint32_t off0 = (blk_ok && key < kend) ? base : 0u;
      const uint32_t off1 = (blk_ok && key + 1 < kend) ? base + row_b : 0u;
      kr[0] = *(const u32x4*)((const char*)a.kc + off0);
      vr[0] = *(const u32x4*)((const char*)a.vc + off0);
      kr[1] = *(const u32x4*)((const char*)a.kc + off1);
      vr[1] = *(const u32x4*)((const char*)a.vc + off1);
    } else {
      const int64_t base = (int64_t)phys * kBlock * tok_stride + thread_off;
      const int64_t off0 = (blk_ok && key < kend) ? base : 0;
      const int64_t off1 = (blk_ok && key + 1 < kend) ? base + tok_stride : 0;
      kr[0] = *(const u32x4*)(a.kc + off0);
      vr[0] = *(const u32x4*)(a.vc + off0);
      kr[1] = *(const u32x4*)(a.kc + off1);
      vr[1] = *(const u32x4*)(a.vc + off1);
    }
  };
  auto store_tile = [&](int buf, bool last) {
    uint16_t* K = Ks + buf * kKsTile;
    uint16_t* V = Vs + buf * kVsTile32;
    if (last) {
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
        if (rr >= dead_from) vr[rr] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      *(u32x4*)&K[(2 * la + rr) * kKsStride + 8 * lb] = kr[rr];
      *(u32x4*)&V[(2 * la + rr) * kVsStride32 + 8 * lb] = vr[rr];
    }
  };
  auto is_last = [&](int tile) { return (tile + 1) * kKeyTile > kend; };
  // V^T fragments by the transposing read: in each 16-lane group, lane i names 4 dims of key row
  // i / 4 of the group's 4 and lane c receives dim c of those 4 rows. Lane (h, d) of the A operand
  // needs, for the 16-key slice s, keys 16s + 4h + 0..3 and 16s + 8 + 4h + 0..3 of dim d -- the keys
  // whose probabilities the score accumulators leave in lane (h, query).
  const int grp = lane >> 4, j = lane & 15;
  const int vt_off = (4 * (grp >> 1) + (j >> 2)) * kVsStride32 + 16 * (grp & 1) + 4 * (j & 3);

  f32x16 acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) acc[dt] = f32x16{};
  float lsum = 0.f;  // this lane's part of the query's sum (its half of the keys)
  float m = -INFINITY;

  load_tile(tile_of(0), table_entry(tile_of(0)));
  const int ph1 = table_entry(tile_of(1));
  store_tile(0, is_last(tile_of(0)));
  if (niter > 1) load_tile(tile_of(1), ph1);
  int ph_next = table_entry(tile_of(2));
  __syncthreads();
  for (int i = 0; i < niter; ++i) {
    const int buf = i & 1;
    const int key0 = tile_of(i) * kKeyTile;
    if (key0 <= wave_last) {
      const uint16_t* K = Ks + buf * kKsTile;
      const uint16_t* V = Vs + buf * kVsTile32;
      f32x16 sT = f32x16{};
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const bf16x8 kf = *(const bf16x8*)&K[qc * kKsStride + 16 * ks + 8 * h];
        sT = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qfrag[ks], sT, 0, 0, 0);
      }
      // value i of this lane: key 8 (i / 4) + 4h + i % 4 of the tile, query qc
      if (key0 + kKeyTile - 1 > wave_first) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (key0 + 8 * (e >> 2) + 4 * h + (e & 3) > qpos) sT[e] = -INFINITY;
      }
      float bm = fmaxf(sT[0], sT[1]);
#pragma unroll
      for (int e = 2; e < 16; e += 2) bm = fmaxf(fmaxf(sT[e], sT[e + 1]), bm);
      bm = xor32_max(bm) * a.scale_log2;
      const float mn = fmaxf(m, bm);
      if (__builtin_amdgcn_ballot_w64(mn > m)) {
        const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
        lsum *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[dt][e] *= alpha;
      }
      m = mn;
      const float mb = mn == -INFINITY ? 0.0f : mn;
      bf16x8 pb[2];
#pragma unroll
      for (int e = 0; e < 16; ++e)
        pb[e >> 3][e & 7] = (__bf16)__builtin_amdgcn_exp2f(__builtin_fmaf(sT[e], a.scale_log2, -mb));
      // the sum of the rounded probabilities, the ones the product uses
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 w = __builtin_bit_cast(u32x4, pb[s]);
#pragma unroll
        for (int e = 0; e < 4; ++e) lsum = dot2_bf16(w[e], 0x3f803f80u, lsum);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          const uint16_t* vp = V + vt_off + 16 * s * kVsStride32 + dt * 32;
          const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)vp);
          const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vp + 8 * kVsStride32));
          const bf16x8 va = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pb[s], acc[dt], 0, 0, 0);
        }
    }
    if (i + 1 < niter) {
      store_tile(buf ^ 1, is_last(tile_of(i + 1)));
      if (i + 2 < niter) load_tile(tile_of(i + 2), ph_next);
      ph_next = table_entry(tile_of(i + 3));
    }
    __syncthreads();
  }
  float l = xor32_sum(lsum);

  // Merge of the key groups, as in the 16-query kernel.
  if (kg > 0) {
    float* xw = (float*)psm + ((kg - 1) * 4 + wave) * kXchFloats32;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) xw[(dt * 16 + e) * 64 + lane] = acc[dt][e];
    xw[64 * 64 + lane] = m;
    xw[65 * 64 + lane] = l;
  }
  __syncthreads();
  if (kg > 0) return;
  float mm = m;  // finite: group 0 saw key 0
#pragma unroll
  for (int o = 1; o < kKeyGroups; ++o) mm = fmaxf(mm, ((float*)psm + ((o - 1) * 4 + wave) * kXchFloats32)[64 * 64 + lane]);
  const float f0 = __builtin_amdgcn_exp2f(m - mm);
  float fo[kKeyGroups];
  l = l * f0;
#pragma unroll
  for (int o = 1; o < kKeyGroups; ++o) {
    const float* xw = (float*)psm + ((o - 1) * 4 + wave) * kXchFloats32;
    const float mo = xw[64 * 64 + lane];
    fo[o] = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - mm);
    l += xw[65 * 64 + lane] * fo[o];
  }
  if (!qvalid) return;
  const float inv = 1.0f / l;
  uint16_t* orow = a.out + (int64_t)(flat + qi) * a.ldo + (int64_t)head * kHeadDim;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[dt][4 * b + r] * f0;
#pragma unroll
        for (int oo = 1; oo < kKeyGroups; ++oo)
          v += ((float*)psm + ((oo - 1) * 4 + wave) * kXchFloats32)[(dt * 16 + 4 * b + r) * 64 + lane] * fo[oo];
        o[r] = v * inv;
      }
      *(uint2*)(orow + dt * 32 + 8 * b + 4 * h) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    }
}

// The key groups' K / V buffers exceed the 64 KB static LDS limit: dynamic LDS, attribute set once.
template <int G, bool OFF32>
static int launch_prefill_kernel(const PrefillArgs& a, dim3 grid, bool wide, hipStream_t s) {
  if (wide) {
    const int rc = allow_dynamic_lds((const void*)paged_prefill32_kernel<G, OFF32>, (int)kPrefillLds32, "paged_prefill32_kernel");
    if (rc != MSA_OK) return rc;
    hipLaunchKernelGGL((paged_prefill32_kernel<G, OFF32>), grid, dim3(256 * kKeyGroups), kPrefillLds32, s, a);
    return MSA_OK;
  }
  const int rc = allow_dynamic_lds((const void*)paged_prefill_kernel<G, OFF32>, (int)kPrefillLds, "paged_prefill_kernel");
  if (rc != MSA_OK) return rc;
  hipLaunchKernelGGL((paged_prefill_kernel<G, OFF32>), grid, dim3(256 * kKeyGroups), kPrefillLds, s, a);
  return MSA_OK;
}

// 32-bit byte offsets when every block of the cache lies within 4 GB of its base (and a block's
// byte size and index both fit __umul24's 24-bit operands).
template <int G>
static int launch_prefill(const PrefillArgs& a, dim3 grid, bool wide, hipStream_t s) {
  const int64_t block_bytes = (int64_t)kBlock * a.kv_heads * kHeadDim * 2;
  const bool off32 = a.num_blocks * block_bytes < ((int64_t)1 << 32) && block_bytes < (1 << 24) &&
                     a.num_blocks <= (1 << 24);
  return off32 ? launch_prefill_kernel<G, true>(a, grid, wide, s) : launch_prefill_kernel<G, false>(a, grid, wide, s);
}

}  // namespace msa

extern "C" size_t msa_paged_attention_decode_workspace_size(int num_seqs, int heads, int head_dim, int max_partitions) {
  if (num_seqs <= 0 || heads <= 0 || head_dim <= 0 || max_partitions <= 1) return 0;
  const size_t slots = (size_t)num_seqs * heads * max_partitions;
  return slots * head_dim * sizeof(float) + slots * 2 * sizeof(float);
}

namespace msa {
constexpr int kDecodeW = 4;  // wavefronts per decode workgroup
// Keys per workgroup-level split: at most 64 blocks per wavefront (one table entry per lane).
constexpr int kDecodeMaxPartTokens = 64 * kDecodeW * kBlock;

// The plain entry point takes eight wavefronts per workgroup for splits of at least this many
// keys: each wavefront then streams fewer blocks of a long context (64 sequences at contexts
// U[128, 2048]: 5.2 against 4.0 TB/s) when G <= 2 (with G = 4, 207 VGPRs, an eight-wavefront
// workgroup fills a CU alone: slower). Shorter splits, and the fused decode-step entry point
// always, take four: their workgroups of a decode batch are all resident at once (three share a
// CU at the kernel's register count for G <= 2), and the fused step's result must not depend on
// the split size its caller derives from a padded block table.
constexpr int kDecodeWideTokens = 1024;

// The fused decode-step kernel (four-wavefront workgroups, 8 KV heads, one split) at up to this
// many sequences: every workgroup is resident at once, and an XCD's CUs receive its workgroups (one
// KV head, a sequence each) in dispatch order, so with the plan's rows longest first CU c would get
// rows c and c + 32 -- the longest contexts together. Taking alternate passes of 32 rows in
// reverse pairs each long context with a short one (the 64-sequence decode step's attention 18.6
// -> 18.2 us). The plain entry point's eight-wavefront workgroups measured slower this way (64
// sequences at contexts U[128, 2048]: 53.8 against 49.6 us) and keep the plan's order.
constexpr int kDecodeSerpentineRows = 64;

template <int G, bool QKV = false, bool ROWS = false>
static void launch_decode(DecodeArgs a, int num_seqs, hipStream_t s, bool narrow = false) {
  a.serpentine = QKV && a.kv_heads == 8 && a.splits == 1 && num_seqs <= kDecodeSerpentineRows;
  // Split-major grid: every sequence's first split, then the second splits, ... The splits past a
  // sequence's context exit at once, and workgroups are handed to an XCD's CUs in dispatch order,
  // so a grid with the split inside the sequence would repeat "real, real, empty, empty" with a
  // period that leaves some CUs all the keys (8B-shaped batch of 256 at contexts U[512, 4096]:
  // 754 us with four 2048-key splits per sequence, 476 with two, 415 split-major with any count).
  const dim3 grid(a.kv_heads, num_seqs, a.splits);
  if constexpr (!QKV && G <= 2) {  // (no eight-wavefront instantiation where it is never launched)
    if (!narrow && a.part_tokens >= kDecodeWideTokens) {
      hipLaunchKernelGGL((paged_decode_kernel<G, 2 * kDecodeW, QKV>), grid, dim3(128 * kDecodeW), 0, s, a);
      return;
    }
  }
  hipLaunchKernelGGL((paged_decode_kernel<G, kDecodeW, QKV, ROWS>), grid, dim3(64 * kDecodeW), 0, s, a);
}

// Shared checks and workspace binding of the two decode entry points.
static int decode_args(const char* who, const uint16_t* q, int64_t ldq, const uint16_t* k_cache, const uint16_t* v_cache,
                       int64_t num_slots, int heads, int kv_heads, int head_dim, int block_size,
                       const int32_t* block_tables, int max_blocks, const int32_t* context_lens, const int32_t* q_rows,
                       int num_seqs, int partition_tokens, int max_partitions, float scale, uint16_t* out, int64_t ldo,
                       void* workspace, size_t workspace_bytes, DecodeArgs& a) {
  const std::string w(who);
  if (!q || !k_cache || !v_cache || !block_tables || !context_lens || !q_rows || !out)
    return fail(MSA_ERR_INVALID, w + ": null pointer");
  if (head_dim != kHeadDim) return fail(MSA_ERR_UNSUPPORTED, w + ": head_dim must be 128");
  if (block_size != kBlock) return fail(MSA_ERR_UNSUPPORTED, w + ": block_size must be 16");
  if (num_seqs < 0 || num_seqs > 65535 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || max_blocks <= 0)
    return fail(MSA_ERR_INVALID, w + ": bad shape (num_seqs <= 65535)");
  if (partition_tokens <= 0 || partition_tokens % kBlock != 0 || max_partitions <= 0 || max_partitions > 65535)
    return fail(MSA_ERR_INVALID, w + ": partition_tokens must be a positive multiple of 16");
  if (partition_tokens > kDecodeMaxPartTokens)
    return fail(MSA_ERR_INVALID, w + ": partition_tokens must be at most 4096");
  if ((int64_t)partition_tokens * max_partitions < (int64_t)max_blocks * kBlock)
    return fail(MSA_ERR_INVALID, w + ": partition_tokens * max_partitions must cover max_blocks * 16");
  if (ldq % 8 != 0 || !aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return fail(MSA_ERR_INVALID, w + ": q/out/caches must be 16-byte aligned");
  a = DecodeArgs{};
  a.q = q; a.ldq = ldq; a.kc = k_cache; a.vc = v_cache; a.num_blocks = num_slots / kBlock;
  a.heads = heads; a.kv_heads = kv_heads; a.bt = block_tables; a.max_blocks = max_blocks;
  a.ctx = context_lens; a.qrows = q_rows; a.part_tokens = partition_tokens; a.splits = max_partitions;
  a.scale_log2 = scale * kLog2e; a.out = out; a.ldo = ldo;
  if (max_partitions > 1) {
    const size_t need = msa_paged_attention_decode_workspace_size(num_seqs, heads, head_dim, max_partitions);
    if (!workspace || workspace_bytes < need) return fail(MSA_ERR_WORKSPACE, w + ": workspace smaller than the workspace size");
    if (!aligned16(workspace)) return fail(MSA_ERR_INVALID, w + ": workspace must be 16-byte aligned");
    const size_t slots = (size_t)num_seqs * heads * max_partitions;
    a.ws_o = (float*)workspace;
    a.ws_ml = a.ws_o + slots * head_dim;
  }
  return MSA_OK;
}
}  // namespace msa

namespace msa {
// The decode entry points' shared body: checks, launch of the decode kernel and, with splits, of
// the split merge.
static int decode_entry(const char* who, const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                        const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads, int head_dim,
                        int block_size, const int32_t* block_tables, int max_blocks, const int32_t* context_lens,
                        const int32_t* q_rows, int num_seqs, int partition_tokens, int max_partitions, float scale,
                        uint16_t* out, int64_t ldo, void* workspace, size_t workspace_bytes, hipStream_t s,
                        bool narrow = false) {
  DecodeArgs a;
  int rc = decode_args(who, q, ldq, k_cache, v_cache, num_slots, heads, kv_heads, head_dim, block_size, block_tables,
                       max_blocks, context_lens, q_rows, num_seqs, partition_tokens, max_partitions, scale, out, ldo,
                       workspace, workspace_bytes, a);
  if (rc != MSA_OK) return rc;
  switch (heads / kv_heads) {
    case 1: launch_decode<1>(a, num_seqs, s, narrow); break;
    case 2: launch_decode<2>(a, num_seqs, s, narrow); break;
    case 4: launch_decode<4>(a, num_seqs, s, narrow); break;
    case 8: launch_decode<8>(a, num_seqs, s, narrow); break;
    default: return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": heads / kv_heads must be 1, 2, 4 or 8");
  }
  rc = check_launch(who);
  if (rc != MSA_OK || max_partitions == 1) return rc;
  launch_reduce(a, num_seqs, s);
  return check_launch("paged attention decode (split merge)");
}

// Scratch of msa_paged_attention_decode_noalloc: the float32 split partials of one call. A
// file-scope device array, one copy per GPU, which holds it until the process ends. In host code
// its name is not a device address: each device's address comes from hipGetSymbolAddress, looked
// up with that device current on the first call there, and only that address reaches kernels.
constexpr size_t kDecodeScratchBytes = MSA_DECODE_NOALLOC_MAX_BYTES;
static __device__ __align__(256) unsigned char scratch[kDecodeScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

// This device's scratch address (the stream's device; the current device for the null stream).
static int decode_scratch(hipStream_t s, void** ptr) {
  int dev = 0;
  hipError_t e = s ? hipStreamGetDevice(s, &dev) : hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MSA_ERR_LAUNCH, std::string("decode scratch: device of the stream: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(MSA_ERR_UNSUPPORTED, "decode scratch: device index past 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    int cur = 0;
    e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
    void* p = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) {
      const hipError_t back = hipSetDevice(cur);
      if (e == hipSuccess) e = back;
    }
    if (e != hipSuccess || p == nullptr)
      return fail(MSA_ERR_LAUNCH, std::string("decode scratch: hipGetSymbolAddress: ") +
                                      (e != hipSuccess ? hipGetErrorString(e) : "null address"));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return MSA_OK;
}
}  // namespace msa

extern "C" int msa_paged_attention_decode(const uint16_t* q, int64_t ldq, const uint16_t* k_cache, const uint16_t* v_cache,
                                          int64_t num_slots, int heads, int kv_heads, int head_dim, int block_size,
                                          const int32_t* block_tables, int max_blocks, const int32_t* context_lens,
                                          const int32_t* q_rows, int num_seqs, int partition_tokens, int max_partitions,
                                          float scale, uint16_t* out, int64_t ldo, void* workspace,
                                          size_t workspace_bytes, msa_stream_t stream) {
  using namespace msa;
  if (num_seqs == 0) return MSA_OK;
  return decode_entry("msa_paged_attention_decode", q, ldq, k_cache, v_cache, num_slots, heads, kv_heads, head_dim,
                      block_size, block_tables, max_blocks, context_lens, q_rows, num_seqs, partition_tokens,
                      max_partitions, scale, out, ldo, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int msa_paged_attention_decode_narrow(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                                 const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                                 int head_dim, int block_size, const int32_t* block_tables,
                                                 int max_blocks, const int32_t* context_lens, const int32_t* q_rows,
                                                 int num_seqs, int partition_tokens, int max_partitions, float scale,
                                                 uint16_t* out, int64_t ldo, void* workspace, size_t workspace_bytes,
                                                 msa_stream_t stream) {
  using namespace msa;
  if (num_seqs == 0) return MSA_OK;
  return decode_entry("msa_paged_attention_decode_narrow", q, ldq, k_cache, v_cache, num_slots, heads, kv_heads,
                      head_dim, block_size, block_tables, max_blocks, context_lens, q_rows, num_seqs, partition_tokens,
                      max_partitions, scale, out, ldo, workspace, workspace_bytes, (hipStream_t)stream, true);
}

extern "C" int msa_paged_attention_decode_noalloc(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                                  const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                                  int head_dim, int block_size, const int32_t* block_tables,
                                                  int max_blocks, const int32_t* context_lens, const int32_t* q_rows,
                                                  int num_seqs, int partition_tokens, int max_partitions, float scale,
                                                  uint16_t* out, int64_t ldo, msa_stream_t stream) {
  using namespace msa;
  if (num_seqs == 0) return MSA_OK;
  const size_t need = msa_paged_attention_decode_workspace_size(num_seqs, heads, head_dim, max_partitions);
  if (need > kDecodeScratchBytes)
    return fail(MSA_ERR_WORKSPACE, "msa_paged_attention_decode_noalloc: the split partials need " + std::to_string(need) +
                                       " bytes, more than the 16 MiB scratch (fewer sequences or partitions per call)");
  void* ws = nullptr;
  if (need > 0) {
    const int rc = decode_scratch((hipStream_t)stream, &ws);
    if (rc != MSA_OK) return rc;
  }
  return decode_entry("msa_paged_attention_decode_noalloc", q, ldq, k_cache, v_cache, num_slots, heads, kv_heads,
                      head_dim, block_size, block_tables, max_blocks, context_lens, q_rows, num_seqs, partition_tokens,
                      max_partitions, scale, out, ldo, ws, need > 0 ? kDecodeScratchBytes : 0, (hipStream_t)stream);
}

namespace msa {
template <bool ROWS>
static int decode_qkv_entry(const char* who, const uint16_t* qkv, int64_t ldqkv, const uint16_t* q_norm_w,
                            const uint16_t* k_norm_w, float qk_eps, const float* cos_table, const float* sin_table,
                            int64_t max_positions, const int64_t* slot_mapping, uint16_t* k_cache, uint16_t* v_cache,
                            int64_t num_slots, int heads, int kv_heads, int head_dim, int block_size,
                            const int32_t* block_tables, int max_blocks, const int32_t* context_lens,
                            const int32_t* q_rows, int num_seqs, int partition_tokens, int max_partitions, float scale,
                            uint16_t* out, int64_t ldo, void* workspace, size_t workspace_bytes, hipStream_t s) {
  if (num_seqs == 0) return MSA_OK;
  DecodeArgs a;
  int rc = decode_args(who, qkv, ldqkv, k_cache, v_cache, num_slots, heads, kv_heads, head_dim, block_size, block_tables,
                       max_blocks, context_lens, q_rows, num_seqs, partition_tokens, max_partitions, scale, out, ldo,
                       workspace, workspace_bytes, a);
  if (rc != MSA_OK) return rc;
  if (!q_norm_w || !k_norm_w || !cos_table || !sin_table || !slot_mapping || max_positions <= 0)
    return fail(MSA_ERR_INVALID, std::string(who) + ": null norm weight / rotary table / slot_mapping");
  if (!aligned16(q_norm_w) || !aligned16(k_norm_w) || !aligned16(cos_table) || !aligned16(sin_table))
    return fail(MSA_ERR_INVALID, std::string(who) + ": norm weights / rotary tables must be 16-byte aligned");
  if (ldqkv < (int64_t)(heads + 2 * kv_heads) * kHeadDim)
    return fail(MSA_ERR_INVALID, std::string(who) + ": ldqkv smaller than (heads + 2 kv_heads) * 128");
  a.qn_w = q_norm_w; a.kn_w = k_norm_w; a.qk_eps = qk_eps; a.cos_t = cos_table; a.sin_t = sin_table;
  a.max_pos = max_positions;
  a.slots = slot_mapping;
  switch (heads / kv_heads) {
    case 1: launch_decode<1, true, ROWS>(a, num_seqs, s); break;
    case 2: launch_decode<2, true, ROWS>(a, num_seqs, s); break;
    case 4: launch_decode<4, true, ROWS>(a, num_seqs, s); break;
    case 8: launch_decode<8, true, ROWS>(a, num_seqs, s); break;
    default: return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": heads / kv_heads must be 1, 2, 4 or 8");
  }
  rc = check_launch(who);
  if (rc != MSA_OK || max_partitions == 1) return rc;
  launch_reduce(a, num_seqs, s);
  return check_launch("msa_paged_attention_decode_qkv (split merge)");
}
}  // namespace msa

extern "C" int msa_paged_attention_decode_qkv(const uint16_t* qkv, int64_t ldqkv, const uint16_t* q_norm_w,
                                              const uint16_t* k_norm_w, float qk_eps, const float* cos_table,
                                              const float* sin_table, int64_t max_positions, const int64_t* slot_mapping,
                                              uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots, int heads,
                                              int kv_heads, int head_dim, int block_size, const int32_t* block_tables,
                                              int max_blocks, const int32_t* context_lens, const int32_t* q_rows,
                                              int num_seqs, int partition_tokens, int max_partitions, float scale,
                                              uint16_t* out, int64_t ldo, void* workspace, size_t workspace_bytes,
                                              msa_stream_t stream) {
  return msa::decode_qkv_entry<false>("msa_paged_attention_decode_qkv", qkv, ldqkv, q_norm_w, k_norm_w, qk_eps, cos_table,
                               sin_table, max_positions, slot_mapping, k_cache, v_cache, num_slots, heads, kv_heads, head_dim,
                               block_size, block_tables, max_blocks, context_lens, q_rows, num_seqs, partition_tokens,
                               max_partitions, scale, out, ldo, workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int msa_paged_attention_decode_qkv_rows(const uint16_t* qkv, int64_t ldqkv, const uint16_t* q_norm_w,
                                                   const uint16_t* k_norm_w, float qk_eps, const float* cos_rows,
                                                   const float* sin_rows, int64_t rows, const int64_t* slot_mapping,
                                                   uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots, int heads,
                                                   int kv_heads, int head_dim, int block_size, const int32_t* block_tables,
                                                   int max_blocks, const int32_t* context_lens, const int32_t* q_rows,
                                                   int num_seqs, int partition_tokens, int max_partitions, float scale,
                                                   uint16_t* out, int64_t ldo, void* workspace, size_t workspace_bytes,
                                                   msa_stream_t stream) {
  return msa::decode_qkv_entry<true>("msa_paged_attention_decode_qkv_rows", qkv, ldqkv, q_norm_w, k_norm_w, qk_eps, cos_rows,
                               sin_rows, rows, slot_mapping, k_cache, v_cache, num_slots, heads, kv_heads, head_dim,
                               block_size, block_tables, max_blocks, context_lens, q_rows, num_seqs, partition_tokens,
                               max_partitions, scale, out, ldo, workspace, workspace_bytes, (hipStream_t)stream);
}

namespace msa {
static int prefill_entry(const char* who, bool wide, const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                         const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads, int head_dim,
                         int block_size, const int32_t* block_tables, int max_blocks, const int32_t* seq_info,
                         const int32_t* work, int num_work, float scale, uint16_t* out, int64_t ldo, hipStream_t s) {
  if (num_work == 0) return MSA_OK;
  if (!q || !k_cache || !v_cache || !block_tables || !seq_info || !work || !out)
    return fail(MSA_ERR_INVALID, std::string(who) + ": null pointer");
  if (head_dim != kHeadDim) return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": head_dim must be 128");
  if (block_size != kBlock) return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": block_size must be 16");
  if (num_work < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || max_blocks <= 0)
    return fail(MSA_ERR_INVALID, std::string(who) + ": bad shape");
  if (ldq % 8 != 0 || ldo % 4 != 0 || !aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return fail(MSA_ERR_INVALID, std::string(who) + ": q/out/caches must be 16-byte aligned");
  PrefillArgs a{};
  a.q = q; a.ldq = ldq; a.kc = k_cache; a.vc = v_cache; a.num_blocks = num_slots / kBlock;
  a.heads = heads; a.kv_heads = kv_heads; a.bt = block_tables; a.max_blocks = max_blocks;
  a.seq_info = seq_info; a.work = work; a.scale_log2 = scale * kLog2e; a.out = out; a.ldo = ldo;
  const dim3 grid(num_work, kv_heads);
  int rc;
  switch (heads / kv_heads) {
    case 1: rc = launch_prefill<1>(a, grid, wide, s); break;
    case 2: rc = launch_prefill<2>(a, grid, wide, s); break;
    case 4: rc = launch_prefill<4>(a, grid, wide, s); break;
    default: return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": heads / kv_heads must be 1, 2 or 4");
  }
  if (rc != MSA_OK) return rc;
  return check_launch(who);
}
}  // namespace msa

extern "C" int msa_paged_attention_prefill(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                           const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                           int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                                           const int32_t* seq_info, const int32_t* work, int num_work, float scale,
                                           uint16_t* out, int64_t ldo, msa_stream_t stream) {
  return msa::prefill_entry("msa_paged_attention_prefill", false, q, ldq, k_cache, v_cache, num_slots, heads, kv_heads,
                            head_dim, block_size, block_tables, max_blocks, seq_info, work, num_work, scale, out, ldo,
                            (hipStream_t)stream);
}

extern "C" int msa_paged_attention_prefill_wide(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                                const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                                int head_dim, int block_size, const int32_t* block_tables,
                                                int max_blocks, const int32_t* seq_info, const int32_t* work,
                                                int num_work, float scale, uint16_t* out, int64_t ldo,
                                                msa_stream_t stream) {
  return msa::prefill_entry("msa_paged_attention_prefill_wide", true, q, ldq, k_cache, v_cache, num_slots, heads,
                            kv_heads, head_dim, block_size, block_tables, max_blocks, seq_info, work, num_work, scale,
                            out, ldo, (hipStream_t)stream);
}
