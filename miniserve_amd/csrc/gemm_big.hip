// Int8 weight-only linear for large prefill GEMMs: 256-token tiles, eight or sixteen wavefronts per
// workgroup (two or four per SIMD).
//
// y[m, n] = sum_k x[m, k] * bf16(q[n, k] * s[n]) with float32 accumulation, as Int8Linear.forward
// (quant/int8.py:35-37) computes it -- the same operands and rounding points as the 128 x 128 GEMM
// (gemm_int8.hip); only the tiling differs.
//
// Why a second tiling: a wavefront tile of TM x TN reads (TM + TN) x K operand bytes from LDS for
// TM x TN x K MACs, and a 256-token tile dequantizes each weight once per 256 tokens instead of per
// 128.
//
//  * Workgroup = WM x WN wavefronts over 256 tokens x BN weight rows: 256 x 256 (2 x 4 wavefronts of
//    128 x 64), 256 x 192 (8 x 2 of 32 x 96) or 256 x 128 (4 x 4 of 64 x 32); the host picks the one
//    that fills the most of the 256 CUs. Per 64-wide K step the workgroup stages the x tile (256 x 64
//    bf16, 32 KB) and the dequantized q tile (BN x 64 -> bf16) in LDS, double buffered. A piece's
//    registers are reloaded for the step after next right after they are stored, so every load has a
//    whole step to arrive (8B-shaped gate_up at 4096 tokens 719 us with the loads at the step's end,
//    704 with this).
//    (256 x 128 in one round of workgroups or with the residual epilogue: 4 x 2 of 64 x 64.)
//  * What bounds it: no unit alone. Per step of a 256 x 128 tile (about 1 us) the MFMAs take 0.47 us
//    of each SIMD, LDS reads 0.34 (1.75 ns per 1 KB read instruction) and writes 0.28 (5.8 ns each),
//    dequantization 0.17; wavefronts that leave a barrier together do the same thing at the same time.
//    Sixteen wavefronts with each slice's fragments read before the previous slice's MFMAs issue
//    overlap them best on the narrow tiles (gate_up at 256 tokens 69.6 us with eight, 69.9 with
//    sixteen that read their own slice's fragments, 65.2 with sixteen that read ahead; qkv at 4096
//    212, 212, 200). On 256 x 256 tiles (128 accumulators a lane) eight wavefronts that read a slice's
//    fragments just before its MFMAs are faster (4096 tokens: 704 us; sixteen 766; reading ahead
//    747; the two wavefronts of a SIMD in alternate memory and MFMA phases 800-821; MFMAs at a raised
//    wavefront priority 784).
//  * Epilogues: bf16 store; residual add (in place allowed); silu(gate) * up with each
//    wavefront's TN weight rows laid out as TN / 2 gate rows then their TN / 2 up rows. Results go
//    through LDS so that each lane writes 16 contiguous bytes (gate and up meet there).
//  * Split-K (256 x 128 tiles, gemm256_split_plan): workgroup (tile, ks) runs K steps
//    [ks k_per, (ks + 1) k_per) and stores its float32 accumulators as partials [ks][m][n]; the
//    caller's merge kernel sums them in split order, as for the 128 x 128 split-K GEMM.
#include <hip/hip_runtime.h>

#include "common.h"

namespace msa {

constexpr int kBM = 256, kBK = 64;
constexpr int kBLd = kBK + 8;  // bf16 elements per LDS row (16 bytes of padding)
template <int BN>
constexpr size_t big_lds_bytes() {
  return 2 * (size_t)(kBM + BN) * kBLd * 2;
}

struct BigGemmArgs {
  const uint16_t* x;
  int64_t ldx;
  const int8_t* w;
  const uint16_t* scale;
  uint16_t* y;
  int64_t ldy;
  const uint16_t* resid;
  int64_t ldr;
  int m, n, k;
  int n_blocks;  // weight-row blocks (BN rows, or BN / 2 gate + BN / 2 up for SILU_MUL)
  int m_blocks;  // token blocks of 256
  int k_per;     // K per split (a multiple of 64; == k without split-K)
  int splits;    // K splits (kBigEpiPartial; 1 otherwise)
  float* part;   // kBigEpiPartial: float32 partials [splits][m][n]
  QkNormOut qk;  // kEpiQkNorm (BN = 128): weight block nb is head slot nb
};

constexpr int kBigEpiPartial = 3;  // split-K: the float32 accumulators of K split ks, no rounding

// Weight row held in LDS row r (0..BN-1) of row block nb. SILU_MUL: wavefront column w holds the
// rows [w TN, (w + 1) TN), its first TN / 2 gate rows and then the matching TN / 2 up rows.
template <int BN, int TN, int EPI>
__device__ __forceinline__ int big_wrow(const BigGemmArgs& a, int nb, int r) {
  if constexpr (EPI == MSA_EPI_SILU_MUL) {
    const int w = r / TN, i = r % TN;
    const int col = nb * (BN / 2) + w * (TN / 2) + (i < TN / 2 ? i : i - TN / 2);
    return (i < TN / 2 ? 0 : a.n / 2) + col;
  } else {
    return nb * BN + r;
  }
}

template <int BN, int WM, int WN, int EPI>
__global__ __launch_bounds__(64 * WM * WN) void int8_gemm256_kernel(BigGemmArgs a) {
  constexpr int NTH = 64 * WM * WN;     // threads
  constexpr int AR = kBM * 8 / NTH;     // 16-byte x pieces per thread per K step
  constexpr int TM = kBM / WM, TN = BN / WN;  // wavefront tile
  constexpr int MT = TM / 32, NT = TN / 32;   // 32 x 32 accumulator tiles
  static_assert((NTH == 512 || NTH == 1024) && TM % 32 == 0 && TN % 32 == 0, "wavefronts of 32 x 32 tiles");
  static_assert(EPI != MSA_EPI_SILU_MUL || (TN / 2) % 8 == 0, "gate and up halves in 16-byte pieces");
  constexpr int BCH = (BN * 4 + NTH - 1) / NTH;  // 16-byte weight chunks per thread per K step
  static_assert(AR <= 4 && BCH <= 2, "two parts of x pieces, two of weight chunks");
  extern __shared__ __attribute__((aligned(16))) uint16_t bsm[];
  uint16_t* As = bsm;                   // [2][256][kBLd]
  uint16_t* Bs = bsm + 2 * kBM * kBLd;  // [2][BN][kBLd]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  // XCD-aware order: the token blocks of one weight block (and K split) run on one XCD
  // (round-robin dispatch), so its weight tiles come from HBM once and from that XCD's L2 after.
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int mb = slot % a.m_blocks, rest = slot / a.m_blocks;
  const int ks = rest % a.splits, nb = (rest / a.splits) * 8 + xcd;
  if (nb >= a.n_blocks) return;  // surplus workgroups of the XCD-rounded grid (whole workgroup)
  const int m0 = mb * kBM;
  const uint32_t kbase = (uint32_t)ks * (uint32_t)a.k_per;  // this split's first K element

  // Loader roles. A: rows tid / 8 + NTH / 8 i (i < AR), 8-element chunk tid % 8. B: chunk
  // c = tid + NTH i (c < 4 BN): row c / 4, 16-byte piece c % 4.
  const int ar = tid >> 3, ac = (tid & 7) * 8;
  // 32-bit byte offsets from the uniform base pointers (the caller checks that they fit): half the
  // registers of per-row 64-bit pointers.
  uint32_t aoff[AR];
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int row = min(m0 + ar + NTH / 8 * i, a.m - 1);  // rows past m repeat row m - 1; outputs dropped
    aoff[i] = (uint32_t)(row * (uint32_t)a.ldx + ac + kbase) * 2u;
  }
  uint32_t boff[BCH];
  float bs[BCH];
#pragma unroll
  for (int i = 0; i < BCH; ++i) {
    const int c = min(tid + NTH * i, BN * 4 - 1);  // chunks past the tile reload the last one (not stored)
    int row = big_wrow<BN, TN, EPI>(a, nb, c / 4);
    row = row < a.n ? row : a.n - 1;
    boff[i] = (uint32_t)row * (uint32_t)a.k + kbase + (c % 4) * 16;
    bs[i] = bf16_to_f32(a.scale[row]);
  }
  // A step's global loads in registers, in four parts: p = 0, 1 the halves of the x pieces, p = 2, 3
  // the weight chunks p - 2 (of BCH).
  u32x4 ra[AR], rb[BCH];  // native vectors: a struct-typed array stays in private memory
  auto load_part = [&](int k0, int p) {
    if (p < 2) {
#pragma unroll
      for (int i = AR / 2 * p; i < AR / 2 * (p + 1); ++i) ra[i] = *(const u32x4*)((const char*)a.x + aoff[i] + 2u * k0);
    } else if (p - 2 < BCH) {
      rb[p - 2] = *(const u32x4*)((const char*)a.w + boff[p - 2] + k0);
    }
  };
  // Part p into LDS buffer buf, the weights dequantized.
  auto store_part = [&](int buf, int p) {
    if (p < 2) {
      uint16_t* A_ = As + buf * kBM * kBLd + ar * kBLd + ac;
#pragma unroll
      for (int i = AR / 2 * p; i < AR / 2 * (p + 1); ++i) *(u32x4*)(A_ + NTH / 8 * i * kBLd) = ra[i];
    } else if (p - 2 < BCH) {
      const int i = p - 2;
      const int c = tid + NTH * i;
      if (BN * 4 % NTH == 0 || c < BN * 4) {  // (a whole wavefront takes one side)
        uint16_t* B_ = Bs + buf * BN * kBLd + (c / 4) * kBLd + (c % 4) * 16;
        // An empty asm redefines rb[i] here, so the compiler cannot start dequantizing the next
        // step's bytes before the barrier that ends the current one (a wait on loads just issued).
        asm volatile("" : "+v"(rb[i]));
        *(bf16x8*)(B_) = dequant8(rb[i].x, rb[i].y, bs[i]);
        *(bf16x8*)(B_ + 8) = dequant8(rb[i].z, rb[i].w, bs[i]);
      }
    }
  };

  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x16{};
  // MFMA operand fragments: lane (h, r) holds row r of a 32-row tile, K elements 8h..8h+7 of the
  // 16-wide slice.
  const int r32 = lane & 31, h = lane >> 5;
  const uint16_t* Afr = As + (wm * TM + r32) * kBLd + h * 8;
  const uint16_t* Bfr = Bs + (wn * TN + r32) * kBLd + h * 8;
  auto read_frags = [&](int buf, int ks, bf16x8(&af)[MT], bf16x8(&bfr)[NT]) {
    const uint16_t* A = Afr + buf * kBM * kBLd + ks * 16;
    const uint16_t* B = Bfr + buf * BN * kBLd + ks * 16;
#pragma unroll
    for (int t = 0; t < MT; ++t) af[t] = *(const bf16x8*)(A + t * 32 * kBLd);
#pragma unroll
    for (int t = 0; t < NT; ++t) bfr[t] = *(const bf16x8*)(B + t * 32 * kBLd);
  };
  auto mfmas = [&](const bf16x8(&af)[MT], const bf16x8(&bfr)[NT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[mt], bfr[nt], acc[mt][nt], 0, 0, 0);
  };

  const int nk = a.k_per / kBK;
  // Top of step kt: LDS buffer kt & 1 holds step kt and the registers step kt + 1. Loads and
  // stores are unconditional (the last steps reload step nk - 1 and stage it into the idle
  // buffer: in bounds, never used) so the prefetch registers stay registers.
#pragma unroll
  for (int p = 0; p < 4; ++p) load_part(0, p);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    store_part(0, p);
    load_part(min(1, nk - 1) * kBK, p);
  }
  __syncthreads();
  if constexpr (BN == 256) {
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        bf16x8 af[MT], bfr[NT];
        read_frags(cur, ks, af, bfr);
        mfmas(af, bfr);
        store_part(cur ^ 1, ks);  // step kt + 1 into the other buffer
        load_part(min(kt + 2, nk - 1) * kBK, ks);
        __builtin_amdgcn_sched_barrier(0);  // keeps each slice's fragments and staging with its MFMAs
      }
      __syncthreads();
    }
  } else {
    // Two fragment sets: each slice's LDS reads are issued before the previous slice's MFMAs.
    // Slices 0 and 1 stage step kt + 1 into the other buffer and reload the registers; the barrier
    // before slice 3 publishes the staged step (and ends every read of the buffer the next step
    // overwrites), and slice 3's MFMAs cover the read of the next step's first slice (at the last
    // step a read of the idle buffer, not used).
    bf16x8 af[2][MT], bfr[2][NT];
    read_frags(0, 0, af[0], bfr[0]);
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        if (ks + 1 < kBK / 16) {
          read_frags(cur, ks + 1, af[(ks + 1) & 1], bfr[(ks + 1) & 1]);
        } else {
          __syncthreads();
          read_frags(cur ^ 1, 0, af[0], bfr[0]);
        }
        mfmas(af[ks & 1], bfr[ks & 1]);
        if (NTH == 1024 && ks < 2) {
#pragma unroll
          for (int p = 2 * ks; p < 2 * ks + 2; ++p) {
            store_part(cur ^ 1, p);
            load_part(min(kt + 2, nk - 1) * kBK, p);
          }
        } else if (ks < 2) {
          // Eight wavefronts: a step's loads together, behind its last store (apart they measured 1%
          // slower over a short K: 0.6B qkv at 900 tokens 17.2 -> 17.4 us).
          store_part(cur ^ 1, ks);
          store_part(cur ^ 1, ks + 2);
          if (ks == 1) {
#pragma unroll
            for (int p = 0; p < 4; ++p) load_part(min(kt + 2, nk - 1) * kBK, p);
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // keeps each slice's reads and staging with its MFMAs
      }
    }
    __syncthreads();  // the last read of the idle buffer precedes the epilogue's reuse of LDS
  }

  if constexpr (EPI == kBigEpiPartial) {
    // value i of lane (h, r) in tile (mt, nt): token row mt*32 + 8(i/4) + 4h + i%4 of the
    // wavefront's TM, weight row nt*32 + r of its TN; 32 lanes write 128 contiguous bytes
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = m0 + wm * TM + mt * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
        if (tok >= a.m) continue;
        float* prow = a.part + ((int64_t)ks * a.m + tok) * a.n;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int col = nb * BN + wn * TN + nt * 32 + r32;
          if (col < a.n) prow[col] = acc[mt][nt][i];
        }
      }
    return;
  }

  if constexpr (EPI == kEpiQkNorm) {
    // The qkv projection: the whole 256-token x 128-dim head tile staged in LDS (free after the
    // loop's last barrier), then the per-head q/k RMSNorm + RoPE + KV-cache write, eight threads
    // per token row.
    static_assert(BN == 128, "a tile is one head slot");
    constexpr int kQLd = 128 + 8;
    static_assert((size_t)kBM * kQLd * 2 <= big_lds_bytes<BN>(), "the head tile fits the tile buffers");
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        uint16_t* c = bsm + (wm * TM + mt * 32 + 8 * (i >> 2) + 4 * h + (i & 3)) * kQLd + wn * TN + r32;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) c[nt * 32] = f32_to_bf16(acc[mt][nt][i]);
      }
    __syncthreads();
    qk_norm_rope_tile<NTH, kBM>(a.qk, bsm, kQLd, nb, m0, a.m, tid);
    return;
  }

  // Epilogue through LDS (free after the loop's last barrier): each wavefront stages its TM x TN
  // tile as bf16 in a region of its own (silu * up: the gate values in columns [0, TN / 2), the up
  // values in [TN / 2, TN)), then stores rows of outputs with 16-byte writes. Value i of lane (h, r)
  // in tile (mt, nt) is token row mt*32 + 8(i/4) + 4h + i%4 and weight row nt*32 + r of the
  // wavefront's TN.
  constexpr int kCLd = TN + 8;
  static_assert((size_t)WM * WN * TM * kCLd * 2 <= big_lds_bytes<BN>(), "epilogue staging fits the tile buffers");
  uint16_t* Cs = bsm + wave * TM * kCLd;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      uint16_t* c = Cs + (mt * 32 + 8 * (i >> 2) + 4 * h + (i & 3)) * kCLd + r32;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) c[nt * 32] = f32_to_bf16(acc[mt][nt][i]);
    }
  __syncthreads();

  constexpr int kOutCols = EPI == MSA_EPI_SILU_MUL ? TN / 2 : TN;
  const int tok0 = m0 + wm * TM;
  const int col0 = EPI == MSA_EPI_SILU_MUL ? nb * (BN / 2) + wn * (TN / 2) : nb * BN + wn * TN;
  const int out_n = EPI == MSA_EPI_SILU_MUL ? a.n / 2 : a.n;
  const bool vec = ((uintptr_t)a.y & 15) == 0 && (a.ldy & 7) == 0 &&
                   (EPI != MSA_EPI_RESIDUAL || (((uintptr_t)a.resid & 15) == 0 && (a.ldr & 7) == 0));
  constexpr int kChunksPerRow = kOutCols / 8;
#pragma unroll 4
  for (int c = lane; c < TM * kChunksPerRow; c += 64) {
    const int row = c / kChunksPerRow, cc = (c % kChunksPerRow) * 8;
    const int tok = tok0 + row, col = col0 + cc;
    if (tok >= a.m || col >= out_n) continue;
    u32x4 v = *(const u32x4*)(Cs + row * kCLd + cc);
    if constexpr (EPI == MSA_EPI_SILU_MUL) {
      // bf16(bf16(silu(bf16(gate))) * bf16(up)), the staged values being the rounded products
      const u32x4 u = *(const u32x4*)(Cs + row * kCLd + TN / 2 + cc);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = pack_bf16x2(round_bf16(silu_f32(bf16lo(v[e]))) * bf16lo(u[e]),
                           round_bf16(silu_f32(bf16hi(v[e]))) * bf16hi(u[e]));
    }
    uint16_t* dst = a.y + (int64_t)tok * a.ldy + col;
    if (vec && col + 8 <= out_n) {
      if constexpr (EPI == MSA_EPI_RESIDUAL) {
        const u32x4 rv = *(const u32x4*)(a.resid + (int64_t)tok * a.ldr + col);
        u32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack_bf16x2(bf16lo(v[e]) + bf16lo(rv[e]), bf16hi(v[e]) + bf16hi(rv[e]));
        *(u32x4*)dst = o;
      } else {
        *(u32x4*)dst = v;
      }
    } else {  // ragged last columns or unaligned output: element by element
      for (int e = 0; e < 8 && col + e < out_n; ++e) {
        float o = e & 1 ? bf16hi(v[e >> 1]) : bf16lo(v[e >> 1]);
        if constexpr (EPI == MSA_EPI_RESIDUAL) o += bf16_to_f32(a.resid[(int64_t)tok * a.ldr + col + e]);
        dst[e] = f32_to_bf16(o);
      }
    }
  }
}

// ---- host side ----------------------------------------------------------------------------------

// Weight rows per tile, in order of preference when two fill the chip equally (larger tiles first).
constexpr int kBigTilings[] = {256, 192, 128};
constexpr int kBigTilingCount = 3;

static int64_t big_n_blocks(int t, int64_t n, int epilogue) {
  const int bn = kBigTilings[t];
  return epilogue == MSA_EPI_SILU_MUL ? (n / 2 + bn / 2 - 1) / (bn / 2) : (n + bn - 1) / bn;
}

// The tiling that keeps the largest share of the 256 CUs' workgroup slots busy over its rounds
// (one workgroup per CU), and its tile count; -1 when none applies (K not a multiple of 64, odd n
// for silu * up).
int gemm256_pick(int64_t m, int64_t n, int64_t k, int epilogue, int64_t* tiles) {
  *tiles = 0;
  if (k % kBK != 0 || (epilogue == MSA_EPI_SILU_MUL && n % 2 != 0)) return -1;
  constexpr int64_t kCUs = 256;
  int best = -1;
  int64_t best_tiles = 0, best_slots = 1;
  for (int t = 0; t < kBigTilingCount; ++t) {
    const int64_t tl = big_n_blocks(t, n, epilogue) * ((m + kBM - 1) / kBM);
    const int64_t slots = (tl + kCUs - 1) / kCUs * kCUs;
    if (best < 0 || tl * best_slots > best_tiles * slots) {  // tl / slots > best_tiles / best_slots
      best = t;
      best_tiles = tl;
      best_slots = slots;
    }
  }
  *tiles = best_tiles;
  return best;
}

template <int BN, int WM, int WN, int EPI>
static int launch_big(const BigGemmArgs& a, int blocks, hipStream_t s) {
  constexpr size_t lds = big_lds_bytes<BN>();
  auto kernel = int8_gemm256_kernel<BN, WM, WN, EPI>;
  const int rc = allow_dynamic_lds((const void*)kernel, (int)lds, "int8_gemm256_kernel");
  if (rc != MSA_OK) return rc;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * WM * WN), lds, s, a);
  return check_launch("msa_int8_gemm (256-token tiles)");
}

template <int BN, int WM, int WN>
static int launch_big_epi(const BigGemmArgs& a, int blocks, int epilogue, hipStream_t s) {
  switch (epilogue) {
    case MSA_EPI_NONE: return launch_big<BN, WM, WN, MSA_EPI_NONE>(a, blocks, s);
    case MSA_EPI_SILU_MUL: return launch_big<BN, WM, WN, MSA_EPI_SILU_MUL>(a, blocks, s);
    default:
      if constexpr (BN == 128) return fail(MSA_ERR_INVALID, "msa_int8_gemm: residual tiling");
      else return launch_big<BN, WM, WN, MSA_EPI_RESIDUAL>(a, blocks, s);
  }
}

// The GEMM on tiling t of gemm256_pick; arguments checked by the caller.
int gemm256_run(int t, const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                const uint16_t* scale, int64_t n, uint16_t* y, int64_t ldy, int epilogue, const uint16_t* residual,
                int64_t ldr, hipStream_t s) {
  if (t < 0 || t >= kBigTilingCount) return fail(MSA_ERR_INVALID, "msa_int8_gemm: no such tiling");
  BigGemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale; a.y = y; a.ldy = ldy; a.resid = residual; a.ldr = ldr;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  a.n_blocks = (int)big_n_blocks(t, n, epilogue);
  a.m_blocks = (int)((m + kBM - 1) / kBM);
  a.k_per = (int)k;
  a.splits = 1;
  const int64_t blocks = (int64_t)((a.n_blocks + 7) / 8) * 8 * a.m_blocks;
  if (blocks > 0x7fffffff) return fail(MSA_ERR_INVALID, "msa_int8_gemm: too many tiles");
  switch (t) {
    case 0: return launch_big_epi<256, 2, 4>(a, (int)blocks, epilogue, s);
    case 1: return launch_big_epi<192, 8, 2>(a, (int)blocks, epilogue, s);
    default:
      // One round of workgroups, and the residual epilogue: eight wavefronts (8B o at 1300 tokens 57.9 us,
      // sixteen 60.1; at 2048 with the residual 71.8, 74.3). More rounds: sixteen (8B qkv at 1300 / 2048
      // tokens 80 / 97, eight 90 / 104).
      // silu * up: eight, but for a longer K on at most three quarters of the CUs (16384 x 5120 at 256 /
      // 512 / 1300 / 4096 tokens, the first 128 tiles: eight 80 / 91 / 257 / 587, sixteen 70 / 95 / 268 / 581;
      // 24576 x 4096 at 256, 192 tiles: 68, 66; 6144 x 1024 at 1000, 192 tiles: 19.5, 20.3).
      if (epilogue == MSA_EPI_RESIDUAL) return launch_big<128, 4, 2, MSA_EPI_RESIDUAL>(a, (int)blocks, s);
      if (epilogue == MSA_EPI_NONE && (int64_t)a.n_blocks * a.m_blocks <= 256)
        return launch_big<128, 4, 2, MSA_EPI_NONE>(a, (int)blocks, s);
      if (epilogue == MSA_EPI_SILU_MUL && (a.k <= 2048 || (int64_t)a.n_blocks * a.m_blocks > 192))
        return launch_big<128, 4, 2, MSA_EPI_SILU_MUL>(a, (int)blocks, s);
      return launch_big_epi<128, 4, 4>(a, (int)blocks, epilogue, s);
  }
}

// The qkv projection with the q/k-norm epilogue on 256 x 128 tiles (one head slot each); arguments
// checked by the caller.
int gemm256_qk_norm_run(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                        const uint16_t* scale, const QkNormOut& qk, hipStream_t s) {
  BigGemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale;
  a.m = (int)m; a.n = (qk.heads + 2 * qk.kv_heads) * 128; a.k = (int)k;
  a.n_blocks = qk.heads + 2 * qk.kv_heads;
  a.m_blocks = (int)((m + kBM - 1) / kBM);
  a.k_per = (int)k;
  a.splits = 1;
  a.qk = qk;
  const int64_t blocks = (int64_t)((a.n_blocks + 7) / 8) * 8 * a.m_blocks;
  if (blocks > 0x7fffffff) return fail(MSA_ERR_INVALID, "msa_int8_gemm_qk_norm_rope_cache: too many tiles");
  return launch_big<128, 4, 4, kEpiQkNorm>(a, (int)blocks, s);
}

// Split-K on 256 x 128 tiles for shapes with too few output tiles to fill the chip unsplit and a
// long K (the 8B-shaped qkv and down at 256 tokens, the 0.6B down at 2048): the fewest splits
// whose workgroups fill 192-320 of the 256 CUs in one round, each split 16+ whole 64-wide K steps;
// 0 when none does or the tiling does not apply (under 192 tokens, K not a multiple of 64). With
// shorter splits the float32 partials (and the merge that reads them) cost more than the tiling
// gains: the 8B-shaped o at 256 tokens in eight 512-wide splits 26.6 us against 25.9 on 128 x 128
// tiles in four; qkv in four 1024-wide splits 29.9 against 33.7, down 44.2 against 50.2.
int gemm256_split_plan(int64_t m, int64_t n, int64_t k) {
  if (m < 192 || k % kBK != 0) return 0;
  const int64_t tiles = ((n + 127) / 128) * ((m + kBM - 1) / kBM);
  const int64_t steps = k / kBK;
  for (int sp = 2; sp <= 16; ++sp) {
    if (steps % sp != 0 || steps / sp < 16) continue;
    if (tiles * sp >= 192 && tiles * sp <= 320) return sp;
  }
  return 0;
}

// float32 partials [splits][m][n] of x @ bf16(q * s)^T on 256 x 128 tiles, splits from
// gemm256_split_plan; arguments (and the 32-bit offsets) checked by the caller.
int gemm256_partials_run(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                         const uint16_t* scale, int64_t n, int splits, float* part, hipStream_t s) {
  BigGemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  a.n_blocks = (int)((n + 127) / 128);
  a.m_blocks = (int)((m + kBM - 1) / kBM);
  a.k_per = (int)(k / splits);
  a.splits = splits;
  a.part = part;
  const int64_t blocks = (int64_t)((a.n_blocks + 7) / 8) * 8 * splits * a.m_blocks;
  if (blocks > 0x7fffffff) return fail(MSA_ERR_INVALID, "msa_int8_gemm: too many tiles");
  return launch_big<128, 4, 4, kBigEpiPartial>(a, (int)blocks, s);
}

}  // namespace msa
