// Int8 weight-only linear for prefill-sized batches (M >= 128 tokens): an LDS-tiled MFMA GEMM.
//
// y[m, n] = sum_k x[m, k] * bf16(q[n, k] * s[n]) with float32 accumulation, as Int8Linear.forward
// (quant/int8.py:35-37) computes it, but the int8 weights are dequantized once per 128 x 64 tile
// into LDS instead of materializing the whole bf16 matrix.
//
//  * Workgroup = 4 wavefronts (2 x 2) owning a 128-token x 128-weight-row output tile; a wavefront
//    owns 64 x 64 = 2 x 2 tiles of v_mfma_f32_32x32x16_bf16 (tokens as the A rows, weight rows as
//    the B columns), each 16-wide K slice's fragments read from LDS before the previous slice's
//    MFMAs issue.
//  * Per 64-wide K step: the workgroup loads the x tile (128 x 64 bf16, 16 KB) and the q tile
//    (128 x 64 int8, 8 KB) into registers, dequantizes q to bf16(q * s) on the way into LDS, and
//    computes the step from the other LDS buffer (double buffered: the next step's global loads
//    are in flight during the MFMAs).
//  * Epilogues: bf16 store; residual add (in place allowed); silu(gate) * up, with the tile's
//    weight rows laid out so that every gate column and its up column land in the same lane.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"

namespace msa {

constexpr int kGBM = 128, kGBN = 128, kGBK = 64;
constexpr int kGLd = kGBK + 8;  // bf16 elements per LDS row (16 bytes of padding)
constexpr size_t kGemmLds = 2 * (size_t)(kGBM + kGBN) * kGLd * 2;

struct GemmArgs {
  const uint16_t* x;
  int64_t ldx;
  const int8_t* w;
  const uint16_t* scale;
  uint16_t* y;
  int64_t ldy;
  const uint16_t* resid;
  int64_t ldr;
  int m, n, k;
  int n_blocks;  // weight-row blocks (of 128 rows, or 64 gate + 64 up for SILU_MUL)
  int m_blocks;  // token blocks of 128
  int k_per;     // K per split (a multiple of 64; == k without split-K)
  float* part;   // split-K: float32 partials [splits][m][n]
  // kEpiQkNorm: the qkv projection's epilogue -- per-head RMSNorm + RoPE of q and k, q rows out,
  // k and v into the paged caches (weight block nb is head slot nb)
  QkNormOut qk;
};

constexpr int kEpiPartial = 3;  // split-K: store the float32 accumulators, no rounding

// Weight row held in LDS row r (0..127) of row block nb.
template <int EPI>
__device__ __forceinline__ int gemm_wrow(const GemmArgs& a, int nb, int r) {
  if constexpr (EPI == MSA_EPI_SILU_MUL) {
    // quarters of 32 rows: gate, up, gate, up -- wavefront column wn owns quarters 2wn, 2wn+1
    const int q = r >> 5, i = r & 31;
    return ((q & 1) ? a.n / 2 : 0) + nb * 64 + (q >> 1) * 32 + i;
  } else {
    return nb * kGBN + r;
  }
}

template <int EPI>
__global__ __launch_bounds__(256) void int8_gemm_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t gsm[];
  uint16_t* As = gsm;                    // [2][128][kGLd]
  uint16_t* Bs = gsm + 2 * kGBM * kGLd;  // [2][128][kGLd]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int nb = blockIdx.x % a.n_blocks, rest = blockIdx.x / a.n_blocks;
  const int mb = rest % a.m_blocks, ks = rest / a.m_blocks;  // ks: the split of K (0 without split-K)
  const int m0 = mb * kGBM;
  const int64_t kbase = (int64_t)ks * a.k_per;

  // Loader roles. A: rows tid/8 + 32i (i < 4), 8-element chunk tid%8. B: rows tid/4 + 64i (i < 2),
  // 16-element chunk tid%4.
  const int ar = tid >> 3, ac = (tid & 7) * 8;
  const uint16_t* ap[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int row = m0 + ar + 32 * i;
    row = row < a.m ? row : a.m - 1;  // rows past m repeat row m-1; their outputs are dropped
    ap[i] = a.x + (int64_t)row * a.ldx + kbase + ac;
  }
  const int br = tid >> 2, bc = (tid & 3) * 16;
  const int8_t* bp[2];
  float bs[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int row = gemm_wrow<EPI>(a, nb, br + 64 * i);
    row = row < a.n ? row : a.n - 1;
    bp[i] = a.w + (int64_t)row * a.k + kbase + bc;
    bs[i] = bf16_to_f32(a.scale[row]);
  }
  // A K step's global tiles in registers: two sets, so that a step's loads are issued two steps
  // before its LDS store -- in flight during two steps of MFMAs.
  uint4 ra0, ra1, ra2, ra3, rb0, rb1, sa0, sa1, sa2, sa3, sb0, sb1;
#define MSA_GEMM_LOAD(p, k0)                  \
  do {                                        \
    p##a0 = *(const uint4*)(ap[0] + (k0));    \
    p##a1 = *(const uint4*)(ap[1] + (k0));    \
    p##a2 = *(const uint4*)(ap[2] + (k0));    \
    p##a3 = *(const uint4*)(ap[3] + (k0));    \
    p##b0 = *(const uint4*)(bp[0] + (k0));    \
    p##b1 = *(const uint4*)(bp[1] + (k0));    \
  } while (0)
#define MSA_GEMM_STORE(p, buf)                                              \
  do {                                                                      \
    uint16_t* A_ = As + (buf) * kGBM * kGLd + ar * kGLd + ac;               \
    *(uint4*)(A_) = p##a0;                                                  \
    *(uint4*)(A_ + 32 * kGLd) = p##a1;                                      \
    *(uint4*)(A_ + 64 * kGLd) = p##a2;                                      \
    *(uint4*)(A_ + 96 * kGLd) = p##a3;                                      \
    uint16_t* B_ = Bs + (buf) * kGBN * kGLd + br * kGLd + bc;               \
    *(bf16x8*)(B_) = dequant8(p##b0.x, p##b0.y, bs[0]);                     \
    *(bf16x8*)(B_ + 8) = dequant8(p##b0.z, p##b0.w, bs[0]);                 \
    *(bf16x8*)(B_ + 64 * kGLd) = dequant8(p##b1.x, p##b1.y, bs[1]);         \
    *(bf16x8*)(B_ + 64 * kGLd + 8) = dequant8(p##b1.z, p##b1.w, bs[1]);     \
  } while (0)

  // 32 x 32 x 16 MFMAs, 2 x 2 tiles per wavefront: lane (h, r) holds row r of a 32-row operand
  // tile, K elements 8h..8h+7 of each 16-wide slice. Two fragment sets: slice ks + 1 is read
  // while slice ks's MFMAs run.
  const int r32 = lane & 31, h = lane >> 5;
  f32x16 acc[2][2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = f32x16{};

#define MSA_GEMM_COMPUTE(cur)                                                                        \
  do {                                                                                               \
    const uint16_t* A = As + (cur) * kGBM * kGLd + (wm * 64 + r32) * kGLd + h * 8;                    \
    const uint16_t* B = Bs + (cur) * kGBN * kGLd + (wn * 64 + r32) * kGLd + h * 8;                    \
    bf16x8 af[2][2], bfr[2][2];                                                                      \
    _Pragma("unroll") for (int t = 0; t < 2; ++t) {                                                  \
      af[0][t] = *(const bf16x8*)(A + t * 32 * kGLd);                                                \
      bfr[0][t] = *(const bf16x8*)(B + t * 32 * kGLd);                                               \
    }                                                                                                \
    _Pragma("unroll") for (int ks = 0; ks < 4; ++ks) {                                               \
      if (ks < 3) {                                                                                  \
        _Pragma("unroll") for (int t = 0; t < 2; ++t) {                                              \
          af[(ks + 1) & 1][t] = *(const bf16x8*)(A + t * 32 * kGLd + (ks + 1) * 16);                 \
          bfr[(ks + 1) & 1][t] = *(const bf16x8*)(B + t * 32 * kGLd + (ks + 1) * 16);                \
        }                                                                                            \
      }                                                                                              \
      _Pragma("unroll") for (int mt = 0; mt < 2; ++mt)                                               \
        _Pragma("unroll") for (int nt = 0; nt < 2; ++nt)                                             \
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][mt], bfr[ks & 1][nt], acc[mt][nt], 0, 0, 0); \
      __builtin_amdgcn_sched_barrier(0);                                                             \
    }                                                                                                \
  } while (0)

  // Step kt computes from LDS buffer kt & 1 while step kt + 1's tiles wait in registers (set
  // (kt + 1) & 1) and step kt + 2's are requested into the other set; then step kt + 1 is stored.
  // Steps past nk load clamped addresses (the last step again) and are never stored.
  const int nk = a.k_per / kGBK;
  const int klast = (nk - 1) * kGBK;
  MSA_GEMM_LOAD(r, 0);
  MSA_GEMM_LOAD(s, min(kGBK, klast));
  MSA_GEMM_STORE(r, 0);
  __syncthreads();
  int kt = 0;
  for (; kt + 2 <= nk; kt += 2) {
    MSA_GEMM_LOAD(r, min((kt + 2) * kGBK, klast));
    MSA_GEMM_COMPUTE(0);
    MSA_GEMM_STORE(s, 1);  // step kt + 1 (exists: kt + 2 <= nk)
    __syncthreads();
    MSA_GEMM_LOAD(s, min((kt + 3) * kGBK, klast));
    MSA_GEMM_COMPUTE(1);
    if (kt + 2 < nk) MSA_GEMM_STORE(r, 0);  // step kt + 2
    __syncthreads();
  }
  if (kt < nk) MSA_GEMM_COMPUTE(0);  // odd nk: the last step, stored at the end of the loop
#undef MSA_GEMM_LOAD
#undef MSA_GEMM_STORE
#undef MSA_GEMM_COMPUTE

  // value i of lane (h, r) in tile (mt, nt): token m0 + wm*64 + mt*32 + 8(i/4) + 4h + i%4, LDS
  // weight row wn*64 + nt*32 + r
  if constexpr (EPI == kEpiPartial) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = m0 + wm * 64 + mt * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
        if (tok >= a.m) continue;
        float* prow = a.part + ((int64_t)ks * a.m + tok) * a.n;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const int col = nb * kGBN + wn * 64 + nt * 32 + r32;
          if (col < a.n) prow[col] = acc[mt][nt][i];
        }
      }
  } else {
    // The tile's bf16 outputs go through LDS (free once every wavefront is past its last K step):
    // rows are then stored 16 bytes per lane, or handed to the q/k-norm epilogue whole.
    constexpr int kCLd = kGBN + 8;
    uint16_t* Cs = gsm;  // [128 tokens][kCLd]
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        uint16_t* c = Cs + (wm * 64 + mt * 32 + 8 * (i >> 2) + 4 * h + (i & 3)) * kCLd + r32;
        if constexpr (EPI == MSA_EPI_SILU_MUL) {
          // the wavefront's 64 weight rows: 32 gate rows (tile 0), then their 32 up rows (tile 1)
          const float gt = round_bf16(acc[mt][0][i]), up = round_bf16(acc[mt][1][i]);
          c[wn * 32] = f32_to_bf16(round_bf16(silu_f32(gt)) * up);
        } else {
#pragma unroll
          for (int nt = 0; nt < 2; ++nt) c[wn * 64 + nt * 32] = f32_to_bf16(acc[mt][nt][i]);
        }
      }
    __syncthreads();
    if constexpr (EPI == kEpiQkNorm) {
      qk_norm_rope_tile<256, kGBM>(a.qk, Cs, kCLd, nb, m0, a.m, tid);
    } else {
      constexpr int kOutCols = EPI == MSA_EPI_SILU_MUL ? 64 : kGBN;
      constexpr int kChunksPerRow = kOutCols / 8;
      const int col0 = EPI == MSA_EPI_SILU_MUL ? nb * 64 : nb * kGBN;
      const int out_n = EPI == MSA_EPI_SILU_MUL ? a.n / 2 : a.n;
      const bool vec = ((uintptr_t)a.y & 15) == 0 && (a.ldy & 7) == 0 &&
                       (EPI != MSA_EPI_RESIDUAL || (((uintptr_t)a.resid & 15) == 0 && (a.ldr & 7) == 0));
#pragma unroll 4
      for (int c = tid; c < kGBM * kChunksPerRow; c += 256) {
        const int row = c / kChunksPerRow, cc = (c % kChunksPerRow) * 8;
        const int tok = m0 + row, col = col0 + cc;
        if (tok >= a.m || col >= out_n) continue;
        const u32x4 v = *(const u32x4*)(Cs + row * kCLd + cc);
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
          const uint16_t* sv = Cs + row * kCLd + cc;
          for (int e = 0; e < 8 && col + e < out_n; ++e) {
            float o = bf16_to_f32(sv[e]);
            if constexpr (EPI == MSA_EPI_RESIDUAL) o += bf16_to_f32(a.resid[(int64_t)tok * a.ldr + col + e]);
            dst[e] = f32_to_bf16(o);
          }
        }
      }
    }
  }
}

template <int EPI>
static int launch_gemm(const GemmArgs& a, int blocks, hipStream_t s) {
  const int rc = allow_dynamic_lds((const void*)int8_gemm_kernel<EPI>, (int)kGemmLds, "int8_gemm_kernel");
  if (rc != MSA_OK) return rc;
  hipLaunchKernelGGL(int8_gemm_kernel<EPI>, dim3(blocks), dim3(256), kGemmLds, s, a);
  return MSA_OK;
}

// Split-K merge: y = bf16(sum of the splits' partials in split order), then the residual add
// bf16(residual + y) when given (in place allowed: each thread reads its residual before writing).
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, int splits, int m,
                                                                 int n, uint16_t* y, int64_t ldy, const uint16_t* resid,
                                                                 int64_t ldr) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int tok = (int)(idx / n), col = (int)(idx % n);
  float v = 0.f;
  for (int s = 0; s < splits; ++s) v += part[((int64_t)s * m + tok) * n + col];
  v = round_bf16(v);
  if (resid) v += bf16_to_f32(resid[(int64_t)tok * ldr + col]);
  y[(int64_t)tok * ldy + col] = f32_to_bf16(v);
}

// K splits of the GEMM: 1 when the output tiles fill the GPU (or for silu * up), else the fewest
// splits (of whole 64-wide steps, at least 512 of K each, at most 8) that give 256+ workgroups,
// or the most such splits when none does.
// Workgroups a split-K launch aims for (splits are added until the tiles times the splits reach it).
#ifndef MSA_SPLITK_TARGET_WGS
#define MSA_SPLITK_TARGET_WGS 256
#endif

// Split-K on the 256-token tiles (gemm_big.hip): the split count, or 0 when that tiling does not
// serve the shape; and its partial pass.
int gemm256_split_plan(int64_t m, int64_t n, int64_t k);
int gemm256_partials_run(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                         const uint16_t* scale, int64_t n, int splits, float* part, hipStream_t s);

// Splits of the 128 x 128 split-K GEMM: enough to reach MSA_SPLITK_TARGET_WGS workgroups when
// fewer than 192 output tiles exist, K per split a multiple of 64 and at least 512.
static int splits128(int64_t m, int64_t n, int64_t k, int epilogue) {
  if (epilogue == MSA_EPI_SILU_MUL || k % kGBK != 0) return 1;
  const int64_t tiles = ((n + kGBN - 1) / kGBN) * ((m + kGBM - 1) / kGBM);
  if (tiles >= 192) return 1;
  const int64_t steps = k / kGBK;
  int best = 1;
  for (int s = 2; s <= 8; ++s) {
    if (steps % s != 0 || k / s < 512) continue;
    best = s;
    if (tiles * s >= MSA_SPLITK_TARGET_WGS) break;
  }
  return best;
}

// The 256 x 128 split-K plan when its 32-bit load offsets fit (x rows at pitch ldx), else 0.
static int splits256(int64_t m, int64_t n, int64_t k, int64_t ldx) {
  if ((m - 1) * ldx * 2 + 2 * k >= (int64_t)1 << 32 || n * k >= (int64_t)1 << 32) return 0;
  return gemm256_split_plan(m, n, k);
}

// Splits on the 256 x 128 tiles where their number is past what splits128 would split but leaves
// much of the chip idle in one unsplit round (96 to 128 tiles on 256 CUs): two splits fill 192 to 256
// of them in one round. 8B-shaped o at 768 / 1024 tokens 52 / 57 us unsplit, 48 / 56 in two splits
// and their merge (with the next norm 56 / 61 and 45 / 51); down 140 / 151, 106 / 123; the 8B-shaped
// qkv with its q/k norm at 385 to 512 tokens 50 / 42-44, at 40 query heads over K = 5120 60 / 54.
// The kernel deals output-row blocks to the eight XCDs, so one round also needs the fullest XCD's
// workgroups to fit its 32 CUs: rows of 20 blocks put three blocks, 36 workgroups at 1300 tokens, on
// four of them, a second round (2560 x 9728: 103 us unsplit, 146 split; with the norm 112 and 145).
static int splits_mid(int64_t m, int64_t n, int64_t k, int epilogue) {
  if (epilogue == MSA_EPI_SILU_MUL || m < 192) return 1;
  const int64_t n_blocks = (n + 127) / 128, m_blocks = (m + 255) / 256;
  const int64_t tiles = n_blocks * m_blocks;
  if (tiles < 96 || tiles > 128 || (n_blocks + 7) / 8 * m_blocks * 2 > 32) return 1;
  return gemm256_split_plan(m, n, k) == 2 ? 2 : 1;
}

// The split count of a GEMM that splits K (1: unsplit): the 256 x 128 tiles' plan where it applies
// (sixteen wavefronts per workgroup), else the 128 x 128 tiles' (four wavefronts).
int gemm_splits(int64_t m, int64_t n, int64_t k, int epilogue) {
  const int s128 = splits128(m, n, k, epilogue);
  if (s128 <= 1) return splits_mid(m, n, k, epilogue);
  const int s256 = gemm256_split_plan(m, n, k);
  return s256 > 1 ? s256 : s128;
}

// Partials for either plan (the 128 x 128 one serves when x's pitch is too large for the 256-token
// kernel's 32-bit offsets).
size_t gemm_workspace_size(int64_t m, int64_t n, int64_t k, int epilogue) {
  const int splits = std::max(gemm_splits(m, n, k, epilogue), splits128(m, n, k, epilogue));
  return splits > 1 ? (size_t)splits * m * n * sizeof(float) : 0;
}

// The middle shapes' two splits pay without a fused consumer of the partials only over a long K (0.6B o /
// down at 4096 tokens, K = 2048 / 3072: 33 / 47 us unsplit, 42 / 53 split; with the norm 39 / 51 and 38 / 48).
static int plain_splits(int64_t m, int64_t n, int64_t k, int epilogue) {
  const int splits = gemm_splits(m, n, k, epilogue);
  return splits > 1 && splits128(m, n, k, epilogue) <= 1 && k < 4096 ? 1 : splits;
}

size_t gemm_plain_workspace_size(int64_t m, int64_t n, int64_t k) {
  return plain_splits(m, n, k, MSA_EPI_NONE) > 1 ? gemm_workspace_size(m, n, k, MSA_EPI_NONE) : 0;
}

// The part without which the GEMM leaves much of the chip idle: the 128-token tiles' splits.
size_t gemm_min_workspace_size(int64_t m, int64_t n, int64_t k) {
  return splits128(m, n, k, MSA_EPI_NONE) > 1 ? gemm_workspace_size(m, n, k, MSA_EPI_NONE) : 0;
}

// The 256-token tilings (gemm_big.hip): the best-filling one and its tile count, and the GEMM on it.
int gemm256_pick(int64_t m, int64_t n, int64_t k, int epilogue, int64_t* tiles);
int gemm256_run(int t, const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                const uint16_t* scale, int64_t n, uint16_t* y, int64_t ldy, int epilogue, const uint16_t* residual,
                int64_t ldr, hipStream_t s);

// Which tiling serves an unsplit GEMM: a 256-token one (gemm256_pick's) when it keeps at least as
// much of the chip's workgroup slots busy over its rounds of workgroups (256 CUs; one 256-token
// workgroup or two 128 x 128 ones per CU) as the 128 x 128 tiling (fewer LDS bytes per MFMA, half
// the dequantization per flop and two wavefronts per SIMD in one workgroup). Returns that tiling,
// or -1.
static int use_gemm256(int64_t m, int64_t n, int64_t k, int64_t ldx, int epilogue) {
  // its loads address x and the weight with 32-bit byte offsets
  if ((m - 1) * ldx * 2 + 2 * k >= (int64_t)1 << 32 || n * k >= (int64_t)1 << 32) return -1;
  int64_t t256 = 0;
  const int t = gemm256_pick(m, n, k, epilogue, &t256);
  if (t < 0 || t256 < 128) return -1;
  const int64_t n128 = epilogue == MSA_EPI_SILU_MUL ? (n / 2 + 63) / 64 : (n + kGBN - 1) / kGBN;
  const int64_t t128 = n128 * ((m + kGBM - 1) / kGBM);
  constexpr int64_t kCUs = 256;
  const int64_t slots256 = (t256 + kCUs - 1) / kCUs * kCUs, slots128 = (t128 + 2 * kCUs - 1) / (2 * kCUs) * 2 * kCUs;
  return t256 * slots128 >= t128 * slots256 ? t : -1;  // t256 / slots256 >= t128 / slots128
}

int gemm256_qk_norm_run(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                        const uint16_t* scale, const QkNormOut& qk, hipStream_t s);

// The qkv projection with its q/k-norm epilogue on 256 x 128 tiles (one head slot each, one
// workgroup of sixteen wavefronts per CU) when they fill at least as much of the chip as the 128 x 128
// tiles (two workgroups per CU).
static bool use_qk_norm256(int64_t m, int64_t k, int64_t ldx, int head_slots) {
  const int64_t n = (int64_t)head_slots * 128;
  if ((m - 1) * ldx * 2 + 2 * k >= (int64_t)1 << 32 || n * k >= (int64_t)1 << 32) return false;
  const int64_t tbig = head_slots * ((m + 255) / 256), t128 = head_slots * ((m + kGBM - 1) / kGBM);
  if (tbig < 128) return false;
  constexpr int64_t kCUs = 256;
  const int64_t slots_big = (tbig + kCUs - 1) / kCUs * kCUs, slots128 = (t128 + 2 * kCUs - 1) / (2 * kCUs) * 2 * kCUs;
  return tbig * slots128 >= t128 * slots_big;
}

// The GEMM with arguments checked by the caller; split-K when planned and the workspace holds it.
int gemm_run(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight, const uint16_t* scale,
             int64_t n, uint16_t* y, int64_t ldy, int epilogue, const uint16_t* residual, int64_t ldr, void* workspace,
             size_t workspace_bytes, hipStream_t s) {
  GemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale; a.y = y; a.ldy = ldy; a.resid = residual; a.ldr = ldr;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  a.n_blocks = (int)(epilogue == MSA_EPI_SILU_MUL ? (n / 2 + 63) / 64 : (n + kGBN - 1) / kGBN);
  a.m_blocks = (int)((m + kGBM - 1) / kGBM);
  int splits = plain_splits(m, n, k, epilogue);
  const bool unsplit_plan = splits == 1 || splits128(m, n, k, epilogue) <= 1;  // planned unsplit but for splits_mid
  if (splits > 1 && (!workspace || workspace_bytes < gemm_workspace_size(m, n, k, epilogue) || !aligned16(workspace)))
    splits = 1;
  const int s256 = splits > 1 ? splits256(m, n, k, ldx) : 0;
  if (splits > 1 && s256 <= 1) splits = splits128(m, n, k, epilogue);
  const int big = splits == 1 && unsplit_plan ? use_gemm256(m, n, k, ldx, epilogue) : -1;
  if (big >= 0) return gemm256_run(big, x, m, k, ldx, qweight, scale, n, y, ldy, epilogue, residual, ldr, s);
  a.k_per = (int)(k / splits);
  a.part = (float*)workspace;
  const int64_t blocks = (int64_t)a.n_blocks * a.m_blocks * splits;
  if (blocks > 0x7fffffff) return fail(MSA_ERR_INVALID, "msa_int8_gemm: too many tiles");
  int rc;
  if (splits > 1) {
    if (s256 > 1) {
      rc = gemm256_partials_run(x, m, k, ldx, qweight, scale, n, s256, a.part, s);
      splits = s256;
    } else {
      rc = launch_gemm<kEpiPartial>(a, (int)blocks, s);
      if (rc == MSA_OK) rc = check_launch("msa_int8_gemm (split-K)");
    }
    if (rc != MSA_OK) return rc;
    const int64_t elems = m * n;
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)((elems + 255) / 256)), dim3(256), 0, s, a.part,
                       splits, a.m, a.n, y, ldy, epilogue == MSA_EPI_RESIDUAL ? residual : nullptr, ldr);
    return check_launch("msa_int8_gemm (split-K merge)");
  }
  switch (epilogue) {
    case MSA_EPI_NONE: rc = launch_gemm<MSA_EPI_NONE>(a, (int)blocks, s); break;
    case MSA_EPI_SILU_MUL: rc = launch_gemm<MSA_EPI_SILU_MUL>(a, (int)blocks, s); break;
    default: rc = launch_gemm<MSA_EPI_RESIDUAL>(a, (int)blocks, s); break;
  }
  if (rc != MSA_OK) return rc;
  return check_launch("msa_int8_gemm");
}

// The split-K partial pass alone: float32 partials [splits][m][n] of x @ bf16(q * s)^T into part,
// with the split count the GEMM would use; returns 1 (nothing launched) when it would not split or
// part is too small.
int gemm_run_partials(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                      const uint16_t* scale, int64_t n, float* part, size_t part_bytes, hipStream_t s) {
  if (gemm_splits(m, n, k, MSA_EPI_NONE) <= 1 || !part || part_bytes < gemm_workspace_size(m, n, k, MSA_EPI_NONE) ||
      !aligned16(part))
    return 1;
  const int s256 = splits256(m, n, k, ldx);
  if (s256 > 1) return gemm256_partials_run(x, m, k, ldx, qweight, scale, n, s256, part, s) == MSA_OK ? s256 : -1;
  const int splits = splits128(m, n, k, MSA_EPI_NONE);
  if (splits <= 1) return 1;
  GemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  a.n_blocks = (int)((n + kGBN - 1) / kGBN);
  a.m_blocks = (int)((m + kGBM - 1) / kGBM);
  a.k_per = (int)(k / splits);
  a.part = part;
  const int64_t blocks = (int64_t)a.n_blocks * a.m_blocks * splits;
  if (blocks > 0x7fffffff) return 1;
  if (launch_gemm<kEpiPartial>(a, (int)blocks, s) != MSA_OK) return -1;
  return splits;
}

// ---- LM head for many rows: gather + RMSNorm once, then a bf16 GEMM with an argmax epilogue ----
//
// When the sampled rows do not fit one LDS activation tile of the streaming LM head (many rows at
// a large hidden size), the rows are normalized once into a workspace and the logits are
// computed tile by tile on MFMA: 128 rows x 128 vocabulary entries x 64-wide K steps, both
// operands bf16 in LDS, double buffered. No logit leaves the workgroup: each one is rounded to
// bf16 (the reference's logits dtype) and the workgroup writes one (max, first index) candidate
// per row for its 128 vocabulary entries.

// One workgroup per row: y[r] = bf16(w * bf16(x[rows[r]] * rsqrt(mean(x^2) + eps))), or the plain
// gathered row when w is null. Squares are exact (bf16 pairs on v_dot2), sums float32.
__global__ __launch_bounds__(256) void lm_rows_prologue_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                               int64_t x_rows, const int64_t* __restrict__ rows,
                                                               const uint16_t* __restrict__ w, float eps, int k,
                                                               uint16_t* __restrict__ y) {
  __shared__ float red[4];
  int64_t src = rows[blockIdx.x];
  src = src < 0 ? 0 : (src >= x_rows ? x_rows - 1 : src);  // memory safety only
  const uint16_t* xr = x + src * ldx;
  uint16_t* yr = y + (int64_t)blockIdx.x * k;
  const int nvec = k / 8;
  if (!w) {
    for (int v = threadIdx.x; v < nvec; v += 256) *(uint4*)(yr + v * 8) = *(const uint4*)(xr + v * 8);
    return;
  }
  float ss = 0.f;
  for (int v = threadIdx.x; v < nvec; v += 256) {
    const uint4 u = *(const uint4*)(xr + v * 8);
    ss = dot2_bf16(u.x, u.x, ss);
    ss = dot2_bf16(u.y, u.y, ss);
    ss = dot2_bf16(u.z, u.z, ss);
    ss = dot2_bf16(u.w, u.w, ss);
  }
  ss = row16_sum(ss);
  ss = xrow_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = red[0] + red[1] + red[2] + red[3];
  const float r = 1.0f / sqrtf(ss / (float)k + eps);
  for (int v = threadIdx.x; v < nvec; v += 256) {
    const uint4 u = *(const uint4*)(xr + v * 8), wv = *(const uint4*)(w + v * 8);
    const uint32_t e[4] = {u.x, u.y, u.z, u.w}, ww[4] = {wv.x, wv.y, wv.z, wv.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = round_bf16(bf16lo(e[i]) * r), hi = round_bf16(bf16hi(e[i]) * r);
      o[i] = pack_bf16x2(bf16lo(ww[i]) * lo, bf16hi(ww[i]) * hi);
    }
    *(uint4*)(yr + v * 8) = uint4{o[0], o[1], o[2], o[3]};
  }
}

struct LmGemmArgs {
  const uint16_t* x;  // [m, k] normalized rows
  const uint16_t* w;  // [n, k] bf16
  float* cand_val;    // [m, n_blocks]
  int32_t* cand_idx;  // [m, n_blocks]
  float* logits;      // [m, ldl] (the logits route)
  int64_t ldl;
  int m, n, k;
  int n_blocks, m_blocks;
};

// Workgroup b: XCD b % 8 takes vocabulary blocks nb = xcd (mod 8) and runs the row blocks of each
// such nb back to back, so repeated weight tiles come from that XCD's L2. LOGITS: the bf16-rounded
// logits are written out as float32 instead of the argmax candidates.
template <bool LOGITS>
__global__ __launch_bounds__(256) void lm_gemm_kernel(LmGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t gsm[];
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int nb = (slot / a.m_blocks) * 8 + xcd, mb = slot % a.m_blocks;
  if (nb >= a.n_blocks) return;  // surplus workgroups of the rounded grid (whole workgroup)
  uint16_t* As = gsm;                    // [2][128][kGLd]
  uint16_t* Bs = gsm + 2 * kGBM * kGLd;  // [2][128][kGLd]
  __shared__ float rv[2][kGBM];
  __shared__ int32_t ri[2][kGBM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, g = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = mb * kGBM, n0 = nb * kGBN;

  // Loader role for both operands: rows tid/8 + 32i (i < 4), 8-element chunk tid%8.
  const int lr = tid >> 3, lc = (tid & 7) * 8;
  const uint16_t* ap[4];
  const uint16_t* bp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ra = min(m0 + lr + 32 * i, a.m - 1), rb = min(n0 + lr + 32 * i, a.n - 1);  // repeats are dropped
    ap[i] = a.x + (int64_t)ra * a.k + lc;
    bp[i] = a.w + (int64_t)rb * a.k + lc;
  }
  uint4 ra0, ra1, ra2, ra3, rb0, rb1, rb2, rb3;
#define MSA_LM_LOAD(k0)                  \
  do {                                   \
    ra0 = *(const uint4*)(ap[0] + (k0)); \
    ra1 = *(const uint4*)(ap[1] + (k0)); \
    ra2 = *(const uint4*)(ap[2] + (k0)); \
    ra3 = *(const uint4*)(ap[3] + (k0)); \
    rb0 = *(const uint4*)(bp[0] + (k0)); \
    rb1 = *(const uint4*)(bp[1] + (k0)); \
    rb2 = *(const uint4*)(bp[2] + (k0)); \
    rb3 = *(const uint4*)(bp[3] + (k0)); \
  } while (0)
#define MSA_LM_STORE(buf)                                             \
  do {                                                                \
    uint16_t* A_ = As + (buf) * kGBM * kGLd + lr * kGLd + lc;         \
    uint16_t* B_ = Bs + (buf) * kGBN * kGLd + lr * kGLd + lc;         \
    *(uint4*)(A_) = ra0;                                              \
    *(uint4*)(A_ + 32 * kGLd) = ra1;                                  \
    *(uint4*)(A_ + 64 * kGLd) = ra2;                                  \
    *(uint4*)(A_ + 96 * kGLd) = ra3;                                  \
    *(uint4*)(B_) = rb0;                                              \
    *(uint4*)(B_ + 32 * kGLd) = rb1;                                  \
    *(uint4*)(B_ + 64 * kGLd) = rb2;                                  \
    *(uint4*)(B_ + 96 * kGLd) = rb3;                                  \
  } while (0)

  f32x4 acc[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nk = a.k / kGBK;
  MSA_LM_LOAD(0);
  MSA_LM_STORE(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) MSA_LM_LOAD((kt + 1) * kGBK);
    const uint16_t* A = As + cur * kGBM * kGLd + (wm * 64 + j) * kGLd + g * 8;
    const uint16_t* B = Bs + cur * kGBN * kGLd + (wn * 64 + j) * kGLd + g * 8;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 af[4], bfr[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        af[t] = *(const bf16x8*)(A + t * 16 * kGLd + ks * 32);
        bfr[t] = *(const bf16x8*)(B + t * 16 * kGLd + ks * 32);
      }
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[mt], bfr[nt], acc[mt][nt], 0, 0, 0);
    }
    if (more) MSA_LM_STORE(cur ^ 1);
    __syncthreads();
  }
#undef MSA_LM_LOAD
#undef MSA_LM_STORE

  // lane (g, j) of tile (mt, nt): row wm*64 + mt*16 + 4g + i, vocabulary entry n0 + wn*64 + nt*16 + j.
  if constexpr (LOGITS) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = m0 + wm * 64 + mt * 16 + 4 * g + i;
        if (r >= a.m) continue;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const int col = n0 + wn * 64 + nt * 16 + j;
          if (col < a.n) a.logits[(int64_t)r * a.ldl + col] = round_bf16(acc[mt][nt][i]);
        }
      }
    return;
  }
  // Per row: the lane's best over nt (increasing entries), then over the 16 lanes j, then over wn.
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = -INFINITY;
      int idx = 0x7fffffff;
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const int col = n0 + wn * 64 + nt * 16 + j;
        const float c = col < a.n ? round_bf16(acc[mt][nt][i]) : -INFINITY;
        if (c > v) {
          v = c;
          idx = col;
        }
      }
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        const float ov = __shfl_xor(v, off);
        const int oi = __shfl_xor(idx, off);
        if (ov > v || (ov == v && oi < idx)) {
          v = ov;
          idx = oi;
        }
      }
      if (j == 0) {
        rv[wn][wm * 64 + mt * 16 + 4 * g + i] = v;
        ri[wn][wm * 64 + mt * 16 + 4 * g + i] = idx;
      }
    }
  __syncthreads();
  if (tid < kGBM && m0 + tid < a.m) {
    float v = rv[0][tid];
    int idx = ri[0][tid];
    if (rv[1][tid] > v || (rv[1][tid] == v && ri[1][tid] < idx)) {
      v = rv[1][tid];
      idx = ri[1][tid];
    }
    a.cand_val[(int64_t)(m0 + tid) * a.n_blocks + nb] = v;
    a.cand_idx[(int64_t)(m0 + tid) * a.n_blocks + nb] = idx;
  }
}

int lm_gemm_vocab_blocks(int64_t vocab) { return (int)((vocab + kGBN - 1) / kGBN); }

// Gather + norm into `xn` ([num_rows, k] bf16), then the GEMM writes [num_rows][n_blocks]
// candidates, or the logits [num_rows][ldl] when `logits` is set. k % 64 == 0.
int launch_lm_gemm(const uint16_t* hidden, int64_t ld_hidden, int64_t hidden_rows, const int64_t* rows, int num_rows,
                   int k, const uint16_t* norm_w, float eps, const uint16_t* weight, int vocab, uint16_t* xn,
                   float* cand_val, int32_t* cand_idx, float* logits, int64_t ldl, hipStream_t s) {
  hipLaunchKernelGGL(lm_rows_prologue_kernel, dim3(num_rows), dim3(256), 0, s, hidden, ld_hidden, hidden_rows, rows,
                     norm_w, eps, k, xn);
  int rc = check_launch("LM head (row prologue)");
  if (rc != MSA_OK) return rc;
  for (const void* f : {(const void*)lm_gemm_kernel<false>, (const void*)lm_gemm_kernel<true>}) {
    rc = allow_dynamic_lds(f, (int)kGemmLds, "lm_gemm_kernel");
    if (rc != MSA_OK) return rc;
  }
  LmGemmArgs a{};
  a.x = xn; a.w = weight; a.cand_val = cand_val; a.cand_idx = cand_idx; a.logits = logits; a.ldl = ldl;
  a.m = num_rows; a.n = vocab; a.k = k;
  a.n_blocks = lm_gemm_vocab_blocks(vocab);
  a.m_blocks = (num_rows + kGBM - 1) / kGBM;
  const int blocks = ((a.n_blocks + 7) / 8) * 8 * a.m_blocks;
  if (logits) hipLaunchKernelGGL(lm_gemm_kernel<true>, dim3(blocks), dim3(256), kGemmLds, s, a);
  else hipLaunchKernelGGL(lm_gemm_kernel<false>, dim3(blocks), dim3(256), kGemmLds, s, a);
  return check_launch("LM head (GEMM)");
}

}  // namespace msa

using namespace msa;

extern "C" size_t msa_int8_gemm_qk_norm_rope_cache_workspace_size(int64_t m, int64_t n, int64_t k) {
  return m > 0 && n > 0 && k > 0 && k % kGBK == 0 ? gemm_workspace_size(m, n, k, MSA_EPI_NONE) : 0;
}

extern "C" int msa_int8_gemm_qk_norm_rope_cache(const uint16_t* x, int64_t m, int64_t k, int64_t ldx,
                                               const int8_t* qweight, const uint16_t* scale, int heads, int kv_heads,
                                               int head_dim, const uint16_t* q_norm_w, const uint16_t* k_norm_w,
                                               float eps, const float* cos, const float* sin,
                                               const int64_t* slot_mapping, uint16_t* q_out, uint16_t* k_cache,
                                               uint16_t* v_cache, int64_t num_slots, void* workspace,
                                               size_t workspace_bytes, msa_stream_t stream) {
  const char* who = "msa_int8_gemm_qk_norm_rope_cache";
  if (m == 0) return MSA_OK;
  if (!x || !qweight || !scale || !q_norm_w || !k_norm_w || !cos || !sin || !slot_mapping || !q_out || !k_cache ||
      !v_cache)
    return fail(MSA_ERR_INVALID, std::string(who) + ": null pointer");
  if (head_dim != 128) return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": head_dim must be 128");
  if (m < 0 || k <= 0 || m > 0x7fffffff || k > 0x7fffffff || heads <= 0 || kv_heads <= 0 || num_slots < 0)
    return fail(MSA_ERR_INVALID, std::string(who) + ": bad shape");
  if (k % kGBK != 0) return fail(MSA_ERR_UNSUPPORTED, std::string(who) + ": in_features must be a multiple of 64");
  if (ldx < k || ldx % 8 != 0 || !aligned16(x) || !aligned16(qweight))
    return fail(MSA_ERR_INVALID, std::string(who) + ": x / qweight must be 16-byte aligned with ldx % 8 == 0");
  if (!aligned16(q_norm_w) || !aligned16(k_norm_w) || !aligned16(cos) || !aligned16(sin) || !aligned16(q_out) ||
      !aligned16(k_cache) || !aligned16(v_cache))
    return fail(MSA_ERR_INVALID, std::string(who) + ": norm weights, cos / sin, q_out and caches must be 16-byte aligned");
  const int64_t n = (int64_t)(heads + 2 * kv_heads) * 128;
  // Few output tiles: split-K partials into the workspace, then the q/k-norm kernel that sums them
  // (the same values: partials summed in split order, rounded to bf16, then normed).
  const int splits = gemm_splits(m, n, k, MSA_EPI_NONE);
  if (splits > 1 && workspace && workspace_bytes >= gemm_workspace_size(m, n, k, MSA_EPI_NONE) && aligned16(workspace)) {
    const int got = gemm_run_partials(x, m, k, ldx, qweight, scale, n, (float*)workspace, workspace_bytes,
                                      (hipStream_t)stream);
    if (got < 0) return MSA_ERR_LAUNCH;  // fail() has recorded why
    if (got > 1)
      return msa_qk_norm_rope_cache_splitk((const float*)workspace, got, m, heads, kv_heads, 128, q_norm_w, k_norm_w,
                                           eps, cos, sin, slot_mapping, q_out, k_cache, v_cache, num_slots, stream);
  }
  const QkNormOut qk{heads, kv_heads, q_norm_w, k_norm_w, eps, cos, sin, slot_mapping, q_out, k_cache, v_cache, num_slots};
  if (use_qk_norm256(m, k, ldx, heads + 2 * kv_heads))
    return gemm256_qk_norm_run(x, m, k, ldx, qweight, scale, qk, (hipStream_t)stream);
  GemmArgs a{};
  a.x = x; a.ldx = ldx; a.w = qweight; a.scale = scale;
  a.m = (int)m; a.n = (int)n; a.k = (int)k;
  a.n_blocks = heads + 2 * kv_heads;
  a.m_blocks = (int)((m + kGBM - 1) / kGBM);
  a.k_per = (int)k;
  a.qk = qk;
  const int64_t blocks = (int64_t)a.n_blocks * a.m_blocks;
  if (blocks > 0x7fffffff) return fail(MSA_ERR_INVALID, std::string(who) + ": too many tiles");
  const int rc = launch_gemm<kEpiQkNorm>(a, (int)blocks, (hipStream_t)stream);
  if (rc != MSA_OK) return rc;
  return check_launch(who);
}

extern "C" int msa_int8_gemm(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                             const uint16_t* scale, int64_t n, uint16_t* y, int64_t ldy, int epilogue,
                             const uint16_t* residual, int64_t ldr, msa_stream_t stream) {
  if (m == 0) return MSA_OK;
  if (!x || !qweight || !scale || !y) return fail(MSA_ERR_INVALID, "msa_int8_gemm: null pointer");
  if (m < 0 || n <= 0 || k <= 0 || m > 0x7fffffff || n > 0x7fffffff || k > 0x7fffffff)
    return fail(MSA_ERR_INVALID, "msa_int8_gemm: bad shape");
  if (k % kGBK != 0) return fail(MSA_ERR_UNSUPPORTED, "msa_int8_gemm: in_features must be a multiple of 64");
  if (ldx < k || ldx % 8 != 0 || !aligned16(x) || !aligned16(qweight))
    return fail(MSA_ERR_INVALID, "msa_int8_gemm: x / qweight must be 16-byte aligned with ldx % 8 == 0");
  if (epilogue < 0 || epilogue > 2) return fail(MSA_ERR_INVALID, "msa_int8_gemm: unknown epilogue");
  if (epilogue == MSA_EPI_SILU_MUL && n % 2 != 0) return fail(MSA_ERR_INVALID, "msa_int8_gemm: SILU_MUL needs an even n");
  const int64_t out_cols = epilogue == MSA_EPI_SILU_MUL ? n / 2 : n;
  if (ldy < out_cols) return fail(MSA_ERR_INVALID, "msa_int8_gemm: ldy too small");
  if (epilogue == MSA_EPI_RESIDUAL && (!residual || ldr < n))
    return fail(MSA_ERR_INVALID, "msa_int8_gemm: the residual epilogue needs residual with ldr >= n");
  return gemm_run(x, m, k, ldx, qweight, scale, n, y, ldy, epilogue, residual, ldr, nullptr, 0, (hipStream_t)stream);
}
