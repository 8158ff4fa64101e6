// Int8 linear for decode batches of up to 64 tokens over weight matrices of tens of megabytes: one
// pass over the weights at the rate of HBM, any K that is a multiple of 64.
//
// A workgroup of eight wavefronts owns units of NT 16-row weight tiles over the whole K. K is dealt
// to the wavefronts in 64-wide chunks (chunk c to wavefront c % 8), so at any time the workgroup
// reads 512 contiguous bytes of each of its rows, and every weight byte is loaded and dequantized
// by exactly one lane of the launch.
//
//  * Per chunk a lane holds 16 bytes of one weight row in each tile (row j, K offsets [16g, 16g + 16)
//    of the chunk) and its share of the 16 MT token rows' 128 bytes of activations (8 lanes per row,
//    whole cache lines). D chunks of both are in flight per wavefront: as a chunk is consumed its
//    registers are refilled with the chunk D further on -- across unit boundaries, so the stream does
//    not drain at a unit's end.
//  * The activations become MFMA A fragments through the wavefront's own LDS region (the LDS
//    operations of one wavefront complete in order: no barrier). They come from L2: a workgroup reads
//    all t x K of them per unit, which is why wider batches take tiles that share them over more rows
//    (the GEMMs).
//  * The weights are dequantized to bf16(q * s), the value of the reference's whole-matrix
//    dequantization (quant/int8.py:36), and multiplied on v_mfma_f32_16x16x32_bf16 with float32
//    accumulation.
//  * The eight partial tiles meet in LDS at a unit's end and are summed in wavefront order; the
//    epilogues (residual add, silu(gate) * up with 8 gate and 8 up rows per tile) round where the
//    reference rounds.
//
// Chunks past K are read out of a buffer descriptor's range, which gives zeros without traffic, so
// every load is unconditional and the compiler's in-order load counter waits for exactly one chunk.
#include <hip/hip_runtime.h>

#include "common.h"

namespace msa {

struct WideArgs {
  const uint16_t* x;
  int64_t ldx;
  int t;  // tokens, 1..16 MT
  int k;  // in features, a multiple of 64
  const int8_t* w;
  const uint16_t* scale;
  int n;      // weight rows ([gate | up] for SILU_MUL)
  int units;  // units of NT tiles
  uint16_t* y;
  int64_t ldy;
  const uint16_t* resid;
  int64_t ldr;
  int k_per;    // K per split (a multiple of 64; k without split-K)
  float* part;  // kWidePartial: float32 partials [splits][t][n], split blockIdx.y
};

constexpr int kWidePartial = 3;

// Weight row of tile `tile` for lane row j (clamped into the matrix; outputs past the end are dropped).
template <int EPI>
__device__ __forceinline__ int wide_row(const WideArgs& a, int tile, int j) {
  if constexpr (EPI == MSA_EPI_SILU_MUL) {
    const int half = a.n / 2;
    return min(8 * tile + (j & 7), half - 1) + (j < 8 ? 0 : half);
  } else {
    return min(16 * tile + j, a.n - 1);
  }
}

template <int W, int NT, int MT, int D, int OCC, int EPI>
__global__ __launch_bounds__(64 * W, W / 4 * OCC) void dec_wide_kernel(WideArgs a) {
  constexpr int XL = 2 * MT;       // activation loads per chunk: eight token rows each
  constexpr int XP = 64 + 8;       // staged row pitch (elements): fragment reads without bank conflicts
  constexpr int kXBytes = MT * 16 * XP * 2, kAccBytes = MT * NT * 1024;
  constexpr int kRegion = kXBytes > kAccBytes ? kXBytes : kAccBytes;
  constexpr int TPW = (MT * NT + W - 1) / W;  // output tiles per wavefront
  extern __shared__ __attribute__((aligned(16))) char s_mem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  uint16_t* xs = (uint16_t*)(s_mem + wave * kRegion);
  const int k0 = (int)blockIdx.y * a.k_per;
  const int nch = min(a.k_per, a.k - k0) / 64;
  const int groups = (nch + W * D - 1) / (W * D);
  constexpr uint32_t kPast = 0x80000000u;  // added to an offset: past every descriptor's range

  const buf_rsrc wrs = make_rsrc(a.w, (uint32_t)a.n * (uint32_t)a.k);
  const buf_rsrc srs = make_rsrc(a.scale, 2u * (uint32_t)a.n);
  const buf_rsrc xrs = make_rsrc(a.x, 2u * ((uint32_t)(a.t - 1) * (uint32_t)a.ldx + (uint32_t)a.k));
  uint32_t xoff[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = min(8 * i + (lane >> 3), a.t - 1);  // rows past t repeat row t - 1: outputs dropped
    xoff[i] = 2u * (mul24(row, (int)a.ldx) + (uint32_t)(k0 + wave * 64 + (lane & 7) * 8));
  }
  auto row_offsets = [&](int unit, uint32_t(&wo)[NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      wo[nt] = mul24(wide_row<EPI>(a, unit * NT + nt, j), a.k) + (uint32_t)(k0 + wave * 64 + g * 16);
  };
  u32x4 xv[D][XL], wv[D][NT];
  auto load_chunk = [&](int s, int group, bool live, const uint32_t(&wo)[NT]) {
    const int i = group * D + s;  // this wavefront's i-th chunk
    const uint32_t past = live && wave + W * i < nch ? 0u : kPast;
    const uint32_t xd = past + (uint32_t)i * (W * 128), wd = past + (uint32_t)i * (W * 64);
#pragma unroll
    for (int l = 0; l < XL; ++l) xv[s][l] = buf_load16(xrs, xoff[l] + xd);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wv[s][nt] = buf_load16(wrs, wo[nt] + wd);
  };
  auto load_scales = [&](int unit, uint32_t(&sc)[NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sc[nt] = buf_load_u16(srs, 2u * wide_row<EPI>(a, unit * NT + nt, j));
  };

  int unit = blockIdx.x;
  uint32_t wo[NT], scb[NT], scn[NT];
  row_offsets(unit, wo);
  load_scales(unit, scb);
#pragma unroll
  for (int s = 0; s < D; ++s) load_chunk(s, 0, true, wo);

  while (true) {
    // The residual values of this wavefront's output tiles: needed last, requested first.
    uint32_t rres[TPW][4] = {};
    if constexpr (EPI == MSA_EPI_RESIDUAL) {
      const buf_rsrc rrs = make_rsrc(a.resid, 2u * ((uint32_t)(a.t - 1) * (uint32_t)a.ldr + (uint32_t)a.n));
#pragma unroll
      for (int o = 0; o < TPW; ++o) {
        const int out = min(wave + o * W, MT * NT - 1), mt_o = out / NT, nt_o = out % NT;
        const int row = wide_row<EPI>(a, unit * NT + nt_o, j);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          rres[o][i] = buf_load_u16(rrs, 2u * (mul24(min(mt_o * 16 + 4 * g + i, a.t - 1), (int)a.ldr) + row));
      }
    }
    f32x4 acc[MT][NT];
    float sf[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      sf[nt] = bf16_to_f32(scb[nt]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int next = unit + (int)gridDim.x;
    for (int gi = 0; gi < groups; ++gi) {
      // What refills the registers: the next group of this unit, or the first of the next.
      const bool last = gi + 1 == groups;
      const int run = last ? next : unit, rgroup = last ? 0 : gi + 1;
      const bool live = !last || next < a.units;
      row_offsets(min(run, a.units - 1), wo);
      if (last) load_scales(min(next, a.units - 1), scn);
#pragma unroll
      for (int s = 0; s < D; ++s) {
#pragma unroll
        for (int l = 0; l < XL; ++l) *(u32x4*)(xs + (8 * l + (lane >> 3)) * XP + (lane & 7) * 8) = xv[s][l];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        bf16x8 xa[MT][2], b[NT][2];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h) xa[mt][h] = *(const bf16x8*)(xs + (mt * 16 + j) * XP + g * 16 + h * 8);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          b[nt][0] = dequant8(wv[s][nt].x, wv[s][nt].y, sf[nt]);
          b[nt][1] = dequant8(wv[s][nt].z, wv[s][nt].w, sf[nt]);
        }
        load_chunk(s, rgroup, live, wo);
        __builtin_amdgcn_sched_barrier(0);  // the refills stay here, ahead of the MFMAs
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[mt][h], b[nt][h], acc[mt][nt], 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // every fragment read precedes the next chunk's LDS writes
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    }
    // The wavefronts' partial tiles, each in its own region, then one wavefront per output tile.
    f32x4* part = (f32x4*)(s_mem + wave * kRegion);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) part[(mt * NT + nt) * 64 + lane] = acc[mt][nt];
    __syncthreads();
#pragma unroll
    for (int o = 0; o < TPW; ++o) {
      const int out = wave + o * W, mt_o = out / NT, nt_o = out % NT;
      if (out >= MT * NT) break;
      f32x4 v = *(const f32x4*)(s_mem + (out * 64 + lane) * 16);
#pragma unroll
      for (int w = 1; w < W; ++w) v += *(const f32x4*)(s_mem + w * kRegion + (out * 64 + lane) * 16);
      // lane (j, g): tokens 4g .. 4g + 3 of the tile, weight row j
      const int tile = unit * NT + nt_o, tok = mt_o * 16 + 4 * g;
      if constexpr (EPI == kWidePartial) {
        const int c = 16 * tile + j;
        float* p = a.part + ((int64_t)blockIdx.y * a.t + tok) * a.n + c;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (tok + i < a.t && c < a.n) p[(int64_t)i * a.n] = v[i];
        continue;
      }
      const buf_rsrc yrs = make_rsrc(
          a.y, 2u * ((uint32_t)(a.t - 1) * (uint32_t)a.ldy + (uint32_t)(EPI == MSA_EPI_SILU_MUL ? a.n / 2 : a.n)));
      f32x4 up{};
      if constexpr (EPI == MSA_EPI_SILU_MUL) {
#pragma unroll
        for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(v[i], 8);
      }
      const int col = EPI == MSA_EPI_SILU_MUL ? 8 * tile + j : 16 * tile + j;
      if (EPI == MSA_EPI_SILU_MUL ? j >= 8 || col >= a.n / 2 : col >= a.n) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (tok + i >= a.t) continue;
        float r = v[i];
        if constexpr (EPI == MSA_EPI_SILU_MUL) {
          const float gt = round_bf16(v[i]), uv = round_bf16(up[i]);
          r = round_bf16(silu_f32(gt)) * uv;
        } else if constexpr (EPI == MSA_EPI_RESIDUAL) {
          r = round_bf16(v[i]) + bf16_to_f32(rres[o][i]);
        }
        buf_store_u16(yrs, 2u * (mul24(tok + i, (int)a.ldy) + col), f32_to_bf16(r));
      }
    }
    unit = next;
    if (unit >= a.units) break;
    __syncthreads();  // the partials are read before the next unit's activations overwrite them
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) scb[nt] = scn[nt];
  }
}

// ---- host side ----------------------------------------------------------------------------------

// Weight matrices of at least this many bytes come here where wide_pays: from there on a launch streams
// for longer than it takes to start. 8B-shaped o [4096 x 4096] at 27 tokens: 12.0 us on the decode kernel (which
// reads the weights once per 16 tokens), 9.1 here; down [4096 x 12288] at 1 / 27 tokens 42.6 / 48.6
// us on the split-K kernel for small batches, 13.1 / 22.2 here; gate_up [24576 x 4096] at 27 / 64
// tokens 48 / 95 us, 27.5 / 38 here. Below (the 0.6B shapes, 1-6 MB) the decode kernel, which has
// every load of the launch in flight at once, is as fast or faster (3072 x 1024 x 16: 3.6 against 3.8).
constexpr int64_t kWideMinWeights = (int64_t)12 << 20;
constexpr int64_t kWideMaxTokens = 64;  // more tokens: the LDS-tiled GEMM shares the activations better

bool dec_wide_eligible(int64_t m, int64_t k, int64_t n, int64_t ldx, int64_t ldy, int64_t ldr) {
  constexpr int64_t kMul = 1 << 24, kRange = (int64_t)1 << 31;  // 24-bit products, 32-bit byte offsets
  const int64_t dims[] = {k, n, ldx, ldy, ldr};
  for (int64_t d : dims)
    if (d >= kMul) return false;
  return m >= 1 && m <= kWideMaxTokens && k % 64 == 0 && n * k >= kWideMinWeights && n * k < kRange &&
         2 * m * ldx < kRange && 2 * m * ldy < kRange && 2 * m * ldr < kRange;
}

constexpr int kWideCUs = 256;
constexpr int kWidePartialNT = 4;

// K splits of the split-K form: 64-row units x splits for about one workgroup per CU, each split at
// least 16 chunks (two per wavefront). 1 when that leaves nothing to split.
int dec_wide_splits(int64_t m, int64_t n, int64_t k) {
  const int64_t units = (n + 16 * kWidePartialNT - 1) / (16 * kWidePartialNT), chunks = k / 64;
  int64_t sp = kWideCUs / units;
  sp = sp < chunks / 16 ? sp : chunks / 16;
  if (sp < 2) return 1;
  const int64_t per = (chunks + sp - 1) / sp;
  return (int)((chunks + per - 1) / per);
}

template <int NT, int MT, int D, int OCC, int EPI>
static int wide_launch(WideArgs a, int tiles, int splits, hipStream_t s) {
  constexpr int W = 8;
  constexpr int kX = MT * 16 * 144, kAcc = MT * NT * 1024;  // as kXBytes, kAccBytes in the kernel
  constexpr size_t lds = (size_t)W * (kX > kAcc ? kX : kAcc);
  static_assert(lds <= 160 * 1024, "the wavefronts' regions fit LDS");
  auto kernel = dec_wide_kernel<W, NT, MT, D, OCC, EPI>;
  if (lds > 64 * 1024) {
    const int rc = allow_dynamic_lds((const void*)kernel, (int)lds, "dec_wide_kernel");
    if (rc != MSA_OK) return rc;
  }
  a.units = (tiles + NT - 1) / NT;
  const int grid = a.units < kWideCUs * OCC ? a.units : kWideCUs * OCC;
  hipLaunchKernelGGL(kernel, dim3(grid, splits), dim3(64 * W), lds, s, a);
  return MSA_OK;
}

// Tiles per unit: rounds of units x tiles x the time of a tile in a unit of that width, which falls with the
// width (a unit's activations are read, and its partial tiles summed, once). Measured per tile and round in
// tenths of the widest unit's, K = 512 to 12288: one token tile 14, 12, 10 for 1, 2, 3 tiles (up to four
// tokens 12, 12, 10, and over a long K, where HBM sets the pace, the same: 17088 x 6144 at one token 28.2
// us in ones, 30.2 in threes); two token tiles 13, 13, 12 for 1, 2, 3 and 10 for 6; three and four 13, 12, 10. Over 800 shapes the pick is 0.3% from the best width (5% with equal times: 65536 x 256 at one
// token 20.3 us in twos, 11.8 in threes). Wide units need registers: six tiles up to 32 tokens, three
// otherwise.
static int wide_nt(int tiles, int tokens, int k) {
  constexpr int kTime[6][4] = {{12, 12, 10, 0}, {14, 12, 10, 0}, {13, 13, 12, 10}, {13, 12, 10, 0}, {13, 12, 10, 0}, {10, 10, 10, 0}};
  constexpr int kWidth[4] = {1, 2, 3, 6};
  const int mt = (tokens + 15) / 16, row = tokens > 4 ? mt : k >= 4096 ? 5 : 0;
  int best = 1;
  int64_t cost = (int64_t)1 << 62;
  for (int i = 0; i < (mt == 2 ? 4 : 3); ++i) {
    const int units = (tiles + kWidth[i] - 1) / kWidth[i];
    const int64_t c = (int64_t)((units + kWideCUs - 1) / kWideCUs) * kWidth[i] * kTime[row][i];
    if (c <= cost) {
      best = kWidth[i];
      cost = c;
    }
  }
  return best;
}

// D, OCC per (NT, MT): as many chunks in flight as the registers hold (measured; deeper than these
// gained nothing: 8B gate_up at 32 tokens, six tiles, 27.5 us with one chunk in flight, 28.1 with two).
template <int EPI>
static int wide_dispatch(const WideArgs& a, int tiles, hipStream_t s) {
  const int mt = (a.t + 15) / 16, nt = wide_nt(tiles, a.t, a.k);
  switch (mt) {
    case 1:
      if (nt == 1) return wide_launch<1, 1, 4, 2, EPI>(a, tiles, 1, s);
      if (nt == 2) return wide_launch<2, 1, 4, 1, EPI>(a, tiles, 1, s);
      return wide_launch<3, 1, 2, 2, EPI>(a, tiles, 1, s);
    case 2:
      if (nt == 1) return wide_launch<1, 2, 2, 2, EPI>(a, tiles, 1, s);
      if (nt == 2) return wide_launch<2, 2, 2, 1, EPI>(a, tiles, 1, s);
      if (nt == 3) return wide_launch<3, 2, 2, 1, EPI>(a, tiles, 1, s);
      return wide_launch<6, 2, 1, 1, EPI>(a, tiles, 1, s);
    case 3:
      if (nt == 1) return wide_launch<1, 3, 2, 1, EPI>(a, tiles, 1, s);
      if (nt == 2) return wide_launch<2, 3, 2, 1, EPI>(a, tiles, 1, s);
      return wide_launch<3, 3, 2, 1, EPI>(a, tiles, 1, s);
    default:
      if (nt == 1) return wide_launch<1, 4, 2, 1, EPI>(a, tiles, 1, s);
      if (nt == 2) return wide_launch<2, 4, 2, 1, EPI>(a, tiles, 1, s);
      return wide_launch<3, 4, 2, 1, EPI>(a, tiles, 1, s);
  }
}

static WideArgs wide_args(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                          const uint16_t* scale, int64_t n) {
  WideArgs a{};
  a.x = x; a.ldx = ldx; a.t = (int)m; a.k = (int)k; a.w = qweight; a.scale = scale; a.n = (int)n; a.k_per = (int)k;
  return a;
}

// Shapes from dec_wide_eligible; other arguments checked by the caller.
int launch_dec_wide(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight, const uint16_t* scale,
                    int64_t n, uint16_t* y, int64_t ldy, int epilogue, const uint16_t* residual, int64_t ldr,
                    hipStream_t s) {
  WideArgs a = wide_args(x, m, k, ldx, qweight, scale, n);
  a.y = y; a.ldy = ldy; a.resid = residual; a.ldr = ldr;
  const int tiles = (int)(epilogue == MSA_EPI_SILU_MUL ? (n / 2 + 7) / 8 : (n + 15) / 16);
  int rc;
  switch (epilogue) {
    case MSA_EPI_NONE: rc = wide_dispatch<MSA_EPI_NONE>(a, tiles, s); break;
    case MSA_EPI_SILU_MUL: rc = wide_dispatch<MSA_EPI_SILU_MUL>(a, tiles, s); break;
    default: rc = wide_dispatch<MSA_EPI_RESIDUAL>(a, tiles, s); break;
  }
  if (rc != MSA_OK) return rc;
  return check_launch("wide decode linear");
}

// float32 partials [splits][m][n], splits from dec_wide_splits: for consumers that merge them in a
// kernel of their own.
int launch_dec_wide_partials(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                             const uint16_t* scale, int64_t n, int splits, float* part, hipStream_t s) {
  WideArgs a = wide_args(x, m, k, ldx, qweight, scale, n);
  a.part = part;
  a.k_per = (int)((k / 64 + splits - 1) / splits * 64);
  const int tiles = (int)((n + 15) / 16), mt = (a.t + 15) / 16;
  int rc;
  switch (mt) {
    case 1:
    case 2: rc = wide_launch<kWidePartialNT, 2, 2, 1, kWidePartial>(a, tiles, splits, s); break;
    case 3: rc = wide_launch<kWidePartialNT, 3, 1, 1, kWidePartial>(a, tiles, splits, s); break;
    default: rc = wide_launch<kWidePartialNT, 4, 1, 1, kWidePartial>(a, tiles, splits, s); break;
  }
  if (rc != MSA_OK) return rc;
  return check_launch("wide decode linear (split-K pass)");
}

}  // namespace msa
